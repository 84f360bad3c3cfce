// Prefill (T > 16 tokens): routing plan and grouped expert GEMMs on MFMA.
//
// Plan (same layout as the decode/bucketing plan, experts ascending, tokens
// ascending within an expert: edge35b/pipeline.py:59-76 _routes,
// block_experts.py:102-121):
//   pf_topk   top-8 per token (or the caller's indices, validated); per block
//             of 8 tokens an 8-bit token mask per expert, built in LDS
//             (no global atomics);
//   pf_scan   (above 2048 tokens; below, pf_fill counts the masks itself) one
//             workgroup per expert: prefix of its mask popcounts over the
//             blocks, and its pair count;
//   pf_fill   expert offsets and ranks, every route placed, and the list of
//             work units (slot, first pair) of at most kPassTok tokens.
//
// Experts (cpu_experts.c:54-69 rounding points; the shared expert is slot 0),
// one persistent launch (pf_experts) whose workgroups take, from 4 or 8 work
// lists, gate/up items and then down items:
//   gate/up   one item per (unit, 128-row tile): 128 gate + 128 up rows
//             of one expert against up to 128 tokens.  Each of the 8 waves
//             streams its 32 weight rows (16 gate, 16 up) from HBM two
//             K-chunks ahead and passes them through an LDS stage of its own
//             into MFMA A operands; the same waves stage the unit's token
//             rows in LDS chunk by chunk, shared by all 8 waves, so a weight
//             byte is read once per 128 tokens and feeds up to 8 16x16x32
//             MFMAs.  SwiGLU in the epilogue, act rows out.
//   down      one item per (unit, 512 output rows): the unit's act rows are
//             staged in LDS once, then 4 tiles of 128 down rows over k = 512
//             stream through registers and a wave's LDS stage, two tiles
//             ahead; y rows out (bf16).
//   The ordered combine is experts.hip's combine_kernel.
//
// A list is a contiguous part of the units, served by the workgroups b with
// b % lists = the list (on XCDs b % 8, one or two per list): a unit's token and
// act rows are fetched into the L2s of its list, and an expert's units
// (consecutive in the plan) run together there, its weight tiles shared.
// Act rows go out and come back with agent-scope stores and loads, so
// results do not depend on that placement.
#include "lrmoe_device.h"
#include "lrmoe_internal.h"

namespace lrmoe {
namespace {

constexpr int kBlkTok = 8;                 // tokens per routing block
constexpr int kGuRows = 128;                // intermediate rows (gate and up) per gate/up workgroup
constexpr int kGuTiles = kInner / kGuRows;  // 4 gate/up tiles per expert
constexpr int kGuChunk = 128;              // k per LDS chunk
constexpr int kGuChunks = kHidden / kGuChunk;
constexpr int kGuSteps = kGuChunk / 32;    // MFMA k-steps (and A loads per lane) per chunk
constexpr int kXsStride = kGuChunk;        // LDS row stride of token and weight chunks (bf16), swizzled (swz)
constexpr int kDnThreads = 512;            // down workgroup: 8 waves of 16 output rows
constexpr int kDnRows = kDnThreads / kWave * 16;  // 128 output rows per down workgroup
constexpr int kDnTiles = kHidden / kDnRows;       // 16 down tiles per expert
constexpr int kDnItemTiles = 4;                   // tiles per split down item
constexpr int kDnItems = kDnTiles / kDnItemTiles; // 4 split down items per unit
constexpr int kDnStage = 2048;                    // bytes of a wave's LDS stage: 16 rows x 64 k
// Work lists of the expert launch, each served by 8 / lists XCDs: fewer share
// weight and token rows of neighbouring items less often in one L2, more end
// less evenly.  Rows read once (non-temporal): 8 lists take 1.02-1.06 times as
// long as 4 up to 512 tokens of a routed prompt and 0.99-1.01 above, 2 lists
// 1.00-1.03.  Rows that an expert's units share (cached): 8 lists 0.95-0.99 of
// 4 (T = 5000-8192 0.98, two units on each of 160 experts 0.95-0.97, 24 experts
// of 257 tokens 0.88), 2 lists 1.02-1.05.
template <bool STREAM>
constexpr int kLists = STREAM ? 4 : 8;
constexpr uint64_t kPfSpinTicks = 5000000; // 50 ms of the 100 MHz wall clock
constexpr int32_t kStatusTimeoutPf = LRMOE_STATUS_TIMEOUT;

// ---- plan ----------------------------------------------------------------------

__global__ __launch_bounds__(256) void pf_topk(const uint16_t* logits, const int64_t* indices_in,
                                               const uint16_t* weights_in, int64_t* indices, uint16_t* weights,
                                               int tokens, Workspace ws) {
    __shared__ uint32_t mask[kExperts];
    __shared__ int32_t bad;
    const int blk = blockIdx.x;
    const int wave = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
    mask[threadIdx.x] = 0u;
    if (threadIdx.x == 0) bad = 0;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int i = 2 * wave + j;
        const int t = blk * kBlkTok + i;
        if (t >= tokens) continue;
        int e = 0;
        bool ok = true;
        if (indices_in == nullptr) {
            const uint64_t packed = *reinterpret_cast<const uint64_t*>(logits + static_cast<size_t>(t) * kExperts + 4 * lane);
            uint32_t w = 0;
            topk8_wave(packed, e, w, static_cast<int>(threadIdx.x & 63));
            if (lane < kTopK) {
                indices[t * kTopK + lane] = e;
                weights[t * kTopK + lane] = static_cast<uint16_t>(w);
            }
        } else if (lane < kTopK) {
            const int64_t v = indices_in[t * kTopK + lane];
            int32_t flags = (v < 0 || v >= kExperts) ? kStatusBadExpert : 0;
            for (int q = 0; q < lane; ++q) flags |= indices_in[t * kTopK + q] == v ? kStatusRepeatedExpert : 0;
            if (flags) atomicOr(&bad, flags);
            ok = flags == 0;
            e = ok ? static_cast<int>(v) : 0;
        }
        if (lane < kTopK && ok) atomicOr(&mask[e], 1u << i);
    }
    __syncthreads();
    uint8_t* row = ws.bmask + static_cast<size_t>(threadIdx.x) * ws.nblk_pad;
    row[blk] = static_cast<uint8_t>(mask[threadIdx.x]);
    if (blk == static_cast<int>(gridDim.x) - 1) {
        for (int b = blk + 1; b < ws.nblk_pad; ++b) row[b] = 0;  // read in whole 16-byte words
    }
    if (threadIdx.x == 0) ws.bstatus[blk] = bad;
}

// Blocks up to which every pf_fill workgroup counts the masks itself (256
// threads x at most 256 bytes each, from L2) and pf_scan is not launched:
// top-k and plan of 40 / 333 / 2048 tokens 11.8 / 11.6 / 11.8 -> 8.4 / 8.7 /
// 10.7 us.  At 1024 blocks the counting would read 256 KiB per workgroup.
constexpr int kScanBlocks = 256;

__global__ __launch_bounds__(256) void pf_scan(int nblk, Workspace ws, Plan plan) {
    __shared__ uint32_t scratch[4];
    const int e = blockIdx.x;
    const int per = (nblk + 255) / 256;
    const int b0 = threadIdx.x * per;
    const int b1 = min(b0 + per, nblk);
    const uint8_t* row = ws.bmask + static_cast<size_t>(e) * ws.nblk_pad;
    uint32_t local = 0;
    for (int b = b0; b < b1; ++b) local += __popc(row[b]);
    uint32_t total = 0;
    uint32_t running = block_scan256(local, scratch, &total, static_cast<int>(threadIdx.x));
    for (int b = b0; b < b1; ++b) {
        ws.blk_base[static_cast<size_t>(e) * ws.nblk_pad + b] = running;
        running += __popc(row[b]);
    }
    if (threadIdx.x == 0) ws.counts[e] = total;
    if (e == 0) {
        int32_t flags = 0;
        for (int b = threadIdx.x; b < nblk; b += 256) flags |= ws.bstatus[b];
        __shared__ int32_t all;
        if (threadIdx.x == 0) all = 0;
        __syncthreads();
        if (flags) atomicOr(&all, flags);
        __syncthreads();
        if (threadIdx.x == 0) *plan.status = all;
    }
}

// SCAN: the masks are counted here (see kScanBlocks), else by pf_scan.
template <bool SCAN>
__global__ __launch_bounds__(256) void pf_fill(const int64_t* indices, int tokens, int shared_present, Workspace ws,
                                               Plan plan) {
    __shared__ uint32_t scratch[4];
    __shared__ uint32_t start[kExperts];  // the block's first pair of each expert
    __shared__ int32_t status_s;
    const int blk = blockIdx.x;
    const int e = threadIdx.x;
    uint32_t count = 0, before = 0;  // the expert's pairs: all, and those of earlier blocks
    int32_t status;
    if constexpr (SCAN) {
        if (threadIdx.x == 0) status_s = 0;
        __syncthreads();
        const uint8_t* row = ws.bmask + static_cast<size_t>(e) * ws.nblk_pad;
        const int nblk = gridDim.x;
        const int32_t flags = e < nblk ? ws.bstatus[e] : 0;  // nblk <= kScanBlocks = 256
#pragma unroll 4
        for (int b = 0; b < ws.nblk_pad; b += 16) {
            const uint4 v = ldg16(row + b);
            const uint32_t word[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                count += __popc(word[i]);
                const int bytes = min(max(blk - b - 4 * i, 0), 4);  // of the word, in blocks before blk
                before += __popc(static_cast<uint32_t>(word[i] & ((1ull << (8 * bytes)) - 1ull)));
            }
        }
        if (flags) atomicOr(&status_s, flags);
        __syncthreads();
        status = status_s;
        if (blk == 0 && threadIdx.x == 0) *plan.status = status;
    } else {
        status = *plan.status;
        count = ws.counts[e];
        before = ws.blk_base[static_cast<size_t>(e) * ws.nblk_pad + blk];
    }
    if (status != 0) {
        for (int i = threadIdx.x; i < kBlkTok * kTopK; i += 256) {
            const int t = blk * kBlkTok + i / kTopK;
            if (t < tokens) plan.route_pair[t * kTopK + i % kTopK] = -1;
        }
        if (blk == 0 && threadIdx.x == 0) {
            *plan.unique = 0;
            plan.offset[0] = 0;
            ws.control->n_units = 0;
        }
        if (blk == 0 && threadIdx.x < 8) ws.control->claim[threadIdx.x] = 0u;
        return;
    }
    if (blk == 0) {
        // pf_experts' claim counters and per-unit gate/up counts, for this call
        for (int i = threadIdx.x; i < ws.max_units; i += 256) ws.unit_done[i] = 0u;
        if (threadIdx.x < 8) ws.control->claim[threadIdx.x] = 0u;
    }
    uint32_t pairs = 0, unique = 0;
    const uint32_t pair0 = block_scan256(count, scratch, &pairs, static_cast<int>(threadIdx.x));
    const uint32_t rank = block_scan256(count ? 1u : 0u, scratch, &unique, static_cast<int>(threadIdx.x));
    start[e] = pair0 + before;
    if (blk == 0) {
        if (count) {
            plan.expert[rank] = e;
            plan.offset[rank] = static_cast<int32_t>(pair0);
        }
        // Work units: the shared expert's passes, then each routed expert's.
        const uint32_t passes = (count + kPassTok - 1) / kPassTok;
        uint32_t unit_total = 0;
        const uint32_t shared_units = shared_present ? (tokens + kPassTok - 1) / kPassTok : 0u;
        const uint32_t first_unit = shared_units + block_scan256(passes, scratch, &unit_total, static_cast<int>(threadIdx.x));
        // A unit names its expert and pair range directly, so an expert
        // workgroup reaches its weight addresses in two dependent loads.
        for (uint32_t j = threadIdx.x; j < shared_units; j += 256) {
            const int first = static_cast<int>(j) * kPassTok;
            ws.units[j] = make_int4(0, kTopK * tokens + first, min(kPassTok, tokens - first), 0);
        }
        for (uint32_t j = 0; j < passes; ++j) {
            const int first = static_cast<int>(j) * kPassTok;
            ws.units[first_unit + j] = make_int4(1 + e, static_cast<int>(pair0) + first,
                                                 min(kPassTok, static_cast<int>(count) - first), 0);
        }
        if (threadIdx.x == 0) {
            plan.offset[unique] = static_cast<int32_t>(pairs);
            *plan.unique = static_cast<int32_t>(unique);
            ws.control->n_units = static_cast<int32_t>(shared_units + unit_total);
        }
    }
    __syncthreads();
    if (threadIdx.x < kBlkTok * kTopK) {
        const int i = threadIdx.x / kTopK;
        const int k = threadIdx.x % kTopK;
        const int t = blk * kBlkTok + i;
        if (t < tokens) {
            const int ex = static_cast<int>(indices[t * kTopK + k]);
            const size_t at = static_cast<size_t>(ex) * ws.nblk_pad + blk;
            const int p = static_cast<int>(start[ex] + __popc(ws.bmask[at] & ((1u << i) - 1u)));
            plan.pair_token[p] = t;
            plan.pair_slot[p] = k;
            int order = 0;
#pragma unroll
            for (int q = 0; q < kTopK; ++q) order += indices[t * kTopK + q] < ex ? 1 : 0;
            plan.route_pair[t * kTopK + order] = p;
        }
    }
}

// ---- experts -------------------------------------------------------------------

struct Unit {
    const uint16_t* gate;
    const uint16_t* up;
    const uint16_t* down;
    const int32_t* tokens;  // token of each pair of the unit, or null for pair index = token (shared)
    int pair0;              // first act/y row of the unit
    int count;              // pairs in the unit, 1..kPassTok
};

// The unit table, the unit count and the expert table are written before
// the expert launch and only read during it: they are read through the
// constant address space, so a wave-uniform lookup is a scalar load, counted
// apart from the vector loads that stream weights and rows.
template <typename T>
__device__ __forceinline__ T ld_const(const T* p) {
    return *reinterpret_cast<const __attribute__((address_space(4))) T*>(reinterpret_cast<uintptr_t>(p));
}

// Weight rows: streamed past the caches where an expert's rows are read once
// per call, cached where several of its units read them (see pf_experts).
template <bool STREAM>
__device__ __forceinline__ uint4 ld_weight(const uint16_t* p) {
    return STREAM ? ldg16_nt(p) : ldg16(p);
}

__device__ __forceinline__ const uint16_t* uniform_ptr(const uint16_t* p) {
    return reinterpret_cast<const uint16_t*>(uniform64(reinterpret_cast<uintptr_t>(p)));
}

__device__ __forceinline__ bool load_unit(const ExpertArgs& a, int u, Unit& w) {
    if (u >= ld_const(&a.ws.control->n_units)) return false;
    const int* rec = reinterpret_cast<const int*>(a.ws.units + u);
    const int4 unit = make_int4(ld_const(rec), ld_const(rec + 1), ld_const(rec + 2), ld_const(rec + 3));
    w.pair0 = unit.y;
    w.count = unit.z;
    if (unit.x == 0) {
        w.gate = a.shared_gate_proj;
        w.up = a.shared_up_proj;
        w.down = a.shared_down;
        w.tokens = nullptr;
        return true;
    }
    const int e = unit.x - 1;
    const uint16_t* gate_up = reinterpret_cast<const uint16_t*>(ld_const(a.expert_ptrs + 2 * e));
    w.gate = gate_up;
    w.up = gate_up + static_cast<size_t>(kInner) * kHidden;
    w.down = reinterpret_cast<const uint16_t*>(ld_const(a.expert_ptrs + 2 * e + 1));
    w.tokens = a.plan.pair_token + unit.y;
    return true;
}

// gate/up workgroup (128 intermediate rows of one work unit): 8 waves, each
// owning two 16-row MFMA tiles (tile r = 8 gate rows and the 8 up rows with
// the same indices).  The waves also move the unit's token rows into LDS,
// one 128-column chunk at a time.
//
// Weights: a load instruction covers 4 rows x 256 contiguous bytes (lane l:
// row 4i + l/16, bytes 16(l%16)), non-temporal, and the 16 rows of a tile pass
// through the wave's own LDS stage into the MFMA layout.  The same bytes
// requested directly in the MFMA layout (16 rows x 64 bytes per instruction,
// cached) stream at 5.1 TB/s over 256 workgroups, this way at 6.2-6.4 (a
// read-only probe over 1.5 GiB).
//
// Per chunk a wave issues its token pieces, then its weights, two to three
// chunks ahead, each into the registers just written to LDS; the waits are
// then for exactly the data used next (the memory counter retires in order),
// and two chunks of weights (16 KiB per wave) stay in flight.  A B operand
// read from LDS feeds both row tiles, and the 4 workgroups of a unit each
// read its token rows once.
constexpr int kGuWaves = kGuRows / 16;
constexpr int kGuThreads = kGuWaves * kWave;
constexpr int kGuPieces = kPassTok * kGuChunk / 8 / kGuThreads;  // 16-byte token pieces per thread per chunk
constexpr int kStRows = 32;                                      // both tiles of a wave
constexpr int kGuClaimChunk = kGuChunks - 4;                     // the last weights are requested: claim the next item

// The next item of a list.  (An increment-with-wrap: the compiler's atomic
// optimiser would turn a lane-0 add into a wave-wide one and wait for it.)
__device__ __forceinline__ uint32_t claim_item(uint32_t* claim) {
    return __builtin_amdgcn_atomic_inc32(claim, 0xffffffffu, __ATOMIC_RELAXED, "agent");
}

// Place of 16-byte piece p of row r in a 256-byte LDS row: ds_read_b128 takes
// 16 lanes at a time, rows r % 16 of k-group g and the others of g ^ 1, and
// with the pieces exchanged by r they fall on all 64 banks once (rows padded
// to 272 bytes spent 40% of the LDS cycles in conflicts).
__device__ __forceinline__ int swz(int r, int p) { return r * kXsStride + 8 * (p ^ (r & 15)); }

// The K loop for NB 16-token column blocks (blocks past the unit's tokens
// read rows whose results are dropped), then SwiGLU.  xoff[j]: byte offset in
// x of this thread's token piece j (unit row tid / 16 + 32 j, 16 bytes at
// column 8 * (tid % 16) of each chunk).  gate_w / up_w: the wave's first gate
// and up row (wave-uniform).  LDS addresses are one base per use, a k-step's
// or load's pieces reached by an xor (4j + g ^ m = (g ^ m) ^ 4j).
//
// claimed (thread 0): the next item, claimed late in this one.  A list's
// workgroups, on two XCDs above all, do not start at the same time: claimed
// as an item starts, the second items of the earlier ones were the first items
// of the others, and a call of about one item per workgroup took two rounds
// (512 tokens on 64 experts, 64 units: 139 us, late 109; one XCD per list,
// claimed at the start, 109).  The streaming loop claims in its last chunks; in the cached one that costs 21
// spills, and the claim's latency falls under the SwiGLU instead.
template <int NB, bool STREAM>
__device__ __forceinline__ void gateup_mfma(const uint16_t* gate_w, const uint16_t* up_w, const uint16_t* x,
                                            const uint32_t* xoff, char* xs, char* stage, uint16_t* act0, uint16_t* act1,
                                            int count, uint32_t* claim, uint32_t& claimed) {
    const int lane = threadIdx.x & 63;
    const int m = lane & 15;
    const int g = lane >> 4;
    // Full units of calls with many tokens per expert: MFMAs and LDS are the
    // larger part there.  (Where the weight stream bounds the call the second
    // barrier per chunk only costs: routed prompts of 1000-2048 tokens 1-3%.)
    constexpr bool kTurns = NB == kPassTok / 16 && !STREAM;
    f32x4 acc[2][NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[0][b] = acc[1][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    uint4 wb[2][2][4];  // two chunks in flight: [chunk parity][tile][load]
    uint4 xr[2][kGuPieces];
    const uint32_t lane_off = static_cast<uint32_t>(g * kHidden + 8 * m);
    uint32_t rd = 2 * swz(m, g);                         // operand row m, k-group g
    uint32_t wr = 2 * swz(g, m);                         // stage row g, piece m
    const uint32_t st = 2 * swz(threadIdx.x >> 4, m);    // token row tid / 16, piece tid % 16
    // Each load's first row, kept in scalar registers (with the lane's 32-bit
    // offset and the chunk as the instruction's immediate).
    const uint16_t* wrow[2][4];
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            wrow[r][i] = (i < 2 ? gate_w : up_w) + (8 * r + 4 * (i & 1)) * kHidden;
            asm volatile("" : "+s"(wrow[r][i]));
        }
    auto load_w = [&](int c) {
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int i = 0; i < 4; ++i) wb[c & 1][r][i] = ld_weight<STREAM>(wrow[r][i] + lane_off + c * kGuChunk);
    };
    auto stage_w = [&](int c) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            char* dst = stage + (wr ^ (64 * i)) + 1024 * i;
#pragma unroll
            for (int r = 0; r < 2; ++r) *reinterpret_cast<uint4*>(dst + 4096 * r) = wb[c & 1][r][i];
        }
    };
    auto load_t = [&](int c) {
#pragma unroll
        for (int j = 0; j < kGuPieces; ++j) xr[c & 1][j] = ldg16(reinterpret_cast<const char*>(x) + c * 2 * kGuChunk + xoff[j]);
    };
    auto store_t = [&](int c) {
#pragma unroll
        for (int j = 0; j < kGuPieces; ++j)
            *reinterpret_cast<uint4*>(xs + (c & 1) * kPassTok * 2 * kXsStride + j * 32 * 2 * kXsStride + st) = xr[c & 1][j];
    };
    auto multiply = [&](int c) {
        const char* xcb = xs + (c & 1) * kPassTok * 2 * kXsStride;
        if constexpr (kTurns) {
            // Pinned order: B operands are read kAhead column blocks ahead of
            // their MFMAs (left to itself the compiler reads two, waits and
            // multiplies).
            constexpr int kAhead = 5;
            uint4 bv[kAhead + 1];
            uint4 av[2][2];
            auto read_a = [&](int j) {
#pragma unroll
                for (int r = 0; r < 2; ++r) av[j & 1][r] = *reinterpret_cast<const uint4*>(stage + 4096 * r + (rd ^ (64 * j)));
            };
            auto read_b = [&](int i) {
                bv[i % (kAhead + 1)] = *reinterpret_cast<const uint4*>(xcb + 16 * (i % NB) * 2 * kXsStride + (rd ^ (64 * (i / NB))));
            };
            __builtin_amdgcn_sched_barrier(0);
            read_a(0);
#pragma unroll
            for (int i = 0; i < kAhead; ++i) read_b(i);
#pragma unroll
            for (int i = 0; i < kGuSteps * NB; ++i) {
                if (i + kAhead < kGuSteps * NB) read_b(i + kAhead);
                if (i % NB == 0 && i / NB + 1 < kGuSteps) read_a(i / NB + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int r = 0; r < 2; ++r) acc[r][i % NB] = mfma16x16x32(av[(i / NB) & 1][r], bv[i % (kAhead + 1)], acc[r][i % NB]);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
#pragma unroll
            for (int j = 0; j < kGuSteps; ++j) {
                const uint32_t at = rd ^ (64 * j);
                const uint4 a0 = *reinterpret_cast<const uint4*>(stage + at);
                const uint4 a1 = *reinterpret_cast<const uint4*>(stage + 4096 + at);
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    const uint4 bv = *reinterpret_cast<const uint4*>(xcb + 16 * b * 2 * kXsStride + at);
                    acc[0][b] = mfma16x16x32(a0, bv, acc[0][b]);
                    acc[1][b] = mfma16x16x32(a1, bv, acc[1][b]);
                }
            }
        }
    };
    if constexpr (kTurns) {
        // The two waves of a SIMD take turns.  In half-step 2c waves
        // 0-3 multiply chunk c while waves 4-7 move data (stage their weight
        // chunk c, store their rows of token chunk c + 1, request the next
        // ones), in half-step 2c + 1 the other way round; a barrier ends every
        // half-step.  With both waves multiplying and then both moving, a chunk
        // took 4430 cycles, 2700 of them MFMAs (2048 at full rate), and the
        // layer 1.02-1.03 times as long at T = 4001-16384 (16 experts of
        // 129-384 tokens 1.02-1.06 times).
        // waves 4-7, which store token rows one chunk further ahead (a scalar:
        // the barriers below sit in branches on it)
        const int late = __builtin_amdgcn_readfirstlane(threadIdx.x >= kGuThreads / 2 ? 1 : 0);
        auto load_late = [&](int c, int set) {  // token chunk c + late (past the end: the last again, dropped)
            const int at = min(c + late, kGuChunks - 1) * 2 * kGuChunk;
#pragma unroll
            for (int j = 0; j < kGuPieces; ++j) {
                uint32_t off = xoff[j];
                asm volatile("" : "+v"(off));  // scalar base + 32-bit offset, not a 64-bit address held per piece
                xr[set][j] = ldg16(reinterpret_cast<const char*>(x) + at + off);
            }
        };
        auto store_late = [&](int c, int set) {  // into chunk c + late's buffer
            char* dst = xs + ((c + late) & 1) * kPassTok * 2 * kXsStride;
#pragma unroll
            for (int j = 0; j < kGuPieces; ++j) *reinterpret_cast<uint4*>(dst + j * 32 * 2 * kXsStride + st) = xr[set][j];
        };
        load_t(0);
        load_w(0);
        load_t(1);
        load_w(1);
        store_t(0);
        load_late(2, 0);
        __syncthreads();
        if (late) {
            store_t(1);
            load_late(1, 1);  // waves 0-3 hold their chunk 1 already
            stage_w(0);
            __syncthreads();
        } else {
            stage_w(0);
        }
        load_w(2);
#pragma unroll
        for (int c = 0; c < kGuChunks; ++c) {
            asm volatile("" : "+v"(rd), "+v"(wr));  // keeps the xor'd addresses from being held across chunks
            multiply(c);
            if (c + 1 < kGuChunks) {
                __syncthreads();
                stage_w(c + 1);
                if (c + 3 < kGuChunks) load_w(c + 3);
                store_late(c + 1, (c + 1) & 1);
                if (c + 3 < kGuChunks) load_late(c + 3, (c + 1) & 1);
                __syncthreads();
            }
        }
        if (!late) __syncthreads();
    } else {
        load_t(0);
        load_w(0);
        load_t(1);
        load_w(1);
        store_t(0);
        load_t(2);
        stage_w(0);
        load_w(2);
#pragma unroll
        for (int c = 0; c < kGuChunks; ++c) {
            asm volatile("" : "+v"(rd), "+v"(wr));
            // Token chunk c is in LDS buffer c & 1; the other buffer is free.
            __syncthreads();
            if (c + 1 < kGuChunks) store_t(c + 1);
            if (c + 3 < kGuChunks) load_t(c + 3);
            multiply(c);
            __builtin_amdgcn_wave_barrier();
            if (c + 1 < kGuChunks) stage_w(c + 1);
            if (c + 3 < kGuChunks) load_w(c + 3);
            if (STREAM && c == kGuClaimChunk && threadIdx.x == 0) claimed = claim_item(claim);
            __builtin_amdgcn_wave_barrier();
        }
    }
    if (!STREAM && threadIdx.x == 0) claimed = claim_item(claim);
    // SwiGLU: lanes g < 2 hold gate rows 4g..4g+3 of a tile's 8, lane + 32 the
    // up rows with the same index.  One lane-half swap per pair of rows gives
    // every lane gate and up of two rows (rows 0, 1 in the low half, 2, 3 in
    // the high half), so all lanes share the activation's arithmetic.
    // act0/act1 point at this lane's first act element of column 0 for tile 0
    // and 1 (2 consecutive intermediate rows).
#pragma unroll
    for (int r = 0; r < 2; ++r) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            uint32_t v[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[r][b][i]), __float_as_uint(acc[r][b][i + 2]),
                                                                false, false);
                v[i] = swiglu_bf16(rbf(__uint_as_float(s[0])), rbf(__uint_as_float(s[1])));
            }
            if (16 * b + m < count) st_agent32((r ? act1 : act0) + static_cast<size_t>(16 * b) * kInner, v[0] | (v[1] << 16));
            __builtin_amdgcn_sched_barrier(0);  // interleaving more of these costs spills
        }
    }
}

// A down item: kDnItemTiles (even) tiles of 128 output rows of one unit, NB
// 16-token column blocks.  (Items of a whole unit while every workgroup gets
// one, with the act rows staged once instead of four times, took 12-21 us
// longer at T = 333-2048: the lists end unevenly.)  The unit's act rows are
// staged in LDS once (rows of 1 KiB, 16-byte piece p of row r at place p ^ r %
// 16: see swz).  Each wave streams its 16 rows of a tile (16 KiB contiguous), 8
// rows x 128 bytes per instruction, two tiles ahead: a piece of 64 k passes from
// its two registers through the wave's LDS stage into MFMA operands (place p ^
// r % 8 of 128-byte rows), and the registers are requested again at once, so
// the stream never waits for a tile to end.  y rows go out through a buffer
// whose range ends at the unit's last row (no branch around a store: one would
// make the compiler wait for every load in flight).  act_bytes, y_bytes: the
// unit's rows.  Returns the next item, claimed (by thread 0) before the last
// two tiles, so that no workgroup holds an unstarted item for long.
template <int NB, bool STREAM>
__device__ __forceinline__ uint32_t down_item(const uint16_t* act, uint32_t act_bytes, const uint16_t* wrow, uint16_t* y,
                                              uint32_t y_bytes, char* lds, char* stage, uint32_t* claim) {
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int m = lane & 15;
    const int g = lane >> 4;
    uint4 wt[2][16];
    f32x4 acc[2][NB];
    const __amdgpu_buffer_rsrc_t yr =
        __builtin_amdgcn_make_buffer_rsrc(y, 0, static_cast<int>(y_bytes), 0x00020000);
    // Load q of a piece: rows 8q + lane / 8, bytes 16 (lane % 8) of the piece.
    const uint32_t lane_off = static_cast<uint32_t>((lane >> 3) * kInner + 8 * (lane & 7));
    constexpr size_t kTile = static_cast<size_t>(kDnRows) * kInner;
    auto load_piece = [&](const uint16_t* tile, int set, int p) {
#pragma unroll
        for (int q = 0; q < 2; ++q) wt[set][2 * p + q] = ld_weight<STREAM>(tile + lane_off + 8 * q * kInner + 64 * p);
    };
    {
        uint4 st[2 * NB];
#pragma unroll
        for (int q = 0; q < 2 * NB; ++q) st[q] = ld_agent16(act, static_cast<uint32_t>((tid + kDnThreads * q) * 16), act_bytes);
#pragma unroll
        for (int p = 0; p < 8; ++p) load_piece(wrow, 0, p);
#pragma unroll
        for (int p = 0; p < 8; ++p) load_piece(wrow + kTile, 1, p);
        // Piece lane of row tid / 64 + 8q (row % 16 alternates with q).
#pragma unroll
        for (int q = 0; q < 2 * NB; ++q) {
            const int r = (tid >> 6) + 8 * q;
            *reinterpret_cast<uint4*>(lds + r * 1024 + 16 * (lane ^ (r & 15))) = st[q];
        }
    }
    __syncthreads();
    uint32_t rd = static_cast<uint32_t>(m * 1024 + 16 * (m ^ g));
    const uint32_t ws = static_cast<uint32_t>(lane * 16) ^ static_cast<uint32_t>(16 * (lane >> 3));  // row lane / 8, place lane % 8 ^ row
    const uint32_t rs = static_cast<uint32_t>(m * 128 + 16 * (g ^ (m & 7)));
    uint32_t yo = static_cast<uint32_t>(m * kHidden + 4 * g) * 2;
    auto tile_mfma = [&](int set, const uint16_t* ahead) {
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[0][b] = acc[1][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int p = 0; p < 8; ++p) {
            __builtin_amdgcn_wave_barrier();
            if (NB == 8) asm volatile("" : "+v"(rd));
#pragma unroll
            for (int q = 0; q < 2; ++q) *reinterpret_cast<uint4*>(stage + ws + 1024 * q) = wt[set][2 * p + q];
            __builtin_amdgcn_wave_barrier();
            if (ahead != nullptr) load_piece(ahead, set, p);
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const uint4 av = *reinterpret_cast<const uint4*>(stage + (rs ^ (64 * k)));
                const uint32_t at = (rd ^ (64 * ((2 * p + k) & 3))) + 256 * ((2 * p + k) >> 2);
#pragma unroll
                for (int b = 0; b < NB; ++b)
                    acc[k][b] = mfma16x16x32(av, *reinterpret_cast<const uint4*>(lds + at + 16384 * b), acc[k][b]);
            }
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const f32x4 v = acc[0][b] + acc[1][b];
            typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
            __builtin_amdgcn_raw_buffer_store_b64(u32x2{pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3])}, yr,
                                                  static_cast<int>(yo + 16 * b * 2 * kHidden), 0, 0);
        }
        yo += kDnRows * 2;
    };
#pragma unroll 1
    for (int t = 2; t < kDnItemTiles; t += 2) {
        wrow += 2 * kTile;
        tile_mfma(0, wrow);
        tile_mfma(1, wrow + kTile);
    }
    uint32_t claimed = 0u;
    if (tid == 0) claimed = claim_item(claim);
    tile_mfma(0, nullptr);
    tile_mfma(1, nullptr);
    return claimed;
}

// The expert stage of a prefill layer in one persistent launch: one
// workgroup per CU.  Workgroup b serves list b % lists (a contiguous part of
// the units, so a unit's items and an expert's units share the L2s of the
// list's XCDs when workgroup b runs on XCD b % 8): first the 4 gate/up items
// of each of its units, then the 4 down items of each, claimed from the list's
// counter one item ahead (a gate/up item claims its successor at its loop's
// end, a down item before its last two tiles).  A down item first waits (bounded) until its unit's 4 gate/up items
// have counted themselves in.  Every gate/up item is claimed before any down
// item of its list and a claimed gate/up item never waits, so the waits end
// whether or not all workgroups are resident.  The claim counters and
// per-unit counts are zeroed by pf_fill.
template <bool STREAM>
__device__ __forceinline__ void expert_items(const ExpertArgs& a, uint16_t* lds, int& claimed_s, int& timeout_s) {
    const int tid = threadIdx.x;
    constexpr int lists = kLists<STREAM>;
    const int list = blockIdx.x % lists;
    const int n_units = ld_const(&a.ws.control->n_units);
    const int first = n_units * list / lists;  // the list's units: [first, first + units)
    const int units = n_units * (list + 1) / lists - first;
    const int n_gu = kGuTiles * units;
    const int n_items = n_gu + kDnItems * units;
    uint32_t* claim = &a.ws.control->claim[list];
    // The claimed item, broadcast to the workgroup (item indices are
    // wave-uniform, so the unit lookups are scalar loads).
    auto publish = [&](uint32_t claimed) -> int {
        if (tid == 0) claimed_s = static_cast<int>(claimed);
        __syncthreads();
        const int item = __builtin_amdgcn_readfirstlane(claimed_s);
        __syncthreads();  // every thread has read claimed_s before it is written again
        return item;
    };
    if (tid == 0) timeout_s = 0;
    int cur = publish(tid == 0 ? claim_item(claim) : 0u);

    // ---- gate/up items (every one claimed before any down item) ----
    while (cur < n_gu) {
        uint32_t claimed = 0u;
        const int u = first + cur / kGuTiles;
        const int tile = cur % kGuTiles;
        // The item's code is written out here rather than called as an
        // inlined function: that form spills registers.
        Unit w;
        if (load_unit(a, u, w)) {  // always: u < n_units
            const int wave = tid >> 6;
            const int lane = tid & 63;
            // Token pieces of this thread: piece tid % 16 of unit rows tid / 16 + 32 j
            // (rows past the unit's count repeat its first token).
            uint32_t xoff[kGuPieces];
#pragma unroll
            for (int j = 0; j < kGuPieces; ++j) {
                const int c = tid / 16 + (kGuThreads / 16) * j;  // token row of the unit, 0..127
                const int cc = c < w.count ? c : 0;
                const int t = w.tokens ? w.tokens[cc] : w.pair0 - kTopK * a.tokens + cc;
                xoff[j] = static_cast<uint32_t>(t) * (2 * kHidden) + 16 * (tid & 15);
            }
            const int m = lane & 15;
            const int g = lane >> 4;
            const int nblk = (w.count + 15) / 16;
            // MFMA row m < 8 of tile r is gate row 128*tile + 16*wave + 8r + m, m >= 8
            // the up row with the same index.
            const size_t row0 = static_cast<size_t>(kGuRows * tile + 16 * __builtin_amdgcn_readfirstlane(wave)) * kHidden;
            const uint16_t* gate_w = uniform_ptr(w.gate + row0);
            const uint16_t* up_w = uniform_ptr(w.up + row0);
            char* xs = reinterpret_cast<char*>(lds);
            char* stage = xs + 2 * (2 * kPassTok + wave * kStRows) * kXsStride;
            uint16_t* act0 = a.ws.act + static_cast<size_t>(w.pair0 + m) * kInner + kGuRows * tile + 16 * wave + 4 * (g & 1) + 2 * (g >> 1);
            uint16_t* act1 = act0 + 8;
            if (nblk <= 2) {
                gateup_mfma<2, STREAM>(gate_w, up_w, a.x, xoff, xs, stage, act0, act1, w.count, claim, claimed);
            } else if (nblk <= 4) {
                gateup_mfma<4, STREAM>(gate_w, up_w, a.x, xoff, xs, stage, act0, act1, w.count, claim, claimed);
            } else {
                gateup_mfma<8, STREAM>(gate_w, up_w, a.x, xoff, xs, stage, act0, act1, w.count, claim, claimed);
            }
        }
        __builtin_amdgcn_s_waitcnt(0);  // this wave's act rows are written
        __syncthreads();
        if (tid == 0) __hip_atomic_fetch_add(a.ws.unit_done + u, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        cur = publish(claimed);
    }

    // ---- down items, one per (unit, quarter of the output rows) ----
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    while (cur < n_items) {
        uint32_t claimed;
        const int j = cur - n_gu;
        const int u = first + j / kDnItems;
        const int tile0 = kDnItemTiles * (j % kDnItems);
        Unit w;
        load_unit(a, u, w);
        // The unit's 4 gate/up items have counted themselves in (bounded wait).
        if (tid == 0 && ld_agent32(a.ws.unit_done + u) < static_cast<uint32_t>(kGuTiles)) {
            const uint64_t start = wall_clock64();
            while (ld_agent32(a.ws.unit_done + u) < static_cast<uint32_t>(kGuTiles)) {
                if (wall_clock64() - start > kPfSpinTicks) {
                    timeout_s = 1;
                    break;
                }
                __builtin_amdgcn_s_sleep(2);
            }
        }
        __syncthreads();  // also: every wave is done with the previous item's act rows
        const int h0 = kDnRows * tile0 + 16 * wave;
        const uint16_t* act = a.ws.act + static_cast<size_t>(w.pair0) * kInner;
        const uint16_t* wrow = uniform_ptr(w.down + static_cast<size_t>(h0) * kInner);
        uint16_t* y = a.ws.y + static_cast<size_t>(w.pair0) * kHidden + h0;
        const uint32_t act_bytes = static_cast<uint32_t>(w.count) * kInner * 2;
        // to the last row's columns of this wave and item
        const uint32_t y_bytes = static_cast<uint32_t>(w.count) * kHidden * 2 - 2 * h0;
        char* rows = reinterpret_cast<char*>(lds);
        char* stage = rows + kPassTok * 1024 + wave * kDnStage;
        if (w.count <= 32) {
            claimed = down_item<2, STREAM>(act, act_bytes, wrow, y, y_bytes, rows, stage, claim);
        } else if (w.count <= 64) {
            claimed = down_item<4, STREAM>(act, act_bytes, wrow, y, y_bytes, rows, stage, claim);
        } else {
            claimed = down_item<8, STREAM>(act, act_bytes, wrow, y, y_bytes, rows, stage, claim);
        }
        cur = publish(claimed);
    }
    if (tid == 0 && timeout_s) atomicOr(&a.ws.control->status, kStatusTimeoutPf);
}

// Weight rows non-temporal while experts are (nearly) one unit each and their
// rows are read once; cached, with the half-step turns of full units, from 1.2
// units per expert on, whose later units find the rows in the caches.  The
// plan has both counts, the host has neither: tokens say little (128 experts
// of 129 tokens each are 2064 tokens and two units per expert, 192 of 127 are
// 3048 and one).  Routed experts, cached over non-temporal time: 0.83-0.97
// from 1.34 units per expert on, at any token count (96 experts of 129 tokens
// 252 -> 205 us, 32 of 129 109 -> 91); 1.01-1.05 at 1.02-1.15, 1.05-1.11 at 1
// (192 of 127 tokens 338 -> 308 us non-temporal); at up to 40 units 0.92-1.05.
__global__ __launch_bounds__(kDnThreads, 1) void pf_experts(ExpertArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
    __shared__ int claimed_s;
    __shared__ int timeout_s;
    if (5 * ld_const(&a.ws.control->n_units) > 6 * ld_const(a.plan.unique)) {
        expert_items<false>(a, lds, claimed_s, timeout_s);
    } else {
        expert_items<true>(a, lds, claimed_s, timeout_s);
    }
}

int max_units(int tokens) {
    return (tokens + kPassTok - 1) / kPassTok + kExperts + (kTopK * tokens + kPassTok - 1) / kPassTok;
}

}  // namespace

size_t prefill_experts_lds() {
    const size_t gateup = static_cast<size_t>(2 * kPassTok + kGuWaves * kStRows) * kXsStride * sizeof(uint16_t);
    const size_t down = static_cast<size_t>(kPassTok) * kInner * sizeof(uint16_t) + kDnThreads / kWave * kDnStage;
    return gateup > down ? gateup : down;
}

hipError_t launch_prefill_plan(const uint16_t* logits, const int64_t* indices_in, const uint16_t* weights_in,
                               int64_t* indices, uint16_t* weights, int tokens, int shared_present,
                               const Workspace& ws, const Plan& plan, hipStream_t stream) {
    if (tokens <= 0) return hipSuccess;
    const int nblk = (tokens + kBlkTok - 1) / kBlkTok;
    hipLaunchKernelGGL(pf_topk, dim3(nblk), dim3(256), 0, stream, logits, indices_in, weights_in, indices, weights,
                       tokens, ws);
    const int64_t* routes = indices_in ? indices_in : indices;
    if (nblk <= kScanBlocks) {
        hipLaunchKernelGGL(pf_fill<true>, dim3(nblk), dim3(256), 0, stream, routes, tokens, shared_present, ws, plan);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(pf_scan, dim3(kExperts), dim3(256), 0, stream, nblk, ws, plan);
    hipLaunchKernelGGL(pf_fill<false>, dim3(nblk), dim3(256), 0, stream, routes, tokens, shared_present, ws, plan);
    return hipGetLastError();
}

hipError_t launch_prefill_experts(const ExpertArgs& a, hipStream_t stream) {
    int device = 0;
    hipError_t err = hipGetDevice(&device);
    if (err != hipSuccess) return err;
    if (device < 0 || device >= 64) return hipErrorInvalidDevice;
    static int cus[64] = {0};  // per device: CU count, 0 until the LDS limit is raised
    if (cus[device] == 0) {
        err = hipFuncSetAttribute(reinterpret_cast<const void*>(pf_experts), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  static_cast<int>(prefill_experts_lds()));
        if (err != hipSuccess) return err;
        int n = 0;
        err = hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device);
        if (err != hipSuccess) return err;
        cus[device] = n;
    }
    // one workgroup per CU (all resident: the down items wait for gate/up
    // items), a multiple of the 8 XCDs
    const int grid = cus[device] / 8 * 8;
    if (grid < 8) return hipErrorNotSupported;
    const StageEvents ev = timing_events(kStageGateUp);
    LRMOE_LAUNCH(pf_experts, dim3(grid), dim3(kDnThreads), prefill_experts_lds(), stream, ev.start, ev.stop, a);
    return hipGetLastError();
}

}  // namespace lrmoe
