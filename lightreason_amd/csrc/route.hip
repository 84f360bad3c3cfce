// Router (softmax/top-k/renormalise) and route bucketing kernels.
//
// Semantics follow the Transformers Qwen3_5MoeTopKRouter.forward that the
// reference patches around (modeling_qwen3_5_moe.py, called from
// SparseMoeBlock.forward; edge35b/expert_stream.py:383-454 receives its
// top_k_index / top_k_weights), and the reference's bucketing:
// edge35b/fused_experts.py:47-54 (routes sorted by expert),
// edge35b/block_experts.py:102-121 (experts ascending, tokens ascending,
// inverse map per token), edge35b/pipeline.py:59-76.
//
// Router logits use one fixed fp32 reduction order so that indices are
// reproducible bit-for-bit: lane l of a wave owns the 32 contiguous elements
// [32l, 32l+32) of the 2048-long dot product and accumulates them in order
// with fmaf from +0, then the 64 partials meet in an xor butterfly with
// offsets 1,2,4,...,32.  Top-k ranks by (bf16 logit desc, expert id asc).
#include "lrmoe_device.h"
#include "lrmoe_internal.h"

namespace lrmoe {
namespace {

constexpr int kTokTile = 16;     // most tokens of a decode call (one tile)
constexpr int kCus = 256;        // CUs of an MI355X (grid sizing only)
constexpr int kXStride = kHidden + 8;  // LDS row stride in bf16 (16-byte pad)

// Stage up to 16 token rows of the router input into LDS, applying the
// RMSNorm (x * r) * (1 + w) with r = 1/sqrt(sum(x^2)/2048 + eps) when `norm`
// is given.  One wave per token; lane l owns elements [32l, 32l+32).
__device__ void stage_tokens(uint16_t* xs, const uint16_t* x, const uint16_t* norm, float eps, int t0, int count,
                             uint16_t* normed_out) {
    const int wave = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
    for (int t = wave; t < count; t += 4) {
        const uint4* src = reinterpret_cast<const uint4*>(x + static_cast<size_t>(t0 + t) * kHidden + 32 * lane);
        uint4 v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = src[i];
        if (norm != nullptr) {
            float f[32];
#pragma unroll
            for (int i = 0; i < 4; ++i) unpack8(v[i], f + 8 * i);
            float acc = 0.0f;
#pragma unroll
            for (int j = 0; j < 32; ++j) acc = __builtin_fmaf(f[j], f[j], acc);
            const float mean = wave_butterfly_sum(acc) / static_cast<float>(kHidden);
            const float r = 1.0f / __builtin_sqrtf(mean + eps);
            const uint4* wsrc = reinterpret_cast<const uint4*>(norm + 32 * lane);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint4 w = wsrc[i];
                float wf[8];
                unpack8(w, wf);
                uint32_t o[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) o[j] = f2bf((f[8 * i + j] * r) * (1.0f + wf[j]));
                v[i] = make_uint4(o[0] | (o[1] << 16), o[2] | (o[3] << 16), o[4] | (o[5] << 16), o[6] | (o[7] << 16));
            }
            if (normed_out != nullptr) {
                uint4* dst = reinterpret_cast<uint4*>(normed_out + static_cast<size_t>(t0 + t) * kHidden + 32 * lane);
#pragma unroll
                for (int i = 0; i < 4; ++i) dst[i] = v[i];
            }
        }
        uint4* dst = reinterpret_cast<uint4*>(xs + t * kXStride + 32 * lane);
#pragma unroll
        for (int i = 0; i < 4; ++i) dst[i] = v[i];
    }
}

// Fixed-order dot of this lane's 32 weights with token row `t` in LDS.
__device__ __forceinline__ float lane_dot(const float* w, const uint16_t* xs, int t, int lane) {
    const uint4* row = reinterpret_cast<const uint4*>(xs + t * kXStride + 32 * lane);
    float acc = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float xf[8];
        unpack8(row[i], xf);
#pragma unroll
        for (int j = 0; j < 8; ++j) acc = __builtin_fmaf(w[8 * i + j], xf[j], acc);
    }
    return acc;
}

// Exclusive scan of one value per thread over threads 0..255 of a workgroup
// of >= 256 threads (every thread must call it; values of threads >= 256 are
// ignored and get 0).  `total` receives the sum over threads 0..255.
__device__ uint32_t scan256(uint32_t value, uint32_t* scratch, uint32_t* total) {
    const int wave = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
    if (threadIdx.x >= kExperts) value = 0;
    uint32_t inclusive = value;
#pragma unroll
    for (int offset = 1; offset < kWave; offset <<= 1) {
        const uint32_t up = static_cast<uint32_t>(__shfl_up(static_cast<int>(inclusive), offset, kWave));
        if (lane >= offset) inclusive += up;
    }
    if (lane == kWave - 1 && wave < 4) scratch[wave] = inclusive;
    __syncthreads();
    uint32_t before = 0;
    for (int w = 0; w < wave && w < 4; ++w) before += scratch[w];
    *total = scratch[0] + scratch[1] + scratch[2] + scratch[3];
    __syncthreads();
    return threadIdx.x < kExperts ? before + inclusive - value : 0u;
}

// Bucket <= 64 tokens held in LDS (ids[t*8 + r], already validated) with one
// 256-thread workgroup: a token bitmap per expert (one LDS atomic per route),
// a block scan for pair offsets and unique ranks, then every route places
// itself in O(1).
__device__ void build_plan_small(const int32_t* ids, int tokens, const Plan& plan) {
    __shared__ unsigned long long tokmask[kExperts];
    __shared__ uint32_t poff[kExperts];
    __shared__ uint32_t scan_scratch[4];
    const int e = threadIdx.x;
    if (e < kExperts) tokmask[e] = 0ull;
    __syncthreads();
    for (int i = threadIdx.x; i < tokens * kTopK; i += blockDim.x) atomicOr(&tokmask[ids[i]], 1ull << (i / kTopK));
    __syncthreads();
    const unsigned long long mask = e < kExperts ? tokmask[e] : 0ull;
    const uint32_t count = static_cast<uint32_t>(__popcll(mask));
    // One scan of (unique flag << 16 | count): counts are <= 64 and pairs <= 512.
    uint32_t packed_total = 0;
    const uint32_t packed = scan256((count ? (1u << 16) : 0u) | count, scan_scratch, &packed_total);
    const uint32_t pair_offset = packed & 0xffffu;
    const uint32_t rank = packed >> 16;
    const uint32_t pairs_total = packed_total & 0xffffu;
    const uint32_t unique_total = packed_total >> 16;
    if (e < kExperts) poff[e] = pair_offset;
    if (count) {
        plan.expert[rank] = e;
        plan.offset[rank] = static_cast<int32_t>(pair_offset);
        unsigned long long m = mask;
        for (int j = 0; m; ++j) {
            const int t = __ffsll(static_cast<long long>(m)) - 1;
            m &= m - 1ull;
            plan.pair_token[pair_offset + j] = t;
        }
    }
    if (e == 0) {
        plan.offset[unique_total] = static_cast<int32_t>(pairs_total);
        *plan.unique = static_cast<int32_t>(unique_total);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < tokens * kTopK; i += blockDim.x) {
        const int t = i / kTopK;
        const int r = i % kTopK;
        const int ex = ids[i];
        const int p = static_cast<int>(poff[ex]) + __popcll(tokmask[ex] & ((1ull << t) - 1ull));
        plan.pair_slot[p] = r;
        int order = 0;
        for (int q = 0; q < kTopK; ++q) order += (ids[t * kTopK + q] < ex) ? 1 : 0;
        plan.route_pair[t * kTopK + order] = p;
    }
}

// Checks ids and returns the status bits for the whole set.
__device__ int32_t validate_ids(const int32_t* ids, int tokens) {
    __shared__ int32_t flags;
    if (threadIdx.x == 0) flags = 0;
    __syncthreads();
    int32_t mine = 0;
    for (int i = threadIdx.x; i < tokens * kTopK; i += blockDim.x) {
        const int e = ids[i];
        if (e < 0 || e >= kExperts) mine |= kStatusBadExpert;
        const int t = i / kTopK;
        for (int q = t * kTopK; q < i; ++q) mine |= (ids[q] == e) ? kStatusRepeatedExpert : 0;
    }
    if (mine) atomicOr(&flags, mine);
    __syncthreads();
    return flags;
}

// Router logits of <= 16 tokens: 4 router rows per workgroup, one per wave
// (the tokens are one tile; the kernel boundary publishes the logits).  With
// norm, the first workgroup also writes the normalised rows.
__global__ __launch_bounds__(256) void router_logits(RouteArgs a) {
    __shared__ __attribute__((aligned(16))) uint16_t xs[kTokTile * kXStride];
    const int wave = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * 4 + wave;
    // Issue this wave's weight loads before staging the tokens.
    uint4 wraw[4];
    if (a.router != nullptr) {
        const uint4* src = reinterpret_cast<const uint4*>(a.router + static_cast<size_t>(row) * kHidden + 32 * lane);
#pragma unroll
        for (int q = 0; q < 4; ++q) wraw[q] = src[q];
    }
    if (a.router != nullptr || (blockIdx.x == 0 && a.norm != nullptr)) {
        stage_tokens(xs, a.x, a.norm, a.eps, 0, a.tokens, blockIdx.x == 0 ? a.normed : nullptr);
    }
    __syncthreads();
    if (a.router == nullptr) return;
    float w[32];
#pragma unroll
    for (int q = 0; q < 4; ++q) unpack8(wraw[q], w + 8 * q);
    for (int t = 0; t < a.tokens; ++t) {
        const float s = wave_butterfly_sum(lane_dot(w, xs, t, lane));
        if (lane == 0) a.logits[static_cast<size_t>(t) * kExperts + row] = static_cast<uint16_t>(f2bf(s));
    }
}

// ---- router of more than 16 tokens --------------------------------------------
//
// The canonical sum of a logit is 64 chains of 32 fmaf, met in a balanced
// binary tree.  v_mfma_f32_16x16x1_4b_f32 runs exactly such chains: with
// K = 1 every accumulator takes one fused multiply-add per instruction, so 32
// of them in element order are the chain from +0, for four chains (the
// instruction's four blocks) of a 16 x 16 tile of (router row, token) at
// once.  Each wave owns 8 consecutive chains (256 of the 2048 columns) of
// every tile of its workgroup; their sums, (b0 + b1) + (b2 + b3) per
// instruction group and then over groups and waves, are the butterfly's tree.
//
// Bound by the fp32 matrix rate (this instruction: 129 TFLOP/s measured, fmaf
// on the VALU 68) and, up to a few hundred tokens, by the latency of one
// tile.  The VALU form it replaces (one wave per row, a butterfly per dot
// product) normalised the tokens 17 times and spent ~90 VALU instructions on
// every 64 x 32 fmaf.  rocprof, averages, T = 40 / 333 / 2048 / 8192 with norm
// and gate: 23 / 34 / 125 / 438 -> 13 / 23 / 48 / 124 us.
//
// Tile: 32 tokens (16 while that gives every tile a CU of its own; their
// normalised rows stay in registers as B operands) against `per` tiles of 16
// router rows; a 17th tile, whose rows all hold the shared-expert gate, gives
// that gate.  Normalising the tokens costs about 1.5 row tiles; the grid's y
// dimension trades repeats of it against idle CUs (launch_route).
typedef float f32x16 __attribute__((ext_vector_type(16)));
constexpr int kRmThreads = 512;
constexpr int kRmWaves = kRmThreads / kWave;
constexpr int kRmRowTiles = kExperts / 16;          // router row tiles; tile 16 is the shared gate

__device__ __forceinline__ float bf_elem(const uint4 (&v)[4], int j) {
    const uint4 p = v[j >> 3];
    const int w = (j & 7) >> 1;
    const uint32_t word = w == 0 ? p.x : w == 1 ? p.y : w == 2 ? p.z : p.w;
    return (j & 1) ? hi_bf(word) : lo_bf(word);
}

// NT column tiles of 16 tokens per workgroup.
template <int NT>
__global__ __launch_bounds__(kRmThreads) void router_tiles(RouteArgs a, int first_tile, int tiles, int per) {
    constexpr int kTok = 16 * NT;
    constexpr int kRows = kTok / kRmWaves;  // token rows whose norm scale a wave computes
    __shared__ __attribute__((aligned(16))) float red[3][kRmWaves][NT][kWave * 4];
    __shared__ float scale[kTok];
    const int wave = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
    const int m = lane & 15;
    const int t0 = blockIdx.x * kTok;
    const int tile0 = first_tile + blockIdx.y * per;
    const int tile1 = min(tile0 + per, first_tile + tiles);
    // This lane's two pieces of 32 columns (chains 8 wave + lane / 16 and + 4).
    const int k0 = 32 * (8 * wave + (lane >> 4));
    uint4 wraw[2][4];
    auto load_rows = [&](int tile, uint4 (*dst)[4]) {
        const uint16_t* row = tile < kRmRowTiles ? a.router + static_cast<size_t>(16 * tile + m) * kHidden : a.shared_gate;
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int i = 0; i < 4; ++i) dst[q][i] = ldg16(row + k0 + 128 * q + 8 * i);
    };
    // Token rows past the last repeat it; their results are dropped.
    uint4 x[NT][2][4];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const uint16_t* row = a.x + static_cast<size_t>(min(t0 + 16 * n + m, a.tokens - 1)) * kHidden;
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int i = 0; i < 4; ++i) x[n][q][i] = ldg16(row + k0 + 128 * q + 8 * i);
    }
    if (a.norm != nullptr) {
        uint4 rows[kRows][4], nw[2][4];
#pragma unroll
        for (int i = 0; i < kRows; ++i) {
            const int t = min(t0 + kRows * wave + i, a.tokens - 1);
#pragma unroll
            for (int q = 0; q < 4; ++q) rows[i][q] = ldg16(a.x + static_cast<size_t>(t) * kHidden + 32 * lane + 8 * q);
        }
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int i = 0; i < 4; ++i) nw[q][i] = ldg16(a.norm + k0 + 128 * q + 8 * i);
        if (tile0 < tile1) load_rows(tile0, wraw);
#pragma unroll
        for (int i = 0; i < kRows; ++i) {
            const float r = row_rms_scale(rows[i], a.eps);
            if (lane == 0) scale[kRows * wave + i] = r;
        }
        __syncthreads();
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const float r = scale[16 * n + m];
            const int t = t0 + 16 * n + m;
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int i = 0; i < 4; ++i) x[n][q][i] = rms_apply8(x[n][q][i], nw[q][i], r);
            if (blockIdx.y == 0 && t < a.tokens) {
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        *reinterpret_cast<uint4*>(a.normed + static_cast<size_t>(t) * kHidden + k0 + 128 * q + 8 * i) = x[n][q][i];
            }
        }
    } else if (tile0 < tile1) {
        load_rows(tile0, wraw);
    }
    // A tile's partial sums meet in LDS.  With three or more tiles the waves
    // 4-7 (`late`) run half a tile behind the others, so that the adding,
    // storing and unpacking between a SIMD's MFMAs of one wave falls under the
    // other's: tile t's barrier is at its end for waves 0-3 and in its middle
    // for waves 4-7, and tile t - 1 is complete after it (three buffers).  In
    // step a tile took 6.4 us, 4.2 of it MFMAs; routing 2048 / 8192 tokens, plan
    // included, took 1.07 / 1.08 times as long.  Fewer tiles only gain the
    // half-tile wait.  A scalar: barriers sit in branches on it.
    const bool late = __builtin_amdgcn_readfirstlane(per >= 3 && wave >= kRmWaves / 2);
    auto finish = [&](int tile) {
        if (threadIdx.x >= NT * 256) return;
        // Thread -> (column tile n, lane, i): row 4 (lane / 16) + i of column lane % 16.
        const int n = threadIdx.x >> 8;
        const int at = threadIdx.x & 255;
        float p[kRmWaves];
#pragma unroll
        for (int w = 0; w < kRmWaves; ++w) p[w] = red[(tile - tile0) % 3][w][n][at];
        const float s = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
        const int t = t0 + 16 * n + ((at >> 2) & 15);
        const int row = 4 * (at >> 6) + (at & 3);
        if (t >= a.tokens) return;
        if (tile < kRmRowTiles) {
            a.logits[static_cast<size_t>(t) * kExperts + 16 * tile + row] = static_cast<uint16_t>(f2bf(s));
        } else if (row == 0) {
            a.sg[t] = static_cast<uint16_t>(f2bf(1.0f / (1.0f + lr_exp(-rbf(s)))));
        }
    };
    for (int tile = tile0; tile < tile1; ++tile) {
        // The next tile's rows are requested and the previous tile's results
        // stored ahead of this tile's MFMAs, which cover both.
        uint4 wnext[2][4];
        load_rows(min(tile + 1, tile1 - 1), wnext);
        if (!late && tile > tile0 + 1) finish(tile - 2);
        f32x4 part[NT];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            f32x16 acc[NT];
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[n][i] = 0.0f;
#pragma unroll
            for (int j = 0; j < 32; ++j) {
                const float w = bf_elem(wraw[q], j);
#pragma unroll
                for (int n = 0; n < NT; ++n)
                    acc[n] = __builtin_amdgcn_mfma_f32_16x16x1f32(w, bf_elem(x[n][q], j), acc[n], 0, 0, 0);
            }
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                f32x4 s;
#pragma unroll
                for (int i = 0; i < 4; ++i) s[i] = (acc[n][i] + acc[n][4 + i]) + (acc[n][8 + i] + acc[n][12 + i]);
                part[n] = q == 0 ? s : part[n] + s;
            }
            if (q == 0 && late) {
                __syncthreads();
                if (tile > tile0) finish(tile - 1);
            }
        }
#pragma unroll
        for (int n = 0; n < NT; ++n) *reinterpret_cast<f32x4*>(&red[(tile - tile0) % 3][wave][n][4 * lane]) = part[n];
        if (!late) __syncthreads();
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int i = 0; i < 4; ++i) wraw[q][i] = wnext[q][i];
    }
    if (tile0 >= tile1) return;
    if (!late && tile1 - tile0 > 1) finish(tile1 - 2);
    __syncthreads();  // the late waves' last sums
    finish(tile1 - 1);
}

// Workgroups per token tile: the count whose rounds over the CUs, each
// costing its row tiles and ~1.5 for the norm, take the least time.
int router_splits(int token_tiles, int row_tiles) {
    int best = 1;
    double best_cost = 1e30;
    for (int y = 1; y <= row_tiles; ++y) {
        const int per = (row_tiles + y - 1) / y;
        const int groups = (row_tiles + per - 1) / per;  // workgroups that have work
        const double cost = static_cast<double>((token_tiles * groups + kCus - 1) / kCus) * (per + 1.5);
        if (cost < best_cost) {
            best_cost = cost;
            best = groups;
        }
    }
    return best;
}

// Top-8 of one token by ballot radix selection.  Lane l holds the logits of
// experts 4l..4l+3 as unique 24-bit keys; the 8th largest key is found bit by
// bit from the top with wave-wide counts.  The eight winners land in LDS with
// their exp() terms (already computed for the softmax denominator), lane k < 8
// ranks entry k, and probabilities and weights take one divide per lane.
// Indices, weights and the LDS expert row are written in rank order.
// Arithmetic and order match topk_token (and the oracle) exactly.
__device__ void topk_token_select(uint64_t packed, int64_t* indices_row, uint16_t* weights_row, int32_t* ids_row,
                                  uint32_t* keys8, float* vals8) {
    const int lane = threadIdx.x & 63;
    uint32_t bits[4], keys[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        bits[j] = static_cast<uint32_t>(packed >> (16 * j)) & 0xffffu;
        keys[j] = route_key(bits[j], 4 * lane + j);
    }
    uint32_t best = keys[0];
#pragma unroll
    for (int j = 1; j < 4; ++j) best = keys[j] > best ? keys[j] : best;
    best = wave_max_u32(best);
    uint32_t threshold = 0;
#pragma unroll 1
    for (int bit = 23; bit >= 0; --bit) {
        const uint32_t candidate = threshold | (1u << bit);
        int above = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) above += __popcll(__ballot(keys[j] >= candidate));
        if (above >= kTopK) threshold = candidate;
    }
    // Softmax terms of this lane's four experts, relative to the top logit.
    const float top = bf2f(key_bits(best));
    float ex[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) ex[j] = lr_exp(bf2f(bits[j]) - top);
    float part = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) part = part + ex[j];
    const float total = wave_butterfly_sum(part);
    // Exactly eight keys are >= threshold (keys are unique); compact them.
    int base = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const bool chosen = keys[j] >= threshold;
        const uint64_t mask = __ballot(chosen);
        if (chosen) {
            const int at = base + __popcll(mask & ((1ull << lane) - 1ull));
            keys8[at] = keys[j];
            vals8[at] = ex[j];
        }
        base += __popcll(mask);
    }
    // LDS accesses of one wave execute in order: the reads see the writes.
    __builtin_amdgcn_wave_barrier();
    const int k = lane & 7;
    const uint32_t my_key = keys8[k];
    int rank = 0;
#pragma unroll
    for (int i = 0; i < kTopK; ++i) rank += keys8[i] > my_key ? 1 : 0;
    const float prob = vals8[k] / total;
    __builtin_amdgcn_wave_barrier();
    if (lane < kTopK) vals8[rank] = prob;
    __builtin_amdgcn_wave_barrier();
    float sum = vals8[0];
#pragma unroll
    for (int i = 1; i < kTopK; ++i) sum = sum + vals8[i];
    const int expert = 255 - static_cast<int>(my_key & 255u);
    if (lane < kTopK) {
        indices_row[rank] = expert;
        weights_row[rank] = static_cast<uint16_t>(f2bf(prob / sum));
        ids_row[rank] = expert;
    }
}

// Decode routing tail in one workgroup of 16 waves (T <= 16): wave t runs
// the top-k of token t (from the router's logits or the caller's) and its
// shared-expert gate; then the workgroup builds the bucketing plan and the
// decode slot records.
__global__ __launch_bounds__(1024) void topk_bucket_small(RouteArgs a) {
    __shared__ int32_t ids[kTokTile * kTopK];
    __shared__ uint32_t keys8[kTokTile][kTopK];
    __shared__ float vals8[kTokTile][kTopK];
    const int t = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
    const uint16_t* logits = a.logits_in != nullptr ? a.logits_in : a.logits;
    if (t < a.tokens) {
        // Issue every load of this wave first: its logits row, and the
        // shared-gate weights and token row.
        const uint64_t packed = reinterpret_cast<const uint64_t*>(logits + static_cast<size_t>(t) * kExperts)[lane];
        const bool gate = a.shared_gate != nullptr;
        uint4 wsg[4], xrow[4];
        if (gate) {
            const uint16_t* x = a.norm != nullptr ? a.normed : a.x;
            const uint4* src = reinterpret_cast<const uint4*>(a.shared_gate + 32 * lane);
            const uint4* row = reinterpret_cast<const uint4*>(x + static_cast<size_t>(t) * kHidden + 32 * lane);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                wsg[q] = src[q];
                xrow[q] = row[q];
            }
        }
        topk_token_select(packed, a.indices + t * kTopK, a.weights + t * kTopK, ids + t * kTopK, keys8[t], vals8[t]);
        if (gate) {
            float acc = 0.0f;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float w[8], xf[8];
                unpack8(wsg[q], w);
                unpack8(xrow[q], xf);
#pragma unroll
                for (int j = 0; j < 8; ++j) acc = __builtin_fmaf(w[j], xf[j], acc);
            }
            const float z = rbf(wave_butterfly_sum(acc));
            if (lane == 0) a.sg[t] = static_cast<uint16_t>(f2bf(1.0f / (1.0f + lr_exp(-z))));
        }
    }
    __syncthreads();
    build_plan_small(ids, a.tokens, a.plan);
    if (threadIdx.x == 0) *a.plan.status = 0;
}

// Standalone bucketing of <= 64 caller-provided tokens in one workgroup.
__global__ __launch_bounds__(256) void bucket_small_kernel(const int64_t* indices, int tokens, Plan plan) {
    __shared__ int32_t ids[64 * kTopK];
    for (int i = threadIdx.x; i < tokens * kTopK; i += blockDim.x) {
        const int64_t e = indices[i];
        ids[i] = (e < 0 || e >= kExperts) ? -1 : static_cast<int32_t>(e);
    }
    __syncthreads();
    const int32_t status = validate_ids(ids, tokens);
    if (status) {
        if (threadIdx.x == 0) {
            *plan.status = status;
            *plan.unique = 0;
            plan.offset[0] = 0;
        }
        for (int i = threadIdx.x; i < tokens * kTopK; i += blockDim.x) plan.route_pair[i] = -1;
        return;
    }
    build_plan_small(ids, tokens, plan);
    if (threadIdx.x == 0) *plan.status = 0;
}

}  // namespace

hipError_t launch_route(const RouteArgs& a, hipStream_t stream) {
    if (a.tokens <= 0) return hipSuccess;
    const StageEvents ev = timing_events(kStageRoute);
    if (a.tokens <= kTokTile) {
        // Decode: router GEMV (one row per wave, 64 workgroups; skipped when
        // logits are given), then top-k + shared gate + bucketing in one
        // workgroup.
        hipEvent_t start = ev.start;
        if (a.router != nullptr || a.norm != nullptr) {
            LRMOE_LAUNCH(router_logits, dim3(a.router != nullptr ? kExperts / 4 : 1), dim3(256), 0, stream, start, nullptr, a);
            start = nullptr;
        }
        LRMOE_LAUNCH(topk_bucket_small, dim3(1), dim3(1024), 0, stream, start, ev.stop, a);
        return hipGetLastError();
    }
    const int row_tiles = (a.router != nullptr ? kRmRowTiles : 0) + (a.shared_gate != nullptr ? 1 : 0);
    hipEvent_t start = ev.start;
    if (row_tiles > 0 || a.norm != nullptr) {
        const int first = a.router != nullptr ? 0 : kRmRowTiles;
        const int tiles16 = (a.tokens + 15) / 16;
        if (tiles16 * row_tiles <= kCus) {
            LRMOE_LAUNCH(router_tiles<1>, dim3(tiles16, row_tiles > 0 ? row_tiles : 1), dim3(kRmThreads), 0, stream,
                         start, nullptr, a, first, row_tiles, 1);
        } else {
            const int tiles32 = (a.tokens + 31) / 32;
            const int splits = row_tiles > 0 ? router_splits(tiles32, row_tiles) : 1;
            LRMOE_LAUNCH(router_tiles<2>, dim3(tiles32, splits), dim3(kRmThreads), 0, stream, start, nullptr, a, first,
                         row_tiles, (row_tiles + splits - 1) / splits);
        }
    } else if (start != nullptr) {
        const hipError_t rec = hipEventRecord(start, stream);
        if (rec != hipSuccess) return rec;
    }
    const hipError_t err = launch_prefill_plan(a.logits_in != nullptr ? a.logits_in : a.logits, nullptr, nullptr,
                                               a.indices, a.weights, a.tokens, a.shared_down != nullptr, a.ws, a.plan,
                                               stream);
    if (err != hipSuccess) return err;
    if (ev.stop != nullptr) return hipEventRecord(ev.stop, stream);
    return hipGetLastError();
}

hipError_t launch_bucket(const int64_t* indices, int tokens, const Workspace& ws, const Plan& plan, hipStream_t stream) {
    if (tokens <= 0) return hipSuccess;
    if (tokens <= 64) {
        hipLaunchKernelGGL(bucket_small_kernel, dim3(1), dim3(256), 0, stream, indices, tokens, plan);
        return hipGetLastError();
    }
    return launch_prefill_plan(nullptr, indices, nullptr, nullptr, nullptr, tokens, false, ws, plan, stream);
}

}  // namespace lrmoe
