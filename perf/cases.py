"""The work a user of this package has it do, as cases that can be timed and
compared: the sparse MoE block at decode, verify and prefill sizes, the routed
experts alone, a chain of blocks, the two mixers of the decoder layer, a whole
verify pass, and the expert gather.

Every call goes through a public entry point (``lightreason_amd.moe``,
``.delta``, ``.attention``, ``.decoder``).  Shapes are the 35B model's; token
counts run from one decode position over verify blocks of 2-16 positions to
prompts of thousands of tokens, odd ones among them.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from lightreason_amd import moe
from lightreason_amd.attention import AttentionDecode
from lightreason_amd.decoder import DecoderLayer, DecoderStack, VerifyPass, is_full_attention
from lightreason_amd.delta import DeltaMixer

HIDDEN, INNER, EXPERTS, TOPK = 2048, 512, 256, 8
EXPERT_BYTES = 3 * INNER * HIDDEN * 2
PAIR_FLOP = 2 * 3 * INNER * HIDDEN
STACK_LAYERS = 8   # two periods of the decoder (three mixers, one attention)
CHAIN_LAYERS = 8   # more weights per pass than any cache holds
MIXER_BYTES = 2 * (12288 * HIDDEN + 64 * HIDDEN + HIDDEN * 4096 + 8192 * 4)
ATTN_BYTES = 2 * (9216 * HIDDEN + HIDDEN * 4096)


def listed():
    return [
        # One decode position through one MoE block: router, RMSNorm, shared
        # expert, residual.  The call a token generator makes per layer.
        {"name": "layer_t1", "kind": "layer", "tokens": 1, "routes": "router"},
        # A verify block of 8 positions whose routes are given as logits with
        # Zipf popularity: the repository's headline decode workload.
        {"name": "layer_t8_zipf", "kind": "layer", "tokens": 8, "routes": "zipf"},
        # The widest verify block through a stack of blocks in one launch.
        {"name": "chain_t16", "kind": "chain", "tokens": 16},
        # Prompts: a chat turn just above the decode sizes, a ragged short
        # prompt, the headline prefill size, and a long prompt in one call.
        {"name": "prefill_t40", "kind": "layer", "tokens": 40, "routes": "router"},
        {"name": "prefill_t333", "kind": "layer", "tokens": 333, "routes": "router"},
        {"name": "prefill_t2048", "kind": "layer", "tokens": 2048, "routes": "router"},
        {"name": "prefill_t8192", "kind": "layer", "tokens": 8192, "routes": "router"},
        # Routed experts for given routes: what a Transformers model whose
        # experts are patched calls per layer of a prompt.
        {"name": "experts_t1000", "kind": "experts", "tokens": 1000},
        # The linear-attention step of a 4-position verify block, with the
        # per-position states that a rollback needs.
        {"name": "mixer_t4_record", "kind": "mixer", "tokens": 4, "record": True, "state": "fp32"},
        # The full-attention step of one decode position after 4096 others.
        {"name": "attention_t1_4k", "kind": "attention", "tokens": 1, "context": 4096},
        # A whole verify pass of 4 positions over 8 decoder layers, replayed
        # from its graph.
        {"name": "decoder_t4", "kind": "decoder", "tokens": 4, "context": 4096},
        # Staging the experts of an 8-position block into one buffer.
        {"name": "gather_t8", "kind": "gather", "tokens": 8},
    ]


def draw(rng):
    kind = rng.choice(["layer", "prefill", "prefill", "prefill", "experts", "chain", "mixer", "attention", "gather"])
    if kind == "layer":
        return {"kind": "layer", "tokens": rng.randint(1, 16), "routes": rng.choice(["router", "zipf"])}
    if kind == "prefill":
        return {"kind": "layer", "tokens": int(round(math.exp(rng.uniform(math.log(17), math.log(8192))))),
                "routes": rng.choice(["router", "router", "zipf"])}
    if kind == "experts":
        return {"kind": "experts", "tokens": int(round(math.exp(rng.uniform(math.log(1), math.log(6000)))))}
    if kind == "chain":
        return {"kind": "chain", "tokens": rng.randint(1, 16)}
    if kind == "mixer":
        return {"kind": "mixer", "tokens": rng.randint(1, 16), "record": rng.random() < 0.5,
                "state": rng.choice(["fp32", "fp32", "bf16"])}
    if kind == "attention":
        return {"kind": "attention", "tokens": rng.randint(1, 16),
                "context": int(round(math.exp(rng.uniform(math.log(50), math.log(20000)))))}
    return {"kind": "gather", "tokens": rng.randint(1, 12)}


# ---- inputs ---------------------------------------------------------------------

class Source:
    """Seeded normal bf16 tensors on the GPU."""

    def __init__(self, seed):
        self.generator = torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)
        self.rng = np.random.default_rng(int(seed) & 0x7FFFFFFF)

    def normal(self, shape, sigma, shift=0.0, dtype=torch.bfloat16):
        t = torch.empty(shape, dtype=dtype, device="cuda").normal_(0.0, sigma, generator=self.generator)
        return t.add_(shift) if shift else t


def _bank(src, layers):
    bank = moe.ExpertBank(layers, "cuda")
    bank.bank.normal_(0.0, 0.02, generator=src.generator)
    return bank


def _layer(src, bank, index, norm=True):
    return moe.LayerWeights(
        router=src.normal((EXPERTS, HIDDEN), 0.02), expert_ptrs=bank.expert_ptrs(index),
        shared_gate_proj=src.normal((INNER, HIDDEN), 0.02), shared_up_proj=src.normal((INNER, HIDDEN), 0.02),
        shared_down_proj=src.normal((HIDDEN, INNER), 0.02), shared_expert_gate=src.normal((HIDDEN,), 0.02),
        norm_weight=src.normal((HIDDEN,), 0.02) if norm else None, eps=1e-6)


def _hidden(src, tokens):
    # A direction common to all tokens gives the experts unequal popularity
    # (the busiest of a long prompt takes about four times the mean).
    return (src.normal((tokens, HIDDEN), 1.0) + src.normal((1, HIDDEN), 0.25)).contiguous()


def _zipf_logits(src, tokens):
    ranks = src.rng.permutation(EXPERTS) + 1
    values = -1.1 * np.log(ranks)[None, :] + src.rng.gumbel(size=(tokens, EXPERTS))
    return torch.from_numpy(values.astype(np.float32)).cuda().to(torch.bfloat16)


def _mixer(src, state_dtype):
    mixer = DeltaMixer(
        in_proj_qkv=src.normal((8192, HIDDEN), 0.02), in_proj_z=src.normal((4096, HIDDEN), 0.02),
        in_proj_b=src.normal((32, HIDDEN), 0.02), in_proj_a=src.normal((32, HIDDEN), 0.02),
        conv1d=src.normal((8192, 4), 0.3), A_log=src.normal((32,), 0.5, 1.5), dt_bias=src.normal((32,), 0.5),
        norm=src.normal((128,), 0.1, 1.0), out_proj=src.normal((HIDDEN, 4096), 0.02))
    return mixer, src.normal((8192, 4), 1.0), src.normal((32, 128, 128), 0.05, dtype=torch.float32).to(state_dtype)


def _attention(src):
    return AttentionDecode(
        q_proj=src.normal((8192, HIDDEN), 0.02), k_proj=src.normal((512, HIDDEN), 0.02),
        v_proj=src.normal((512, HIDDEN), 0.02), o_proj=src.normal((HIDDEN, 4096), 0.02),
        q_norm=src.normal((256,), 0.1), k_norm=src.normal((256,), 0.1))


def _cache(src, context):
    # Room for the block and some growth, as a server's cache has.
    return src.normal((2, context + 64, 256), 1.0)


def _rope(tokens, start):
    pos = torch.arange(start, start + tokens, device="cuda", dtype=torch.float32)
    inv = 1.0 / (10000.0 ** (torch.arange(0, 64, 2, device="cuda", dtype=torch.float32) / 64))
    ang = torch.cat([pos[:, None] * inv[None]] * 2, dim=1)
    return ang.cos().to(torch.bfloat16).contiguous(), ang.sin().to(torch.bfloat16).contiguous()


def prepare(case, seed):
    src = Source(seed)
    kind, tokens = case["kind"], case["tokens"]
    s = {"case": case, "keep": []}
    if kind in ("layer", "chain", "experts"):
        layers = CHAIN_LAYERS if kind == "chain" else 1
        s["bank"] = _bank(src, layers)
        # Caller logits come with rows that are normalised already.
        s["layers"] = [_layer(src, s["bank"], i, norm=case.get("routes") != "zipf") for i in range(layers)]
        s["x"] = _hidden(src, tokens)
        s["out"] = torch.empty_like(s["x"])
        s["logits"] = _zipf_logits(src, tokens) if case.get("routes") == "zipf" else None
        if kind == "experts":
            logits = _zipf_logits(src, tokens).float()
            top, s["indices"] = torch.topk(logits, TOPK, dim=-1)
            s["weights"] = torch.softmax(top, dim=-1).to(torch.bfloat16)
        else:
            shape = (layers, tokens, TOPK) if kind == "chain" else (tokens, TOPK)
            s["indices"] = torch.zeros(shape, dtype=torch.int64, device="cuda")
            s["weights"] = torch.zeros(shape, dtype=torch.bfloat16, device="cuda")
        s["workspace"] = moe.Workspace("cuda", tokens)
    elif kind == "mixer":
        s["mixer"], s["conv"], s["state"] = _mixer(src, torch.float32 if case["state"] == "fp32" else torch.bfloat16)
        s["x"] = src.normal((tokens, HIDDEN), 1.0)
        s["conv_record"] = s["state_record"] = None
        if case["record"]:
            s["conv_record"] = torch.zeros((tokens, 8192, 4), dtype=torch.bfloat16, device="cuda")
            s["state_record"] = torch.zeros((tokens, 32, 128, 128), dtype=s["state"].dtype, device="cuda")
    elif kind == "attention":
        s["attention"] = _attention(src)
        s["x"] = src.normal((tokens, HIDDEN), 1.0)
        s["k"], s["v"] = _cache(src, case["context"]), _cache(src, case["context"])
        s["cos"], s["sin"] = _rope(tokens, case["context"])
    elif kind == "decoder":
        bank = _bank(src, STACK_LAYERS)
        layers = []
        for l in range(STACK_LAYERS):
            part = dict(input_norm=src.normal((HIDDEN,), 0.02), moe=_layer(src, bank, l))
            if is_full_attention(l):
                part.update(attention=_attention(src), k_cache=_cache(src, case["context"]),
                            v_cache=_cache(src, case["context"]))
            else:
                part["mixer"], part["conv_state"], part["state"] = _mixer(src, torch.float32)
            layers.append(DecoderLayer(**part))
        s["bank"], s["layers"] = bank, layers
        s["x"] = src.normal((tokens, HIDDEN), 1.0)
        s["cos"], s["sin"] = _rope(tokens, case["context"])
        before = [(l.conv_state.clone(), l.state.clone()) for l in layers if l.mixer is not None]
        s["verify"] = VerifyPass(DecoderStack(layers, "cuda"), [tokens], case["context"])
        # Capturing runs the step once; the caches' states start as drawn.
        for l, (conv, state) in zip([l for l in layers if l.mixer is not None], before):
            l.conv_state.copy_(conv)
            l.state.copy_(state)
    else:
        s["bank"] = _bank(src, 1)
        # As many experts as a block of that many positions selects on average.
        rows = round(_unique_experts(tokens, False))
        chosen = sorted(src.rng.choice(EXPERTS, rows, replace=False).tolist())
        s["chosen"] = chosen
        s["staging"] = torch.zeros((len(chosen), EXPERT_BYTES // 2), dtype=torch.bfloat16, device="cuda")
        pointers = s["bank"].expert_ptrs(0)[:, 0]
        s["descriptors"] = torch.stack([pointers, torch.full_like(pointers, -1), torch.zeros_like(pointers)], 1)[None].contiguous()
        s["destinations"] = torch.tensor([s["staging"].data_ptr()], device="cuda")
        s["sizes"] = torch.tensor([EXPERT_BYTES], device="cuda")
        s["src"] = torch.tensor(chosen, dtype=torch.int32, device="cuda")
        s["dst"] = torch.arange(len(chosen), dtype=torch.int32, device="cuda")
        s["count"] = torch.tensor([len(chosen)], device="cuda")
    return s


def run(s):
    kind = s["case"]["kind"]
    if kind == "layer":
        moe.moe_layer(s["x"], s["layers"][0], out=s["out"], indices=s["indices"], weights=s["weights"],
                      logits_in=s["logits"], workspace=s["workspace"])
        return {"out": s["out"], "indices": s["indices"], "weights": s["weights"]}
    if kind == "chain":
        moe.moe_chain(s["x"], s["layers"], out=s["out"], indices=s["indices"], weights=s["weights"],
                      workspace=s["workspace"])
        return {"out": s["out"], "indices": s["indices"], "weights": s["weights"]}
    if kind == "experts":
        return moe.moe_experts(s["x"], s["indices"], s["weights"], s["layers"][0].expert_ptrs, out=s["out"],
                               workspace=s["workspace"])
    if kind == "mixer":
        out = s["mixer"].step(s["x"], s["conv"], s["state"], conv_record=s["conv_record"],
                              state_record=s["state_record"])
        return {"out": out, "conv": s["conv"], "state": s["state"], "conv_record": s["conv_record"],
                "state_record": s["state_record"]}
    if kind == "attention":
        out = s["attention"].step(s["x"], s["cos"], s["sin"], s["k"], s["v"], s["case"]["context"])
        return {"out": out, "k": s["k"], "v": s["v"]}
    if kind == "decoder":
        out = s["verify"].verify(s["x"], s["cos"], s["sin"], length=s["case"]["context"], check=False)
        states = [(l.conv_state, l.state) if l.mixer is not None else (l.k_cache, l.v_cache) for l in s["layers"]]
        return {"out": out, "states": states}
    moe.gather(s["descriptors"], s["destinations"], s["sizes"], s["src"], s["dst"], s["count"],
               max_copies=len(s["chosen"]), experts=EXPERTS, stripes=48)
    return s["staging"]


# ---- what a pass cannot do without ----------------------------------------------

def _unique_experts(tokens, zipf):
    if not zipf:
        return EXPERTS * (1.0 - (1.0 - TOPK / EXPERTS) ** tokens)
    rng = np.random.default_rng(0)
    logits = -1.1 * np.log(np.arange(1, EXPERTS + 1)) + rng.gumbel(size=(tokens, EXPERTS))
    return len(np.unique(np.argpartition(-logits, TOPK, axis=1)[:, :TOPK]))


def _moe_work(tokens, zipf=False, router=True, shared=True):
    rows = 2 * HIDDEN * tokens
    nbytes = _unique_experts(tokens, zipf) * EXPERT_BYTES + 2 * rows + (2 + 8) * TOPK * tokens
    flops = TOPK * tokens * PAIR_FLOP
    if shared:
        nbytes += EXPERT_BYTES + 2 * HIDDEN
        flops += tokens * PAIR_FLOP
    if router:
        nbytes += 2 * EXPERTS * HIDDEN
        flops += 2 * EXPERTS * HIDDEN * tokens
    elif shared:
        nbytes += 2 * EXPERTS * tokens
    return nbytes, flops


def _mixer_work(tokens, record, state_bytes):
    state = 32 * 128 * 128 * state_bytes
    nbytes = MIXER_BYTES + 2 * state + 2 * 8192 * 4 * 2 + 2 * 2 * HIDDEN * tokens
    if record:
        nbytes += tokens * (state + 8192 * 4 * 2)
    flops = 2 * tokens * (12352 * HIDDEN + HIDDEN * 4096) + 8 * tokens * 32 * 128 * 128
    return nbytes, flops


def _attention_work(tokens, context):
    nbytes = ATTN_BYTES + (context + tokens) * 2 * 2 * 256 * 2 + 2 * 2 * HIDDEN * tokens
    flops = 2 * tokens * (9216 * HIDDEN + HIDDEN * 4096) + 4 * tokens * 16 * 256 * (context + tokens)
    return nbytes, flops


def work(case):
    kind, tokens = case["kind"], case["tokens"]
    if kind == "layer":
        zipf = case["routes"] == "zipf"
        nbytes, flops = _moe_work(tokens, zipf, router=not zipf)
    elif kind == "chain":
        nbytes, flops = (CHAIN_LAYERS * v for v in _moe_work(tokens))
    elif kind == "experts":
        nbytes, flops = _moe_work(tokens, zipf=True, router=False, shared=False)
    elif kind == "mixer":
        nbytes, flops = _mixer_work(tokens, case["record"], 4 if case["state"] == "fp32" else 2)
    elif kind == "attention":
        nbytes, flops = _attention_work(tokens, case["context"])
    elif kind == "decoder":
        parts = [_moe_work(tokens)] * STACK_LAYERS
        parts += [_attention_work(tokens, case["context"])] * (STACK_LAYERS // 4)
        parts += [_mixer_work(tokens, False, 4)] * (STACK_LAYERS * 3 // 4)
        nbytes, flops = sum(p[0] for p in parts), sum(p[1] for p in parts)
    else:
        nbytes, flops = 2 * round(_unique_experts(tokens, False)) * EXPERT_BYTES, 0
    return {"bytes": nbytes, "flops": flops}


# ---- what another correct implementation may differ by --------------------------

def tolerance(case):
    kind = case["kind"]
    if kind == "gather":
        return "exact"  # bytes are copied
    if kind in ("chain", "decoder"):
        # Rounding of one layer travels through the eight: a changed sum order
        # in bf16, and now and then a route that was nearly tied.
        return {"rel": 3e-2, "differ": 0.05}
    # Against 64 bits these measure 0.002 (rows with a residual) to 0.007 (the
    # mixer's and the attention's outputs): bf16 results of bf16 factors.
    return {"rel": 1e-2, "differ": 2e-3}


# ---- the same in 64 bits --------------------------------------------------------

def _d(t):
    return t.double()


def _swiglu(x, gate, up, down):
    g = x @ _d(gate).T
    return (torch.nn.functional.silu(g) * (x @ _d(up).T)) @ _d(down).T


def _exact_experts(bank, x, indices, weights):
    out = torch.zeros_like(x)
    for e in range(EXPERTS):
        token, slot = torch.nonzero(indices == e, as_tuple=True)
        if token.numel():
            gate_up, down = bank.expert(0, e)
            y = _swiglu(x[token], gate_up[:INNER], gate_up[INNER:], down)
            out.index_add_(0, token, y * _d(weights)[token, slot][:, None])
    return out


def _rms(x, weight, eps):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * (1.0 + _d(weight))


def _exact_layer(s):
    layer, x = s["layers"][0], _d(s["x"])
    # The router's rows and its logits are bf16 values by definition: routes
    # rank (logit descending, expert ascending).
    rows = x if layer.norm_weight is None else _d(_rms(x, layer.norm_weight, layer.eps).to(torch.bfloat16))
    logits = _d(s["logits"]) if s["logits"] is not None else _d((rows @ _d(layer.router).T).to(torch.bfloat16))
    order = torch.sort(logits, dim=-1, descending=True, stable=True).indices[:, :TOPK]
    p = torch.softmax(logits, dim=-1).gather(1, order)
    weights = p / p.sum(-1, keepdim=True)
    out = _exact_experts(s["bank"], rows, order, weights)
    gate = torch.sigmoid(rows @ _d(layer.shared_expert_gate))
    out += gate[:, None] * _swiglu(rows, layer.shared_gate_proj, layer.shared_up_proj, layer.shared_down_proj)
    if layer.norm_weight is not None:
        out += x
    return {"out": out, "indices": order, "weights": weights}


def _exact_mixer(s):
    m, x = s["mixer"], _d(s["x"])
    tokens = x.shape[0]
    inputs = torch.cat([_d(s["conv"]), (x @ _d(m.in_proj_qkv).T).T], dim=1)  # [8192, 4 + T]
    z = (x @ _d(m.in_proj_z).T).view(tokens, 32, 128)
    beta = torch.sigmoid(x @ _d(m.in_proj_b).T)
    decay = torch.exp(-_d(m.A_log).exp() * torch.nn.functional.softplus(x @ _d(m.in_proj_a).T + _d(m.dt_bias)))
    state = _d(s["state"])
    core, convs, states = [], [], []
    for t in range(tokens):
        window = inputs[:, t + 1:t + 5]
        act = torch.nn.functional.silu((window * _d(m.conv1d)).sum(1))
        q, k, v = act[:2048].view(16, 128), act[2048:4096].view(16, 128), act[4096:].view(32, 128)
        q, k = (u * torch.rsqrt(u.pow(2).sum(-1, keepdim=True) + 1e-6) for u in (q, k))
        q, k = q.repeat_interleave(2, 0) / math.sqrt(128.0), k.repeat_interleave(2, 0)
        state = state * decay[t][:, None, None]
        delta = (v - (state * k[:, :, None]).sum(1)) * beta[t][:, None]
        state = state + k[:, :, None] * delta[:, None, :]
        core.append((state * q[:, :, None]).sum(1))
        convs.append(window.clone())
        states.append(state)
    core = torch.stack(core)
    normed = core * torch.rsqrt(core.pow(2).mean(-1, keepdim=True) + m.eps) * _d(m.norm) * torch.nn.functional.silu(z)
    record = s["conv_record"] is not None
    return {"out": normed.reshape(tokens, 4096) @ _d(m.out_proj).T, "conv": convs[-1], "state": states[-1],
            "conv_record": torch.stack(convs) if record else None,
            "state_record": torch.stack(states) if record else None}


def _exact_attention(s):
    a, x, length = s["attention"], _d(s["x"]), s["case"]["context"]
    tokens = x.shape[0]
    qg = (x @ _d(a.q_proj).T).view(tokens, 16, 512)
    k, v = ((x @ _d(w).T).view(tokens, 2, 256) for w in (a.k_proj, a.v_proj))

    def norm_rope(h, weight):
        n = _rms(h, weight, a.eps)
        c, sn = _d(s["cos"])[:, None, :], _d(s["sin"])[:, None, :]
        rotated = torch.cat([-n[..., 32:64], n[..., :32]], dim=-1)
        return torch.cat([n[..., :64] * c + rotated * sn, n[..., 64:]], dim=-1)

    q, k = norm_rope(qg[..., :256], a.q_norm), norm_rope(k, a.k_norm)
    keys, values = _d(s["k"]), _d(s["v"])
    keys[:, length:length + tokens], values[:, length:length + tokens] = k.transpose(0, 1), v.transpose(0, 1)
    reach = torch.arange(length + tokens, device=x.device)[None] > length + torch.arange(tokens, device=x.device)[:, None]
    att = torch.empty((tokens, 16, 256), dtype=torch.float64, device=x.device)
    for h in range(16):
        scores = (q[:, h] @ keys[h // 8, :length + tokens].T / 16.0).masked_fill(reach, float("-inf"))
        att[:, h] = torch.softmax(scores, dim=-1) @ values[h // 8, :length + tokens]
    att = (att * torch.sigmoid(qg[..., 256:])).reshape(tokens, 4096)
    return {"out": att @ _d(a.o_proj).T, "k": keys, "v": values}


def exact(case, seed):
    kind = case["kind"]
    # A stack's routes follow its own rounding, so it has no value in 64 bits.
    if kind in ("chain", "decoder"):
        return None
    s = prepare(case, seed)
    if kind == "layer":
        return _exact_layer(s)
    if kind == "experts":
        return _exact_experts(s["bank"], _d(s["x"]), s["indices"], s["weights"])
    if kind == "mixer":
        return _exact_mixer(s)
    if kind == "attention":
        return _exact_attention(s)
    return s["bank"].bank[0, s["chosen"]]
