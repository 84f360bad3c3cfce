"""The router of more than 16 tokens (fp32 MFMA chains) against the oracle,
bit for bit: logits, routes, shared gate and normalised rows (needs an
MI355X).

Sizes: one and two column tiles of 16 tokens (the single-tile kernel serves
up to 240 tokens with a shared gate, 256 without), remainders on both sides
of a tile, and the row tiles (16, and one for the gate) split over 17, 16, 9,
6, 5, 4, 3 and 1 workgroups per token tile.  From three row tiles per
workgroup on, half of the waves run half a tile behind: workgroups of one row
tile (1100 tokens without a gate: 3 x 5 + 1; 1400 with: 4 x 4 + 1) meet the end
of that loop at its start.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import to_u16

pytestmark = pytest.mark.gpu


def _check(x, router, norm, gate, oracle, eps=1e-6, sample=None):
    """``sample``: the tokens to compare (all when None)."""
    from lightreason_amd.moe import Workspace, route_topk

    tokens = x.shape[0]
    sample = slice(None) if sample is None else torch.from_numpy(sample).to(x.device)
    ws = Workspace(x.device, tokens)
    indices, weights, logits, sg, normed = route_topk(x, router, norm_weight=norm, eps=eps, shared_expert_gate=gate,
                                                      workspace=ws)
    torch.cuda.synchronize()
    rows = to_u16(x[sample])
    if norm is not None:
        rows = oracle.rmsnorm(rows, to_u16(norm), eps)
        np.testing.assert_array_equal(to_u16(normed[sample]), rows)
    o_logits, o_idx, o_w = oracle.route(rows, to_u16(router))
    np.testing.assert_array_equal(to_u16(logits[sample]), o_logits)
    np.testing.assert_array_equal(indices[sample].cpu().numpy(), o_idx)
    np.testing.assert_array_equal(to_u16(weights[sample]), o_w)
    if gate is not None:
        np.testing.assert_array_equal(to_u16(sg[sample]), oracle.shared_gate(rows, to_u16(gate)))
    assert ws.status() == 0


FORMS = [(True, True), (False, True), (True, False), (False, False)]


@pytest.mark.parametrize("tokens,norm,gate",
                         [(t, *form) for t in (17, 31, 32, 33, 240, 241, 257) for form in FORMS]
                         + [(t, True, True) for t in (600, 1400, 2080, 4100)]  # the oracle takes seconds there
                         + [(1100, False, False), (1100, True, False)])
def test_router_tiles_bit_exact(model, oracle, tokens, norm, gate):
    layer = model.layers[0]
    print(f"[router] T={tokens} norm={norm} gate={gate}", flush=True)
    _check(model.hidden(tokens, step=7000 + tokens), layer.router, layer.norm_weight if norm else None,
           layer.shared_expert_gate if gate else None, oracle, layer.eps)


@pytest.mark.parametrize("tokens,norm,gate", [(6200, True, True), (6200, False, False)])
def test_one_workgroup_per_token_tile(model, oracle, tokens, norm, gate):
    """All row tiles in one workgroup: every column of the first, a middle and
    the last two token tiles."""
    layer = model.layers[0]
    sample = np.r_[0:32, 3104:3136, 6144:tokens]
    print(f"[router] T={tokens} norm={norm} gate={gate}", flush=True)
    _check(model.hidden(tokens, step=7000 + tokens), layer.router, layer.norm_weight if norm else None,
           layer.shared_expert_gate if gate else None, oracle, layer.eps, sample=sample)


@pytest.mark.parametrize("tokens", [50, 300])
@pytest.mark.parametrize("scale_x,scale_w", [(-70, -62), (40, 30), (-130, 100), (0, -125)])
def test_router_tiles_extreme_exponents(model, oracle, tokens, scale_x, scale_w):
    """Products and sums near the subnormal range, and far above 1; subnormal
    rows and subnormal router rows."""
    layer = model.layers[0]
    x = (model.hidden(tokens, step=7777).float() * 2.0**scale_x).to(torch.bfloat16)
    router = (layer.router.float() * 2.0**scale_w).to(torch.bfloat16)
    if scale_x == -130 or scale_w == -125:
        tiny = (x if scale_x == -130 else router).float().abs()
        assert bool(((tiny > 0) & (tiny < 2.0**-126)).any())
    print(f"[router] T={tokens} exponents {scale_x} {scale_w}", flush=True)
    _check(x, router, None, layer.shared_expert_gate, oracle)


@pytest.mark.parametrize("tokens", [40, 300])
@pytest.mark.parametrize("norm", [False, True])
def test_router_tiles_inf_and_nan(model, oracle, tokens, norm):
    """Infinities and NaN in token rows and router rows: they reach exactly
    the logits that the oracle's do, every other logit keeps its bits, and the
    routes are those of the logits.  (The sign and payload of a NaN are the
    processor's.)"""
    from lightreason_amd.moe import Workspace, route_topk

    layer = model.layers[0]
    inf, nan = float("inf"), float("nan")
    x, router = model.hidden(tokens, step=7600 + tokens), layer.router.clone()
    last = tokens - 1
    x[3, 5], x[17, 700], x[20, 2047], x[last, 1000] = inf, -inf, nan, inf
    x[last, 1001] = -inf
    router[9, 33], router[100, 1500], router[255, 0] = inf, nan, -inf
    print(f"[router] inf and nan T={tokens} norm={norm}", flush=True)
    indices, weights, logits, _, normed = route_topk(x, router, norm_weight=layer.norm_weight if norm else None,
                                                     eps=layer.eps, workspace=Workspace(x.device, tokens))
    torch.cuda.synchronize()

    def masked(bits):  # NaN -> one value
        return np.where((bits & 0x7FFF) > 0x7F80, 0x7FC0, bits)

    rows = to_u16(x)
    if norm:
        rows = oracle.rmsnorm(rows, to_u16(layer.norm_weight), layer.eps)
        np.testing.assert_array_equal(masked(to_u16(normed)), masked(rows))
    want, _, _ = oracle.route(rows, to_u16(router))
    got = to_u16(logits)
    np.testing.assert_array_equal(masked(got), masked(want))
    idx, wts = oracle.route_logits(got)
    np.testing.assert_array_equal(indices.cpu().numpy(), idx)
    np.testing.assert_array_equal(masked(to_u16(weights)), masked(wts))


@pytest.mark.parametrize("tokens", [40, 300])
def test_norm_and_gate_with_caller_logits(model, oracle, tokens):
    """Caller logits: the rows are still normalised and the gate computed."""
    from lightreason_amd.moe import Workspace, route_topk

    layer = model.layers[0]
    x = model.hidden(tokens, step=7900 + tokens)
    logits = model.hidden(tokens, step=7950 + tokens)[:, :256].contiguous()
    print(f"[router] caller logits T={tokens}", flush=True)
    indices, _, _, sg, normed = route_topk(x, None, logits_in=logits, norm_weight=layer.norm_weight, eps=layer.eps,
                                           shared_expert_gate=layer.shared_expert_gate,
                                           workspace=Workspace(x.device, tokens))
    torch.cuda.synchronize()
    rows = oracle.rmsnorm(to_u16(x), to_u16(layer.norm_weight), layer.eps)
    np.testing.assert_array_equal(to_u16(normed), rows)
    np.testing.assert_array_equal(to_u16(sg), oracle.shared_gate(rows, to_u16(layer.shared_expert_gate)))
    np.testing.assert_array_equal(indices.cpu().numpy(), oracle.route_logits(to_u16(logits))[0])
