"""The router of more than 16 tokens (fp32 MFMA chains) against the oracle,
bit for bit: logits, routes, shared gate and normalised rows (needs an
MI355X).

Sizes: one and two column tiles of 16 tokens (the single-tile kernel serves
up to 240 tokens with a shared gate, 256 without), remainders on both sides
of a tile, and row tiles split over 8, 4 and 1 workgroups per token tile.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import to_u16

pytestmark = pytest.mark.gpu


def _check(x, router, norm, gate, oracle, eps=1e-6):
    from lightreason_amd.moe import Workspace, route_topk

    tokens = x.shape[0]
    ws = Workspace(x.device, tokens)
    indices, weights, logits, sg, normed = route_topk(x, router, norm_weight=norm, eps=eps, shared_expert_gate=gate,
                                                      workspace=ws)
    torch.cuda.synchronize()
    rows = to_u16(x)
    if norm is not None:
        rows = oracle.rmsnorm(rows, to_u16(norm), eps)
        np.testing.assert_array_equal(to_u16(normed), rows)
    o_logits, o_idx, o_w = oracle.route(rows, to_u16(router))
    np.testing.assert_array_equal(to_u16(logits), o_logits)
    np.testing.assert_array_equal(indices.cpu().numpy(), o_idx)
    np.testing.assert_array_equal(to_u16(weights), o_w)
    if gate is not None:
        np.testing.assert_array_equal(to_u16(sg), oracle.shared_gate(rows, to_u16(gate)))
    assert ws.status() == 0


FORMS = [(True, True), (False, True), (True, False), (False, False)]


@pytest.mark.parametrize("tokens,norm,gate",
                         [(t, *form) for t in (17, 31, 32, 33, 240, 241, 257) for form in FORMS]
                         + [(t, True, True) for t in (600, 2080, 4100)])  # the oracle takes seconds there
def test_router_tiles_bit_exact(model, oracle, tokens, norm, gate):
    layer = model.layers[0]
    print(f"[router] T={tokens} norm={norm} gate={gate}", flush=True)
    _check(model.hidden(tokens, step=7000 + tokens), layer.router, layer.norm_weight if norm else None,
           layer.shared_expert_gate if gate else None, oracle, layer.eps)


@pytest.mark.parametrize("scale_x,scale_w", [(-70, -62), (40, 30)])
def test_router_tiles_extreme_exponents(model, oracle, scale_x, scale_w):
    """Products and sums near the subnormal range, and far above 1."""
    layer = model.layers[0]
    x = model.hidden(50, step=7777) * 2.0**scale_x
    print(f"[router] exponents {scale_x} {scale_w}", flush=True)
    _check(x, layer.router * 2.0**scale_w, None, layer.shared_expert_gate, oracle)


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
