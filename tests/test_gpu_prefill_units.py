"""The prefill expert stage at the edges of its work units (needs an MI355X).

All tokens go to the same 8 experts, so every unit's size is known: one
column block, the edges of the 2-, 4- and 8-block variants (32, 64 and 128
rows of a unit).  Up to 128 tokens an expert is one unit and its weight rows
are non-temporal, above that they are cached: 129-256 tokens are a full unit and
one at the same edges.
Outputs of a token sample (every token up to 130) against the oracle within
helpers.assert_layer_close (1e-2, bf16 storage with fp32 accumulation).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import assert_layer_close, oracle_layer_rows, to_u16

pytestmark = pytest.mark.gpu

HOT = np.array([0, 31, 64, 127, 128, 200, 254, 255])


@pytest.mark.parametrize("tokens", [17, 32, 33, 48, 49, 64, 65, 127, 128, 129, 159, 160, 161, 192, 193,
                                    255, 256, 257, 2559, 2561])
@pytest.mark.parametrize("norm", [False, True])
def test_units_of_known_size(model, oracle, host_experts, tokens, norm):
    from lightreason_amd.moe import LayerWeights, Workspace, moe_layer

    rng = np.random.default_rng(tokens)
    logits = rng.normal(0.0, 1.0, size=(tokens, 256))
    logits[:, HOT] += 14.0
    x = model.hidden(tokens, step=8000 + tokens)
    logits = torch.from_numpy(logits.astype(np.float32)).to(torch.bfloat16).to(x.device)
    base = model.layers[0]
    layer = LayerWeights(**{**base.__dict__, "norm_weight": base.norm_weight if norm else None})
    ws = Workspace(x.device, tokens)
    idx = torch.empty((tokens, 8), dtype=torch.int64, device=x.device)
    print(f"[units] T={tokens} norm={norm}", flush=True)
    out = moe_layer(x, layer, indices=idx, logits_in=logits, workspace=ws)
    torch.cuda.synchronize()
    assert ws.status() == 0
    assert set(np.unique(idx.cpu().numpy()).tolist()) == set(HOT.tolist())
    xb = to_u16(x)
    if tokens <= 130:
        rows = np.arange(tokens)
    else:
        last = tokens // 128 * 128
        rows = np.unique([0, 15, 16, 127, 128, 129, last - 1, min(last, tokens - 1), tokens - 1])
    want, _, _ = oracle_layer_rows(oracle, layer, xb, host_experts, rows=rows, logits_bits=to_u16(logits))
    assert_layer_close(to_u16(out)[rows], want, xb[rows] if norm else None, what=f"units T={tokens}")


@pytest.mark.parametrize("tokens", [65, 121, 128, 129, 2041, 2048, 2049, 2100])
def test_plan_around_the_scan_launch(device, oracle, tokens):
    """Up to 2048 tokens (256 blocks) the plan's last kernel counts the block
    masks itself, above that a scan launch does: whole 16-byte words of masks,
    their remainders, and both sides of the switch, against the oracle; then
    a bad route in the last block of each."""
    from helpers import uniform_routes, zipf_routes
    from lightreason_amd.moe import Workspace, bucket

    idx, _ = (zipf_routes if tokens % 2 else uniform_routes)(tokens, 100 + tokens)
    ws = Workspace(device, tokens)
    ws.buffer.fill_(0xA5)  # nothing may be read that the call did not write
    print(f"[plan] T={tokens}", flush=True)
    plan = bucket(torch.from_numpy(idx).to(device), ws)
    torch.cuda.synchronize()
    ref = oracle.bucket(idx)
    unique = int(plan["unique"].item())
    assert int(plan["status"].item()) == 0 and unique == ref["unique"]
    np.testing.assert_array_equal(plan["expert"][:unique].cpu().numpy(), ref["expert"])
    np.testing.assert_array_equal(plan["offset"][:unique + 1].cpu().numpy(), ref["offset"])
    for name in ("pair_token", "pair_slot", "route_pair"):
        np.testing.assert_array_equal(plan[name].cpu().numpy(), ref[name])
    idx[-1, 3] = 256
    plan = bucket(torch.from_numpy(idx).to(device), ws)
    assert int(plan["status"].item()) == 1 and int(plan["unique"].item()) == 0
    assert bool((plan["route_pair"] == -1).all())


def _two_sizes(model, small, large, routes, weights, x, what):
    """Routed experts of the first ``small`` and of all ``large`` tokens of
    every set of ``routes``: a token's row is the same bits in both calls.
    Returns the best us per call of each size, the sets in turn (more weights
    than the caches hold)."""
    from lightreason_amd.moe import Workspace, moe_experts

    sets = len(routes)
    ptrs = model.layers[0].expert_ptrs
    ws = {t: Workspace(x.device, t) for t in (small, large)}

    def call(tokens, s):
        return moe_experts(x[:tokens], routes[s][:tokens], weights[:tokens], ptrs, workspace=ws[tokens])

    def time(tokens):
        start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        for s in range(sets):
            call(tokens, s)
        start.record()
        for i in range(4 * sets):
            call(tokens, i % sets)
        stop.record()
        stop.synchronize()
        return start.elapsed_time(stop) / (4 * sets) * 1e3

    print(f"[units] {what}", flush=True)
    for s in range(sets):
        assert torch.equal(call(small, s).view(torch.int16), call(large, s)[:small].view(torch.int16))
    assert ws[small].status() == 0 and ws[large].status() == 0
    times = [(time(small), time(large)) for _ in range(7)]
    best = [min(t) for t in zip(*times)]
    print(f"[units] {small} tokens {best[0]:.1f} us, {large} tokens {best[1]:.1f} us", flush=True)
    return best


def test_one_item_per_workgroup_takes_one_round(model):
    """1000 tokens on 8 experts are 64 units, 256 gate/up items for 256
    workgroups; 512 tokens are 128 items.  The larger call must not take a
    second round (measured 1.08 times the smaller call's time; 1.42 when a
    workgroup claimed its second item before every one had a first)."""
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("sizes are chosen for 256 workgroups")
    rng = np.random.default_rng(88)
    x = model.hidden(1000, step=8800)
    experts = rng.permutation(256)[:48].reshape(6, 8)
    routes = [torch.from_numpy(np.stack([rng.permutation(e) for _ in range(1000)]).astype(np.int64)).to(x.device)
              for e in experts]
    weights = torch.softmax(torch.from_numpy(rng.normal(size=(1000, 8))), dim=1).to(torch.bfloat16).to(x.device)
    best = _two_sizes(model, 512, 1000, routes, weights, x, "one item per workgroup")
    assert best[1] < 1.25 * best[0], best


def test_second_units_find_their_rows_cached(model):
    """96 experts of 128 tokens are one unit each, of 129 two: twice the
    weight rows read, the second time through the caches (measured 1.24 times
    the smaller call's time; 1.48 with all rows non-temporal).  The two calls
    fall on the two sides of the rule that chooses."""
    rng = np.random.default_rng(96)
    x = model.hidden(12 * 129, step=8900)
    token = 8 * np.arange(12 * 129)[:, None] + np.arange(8)[None]  # expert e: tokens e/8, e/8 + 12, ..
    routes = [torch.from_numpy(rng.permutation(256)[:96][token % 96].astype(np.int64)).to(x.device) for _ in range(2)]
    weights = torch.softmax(torch.from_numpy(rng.normal(size=(12 * 129, 8))), dim=1).to(torch.bfloat16).to(x.device)
    best = _two_sizes(model, 12 * 128, 12 * 129, routes, weights, x, "second units")
    assert best[1] < 1.36 * best[0], best


def test_lists_of_one_xcd_share_cached_rows(model):
    """24 experts of 256 tokens are two units each, of 257 three: 288 gate/up
    items for 256 workgroups, the third units of one row (measured 1.07 times
    the smaller call's time; 1.20 with lists over two XCDs, whose L2s each
    fetched an expert's rows)."""
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("sizes are chosen for 256 workgroups")
    rng = np.random.default_rng(24)
    x = model.hidden(3 * 257, step=9000)
    token = 8 * np.arange(3 * 257)[:, None] + np.arange(8)[None]
    experts = rng.permutation(256)[:240].reshape(10, 24)
    routes = [torch.from_numpy(e[token % 24].astype(np.int64)).to(x.device) for e in experts]
    weights = torch.softmax(torch.from_numpy(rng.normal(size=(3 * 257, 8))), dim=1).to(torch.bfloat16).to(x.device)
    best = _two_sizes(model, 3 * 256, 3 * 257, routes, weights, x, "lists of one XCD")
    assert best[1] < 1.14 * best[0], best


def test_captured_call_chooses_at_each_replay(model):
    """The form of the expert kernel is chosen from the plan on the device: a
    captured call replays routes on either side of the rule, and bad ones,
    as an eager call answers them."""
    from lightreason_amd.moe import Workspace, moe_experts

    tokens = 200
    rng = np.random.default_rng(200)
    x = model.hidden(tokens, step=9100)
    device = x.device
    few = np.stack([rng.permutation(HOT) for _ in range(tokens)])  # two units per expert: cached rows
    wide = np.stack([rng.permutation(256)[:8] for _ in range(tokens)])  # one: non-temporal rows
    bad = wide.copy()
    bad[77, 2] = 256
    weights = torch.softmax(torch.from_numpy(rng.normal(size=(tokens, 8))), dim=1).to(torch.bfloat16).to(device)
    ptrs = model.layers[0].expert_ptrs
    indices = torch.from_numpy(wide.astype(np.int64)).to(device)
    out = torch.empty_like(x)
    ws, eager = Workspace(device, tokens), Workspace(device, tokens)
    print("[units] captured call", flush=True)
    moe_experts(x, indices, weights, ptrs, out=out, workspace=ws)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        moe_experts(x, indices, weights, ptrs, out=out, workspace=ws)
    for routes, status in ((few, 0), (wide, 0), (bad, 1), (few, 0), (few, 0), (wide, 0)):
        indices.copy_(torch.from_numpy(routes.astype(np.int64)))
        out.fill_(7.0)
        graph.replay()
        want = moe_experts(x, indices, weights, ptrs, workspace=eager)
        torch.cuda.synchronize()
        assert ws.status() == status and eager.status() == status
        assert torch.equal(out.view(torch.int16), want.view(torch.int16))
        assert bool(want.any()) == (status == 0)
