"""The prefill expert stage at the edges of its work units (needs an MI355X).

All tokens go to the same 8 experts, so every unit's size is known: one
column block, the edges of the 2-, 4- and 8-block variants (32, 64 and 128
rows of a unit), a second unit of one row, and the sizes around the switch
from non-temporal to cached weight rows (2560 tokens).  Outputs of a token
sample (every token up to 130) against the oracle within
helpers.assert_layer_close (1e-2, bf16 storage with fp32 accumulation).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import assert_layer_close, oracle_layer_rows, to_u16

pytestmark = pytest.mark.gpu

HOT = np.array([0, 31, 64, 127, 128, 200, 254, 255])


@pytest.mark.parametrize("tokens", [17, 32, 33, 48, 49, 64, 65, 127, 128, 129, 2559, 2561])
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
