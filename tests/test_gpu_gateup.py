"""The matrix-core gate/up GEMM at the edges of its tiles, against the oracle."""
import numpy as np
import pytest

from jxai_amd import formats as F
from jxai_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def moe():
    from jxai_amd import moe as M
    M.init(0)
    return M


# d: one half-unit of 128 columns, an odd number of them, several super-blocks; d_ff: row tiles that leave
# waves of the last workgroup without one; tokens: either side of a workgroup's 64 pairs and of a dispatch tile's
# 128 (both experts see every token)
@pytest.mark.parametrize("fmt,d,ff", [(F.Q4_0, 128, 32), (F.Q4_0, 384, 416), (F.Q8_0, 128, 32), (F.Q8_0, 640, 288),
                                      (F.Q4_K, 256, 256), (F.Q4_K, 768, 1280), (F.Q5_K, 256, 256), (F.Q5_K, 512, 768)])
def test_gateup_tile_edges(moe, port, fmt, d, ff):
    cfg = synth.LayerConfig(f"gu_{fmt}_{d}_{ff}", d, 2, 2, ff, fmt)
    lw = synth.make_layer(cfg)
    L = moe.MoELayer.from_weights(lw)
    for n in (1, 33, 64, 65, 127, 130):
        print(f"[gpu] gate/up {fmt} d={d} ff={ff} n={n}", flush=True)
        x = synth.make_tokens(cfg, n)
        x[n // 2, :32] = 0.0  # a zero block
        out, ids, _, _ = L.forward(x, regime="mfma")
        want, ids_o, _, _ = port.moe_forward(lw, x)
        assert np.array_equal(ids, ids_o)
        # the layer bar: a last-bit difference in a gate/up sum moves a value of h by one of 127 steps
        assert (np.abs(out - want).max(axis=1) / np.abs(want).max(axis=1)).max() <= 1e-3
    L.close()
