"""Router logits on the matrix cores (more than 16 rows, many tokens): bit-exact, at the edges of its blocks."""
import numpy as np
import pytest

from jxai_amd import formats as F
from jxai_amd import synth

pytestmark = pytest.mark.gpu


# rows: one more than a block's 16, a ragged last block with the shared gate's row, several full ones; tokens: 64 a
# block; d: fewer chunks than buffers and more (64 floats a chunk)
@pytest.mark.parametrize("E,shared,d", [(17, False, 128), (24, True, 704), (64, False, 2304)])
@pytest.mark.parametrize("n", [512, 575, 641])
def test_router_logits_bitexact(port, E, shared, d, n):
    from jxai_amd import moe
    moe.init(0)
    print(f"[gpu] router E={E} shared={shared} d={d} n={n}", flush=True)
    cfg = synth.LayerConfig(f"rm_{E}_{d}", d, E, 4, 256, F.Q4_0, d_ff_shared=256 if shared else 0, shared_gate=shared)
    lw = synth.make_layer(cfg)
    x = synth.make_tokens(cfg, n)
    x[3] = 0.0
    x[5] *= np.float32(1e-37)  # subnormal products, and some that vanish
    products = np.abs(lw.router.astype(np.float64) * x[5].astype(np.float64))
    tiny = np.finfo(np.float32).tiny
    assert (products < tiny).mean() > 0.9 and (products > 2.0 ** -149).mean() > 0.9
    L = moe.MoELayer.from_weights(lw)
    _, ids, w, _ = L.forward(x)
    lg_o, ids_o, w_o = port.route(lw, x)
    assert np.array_equal(L.last_logits(n).view(np.uint32), lg_o.view(np.uint32))
    assert np.array_equal(ids, ids_o)
    np.testing.assert_allclose(w, w_o, rtol=2e-6, atol=0)
    L.close()


@pytest.mark.parametrize("n", [130, 512, 600])
def test_router_unaligned_x(port, n):
    """A caller's x on the alignment of a float only: the same logits and outputs, bit for bit."""
    from jxai_amd import moe
    moe.init(0)
    cfg = synth.LayerConfig("rm_off", 256, 24, 4, 256, F.Q4_0)
    lw = synth.make_layer(cfg)
    L = moe.MoELayer.from_weights(lw)
    x = synth.make_tokens(cfg, n)
    got = []
    for at in (0, 1, 2, 4):  # floats
        print(f"[gpu] router x off by {4 * at} bytes n={n}", flush=True)
        xb = moe.DeviceBuffer(x.nbytes + 64).upload(np.concatenate([np.zeros(at, np.float32), x.reshape(-1)]))
        xb.ptr = type(xb.ptr)(xb.ptr.value + 4 * at)
        out = moe.DeviceBuffer(x.nbytes)
        L.forward_device(xb, n, out)
        xb.ptr = type(xb.ptr)(xb.ptr.value - 4 * at)
        got.append((L.last_logits(n), out.download(np.empty_like(x))))
    assert np.array_equal(got[0][0].view(np.uint32), port.route(lw, x)[0].view(np.uint32))
    for logits, out in got[1:]:
        assert np.array_equal(logits.view(np.uint32), got[0][0].view(np.uint32))
        assert np.array_equal(out, got[0][1])
    L.close()
