"""The matrix-core gate/up GEMM and the projection launch at the edges of their tiles, against the oracle."""
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
        # A last-bit difference in a gate/up sum can move a value of h by one step, amax / 127 of its block.  One
        # step of a block with amax = 4 sigma_h against a weight of 3 sigma_w changes an output by 12 sigma_w
        # sigma_h / 127, and the largest of a row's outputs is about 3 sqrt(d_ff) sigma_w sigma_h: 1 / (32 sqrt(d_ff))
        # of it, the layer bar of 1e-3 from d_ff = 1024 on.  Most tokens have no such step.
        err = np.abs(out - want).max(axis=1) / np.abs(want).max(axis=1)
        assert err.max() <= max(1e-3, 1 / (32 * np.sqrt(ff)))
        assert np.median(err) <= 1e-3
    L.close()


# d: an odd number of the down's row tiles, so the last wave's second one is past the matrix; d_ff: odd numbers of its
# half-units, and (from 8192 columns) K in two parts, for Q4_0 and Q8_0 the second an odd number of half-units.  Pairs
# per expert as the tokens: one, either side of a pair tile, of a workgroup, and many (from 24 the FP6 forms' two-tile loop)
@pytest.mark.parametrize("codes", ["1", "0"])
@pytest.mark.parametrize("fmt,d,ff", [(F.Q4_0, 160, 384), (F.Q8_0, 160, 384), (F.Q4_0, 96, 8320), (F.Q8_0, 96, 8320),
                                      (F.Q4_K, 288, 512), (F.Q5_K, 288, 512), (F.Q4_K, 32, 8448), (F.Q5_K, 32, 8448)])
def test_down_tile_edges(moe, port, monkeypatch, fmt, d, ff, codes):
    monkeypatch.setenv("JX_GEMM_CODES", codes)
    cfg = synth.LayerConfig(f"dn_{fmt}_{d}_{ff}", d, 2, 2, ff, fmt)
    lw = synth.make_layer(cfg)
    L = moe.MoELayer.from_weights(lw)
    for n in (1, 23, 32, 33, 65):
        print(f"[gpu] down {fmt} d={d} ff={ff} codes={codes} n={n}", flush=True)
        x = synth.make_tokens(cfg, n)
        out, ids, _, _ = L.forward(x, regime="mfma")
        want, ids_o, _, _ = port.moe_forward(lw, x)
        assert np.array_equal(ids, ids_o)
        # one step of h in a row's output, as test_gateup_tile_edges (K-quants with d off whole super-blocks have
        # their gate/up on fp32 activations)
        err = np.abs(out - want).max(axis=1) / np.abs(want).max(axis=1)
        assert err.max() <= max(1e-3, 1 / (32 * np.sqrt(ff)))
        assert np.median(err) <= 1e-3
    L.close()


def extreme_blocks(fmt, rows, cols, seed):
    """A matrix whose 32-blocks each hold one extreme quant throughout (each sign where the format has one), or both."""
    raw = synth.quant_matrix(seed, fmt, rows, cols).reshape(-1, F.BLOCK[fmt][1]).copy()
    pick = synth.random_bytes(seed ^ 0x77, raw.shape[0]) % 3
    lo, hi = (0x81, 0x7F) if fmt == F.Q8_0 else (0x00, 0xFF)
    at = {F.Q4_0: 2, F.Q8_0: 2, F.Q4_K: 16, F.Q5_K: 16}[fmt]
    fill = np.where(pick == 0, lo, hi).astype(np.uint8)[:, None]
    body = np.broadcast_to(fill, (raw.shape[0], raw.shape[1] - at)).copy()
    mixed = pick == 2
    body[mixed, ::2] = lo
    body[mixed, 1::2] = hi
    raw[:, at:] = body
    return raw.reshape(-1)


@pytest.mark.parametrize("codes", ["1", "0"])
@pytest.mark.parametrize("fmt", [F.Q4_0, F.Q8_0, F.Q4_K, F.Q5_K])
def test_extreme_quants(moe, port, monkeypatch, fmt, codes):
    """Whole blocks of the weights' largest quants against activations of +-127: the block sums of the greatest
    magnitude (a down of one-hot columns would hide them: h is what the gate/up leaves)."""
    monkeypatch.setenv("JX_GEMM_CODES", codes)
    cfg = synth.LayerConfig(f"ext_{fmt}", 512, 2, 2, 1280, fmt)
    lw = synth.make_layer(cfg)
    lw.gate = extreme_blocks(fmt, 2 * 1280, 512, synth.sub_seed("ext", "gate"))
    lw.up = extreme_blocks(fmt, 2 * 1280, 512, synth.sub_seed("ext", "up"))
    lw.down = extreme_blocks(fmt, 2 * 512, 1280, synth.sub_seed("ext", "down"))
    L = moe.MoELayer.from_weights(lw)
    n = 70
    print(f"[gpu] extreme quants {fmt} codes={codes}", flush=True)
    sign = np.where(synth.random_bytes(synth.sub_seed("ext", "x"), n * 512) & 1, 1, -1).reshape(n, 512)
    x = (sign * np.repeat(0.5 + synth.uniform01(synth.sub_seed("ext", "s"), n * 16), 32).reshape(n, 512)).astype(np.float32)
    x[:8] = np.abs(x[:8])
    x[8:16, ::2] = np.abs(x[8:16, ::2])
    x[8:16, 1::2] = -np.abs(x[8:16, 1::2])
    x *= np.float32(0.02)
    out, ids, _, _ = L.forward(x, regime="mfma")
    q = L.last_xq8(n).reshape(n, 16, 34)[:, :, 2:].view(np.int8)
    assert (np.abs(q.astype(np.int32)) == 127).all()
    want, ids_o, _, _ = port.moe_forward(lw, x)
    assert np.array_equal(ids, ids_o)
    err = np.abs(out - want).max(axis=1) / np.abs(want).max(axis=1)
    # d_ff past 1024: the layer bar (a step of h against the down's extreme weights stays in proportion to the output)
    assert err.max() <= 1e-3, err
    L.close()


# the largest batch of the GEMVs and the smallest of the GEMMs: 10 pairs per expert (Q4_0; 7 where the gate/up workgroups
# fill the chip once, or beside a shared expert of four times the size), 12 (K-quants), 12 tokens (Q8_0); the same with a
# down that has no block GEMM
@pytest.mark.parametrize("fmt,n,kw", [(F.Q4_0, 40, {}), (F.Q4_0, 28, dict(n_experts=16, top_k=4, d_ff=1024)),
                                      (F.Q4_0, 40, dict(n_experts=64, top_k=16, d_ff=1152)),
                                      (F.Q4_0, 28, dict(d_ff=256, d_ff_shared=1024)),
                                      (F.Q4_0, 40, dict(down_wtype=F.Q6_K)), (F.Q4_0, 40, dict(down_wtype=F.Q5_0)),
                                      (F.Q4_K, 48, {}), (F.Q8_0, 12, {}), (F.Q8_0, 12, dict(down_wtype=F.Q6_K))])
def test_regime_edge(moe, port, fmt, n, kw):
    """Either side of the line the layer's own choice is that regime's result bit for bit, and the oracle's."""
    kw = dict(dict(n_experts=8, top_k=2, d_ff=1280), **kw)
    cfg = synth.LayerConfig("edge_" + "_".join(str(v) for v in (fmt, *kw.values())), 512, wtype=fmt, **kw)
    lw = synth.make_layer(cfg)
    L = moe.MoELayer.from_weights(lw)
    for m, regime in ((n - 1, "gemv"), (n, "mfma")):
        print(f"[gpu] regime edge {fmt} {kw} n={m}", flush=True)
        x = synth.make_tokens(cfg, m)
        out, ids, _, _ = L.forward(x)
        assert np.array_equal(out, L.forward(x, regime=regime)[0])
        want, ids_o, _, _ = port.moe_forward(lw, x)
        assert np.array_equal(ids, ids_o)
        # the layer bar from d_ff = 1024 on (one step of h below it: 1 / (32 sqrt(d_ff)) of a row's largest output)
        err = np.abs(out - want).max(axis=1) / np.abs(want).max(axis=1)
        assert err.max() <= max(1e-3, 1 / (32 * np.sqrt(cfg.d_ff))) and np.median(err) <= 1e-3
    L.close()


@pytest.mark.parametrize("fmt,n,kw", [(F.Q4_0, 160, {}), (F.Q4_0, 128, dict(sh_down_wtype=F.Q5_0)), (F.Q4_K, 128, {}),
                                      (F.Q8_0, 128, {}), (F.Q6_K, 64, {}), (F.Q5_0, 64, {})])
def test_shared_regime_edge(moe, monkeypatch, fmt, n, kw):
    """The shared expert's own line: below it the GEMVs' result, from it the GEMMs'."""
    cfg = synth.LayerConfig(f"shedge_{fmt}_{len(kw)}", 512, 4, 2, 256, fmt, d_ff_shared=512, **kw)
    lw = synth.make_layer(cfg)
    layers = []
    for line in (None, "1000000", "1"):
        if line:
            monkeypatch.setenv("JX_SMFMA_MIN", line)
        layers.append(moe.MoELayer.from_weights(lw))
    print(f"[gpu] shared regime edge {fmt} {kw} n={n}", flush=True)
    for m, same, other in ((n - 1, 1, 2), (n, 2, 1)):
        x = synth.make_tokens(cfg, m)
        out = [L.forward(x)[0] for L in layers]
        assert np.array_equal(out[0], out[same])
        assert not np.array_equal(out[0], out[other])  # (the two round differently)
    for L in layers:
        L.close()


@pytest.mark.parametrize("fmt", [F.Q4_0, F.Q8_0, F.Q4_K, F.Q5_K, F.Q6_K])
@pytest.mark.parametrize("cols,rows", [(256, (8, 33, 1)), (4352, (160, 32, 64))])
def test_projection_launch(moe, port, fmt, cols, rows):
    """q, k and v in one launch (ragged row counts, more columns than one pass of the staged quantization) equal
    the one-matrix call bit for bit: the same block sums in the same order."""
    print(f"[gpu] projection {fmt} cols={cols} rows={rows}", flush=True)
    x = synth.normal_f32(synth.sub_seed("qkvp", f"x{cols}"), cols, 1.0)
    mats = [synth.quant_matrix(synth.sub_seed("qkvp", f"{i}{cols}"), fmt, r, cols) for i, r in enumerate(rows)]
    qm = [moe.QMatrix(fmt, m, r, cols) for m, r in zip(mats, rows)]
    xb = moe.DeviceBuffer(x.nbytes).upload(x)
    outs = [moe.DeviceBuffer(r * 4) for r in rows]
    assert moe.lib().jx_matmul_qkv_quant_f32_dev(*[q.handle for q in qm], xb.ptr, *[o.ptr for o in outs], None) == 0
    moe.lib().jx_device_synchronize()
    for m, r, o, q in zip(mats, rows, outs, qm):
        got = o.download(np.empty(r, np.float32))
        if r >= 8:  # fewer rows alone take fp32 activations
            one = moe.DeviceBuffer(r * 4)
            assert moe.lib().jx_matmul_quant_f32_dev(q.handle, xb.ptr, one.ptr, None) == 0
            moe.lib().jx_device_synchronize()
            assert np.array_equal(got, one.download(np.empty(r, np.float32)))
        want = port.matmul_qkv_quant_f32([(fmt, m, r), (fmt, mats[0], rows[0]), None], x)[0]
        assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()
    for q in qm:
        q.close()


# the projections on one format and on mixed ones (Q5_0 takes fp32 activations)
@pytest.mark.parametrize("fmts", [(F.Q4_K, F.Q4_K, F.Q4_K), (F.Q4_0, F.Q8_0, F.Q4_0), (F.Q8_0, F.Q5_0, F.Q6_K)])
@pytest.mark.parametrize("at", [0, 100, 4000])
def test_projection_outputs_over_x(moe, fmts, at):
    """An output that shares memory with x (its start, its middle, its end) changes nothing: every product uses x
    as it was before the call.  Where k and v share memory, v stands."""
    cols, rows = 4096, (2048, 96, 320)
    print(f"[gpu] projection over x {fmts} at {at}", flush=True)
    x = synth.normal_f32(synth.sub_seed("qkvo", "x"), cols, 1.0)
    qm = [moe.QMatrix(f, synth.quant_matrix(synth.sub_seed("qkvo", f"{i}"), f, r, cols), r, cols)
          for i, (f, r) in enumerate(zip(fmts, rows))]
    buf = moe.DeviceBuffer(4 * (cols + 8192))
    sep = [moe.DeviceBuffer(r * 4) for r in rows]

    def call(ptrs):
        buf.upload(x)
        assert moe.lib().jx_matmul_qkv_quant_f32_dev(*[q.handle for q in qm], buf.ptr, *ptrs, None) == 0
        moe.lib().jx_device_synchronize()

    call([b.ptr for b in sep])
    want = [b.download(np.empty(r, np.float32)) for b, r in zip(sep, rows)]
    for over in range(3):
        for b in sep:
            b.upload(np.zeros(b.nbytes // 4, np.float32))
        call([buf.ptr.value + 4 * at if i == over else b.ptr for i, b in enumerate(sep)])
        whole = buf.download(np.empty(cols + 8192, np.float32))
        for i, (b, r) in enumerate(zip(sep, rows)):
            got = whole[at:at + r] if i == over else b.download(np.empty(r, np.float32))
            assert np.array_equal(got, want[i]), (over, i)
    call([sep[0].ptr, sep[2].ptr, sep[2].ptr])
    assert np.array_equal(sep[2].download(np.empty(rows[2], np.float32)), want[2])
    for q in qm:
        q.close()
