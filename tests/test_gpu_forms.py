"""What the block GEMM holds beside the weights: its bounds in device memory, and the same results with and without."""
import ctypes as C

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


def free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    assert C.CDLL("libamdhip64.so").hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value, total.value


def held(moe, lw):
    """Device bytes that a layer of these weights takes, per weight, beyond 32 MB for its small buffers and streams (each
    allocation takes whole pages of 2 MB)."""
    before = free_bytes()[0]
    L = moe.MoELayer.from_weights(lw)
    used = before - free_bytes()[0]
    L.close()
    return (used - (32 << 20)) / (3.0 * lw.cfg.n_experts * lw.cfg.d_model * lw.cfg.d_ff)


# bytes per weight of the blocks and (K-quants) the 0.25 or 0.31 of the table; the codes take 0.75 to 0.88 more
@pytest.mark.parametrize("fmt,least,codes", [(F.Q4_0, 0.5625, 0.875), (F.Q4_K, 0.8125, 0.75), (F.Q5_K, 1.0, 0.75),
                                             (F.Q8_0, 1.0625, 0.0)])
def test_memory_without_codes(moe, monkeypatch, fmt, least, codes):
    """The second copy of the weights is only built while three quarters of the device stay free behind it."""
    lw = synth.make_layer(synth.LayerConfig(f"mem_{fmt}", 2048, 8, 2, 4096, fmt))
    print(f"[gpu] layer memory {fmt}", flush=True)
    held(moe, lw)  # (the first layer also loads the library's kernels)
    free, total = free_bytes()
    assert free > 0.9 * total
    assert held(moe, lw) <= least + codes
    if codes:
        fill = moe.DeviceBuffer(free - int(0.74 * total))  # less than three quarters free from here on
        assert held(moe, lw) <= least
        fill.free()
    monkeypatch.setenv("JX_GEMM_CODES", "0")
    assert held(moe, lw) <= least


# the same edges as the gate/up's: half-units, ragged row tiles, 64-pair parts; 24 pairs per expert and more take
# the two-tile loop throughout
@pytest.mark.parametrize("fmt,d,ff", [(F.Q4_0, 128, 32), (F.Q4_0, 384, 416), (F.Q4_0, 640, 384), (F.Q4_K, 256, 256),
                                      (F.Q4_K, 768, 1280), (F.Q5_K, 256, 256), (F.Q5_K, 768, 1280)])
def test_forms_same_bits(moe, monkeypatch, fmt, d, ff):
    """Products from the FP6 codes and from the blocks: the same integer sums, scale products and order."""
    lw = synth.make_layer(synth.LayerConfig(f"forms_{fmt}_{d}_{ff}", d, 3, 2, ff, fmt, d_ff_shared=256))
    monkeypatch.setenv("JX_GEMM_CODES", "1")
    with_codes = moe.MoELayer.from_weights(lw)
    monkeypatch.setenv("JX_GEMM_CODES", "0")
    without = moe.MoELayer.from_weights(lw)
    for n in (1, 2, 33, 48, 65, 130, 200):
        print(f"[gpu] forms {fmt} d={d} ff={ff} n={n}", flush=True)
        x = synth.make_tokens(lw.cfg, n)
        a, b = with_codes.forward(x, regime="mfma"), without.forward(x, regime="mfma")
        for u, v in zip(a, b):
            assert np.array_equal(u, v)
    with_codes.close()
    without.close()


def spoil(blocks, fmt, at):
    """Block `at` of a Q4_K / Q5_K matrix: scales d * 63 past fp16 on quants that are all zero, no minimum."""
    size = F.BLOCK[fmt][1]
    b = blocks.reshape(-1)[at * size:(at + 1) * size]
    b[:] = 0
    b[0:2] = np.frombuffer(np.float16(1100).tobytes(), np.uint8)
    b[4:12] = 0xFF  # scales 0..3 are 63, and the upper bits of 4..7
    b[12:16] = 0x0F  # their lower bits, minima 4..7 zero but for the upper bits (dmin is zero)


@pytest.mark.parametrize("fmt", [F.Q4_K, F.Q5_K])
@pytest.mark.parametrize("which", ["gate", "up", "down"])
def test_scale_past_fp16(moe, port, fmt, which):
    """A matrix with a scale past fp16 has no table for the block GEMM: prompts still give the oracle's results."""
    cfg = synth.LayerConfig(f"over_{fmt}_{which}", 512, 2, 2, 512, fmt)
    lw = synth.make_layer(cfg)
    m = np.array(getattr(lw, which))
    spoil(m, fmt, 777)
    setattr(lw, which, m)
    L = moe.MoELayer.from_weights(lw)
    for n in (3, 64, 130):
        print(f"[gpu] scale past fp16 {fmt} {which} n={n}", flush=True)
        x = synth.make_tokens(cfg, n)
        out, ids, _, _ = L.forward(x, regime="mfma")
        want, ids_o, _, _ = port.moe_forward(lw, x)
        assert np.array_equal(ids, ids_o)
        err = np.abs(out - want).max(axis=1) / np.abs(want).max(axis=1)
        # one step of h moves an output by 1 / (32 sqrt(d_ff)) of the row's largest; the fp16 down holds h in 11 bits
        assert err.max() <= max(1e-3, 1 / (32 * np.sqrt(cfg.d_ff))) and np.median(err) <= 1e-3
    L.close()


def test_fp16_down_workspace(moe):
    """The fp16 down GEMM's rows of h take 2 bytes per element, and what its kernels read is laid out by that."""
    cfg = synth.LayerConfig("ws_q6k", 256, 2, 2, 8192, F.Q4_K, down_wtype=F.Q6_K)
    lw = synth.make_layer(cfg)
    L = moe.MoELayer.from_weights(lw)
    n = 4096
    print(f"[gpu] workspace of {n} tokens, Q6_K down", flush=True)
    x = synth.make_tokens(cfg, n)
    L.forward(x[:1])
    before = free_bytes()[0]
    L.forward(x, regime="mfma")
    used = before - free_bytes()[0]
    pairs = n * cfg.top_k
    # per pair: h in Q8_0 (1 byte an element, 8 a block) and in the fp16 form (2, pieces 48 a super-block, 4 a half-unit),
    # the down's output in two parts; per token: x three times, its Q8_0 form and codes (2 bytes) and pieces
    h = cfg.d_ff * (1 + 8 / 32 + 2 + 48 / 256 + 4 / 128) + 2 * 4 * cfg.d_model
    want = pairs * h + n * cfg.d_model * (3 * 4 + 1 + 8 / 32 + 2 + 48 / 256)
    assert used <= 1.02 * want + (32 << 20), (used, want)
    L.close()


@pytest.mark.parametrize("name,n", [("qwen3moe", 600), ("dsv2lite_q50", 150), ("toy_q5k", 200)])
def test_repeats_bit_for_bit(moe, name, n):
    """The same call gives the same bits, also after calls of other sizes and values on the same workspace."""
    cfg = synth.CONFIGS[name]
    L = moe.MoELayer.from_weights(synth.make_layer(cfg))
    x = synth.make_tokens(cfg, n)
    print(f"[gpu] repeats {name} n={n}", flush=True)
    first = L.forward(x)
    for m, scale in ((n + 70, 1e4), (n - 33, 1e-4), (1, 1.0)):
        L.forward(synth.make_tokens(cfg, m, seed=m) * np.float32(scale))
        for a, b in zip(L.forward(x), first):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    L.close()
