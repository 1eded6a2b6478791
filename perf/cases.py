"""What a user of this framework has it do, as cases that a timing program can run.

The framework's main path is one MoE layer resident on the GPU (`MoELayer.forward_device`, or
`jx_moe_forward` of the C interface where the routing is wanted too): a few tokens at a time while
text is generated, tens of tokens where requests are batched, hundreds to thousands of tokens of
prompt.  Beside it stands the attention projection of one token (`jx_matmul_qkv_quant_f32_dev`).
Layer shapes are those of `jxai_amd.synth.CONFIGS`; weights and tokens are drawn on the GPU from the
seed in the distributions that `jxai_amd.synth` gives them.
"""
import ctypes as C
import math

import torch

from jxai_amd import formats as F
from jxai_amd import moe, synth
from jxai_amd._lib import JX_FWD_ASYNC, JX_FWD_DEVICE_PTRS, JX_FWD_RESIDUAL, check, lib


def _layer(name, config, tokens, residual=False, routing=False):
    return {"name": name, "path": "layer", "config": config, "tokens": tokens, "residual": residual,
            "routing": routing}


def listed():
    return [
        # one token of a tiny model: nothing but launches and hand-overs between them
        _layer("toy-1", "toy", 1),
        # the attention projection beside the layer: one token through q, k and v
        {"name": "qkv-4096", "path": "qkv", "config": "Q4_K", "cols": 4096, "q_rows": 4096, "kv_rows": 1024},
        # generating text for one user: many small experts with a shared one; two large experts
        _layer("qwen15-1", "qwen15moe", 1),
        _layer("mixtral-1", "mixtral", 1),
        # a handful of users, or the draft tokens of one, through a Q4_K_M file's layer
        _layer("mixtral-q6k-5", "mixtral_q6k", 5),
        # batched generation: an odd batch with the steps either side of the block and its routing kept for
        # telemetry; two usual batch sizes on layers with a shared expert
        _layer("qwen3-37-residual", "qwen3moe", 37, residual=True, routing=True),
        _layer("dsv2lite-32", "dsv2lite", 32),
        _layer("qwen15-64", "qwen15moe", 64),
        # prompts: a short and a long one over large experts, many small Q8_0 experts under skewed routing,
        # and a ragged length through a Q4_K_M file's small experts
        _layer("mixtral-512", "mixtral", 512),
        _layer("mixtral-2048", "mixtral", 2048),
        _layer("qwen3-2048", "qwen3moe", 2048),
        _layer("dsv2lite-q50-1555", "dsv2lite_q50", 1555),
    ]


def draw(rng):
    if rng.random() < 0.1:
        cols = 256 * rng.randint(8, 32)
        return {"path": "qkv", "config": rng.choice(["Q4_0", "Q8_0", "Q4_K", "Q6_K"]), "cols": cols,
                "q_rows": 32 * rng.randint(32, 160), "kv_rows": 32 * rng.randint(8, 64)}
    config = rng.choice(["toy", "qwen15moe", "mixtral", "mixtral_q6k", "qwen3moe", "dsv2lite", "dsv2lite_q50"])
    most = {"mixtral": 1900, "mixtral_q6k": 1024}.get(config, 2048)
    tokens = min(most, int(round(math.exp(rng.uniform(0.0, math.log(most + 0.5))))))
    case = _layer("", config, tokens, residual=rng.random() < 0.25, routing=rng.random() < 0.25)
    del case["name"]
    return case


# ------------------------------------------------------------------------------------------ inputs


def _rng(seed, name):
    return torch.Generator(device="cuda").manual_seed(synth.sub_seed("perf", name, seed) >> 1)


def _matrix(g, t, rows, cols):
    """A [rows][cols] matrix in GGML block layout on the GPU, [blocks][bytes], as synth.quant_matrix draws it."""
    blk, size = F.BLOCK[t]
    n = rows * ((cols + blk - 1) // blk)
    raw = torch.randint(0, 256, (n, size), dtype=torch.uint8, device="cuda", generator=g)

    def scales(at, k):
        v = (0.005 + 0.015 * torch.rand(n, device="cuda", generator=g)) * k
        raw[:, at:at + 2] = v.half().view(torch.uint8).reshape(n, 2)

    if t == F.Q8_0:
        raw[:, 2:] = torch.randint(-127, 128, (n, 32), dtype=torch.int8, device="cuda", generator=g).view(torch.uint8)
    scales(208 if t == F.Q6_K else 0, {F.Q6_K: 1 / 16, F.Q5_0: 0.5}.get(t, 1.0))
    if t == F.Q4_K:
        scales(2, 1.0)
    return raw


def _normal(g, shape, std=1.0, mean=0.0):
    return torch.randn(shape, device="cuda", generator=g) * std + mean


def _inputs(case, seed):
    """Every input of a case, on the GPU (weights as [blocks][bytes])."""
    if case["path"] == "qkv":
        t = F.BY_NAME[case["config"]]
        rows = {"q": case["q_rows"], "k": case["kv_rows"], "v": case["kv_rows"]}
        w = {m: _matrix(_rng(seed, m), t, r, case["cols"]) for m, r in rows.items()}
        return dict(t=t, rows=rows, w=w, x=_normal(_rng(seed, "x"), (case["cols"],)))
    cfg = synth.CONFIGS[case["config"]]
    d, E, Fd, Fs = cfg.d_model, cfg.n_experts, cfg.d_ff, cfg.d_ff_shared
    i = {"cfg": cfg, "router": _normal(_rng(seed, "router"), (E, d), 0.02), "bias": None,
         "gate": _matrix(_rng(seed, "gate"), cfg.wtype, E * Fd, d),
         "up": _matrix(_rng(seed, "up"), cfg.wtype, E * Fd, d),
         "down": _matrix(_rng(seed, "down"), cfg.down_t, E * d, Fd),
         "x": _normal(_rng(seed, "x"), (case["tokens"], d)), "norm": None, "sh_inp": None}
    if cfg.zipf_gamma > 0:
        i["bias"] = torch.from_numpy(synth.zipf_bias(cfg, seed)).cuda()
    if case["residual"]:
        i["norm"] = _normal(_rng(seed, "norm"), (d,), 0.1, 1.0)
    if Fs:
        i["sh_gate"] = _matrix(_rng(seed, "sh_gate"), cfg.wtype, Fs, d)
        i["sh_up"] = _matrix(_rng(seed, "sh_up"), cfg.wtype, Fs, d)
        i["sh_down"] = _matrix(_rng(seed, "sh_down"), cfg.sh_down_t, d, Fs)
        if cfg.shared_gate:
            i["sh_inp"] = _normal(_rng(seed, "sh_inp"), (d,), 0.02)
    return i


class _Buffer:
    """A tensor handed to the library as a device buffer."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = C.c_void_p(tensor.data_ptr())


_stream = []


def _the_stream():
    """The one stream that the program runs its layers on."""
    if not _stream:
        _stream.append(torch.cuda.Stream())
    return _stream[0].cuda_stream


def _host(a):
    return None if a is None else a.cpu().numpy()


def prepare(case, seed):
    moe.init(0)
    i = _inputs(case, seed)
    if case["path"] == "qkv":
        s = {"W": [moe.QMatrix(i["t"], _host(i["w"][m]).reshape(-1), r, case["cols"]) for m, r in i["rows"].items()],
             "x": _Buffer(i["x"]),
             "out": [_Buffer(torch.empty(r, device="cuda")) for r in i["rows"].values()]}
    else:
        cfg = i["cfg"]
        more = {}
        if cfg.has_shared:
            more = dict(d_ff_shared=cfg.d_ff_shared, sh_gate_type=cfg.wtype, sh_up_type=cfg.wtype,
                        sh_down_type=cfg.sh_down_t, sh_gate=_host(i["sh_gate"]), sh_up=_host(i["sh_up"]),
                        sh_down=_host(i["sh_down"]), sh_gate_inp=_host(i["sh_inp"]))
        n, k, E = case["tokens"], cfg.top_k, cfg.n_experts
        s = {"layer": moe.MoELayer(n_experts=E, top_k=k, d_model=cfg.d_model, d_ff=cfg.d_ff, gate_type=cfg.wtype,
                                   up_type=cfg.wtype, down_type=cfg.down_t, router=_host(i["router"]),
                                   router_bias=_host(i["bias"]), gate_exps=_host(i["gate"]), up_exps=_host(i["up"]),
                                   down_exps=_host(i["down"]), ffn_norm=_host(i["norm"]), activation=cfg.act, **more),
             "x": _Buffer(i["x"]), "out": _Buffer(torch.empty_like(i["x"])), "n": n,
             "flags": JX_FWD_RESIDUAL if case["residual"] else 0}
        if case["routing"]:
            s["routing"] = [_Buffer(torch.empty(n, k, dtype=torch.int32, device="cuda")),
                            _Buffer(torch.empty(n, k, device="cuda")),
                            _Buffer(torch.empty(E, dtype=torch.int32, device="cuda"))]
    s["stream"] = _the_stream()
    return s


def run(s):
    if "W" in s:
        check(lib().jx_matmul_qkv_quant_f32_dev(*[w.handle for w in s["W"]], s["x"].ptr, *[b.ptr for b in s["out"]],
                                                C.c_void_p(s["stream"])), "jx_matmul_qkv_quant_f32_dev")
        return [b.tensor for b in s["out"]]
    if "routing" not in s:
        s["layer"].forward_device(s["x"], s["n"], s["out"], sync=False, stream=s["stream"], extra_flags=s["flags"])
        return s["out"].tensor
    ids, weights, counts = s["routing"]
    check(lib().jx_moe_forward(s["layer"].handle, s["x"].ptr, s["n"], s["out"].ptr, ids.ptr, weights.ptr, counts.ptr,
                               C.c_void_p(s["stream"]), JX_FWD_DEVICE_PTRS | JX_FWD_ASYNC | s["flags"]),
          "jx_moe_forward")
    return {"out": s["out"].tensor, "ids": ids.tensor, "weights": weights.tensor, "counts": counts.tensor}


# ------------------------------------------------------------------------------------------ what a pass needs


def work(case):
    if case["path"] == "qkv":
        t, rows, cols = F.BY_NAME[case["config"]], case["q_rows"] + 2 * case["kv_rows"], case["cols"]
        return {"bytes": F.matrix_bytes(t, rows, cols) + 4 * (cols + rows), "flops": 2 * rows * cols}
    cfg = synth.CONFIGS[case["config"]]
    n, d, E, k = case["tokens"], cfg.d_model, cfg.n_experts, cfg.top_k
    # experts that at least one token is expected to choose
    share = [(e + 1) ** (-1.1 * cfg.zipf_gamma) for e in range(E)]
    distinct = sum(1 - (1 - min(1.0, k * s / sum(share))) ** n for s in share)
    nbytes = distinct * synth.expert_bytes(cfg) + synth.shared_bytes(cfg) + 4 * E * d + 8 * n * d
    flops = 2 * n * 3 * d * (k * cfg.d_ff + cfg.d_ff_shared) + 2 * n * E * d
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # Four times what differs from 64 bits at most.  The projection is 32-bit sums of exact block products
    # (1.7e-7).  A layer quantizes the activations between its two products again, where a last-bit
    # difference in a sum can move a value by one of 127 steps (5e-5 of a single token's output), and the
    # prompt form of the second product holds its input in 12 bits (2.7e-4).
    return {"rel": 7e-7} if case["path"] == "qkv" else {"rel": 1e-3}


# ------------------------------------------------------------------------------------------ in 64 bits


def _weights64(raw, t, rows, cols):
    """The matrix of GGML blocks in 64 bits (the block formats as the GGUF files hold them)."""
    n = raw.shape[0]

    def half(at):
        return raw[:, at:at + 2].contiguous().view(torch.float16).double().reshape(n, 1)

    def nibbles(b):
        return torch.cat([b & 15, b >> 4], -1)

    if t == F.Q4_0:
        w = (nibbles(raw[:, 2:18]).double() - 8) * half(0)
    elif t == F.Q5_0:
        high = (raw[:, 2:6, None] >> torch.arange(8, device=raw.device, dtype=torch.uint8)) & 1
        w = ((nibbles(raw[:, 6:22]) | high.reshape(n, 32) << 4).double() - 16) * half(0)
    elif t == F.Q8_0:
        w = raw[:, 2:].contiguous().view(torch.int8).double() * half(0)
    elif t == F.Q4_K:
        s = raw[:, 4:16]
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | (s[:, 0:4] >> 6) << 4], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | (s[:, 4:8] >> 6) << 4], 1).double()
        q = nibbles(raw[:, 16:144].reshape(n, 4, 32)).reshape(n, 8, 32).double()
        w = q * (half(0) * sc)[:, :, None] - (half(2) * mn)[:, :, None]
    else:  # Q6_K
        ql, qh = nibbles_6k(raw[:, 0:128].reshape(n, 2, 64)), raw[:, 128:192].reshape(n, 2, 1, 32)
        high = (qh >> torch.tensor([0, 2, 4, 6], device=raw.device, dtype=torch.uint8)[:, None]) & 3
        q = (ql | high << 4).double().reshape(n, 16, 16) - 32
        w = q * (half(208) * raw[:, 192:208].contiguous().view(torch.int8).double())[:, :, None]
    return w.reshape(rows, -1)[:, :cols]


def nibbles_6k(b):
    """[n][2][64] low-bit bytes of Q6_K as [n][2][4 groups of 32]."""
    lo, hi = b & 15, b >> 4
    return torch.stack([lo[..., :32], lo[..., 32:], hi[..., :32], hi[..., 32:]], 2)


def _q8(x):
    """Activations as the path's definition quantizes them (blocks of 32 in 8 bits, the scale cut to fp16)."""
    b = x.float().reshape(-1, 32)
    d = b.abs().amax(1, keepdim=True) / 127
    h = d.half()
    h = torch.where(h.float() > d, (h.view(torch.int16) - 1).view(torch.float16), h)
    q = torch.where(h != 0, b * (1 / d), torch.zeros_like(b))
    q = (q.double().abs() + 0.5).floor().clamp(max=127) * q.sign().double()
    return (q * h.double()).reshape(x.shape)


def _input64(x, t, cols):
    return _q8(x) if F.supports_q8_activation(t, cols) else x.float().double()


def _ffn64(x, gate, up, down, types, d, ff):
    xin = _input64(x, types[0], d)
    g = xin @ _weights64(gate, types[0], ff, d).T
    h = g * torch.sigmoid(g) * (xin @ _weights64(up, types[0], ff, d).T)
    return _input64(h, types[1], ff) @ _weights64(down, types[1], d, ff).T


def exact(case, seed):
    i = _inputs(case, seed)
    if case["path"] == "qkv":
        x = _input64(i["x"], i["t"], case["cols"])
        return [_weights64(i["w"][m], i["t"], r, case["cols"]) @ x for m, r in i["rows"].items()]
    cfg = i["cfg"]
    d, E, k, ff = cfg.d_model, cfg.n_experts, cfg.top_k, cfg.d_ff
    x = i["x"].double()
    if case["residual"]:
        x = x / (x.square().mean(1, keepdim=True) + cfg.rms_eps).sqrt() * i["norm"].double()
    logits = x @ i["router"].double().T
    if i["bias"] is not None:
        logits = logits + i["bias"].double()
    top, ids = logits.topk(k, 1)
    weights = torch.softmax(top, 1)
    out = i["x"].double() if case["residual"] else torch.zeros_like(x)
    for e in range(E):
        tok, slot = (ids == e).nonzero(as_tuple=True)
        if tok.numel():
            one = [m.view(E, -1, m.shape[1])[e] for m in (i["gate"], i["up"], i["down"])]
            y = _ffn64(x[tok], *one, (cfg.wtype, cfg.down_t), d, ff)
            out.index_add_(0, tok, y * weights[tok, slot][:, None])
    if cfg.has_shared:
        y = _ffn64(x, i["sh_gate"], i["sh_up"], i["sh_down"], (cfg.wtype, cfg.sh_down_t), d, cfg.d_ff_shared)
        out += y if i["sh_inp"] is None else y * torch.sigmoid(x @ i["sh_inp"].double())[:, None]
    if not case["routing"]:
        return out
    return {"out": out, "ids": None, "weights": weights, "counts": None}
