"""The work that users of the reactor have it do, as cases that can be timed and checked.

Every case goes through a public entry of ``oct_amd.prometheus.NativeRuntime``:
the fp32 and bf16 products, the matrix-vector product, the row reductions and
RMSNorm, the two transformer layers and the binary64 transform, on
device-resident operands as a model holds them, and Oct's own ``@`` on host
matrices with its copies.

``listed()`` names the fixed cases, ``draw(rng)`` gives more of the same ranges,
``prepare`` makes what a program has in hand before the call, ``run`` is one call,
``work`` the bytes and operations it cannot do without, ``exact`` the same result
in 64 bits from plain torch or numpy, ``tolerance`` how far two correct
implementations at this precision may differ.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from oct_amd import prometheus as p

# The Gemma-2B layer (fp32): width, query heads, head width, FFN width.
GEMMA = {"hidden": 2048, "heads": 8, "head_dim": 256, "ffn": 16384}
# The Z-Image main block (bf16): width, heads of 128, FFN width, condition width.
DIT = {"hidden": 3840, "heads": 30, "ffn": 10240, "cond": 256}
OPS = {"sum": p.OP_SUM, "max": p.OP_MAX, "softmax": p.OP_SOFTMAX}

_runtime = None


def runtime() -> p.NativeRuntime:
    """The one runtime handle a program opens and keeps."""
    global _runtime
    if _runtime is None:
        _runtime = p.NativeRuntime()
        _runtime.require_hardware_gpu()
    return _runtime


def listed() -> list:
    return [
        # A large dense fp32 product, the library's headline size.
        {"name": "sgemm_4096", "kind": "sgemm", "m": 4096, "n": 4096, "k": 4096},
        # No side a multiple of a tile, two of them odd: data as it comes.
        {"name": "sgemm_ragged", "kind": "sgemm", "m": 4097, "n": 3001, "k": 513},
        # A short prompt's query projection (15 tokens of a 1536-wide model).
        {"name": "sgemm_tokens15", "kind": "sgemm", "m": 15, "n": 2048, "k": 1536},
        # One vector through a resident matrix.
        {"name": "gemv_8192x4096", "kind": "sgemm", "m": 8192, "n": 1, "k": 4096},
        # Oct's `@` on host matrices, copies both ways in the call.
        {"name": "host_matmul_1024", "kind": "host", "m": 1024, "n": 1024, "k": 1024},
        # The FFN down projection of a 1056-token image block, bf16 operands.
        {"name": "gemm_bf16_1056", "kind": "bf16", "m": 1056, "n": 3840, "k": 10240},
        # Attention-sized softmax over a large batch of rows.
        {"name": "softmax_8192x4096", "kind": "reduction", "op": "softmax", "rows": 8192, "width": 4096},
        # The smallest call: an image block's norm over its 1056 tokens.
        {"name": "rmsnorm_1056x3840", "kind": "reduction", "op": "rmsnorm", "rows": 1056, "width": 3840},
        # A whole decoder layer over a long prompt.
        {"name": "decoder_t512", "kind": "decoder", "tokens": 512, "offset": 0},
        # The same layer over a short prompt: every weight is read for few rows.
        {"name": "decoder_t15", "kind": "decoder", "tokens": 15, "offset": 0},
        # The image block at its largest: a 64x64 latent grid and 128 text tokens.
        {"name": "dit_t4224", "kind": "dit", "grid_h": 64, "grid_w": 64, "text": 128},
        # A long binary64 transform.
        {"name": "fft64_2p20", "kind": "fft64", "log2": 20},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(("sgemm", "tokens", "gemv", "host", "bf16", "reduction", "decoder", "dit", "fft64"))
    if kind == "sgemm":
        return {"kind": "sgemm", "m": _log_int(rng, 64, 4096), "n": _log_int(rng, 64, 4096),
                "k": _log_int(rng, 64, 4096)}
    if kind == "tokens":
        # 1 to 33 rows (a decode step, a short prompt) against a weight matrix.
        n, k = _log_int(rng, 512, 16384), _log_int(rng, 512, 8192)
        if rng.random() < 0.75:  # most models' widths are multiples of 128
            n, k = n // 128 * 128, k // 128 * 128
        return {"kind": "sgemm", "m": _log_int(rng, 1, 33), "n": n, "k": k}
    if kind == "gemv":
        return {"kind": "sgemm", "m": _log_int(rng, 1024, 16384), "n": 1, "k": _log_int(rng, 1024, 8192)}
    if kind == "host":
        return {"kind": "host", "m": _log_int(rng, 32, 1536), "n": _log_int(rng, 32, 1536),
                "k": _log_int(rng, 32, 1536)}
    if kind == "bf16":
        n, k = _log_int(rng, 256, 11520), _log_int(rng, 256, 10240)
        if rng.random() < 0.75:
            n, k = n // 128 * 128, k // 128 * 128
        return {"kind": "bf16", "m": _log_int(rng, 32, 4224), "n": n, "k": k}
    if kind == "reduction":
        # From a few vocabulary-sized rows to many short ones, 16 to 128 MB in all.
        total = _log_int(rng, 1 << 22, 1 << 25)
        width = _log_int(rng, 256, min(262144, total // 8))
        if rng.random() < 0.5:
            width = width // 64 * 64
        rows = total // width
        return {"kind": "reduction", "op": rng.choice(("sum", "max", "softmax", "rmsnorm")), "rows": rows,
                "width": width}
    if kind == "decoder":
        return {"kind": "decoder", "tokens": _log_int(rng, 1, 512), "offset": rng.randrange(0, 4096)}
    if kind == "dit":
        return {"kind": "dit", "grid_h": rng.randrange(16, 65), "grid_w": rng.randrange(16, 65),
                "text": rng.randrange(1, 129)}
    return {"kind": "fft64", "log2": rng.randrange(10, 21)}


# ------------------------------------------------------------------ inputs
def _generator(seed: int, device: str = "cuda") -> torch.Generator:
    return torch.Generator(device=device).manual_seed(int(seed))


def _uniform(g, shape, device="cuda"):
    return torch.rand(shape, generator=g, device=device, dtype=torch.float32).mul_(2.0).sub_(1.0)


def _normal(g, shape, mean=0.0, std=1.0):
    t = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
    return t.mul_(std).add_(mean) if (mean, std) != (0.0, 1.0) else t


def _tokens(case) -> int:
    return case["grid_h"] * case["grid_w"] + case["text"]


def _coordinates(case) -> torch.Tensor:
    """(frame, row, column): the image grid one frame after the padded text, then the text."""
    h, w, text = case["grid_h"], case["grid_w"], case["text"]
    frame = text + (32 - text % 32) % 32 + 1
    i = torch.arange(h * w)
    image = torch.stack((torch.full_like(i, frame), i // w, i % w), dim=1)
    t = torch.arange(1, text + 1)
    words = torch.stack((t, torch.zeros_like(t), torch.zeros_like(t)), dim=1)
    return torch.cat((image, words)).to(torch.float32).cuda()


def _inputs(case, seed) -> dict:
    kind = case["kind"]
    if kind == "host":
        g = _generator(seed, "cpu")
        return {"a": _uniform(g, (case["m"], case["k"]), "cpu").numpy(),
                "b": _uniform(g, (case["k"], case["n"]), "cpu").numpy()}
    g = _generator(seed)
    if kind == "sgemm":
        return {"a": _uniform(g, (case["m"], case["k"])), "b": _uniform(g, (case["k"], case["n"]))}
    if kind == "bf16":
        return {"a": _normal(g, (case["m"], case["k"])).to(torch.bfloat16),
                "b": _normal(g, (case["k"], case["n"]), 0.0, 0.02).to(torch.bfloat16)}
    if kind == "reduction":
        x = {"x": _normal(g, (case["rows"], case["width"]))}
        if case["op"] == "rmsnorm":
            x["w"] = _normal(g, (case["width"],), 1.0, 0.02)
        return x
    if kind == "decoder":
        D, H, d, F = GEMMA["hidden"], GEMMA["heads"], GEMMA["head_dim"], GEMMA["ffn"]
        return {"input": _normal(g, (case["tokens"], D)),
                "attn_norm_weight": _normal(g, (D,), 1.0, 0.02),
                "w_qkv": _normal(g, (D, (H + 2) * d), 0.0, 0.02),
                "w_o": _normal(g, (H * d, D), 0.0, 0.02),
                "ffn_norm_weight": _normal(g, (D,), 1.0, 0.02),
                "w_gate_up": _normal(g, (D, 2 * F), 0.0, 0.02),
                "w_down": _normal(g, (F, D), 0.0, 0.02)}
    if kind == "dit":
        D, F, C = DIT["hidden"], DIT["ffn"], DIT["cond"]
        bf16 = lambda shape: _normal(g, shape, 0.0, 0.02).to(torch.bfloat16)  # noqa: E731
        norm = lambda n: _normal(g, (n,), 1.0, 0.02)  # noqa: E731
        return {"input": _normal(g, (_tokens(case), D)), "coordinates": _coordinates(case),
                "condition": _normal(g, (C,)), "w_adaln": bf16((C, 4 * D)), "b_adaln": _normal(g, (4 * D,), 0.0, 0.02),
                "attn_norm1": norm(D), "attn_norm2": norm(D), "ffn_norm1": norm(D), "ffn_norm2": norm(D),
                "q_norm": norm(128), "k_norm": norm(128), "w_qkv": bf16((D, 3 * D)), "w_out": bf16((D, D)),
                "w_13": bf16((D, 2 * F)), "w_2": bf16((F, D))}
    return {"x": torch.randn((1 << case["log2"], 2), generator=g, device="cuda", dtype=torch.float64)}


def prepare(case, seed) -> dict:
    rt = runtime()
    kind = case["kind"]
    s = dict(_inputs(case, seed), case=case, rt=rt)
    new = lambda *shape: torch.empty(shape, dtype=torch.float32, device="cuda")  # noqa: E731
    if kind in ("sgemm", "bf16"):
        s["c"] = new(case["m"], case["n"])
    elif kind == "reduction":
        rows, width = case["rows"], case["width"]
        s["out"] = new(rows) if case["op"] in ("sum", "max") else new(rows, width)
        if case["op"] == "rmsnorm":
            s["inv"] = new(rows)
    elif kind == "decoder":
        s["output"] = torch.empty_like(s["input"])
        ptrs = {k: v.data_ptr() for k, v in s.items() if isinstance(v, torch.Tensor)}
        s["request"] = rt.decoder_layer_request(case["tokens"], GEMMA["hidden"], GEMMA["heads"], GEMMA["head_dim"],
                                                GEMMA["ffn"], ptrs, position_offset=case["offset"])
    elif kind == "dit":
        s["output"] = torch.empty_like(s["input"])
        ptrs = {k: v.data_ptr() for k, v in s.items() if isinstance(v, torch.Tensor)}
        s["request"] = rt.dit_block_request(_tokens(case), DIT["hidden"], DIT["heads"], DIT["ffn"], DIT["cond"], ptrs)
    elif kind == "fft64":
        s["out"] = torch.empty_like(s["x"])
    # The reactor works on its own stream: what torch still has queued comes first.
    torch.cuda.synchronize()
    return s


def run(s):
    case, rt = s["case"], s["rt"]
    kind = case["kind"]
    if kind == "sgemm":
        rt.sgemm_device(s["a"].data_ptr(), s["b"].data_ptr(), s["c"].data_ptr(), case["m"], case["n"], case["k"])
        return s["c"]
    if kind == "host":
        return rt.sgemm(case["m"], case["n"], case["k"], s["a"], s["b"])[0]
    if kind == "bf16":
        rt.gemm_bf16_device(s["a"].data_ptr(), s["b"].data_ptr(), s["c"].data_ptr(), case["m"], case["n"], case["k"])
        return s["c"]
    if kind == "reduction":
        if case["op"] == "rmsnorm":
            rt.rmsnorm_device(s["x"].data_ptr(), s["w"].data_ptr(), s["out"].data_ptr(), s["inv"].data_ptr(),
                              case["rows"], case["width"], case["width"], 1e-6)
            return {"out": s["out"], "inv": s["inv"]}
        rt.reduction_device(s["x"].data_ptr(), s["out"].data_ptr(), case["rows"], case["width"], OPS[case["op"]])
        return s["out"]
    if kind == "decoder":
        rt.decoder_layer_f32_device(s["request"])
        return s["output"]
    if kind == "dit":
        rt.dit_block_bf16_device(s["request"])
        return s["output"]
    rt.fft64_device(s["x"].data_ptr(), s["out"].data_ptr(), 1 << case["log2"])
    return s["out"]


def work(case) -> dict:
    kind = case["kind"]
    if kind in ("sgemm", "host", "bf16"):
        m, n, k = case["m"], case["n"], case["k"]
        e = 2 if kind == "bf16" else 4
        return {"bytes": e * (m * k + k * n) + 4 * m * n, "flops": 2 * m * n * k}
    if kind == "reduction":
        rows, width = case["rows"], case["width"]
        wide = case["op"] in ("softmax", "rmsnorm")
        extra = 4 * (width + rows) if case["op"] == "rmsnorm" else (0 if wide else 4 * rows)
        return {"bytes": 4 * rows * width * (2 if wide else 1) + extra, "flops": 2 * rows * width}
    if kind == "decoder":
        D, H, d, F, T = GEMMA["hidden"], GEMMA["heads"], GEMMA["head_dim"], GEMMA["ffn"], case["tokens"]
        weights = D * (H + 2) * d + H * d * D + 3 * D * F
        return {"bytes": 4 * (weights + 2 * D + 2 * T * D), "flops": 2 * T * weights + 2 * T * (T + 1) * H * d}
    if kind == "dit":
        D, F, C, T = DIT["hidden"], DIT["ffn"], DIT["cond"], _tokens(case)
        weights = 4 * D * D + 3 * D * F
        return {"bytes": 2 * (weights + 4 * C * D) + 4 * (8 * D + 2 * T * D + 3 * T),
                "flops": 2 * T * weights + 4 * T * T * D + 8 * C * D}
    n = 1 << case["log2"]
    return {"bytes": 32 * n, "flops": 5 * n * case["log2"]}


def tolerance(case):
    kind = case["kind"]
    if kind in ("sgemm", "host"):
        return {"rel": 5e-6}
    if kind == "bf16":
        return {"rel": 3e-6}
    if kind == "reduction":
        return {"rel": 5e-7}
    if kind == "decoder":
        return {"rel": 5e-6}
    if kind == "dit":
        return {"rel": 8e-3}
    return {"rel": 4e-15}


# ------------------------------------------------------- the same in 64 bits
def _rms(x, w, eps):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _exact_decoder(case, w):
    D, H, d, F, T = GEMMA["hidden"], GEMMA["heads"], GEMMA["head_dim"], GEMMA["ffn"], case["tokens"]
    f = {k: v.double() for k, v in w.items()}
    x = f["input"]
    qkv = _rms(x, f["attn_norm_weight"], 1e-6) @ f["w_qkv"]
    q, k, v = qkv[:, :H * d].reshape(T, H, d), qkv[:, H * d:(H + 1) * d].reshape(T, 1, d), qkv[:, (H + 1) * d:]
    inv = 10000.0 ** (-2.0 * torch.arange(d // 2, device="cuda", dtype=torch.float64) / d)
    ang = (case["offset"] + torch.arange(T, device="cuda", dtype=torch.float64))[:, None] * inv
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]
    turn = lambda t: torch.cat((t[..., :d // 2] * cos - t[..., d // 2:] * sin,  # noqa: E731
                                t[..., d // 2:] * cos + t[..., :d // 2] * sin), -1)
    q, k = turn(q), turn(k)[:, 0]
    later = torch.ones((T, T), dtype=torch.bool, device="cuda").triu(1)
    heads = []
    for h in range(H):
        scores = (q[:, h] @ k.t().contiguous() / math.sqrt(d)).masked_fill(later, -math.inf)
        heads.append(torch.softmax(scores, -1) @ v)
    hid = x + torch.cat(heads, -1) @ f["w_o"]
    gu = _rms(hid, f["ffn_norm_weight"], 1e-6) @ f["w_gate_up"]
    g = gu[:, :F]
    gelu = 0.5 * g * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (g + 0.044715 * g ** 3)))
    return hid + (gelu * gu[:, F:]) @ f["w_down"]


def _exact_dit(case, w):
    D, H, F, T = DIT["hidden"], DIT["heads"], DIT["ffn"], _tokens(case)
    f = {k: v.double() for k, v in w.items()}
    mod = f["condition"] @ f["w_adaln"] + f["b_adaln"]
    scale_a, gate_a, scale_m, gate_m = mod.reshape(4, D)
    x = f["input"]
    qkv = (_rms(x, f["attn_norm1"], 1e-5) * (1.0 + scale_a)) @ f["w_qkv"]
    ang = []
    for axis, width in enumerate((32, 48, 48)):
        pair = torch.arange(width // 2, device="cuda", dtype=torch.float64)
        ang.append(f["coordinates"][:, axis:axis + 1] / 256.0 ** (2.0 * pair / width))
    ang = torch.cat(ang, -1)
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]

    def turn(t, norm):
        t = _rms(t.reshape(T, H, 128), norm, 1e-5)
        even, odd = t[..., 0::2], t[..., 1::2]
        return torch.stack((even * cos - odd * sin, even * sin + odd * cos), -1).reshape(T, H, 128)

    q, k, v = turn(qkv[:, :D], f["q_norm"]), turn(qkv[:, D:2 * D], f["k_norm"]), qkv[:, 2 * D:].reshape(T, H, 128)
    heads = []
    for h in range(H):
        scores = q[:, h] @ k[:, h].t().contiguous() / math.sqrt(128.0)
        heads.append(torch.softmax(scores, -1) @ v[:, h])
    r = x + torch.tanh(gate_a) * _rms(torch.cat(heads, -1) @ f["w_out"], f["attn_norm2"], 1e-5)
    gu = (_rms(r, f["ffn_norm1"], 1e-5) * (1.0 + scale_m)) @ f["w_13"]
    hid = torch.nn.functional.silu(gu[:, :F]) * gu[:, F:]
    return r + torch.tanh(gate_m) * _rms(hid @ f["w_2"], f["ffn_norm2"], 1e-5)


def exact(case, seed):
    kind = case["kind"]
    s = _inputs(case, seed)
    if kind == "host":
        return (s["a"].astype(np.float64) @ s["b"].astype(np.float64)).reshape(-1)
    if kind in ("sgemm", "bf16"):
        return s["a"].double() @ s["b"].double()
    if kind == "reduction":
        x = s["x"].double()
        if case["op"] == "sum":
            return x.sum(-1)
        if case["op"] == "max":
            return x.amax(-1)
        if case["op"] == "softmax":
            return torch.softmax(x, -1)
        return {"out": _rms(x, s["w"].double(), 1e-6), "inv": 1.0 / torch.sqrt(x.square().mean(-1) + 1e-6)}
    if kind == "decoder":
        return _exact_decoder(case, s)
    if kind == "dit":
        return _exact_dit(case, s)
    x = s["x"].cpu().numpy().view(np.complex128).reshape(-1)
    return np.fft.fft(x).view(np.float64).reshape(-1, 2)
