"""The work that this package has to do fast, as its callers issue it.

A case is a plain dict; `prepare` makes what a serving process holds before the call (activations, resident
weights, output buffers), `run` is one pass through the public entry points.  Three families:

* `linear`: one quantized linear layer, any of the resident weight formats, from one decode row over small
  batches and chunked prefill to a full prefill of 2048 rows;
* `norm_linear`: residual add + RMS norm + linear of a decode step, one fused call;
* `moe_block`, `moe_full`, `moe_gguf`: a mixture-of-experts layer (128 experts, top 8): block-FP8 experts with
  and without quantised activations, the fused op with a shared expert, and GGUF experts over sorted chunks.

Weights are made on the device from the seed: uniform integer codes for the integer formats (every code occurs),
e4m3 codes of N(0, 0.02) weights for FP8, scales of the size that quantizing such weights gives.
"""
import math
import os
import sys

import torch

_PKG = os.path.abspath("llm-scaler_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import custom_esimd_kernels_sglang as s  # noqa: E402
import custom_esimd_kernels_vllm as v  # noqa: E402
from custom_esimd_kernels_sglang import moe_grouped_gguf_xpu as mg  # noqa: E402

E, TOPK, H, I = 128, 8, 2048, 768           # the mixture-of-experts layer of the benchmark
_DT = {"f16": torch.float16, "bf16": torch.bfloat16}


def listed():
    return [
        # attention output / q projection of a 4096-wide model, one token: the smallest call of a decode step
        dict(name="int4_decode", family="linear", fmt="int4", M=1, K=4096, N=4096, dtype="f16"),
        # MLP up projection of the same decode step on per-channel FP8 weights
        dict(name="fp8_decode", family="linear", fmt="fp8_channel", M=1, K=4096, N=14336, dtype="bf16"),
        # norm + projection of a decode step in one call, the form the serving patch issues per layer
        dict(name="norm_fp8_decode", family="norm_linear", fmt="fp8_tensor", M=1, K=4096, N=14336, dtype="f16"),
        # 32 sequences decoding together
        dict(name="fp8_batch", family="linear", fmt="fp8_channel", M=32, K=4096, N=14336, dtype="bf16"),
        # 64 sequences on GGUF weights
        dict(name="q4k_batch", family="linear", fmt="q4_k", M=64, K=5120, N=5120, dtype="f16"),
        # a prefill chunk of ragged length, block-scaled FP8, the fused linear-attention input projection
        dict(name="fp8_block_chunk", family="linear", fmt="fp8_block", M=201, K=2048, N=12288, dtype="bf16"),
        # a short prompt on the format that mixed GGUF files keep their most sensitive matrices in
        dict(name="q6k_prefill", family="linear", fmt="q6_k", M=500, K=5120, N=5120, dtype="f16"),
        # a long prompt, asymmetric INT4
        dict(name="int4_prefill", family="linear", fmt="int4_zp", M=2048, K=4096, N=14336, dtype="bf16"),
        # one token through a mixture-of-experts layer with its shared expert
        dict(name="moe_decode", family="moe_full", T=1, dtype="bf16"),
        # 512 tokens, activations quantised to e4m3 on the way into both matrix products
        dict(name="moe_batch", family="moe_block", T=512, act_quant=True, dtype="bf16"),
        # a long prompt with 16-bit activations
        dict(name="moe_prefill", family="moe_block", T=4096, act_quant=False, dtype="bf16"),
        # a prompt on GGUF experts: Q4_K gate / up, SiLU, Q6_K down, weighted sum
        dict(name="moe_gguf_prefill", family="moe_gguf", T=2048, dtype="f16"),
    ]


# rows over which each weight format is used: every format decodes and prefills; no drawn case is heavier than
# the long prompts listed above
_LINEAR = {"int4": 2048, "int4_zp": 2048, "fp8_channel": 2048, "fp8_tensor": 2048, "fp8_block": 2048, "q4_k": 2048,
           "q4_0": 1024, "q8_0": 1024, "q5_k": 1024, "q6_k": 1024}
_MAX_FLOPS = 2.0 * 2048 * 4096 * 14336


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear"] * 7 + ["norm_linear", "moe_block", "moe_full", "moe_gguf"])
    if kind in ("linear", "norm_linear"):
        fmt = rng.choice(["int4", "fp8_tensor"] if kind == "norm_linear" else sorted(_LINEAR))
        gguf = fmt.startswith("q")
        K = 512 * rng.randint(2, 12)
        if fmt not in ("q5_k", "q6_k"):              # whole groups of the format, not whole tiles
            K += 256 * rng.randint(0, 1) if fmt == "q4_k" else 128 * rng.randint(0, 3)
        N = _log(rng, 1024, 14336)
        N = N | 1 if rng.random() < 0.15 else N // 8 * 8
        M = 1 if kind == "norm_linear" else _log(rng, 1, _LINEAR[fmt])
        while 2.0 * M * K * N > _MAX_FLOPS * (0.5 if gguf else 1.0):
            M //= 2
        return dict(family=kind, fmt=fmt, M=M, K=K, N=N, dtype="f16" if gguf or kind == "norm_linear" else
                    rng.choice(["f16", "bf16"]))
    if kind == "moe_full":
        return dict(family=kind, T=_log(rng, 1, 64), dtype=rng.choice(["f16", "bf16"]))
    if kind == "moe_block":
        quant = rng.random() < 0.5
        return dict(family=kind, T=_log(rng, 16, 1024 if quant else 4096), act_quant=quant, dtype=rng.choice(["f16", "bf16"]))
    return dict(family=kind, T=_log(rng, 16, 2048), dtype="f16")


# ---------------------------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _u8(g, *shape):
    return torch.randint(0, 256, shape, dtype=torch.uint8, generator=g, device="cuda")


def _uni(g, lo, hi, *shape):
    return torch.rand(*shape, generator=g, device="cuda") * (hi - lo) + lo


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _fp8(w, scale):
    return (w / scale).clamp_(-448, 448).to(torch.float8_e4m3fn)


def _block_fp8(g, *shape):
    """N(0, 0.02) weights [..., N, K] as e4m3 with one scale = absmax / 448 per 128 x 128 block."""
    n, k = shape[-2:]
    pad = -n % 128
    lead = shape[:-2]
    qs, ss = [], []
    for _ in range(math.prod(lead)):
        w = _randn(g, n, k) * 0.02
        b = torch.nn.functional.pad(w, (0, 0, 0, pad)).view((n + pad) // 128, 128, k // 128, 128)
        sc = b.abs().amax(dim=(1, 3)) / 448.0
        qs.append(_fp8(b, sc[:, None, :, None]).reshape(n + pad, k)[:n])
        ss.append(sc)
    if not lead:
        return qs[0].contiguous(), ss[0].contiguous()
    return torch.stack([q.view(torch.uint8) for q in qs]).view(torch.float8_e4m3fn).view(*shape), torch.stack(ss)


def _q4k(g, *shape):
    """Repacked Q4_K: nibbles [..., N, K/2], fp16 scale = d x 6-bit and min = dmin x 6-bit per 32 values."""
    n, k = shape[-2:]
    lead = shape[:-2]
    d, dm = _uni(g, 0.001, 0.01, *lead, n, k // 256, 1), _uni(g, 0.0, 0.005, *lead, n, k // 256, 1)
    six = [torch.randint(0, 64, (*lead, n, k // 256, 8), generator=g, device="cuda").float() for _ in range(2)]
    return (_u8(g, *lead, n, k // 2), (d * six[0]).reshape(*lead, n, k // 32).half(),
            (dm * six[1]).reshape(*lead, n, k // 32).half())


def _linear_weight(g, fmt, N, K):
    """The op's operands between the input and the output."""
    if fmt in ("int4", "int4_zp"):
        w = (_u8(g, N, K // 2), _uni(g, 0.005, 0.02, N, K // 128).half())
        return w if fmt == "int4" else w + (torch.randint(0, 16, (N, K // 128), dtype=torch.uint8, generator=g, device="cuda"),)
    if fmt == "fp8_block":
        return _block_fp8(g, N, K)
    if fmt.startswith("fp8"):
        w = _randn(g, N, K) * 0.02
        sc = (w.abs().amax(dim=1) if fmt == "fp8_channel" else w.abs().amax().reshape(1)) / 448.0
        return _fp8(w, sc[:, None]), sc.float()
    if fmt == "q4_k":
        return _q4k(g, N, K)
    if fmt == "q4_0":
        return _u8(g, N, K // 2), _uni(g, -0.02, 0.02, N, K // 32).half()
    if fmt == "q8_0":
        return _u8(g, N, K).view(torch.int8), _uni(g, -0.002, 0.002, N, K // 32).half()
    if fmt == "q5_k":
        ql, sc, mn = _q4k(g, N, K)
        return ql, _u8(g, N, K // 8), sc * 0.5, mn * 0.5
    sc = (_uni(g, 0.00002, 0.0002, N, K // 256, 1) * torch.randint(-128, 128, (N, K // 256, 16), generator=g, device="cuda"))
    return _u8(g, N, K // 2), _u8(g, N, K // 4), sc.reshape(N, K // 16).half()


def prepare(case, seed):
    g = _gen(seed)
    st = dict(case)
    dt = _DT[case["dtype"]]
    fam = case["family"]
    if fam == "linear":
        st["x"] = _randn(g, case["M"], case["K"]).to(dt)
        st["w"] = _linear_weight(g, case["fmt"], case["N"], case["K"])
        st["out"] = torch.empty(case["M"], case["N"], dtype=dt, device="cuda")
    elif fam == "norm_linear":
        K, N = case["K"], case["N"]
        st["x"], st["residual"] = _randn(g, 1, K).to(dt), _randn(g, 1, K).to(dt)
        st["norm_w"] = (_randn(g, K) * 0.1 + 1.0).to(dt)
        st["w"] = _linear_weight(g, case["fmt"], N, K)
        st["out"], st["normed"] = torch.empty(1, N, dtype=dt, device="cuda"), torch.empty(1, K, dtype=dt, device="cuda")
    else:
        T = case["T"]
        st["x"] = (_randn(g, T, H) * (0.1 if fam == "moe_gguf" else 1.0)).to(dt)
        st["logits"] = _randn(g, T, E).to(dt)
        if fam == "moe_gguf":
            _prepare_gguf(st, g, T)
        else:
            st["w13"], st["s13"] = _block_fp8(g, E, 2 * I, H)
            st["w2"], st["s2"] = _block_fp8(g, E, H, I)
            if fam == "moe_full":
                st["sw13"], st["ss13"] = _block_fp8(g, 2 * I, H)
                st["sw2"], st["ss2"] = _block_fp8(g, H, I)
                st["gate"] = (_randn(g, 1, H) * 0.05).to(dt)
            st["out"] = torch.empty(T, H, dtype=dt, device="cuda")
    return st


def _prepare_gguf(st, g, T):
    """Expert stacks, and the routing as the caller's own code leaves it: routes sorted by expert, cut into chunks of
    one expert and at most 64 rows (one row per expert and the 16-row form for a handful of tokens)."""
    gate, up = _q4k(g, E, I, H), _q4k(g, E, I, H)
    sc = _uni(g, 0.00002, 0.0002, E, H, I // 256, 1) * torch.randint(-128, 128, (E, H, I // 256, 16), generator=g, device="cuda")
    st["gate"], st["up"] = gate, up
    st["down"] = (_u8(g, E, H, I // 2), _u8(g, E, H, I // 4), sc.reshape(E, H, I // 16).half())
    weights, ids = torch.topk(torch.softmax(st["logits"].float(), dim=1), TOPK, dim=1)
    flat = ids.reshape(-1)
    order = torch.sort(flat, stable=True).indices
    st["tok_ids"] = (order // TOPK).to(torch.int32)
    st["pos"] = torch.argsort(order).to(torch.int32).reshape(T, TOPK).contiguous()
    st["w_sorted"] = (weights / weights.sum(1, keepdim=True)).reshape(-1)[order].half()
    counts = torch.bincount(flat, minlength=E).tolist()
    st["smallm"] = T <= 16
    rows, at = [], 0
    for e, n in enumerate(counts):
        step = max(n, 1) if st["smallm"] else 64
        for t0 in range(0, max(n, 1) if st["smallm"] else n, step):
            rows.append([e, at + t0, min(step, n - t0)])
        at += n
    st["chunks"] = torch.tensor(rows, dtype=torch.int32, device="cuda")
    P = T * TOPK
    st["gate_buf"] = torch.zeros(P, 2 * I, dtype=torch.float16, device="cuda")
    st["inter"] = torch.empty(P, I, dtype=torch.float16, device="cuda")
    st["routes"] = torch.zeros(P, H, dtype=torch.float16, device="cuda")
    st["out"] = torch.empty(T, H, dtype=torch.float16, device="cuda")


# ------------------------------------------------------------------------------------------------ passes
def run(st):
    fam, x, out = st["family"], st["x"], st["out"]
    if fam == "linear":
        fmt, w = st["fmt"], st["w"]
        if fmt == "int4":
            (v.esimd_gemv_int4 if st["M"] == 1 else v.esimd_gemm_int4_pgrp)(x, *w, out)
        elif fmt == "int4_zp":
            v.esimd_gemm_int4_pgrp_zp(x, *w, out)
        elif fmt == "fp8_channel":
            v.esimd_gemv_fp8_pern(x, *w, out, st["N"], st["K"])
        elif fmt == "fp8_tensor":
            (v.esimd_gemv_fp8_pert if st["M"] == 1 else v.esimd_gemm_fp8_pert)(x, *w, out)
        elif fmt == "fp8_block":
            v.esimd_gemm_fp8_blockscale(x, *w, out)
        elif fmt == "q4_k":
            s.esimd_gemv_q4_k(x, *w, out)
        elif fmt == "q4_0":
            (s.esimd_gemv_q4_0 if st["M"] == 1 else s.esimd_gemm_q4_0)(x, *w, out)
        elif fmt == "q8_0":
            (s.esimd_gemv_q8_0 if st["M"] == 1 else s.esimd_gemv_q8_0_m)(x, *w, out)
        elif fmt == "q5_k":
            s.esimd_gemv_q5_k(x, *w, out)
        else:
            (s.esimd_gemv_q6_k if st["M"] == 1 else s.esimd_gemv_q6_k_m)(x, *w, out)
        return out
    if fam == "norm_linear":
        op = v.esimd_resadd_norm_gemv_int4_pert if st["fmt"] == "int4" else v.esimd_resadd_norm_gemv_fp8_pert
        op(x, st["residual"], st["norm_w"], *st["w"], out, st["normed"], 1e-6)
        return out, st["normed"], st["residual"]
    if fam == "moe_full":
        torch.ops.moe_ops.moe_forward_full_fp8_block(x, st["logits"], out, st["w13"], st["s13"], st["sw13"], st["ss13"],
                                                     st["w2"], st["s2"], st["sw2"], st["ss2"], st["gate"], TOPK, 1, E)
        return out
    if fam == "moe_block":
        v.moe_forward_fp8_block(x, st["logits"], st["w13"], st["s13"], st["w2"], st["s2"], out, TOPK, st["act_quant"])
        return out
    P = st["T"] * TOPK
    mg.moe_up_q4k_ggemv(x, *st["gate"], *st["up"], st["gate_buf"], st["chunks"], H, I, st["tok_ids"], smallm=st["smallm"])
    v.esimd_moe_silu_mul(st["gate_buf"], st["inter"], 2 * I, I, P)
    mg.moe_down_q6k_ggemv(st["inter"], *st["down"], st["routes"], st["chunks"], I, H, smallm=st["smallm"])
    v.esimd_moe_gather(st["routes"], st["pos"], st["w_sorted"], out, H, TOPK, st["T"])
    return out, st["gate_buf"], st["routes"]


# ---------------------------------------------------------------------------------- what a pass cannot do without
_BITS = {"int4": 4 + 16 / 128, "int4_zp": 4 + 24 / 128, "fp8_channel": 8, "fp8_tensor": 8, "fp8_block": 8, "q4_k": 5, "q4_0": 4.5,
         "q8_0": 8.5, "q5_k": 6, "q6_k": 7}


def work(case):
    fam = case["family"]
    if fam in ("linear", "norm_linear"):
        M, K, N = case["M"], case["K"], case["N"]
        scales = 4 * N if case["fmt"] == "fp8_channel" else 0
        rows = 2 * M * K if fam == "linear" else 5 * 2 * K
        return {"bytes": N * K * _BITS[case["fmt"]] / 8 + scales + rows + 2 * M * N, "flops": 2.0 * M * N * K}
    T = case["T"]
    P = T * TOPK
    used = E * (1.0 - (1.0 - TOPK / E) ** T)         # experts that have a row
    bits = {"moe_gguf": (5 * 2 + 7)}.get(fam, 24)    # gate + up + down, per (expert, hidden, intermediate)
    shared = 1 if fam == "moe_full" else 0
    # the GGUF stages are separate calls: each stage's output rows are results too
    rows = 4 * T * H + 2 * T * E + (2 * P * (2 * I + H) if fam == "moe_gguf" else 0)
    return {"bytes": (used + shared) * H * I * bits / 8 + rows, "flops": 2.0 * (P + shared * T) * 3 * H * I}


# ------------------------------------------------------------- the same pass in 64 bits, from the formats' definitions
def _nibbles(b):
    return torch.stack([b & 15, b >> 4], -1).flatten(-2)                  # low nibble first


def _fields(b, bits, tile):
    """High bits: byte t of a tile of 512 values holds values p x tile + t in its fields p; tile 0: consecutive values."""
    f = torch.stack([b >> s & (1 << bits) - 1 for s in range(0, 8, bits)], -1)
    return f.flatten(-2) if not tile else f.unflatten(-2, (-1, tile)).transpose(-1, -2).flatten(-3)


def _scaled(u, s, m=None):
    s = s.double().repeat_interleave(u.shape[-1] // s.shape[-1], -1)
    return u * s if m is None else u * s - m.double().repeat_interleave(u.shape[-1] // m.shape[-1], -1)


def _blocks(q, s):
    s = s.double().repeat_interleave(128, -2)[..., :q.shape[-2], :]
    return _scaled(q.float().double(), s)


def _weight64(fmt, w, shuffled=True):
    if fmt in ("int4", "int4_zp"):
        z = w[2].double().repeat_interleave(128, -1) if fmt == "int4_zp" else 8.0
        return _scaled(_nibbles(w[0]).double() - z, w[1])
    if fmt == "fp8_block":
        return _blocks(*w)
    if fmt.startswith("fp8"):
        return w[0].float().double() * w[1].double()[:, None]
    if fmt == "q8_0":
        return _scaled(w[0].double(), w[1])
    u = _nibbles(w[0])
    if fmt == "q4_0":
        return _scaled(u.double() - 8.0, w[1])
    if fmt == "q4_k":
        return _scaled(u.double(), *w[1:])
    if fmt == "q5_k":
        return _scaled((u + 16 * _fields(w[1], 1, 64 * shuffled)).double(), *w[2:])
    return _scaled((u + 16 * _fields(w[1], 2, 128 * shuffled)).double() - 32.0, w[2])


def _quant64(a):
    """One scale = absmax / 448 per 128 values, e4m3 codes, and back."""
    b = a.unflatten(-1, (-1, 128))
    s = b.abs().amax(-1, keepdim=True).clamp(min=1e-12) / 448.0
    return ((b / s).float().to(torch.float8_e4m3fn).double() * s).flatten(-2)


def _act(g, u):
    return g * torch.sigmoid(g) * u


def _experts64(st, x, ids, w, quant):
    """sum over the routes of weight x expert(x), from block-FP8 stacks."""
    f = (lambda a: _quant64(a.to(_DT[st["dtype"]]).double())) if quant else (lambda a: a)
    xq, y = f(x), torch.zeros_like(x)
    for e in range(E):
        t, j = (ids == e).nonzero(as_tuple=True)
        if t.numel():
            gu = xq[t] @ _blocks(st["w13"][e], st["s13"][e]).t()
            y.index_add_(0, t, w[t, j, None] * (f(_act(*gu.chunk(2, 1))) @ _blocks(st["w2"][e], st["s2"][e]).t()))
    return y


def exact(case, seed):
    st, fam = prepare(case, seed), case["family"]
    x = st["x"].double()
    if fam == "linear":
        return x @ _weight64(st["fmt"], st["w"]).t()
    if fam == "norm_linear":
        a = x + st["residual"].double()
        n = a * torch.rsqrt(a.pow(2).mean(-1, keepdim=True) + 1e-6) * st["norm_w"].double()
        return n @ _weight64(st["fmt"], st["w"]).t(), n, a
    if fam == "moe_gguf":
        P, tok = st["T"] * TOPK, st["tok_ids"].long()
        gate, inter = torch.empty(P, 2 * I, dtype=torch.float64, device="cuda"), torch.empty(P, I, dtype=torch.float64, device="cuda")
        routes = torch.empty(P, H, dtype=torch.float64, device="cuda")
        for e, at, n in st["chunks"].tolist():
            r = slice(at, at + n)
            for h, k in enumerate(("gate", "up")):
                gate[r, h * I:(h + 1) * I] = x[tok[r]] @ _weight64("q4_k", [t[e] for t in st[k]]).t()
            inter[r] = _act(*gate[r].chunk(2, 1))
            routes[r] = inter[r] @ _weight64("q6_k", [t[e] for t in st["down"]], shuffled=False).t()
        pos = st["pos"].long()
        return (routes[pos] * st["w_sorted"].double()[pos][..., None]).sum(1), gate, routes
    order = torch.sort(st["logits"].double(), dim=1, descending=True, stable=True)
    ids, w = order.indices[:, :TOPK], torch.softmax(order.values[:, :TOPK], 1)
    y = _experts64(st, x, ids, w, case.get("act_quant", False))
    if fam == "moe_full":
        gu = x @ _blocks(st["sw13"], st["ss13"]).t()
        y += torch.sigmoid(x @ st["gate"].double().t()) * (_act(*gu.chunk(2, 1)) @ _blocks(st["sw2"], st["ss2"]).t())
    return y


# Four times the largest relative error (2-norm of the difference) seen against the same formula in 64 bits on the
# dequantized weights, over the listed cases and 24 drawn ones: linear fp16 4.2e-4, bf16 2.4e-3 (the output's rounding,
# and the weights' where the matrix cores take them); experts fp16 6.6e-4, bf16 4.4e-3 (the intermediate's rounding as
# well); experts with quantised activations 1.4e-2 in norm and 0.14 at most (an intermediate that rounds to the other
# neighbour in fp16 / bf16 may cross a boundary of e4m3, where a step is 2^-4).
def tolerance(case):
    bf16 = case["dtype"] == "bf16"
    if case["family"] == "moe_block" and case["act_quant"]:
        return {"rel": 0.03, "max": 0.55}
    if case["family"].startswith("moe"):
        return {"rel": 0.0176 if bf16 else 0.0027}
    return {"rel": 0.0095 if bf16 else 0.0017}
