"""The launches of the fused block-FP8 MoE decode step by themselves, against plain fp32 math on the dequantized weights."""
import pytest
import torch

from oracle import qlinear_oracle as O

pytestmark = pytest.mark.gpu


def _fp8(*shape, g):
    w, s = O.fp8_quantize_block(torch.randn(*shape, generator=g) * 0.1)
    return w, s, O.fp8_dequant_block(w, s).float()


# one piece per lane at most; more pieces than one batch of loads; rows that do not fill a workgroup; 1, 2 and 4 rows per wavefront
@pytest.mark.parametrize("T,k,E,H,I", [(1, 1, 2, 128, 128), (1, 8, 16, 2048, 768), (2, 8, 16, 2048, 384), (3, 3, 5, 2048, 256),
                                       (12, 4, 8, 1152, 256), (2, 10, 12, 256, 1024), (1, 64, 64, 128, 128)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_down_projections_and_their_sum(dev, dt, T, k, E, H, I):
    from mi355x_qlinear import capi
    g = torch.Generator().manual_seed(T * 100 + k + I)
    gu = torch.randn(T * k + T, 2 * I, generator=g).to(dt)
    w, ws, wd = _fp8(E, H, I, g=g)
    sw, sws, swd = _fp8(H, I, g=g)
    ids = torch.randint(0, E, (T, k), generator=g).to(torch.int32)
    ids[0, 0], ids[-1, -1] = -3, E + 5                      # held into the range
    tw, gate = torch.rand(T, k, generator=g).to(dt), torch.rand(T, generator=g)
    out = torch.full((T, H), 7.0, dtype=dt, device=dev)
    d = [t.to(dev) for t in (gu, w, ws, sw, sws, ids, tw, gate)]
    capi.call("mi_moe_down_sum_fp8_block", d[0], *[capi.ptr(t) for t in d], capi.ptr(out), T, k, E, H, I, capi.act_dtype(d[0]))
    a = gu.float()
    a = (a[:, :I] / (1 + torch.exp(-a[:, :I])) * a[:, I:]).to(dt).double()
    ref, scale = torch.zeros(T, H, dtype=torch.float64), torch.zeros(T, H, dtype=torch.float64)
    for t in range(T):
        for j in range(k):
            e = min(max(int(ids[t, j]), 0), E - 1)
            ref[t] += tw[t, j].double() * (wd[e].double() @ a[t * k + j])
            scale[t] += tw[t, j].double() * (wd[e].double().abs() @ a[t * k + j].abs())
        ref[t] += gate[t].double() * (swd.double() @ a[T * k + t])
        scale[t] += gate[t].double() * (swd.double().abs() @ a[T * k + t].abs())
    # the output's rounding, fp32 sums, and an activation that the device's expf rounds to the other neighbour
    eps = 2.0 ** -11 if dt == torch.float16 else 2.0 ** -8
    assert bool(((out.cpu().double() - ref).abs() <= eps * ref.abs() + (2.0 ** -18 + eps / 16) * scale).all())


# 80, 496 and 432 pieces past the end; 8 of them behind 65 280 bytes of activations, none behind 65 536
@pytest.mark.parametrize("T,k,E,H,I", [(1, 8, 16, 256, 768), (3, 1, 2, 128, 128), (12, 4, 8, 1152, 256), (1, 50, 51, 128, 640), (1, 63, 64, 128, 512)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_an_infinity_stays_one(dev, dt, T, k, E, H, I):
    """An activation of the shared expert's last piece overflows: its products are infinite, of the weight's sign, and no lane beyond
    the sequence's end may turn them into NaN."""
    from mi355x_qlinear import capi
    g = torch.Generator().manual_seed(T + k + I)
    gu = torch.randn(T * k + T, 2 * I, generator=g).to(dt)
    gu[-1, I - 1], gu[-1, 2 * I - 1] = torch.finfo(dt).max, 4.0          # the last token's shared expert: silu(max) x 4
    w, ws, _ = _fp8(E, H, I, g=g)
    sw, sws, swd = _fp8(H, I, g=g)
    sign = torch.where(torch.arange(H) % 2 == 0, 0x38, 0xB8).to(torch.uint8)    # 1 and -1
    sw[:, -1] = sign.view(sw.dtype) if sw.dtype != torch.uint8 else sign
    ids, tw, gate = torch.randint(0, E, (T, k), generator=g).to(torch.int32), torch.rand(T, k, generator=g).to(dt), torch.rand(T, generator=g) + 0.1
    out = torch.zeros(T, H, dtype=dt, device=dev)
    d = [t.to(dev) for t in (gu, w, ws, sw, sws, ids, tw, gate)]
    capi.call("mi_moe_down_sum_fp8_block", d[0], *[capi.ptr(t) for t in d], capi.ptr(out), T, k, E, H, I, capi.act_dtype(d[0]))
    want = torch.where(torch.arange(H) % 2 == 0, float("inf"), float("-inf")).to(dt)
    assert torch.equal(out[-1].cpu(), want) and bool(out[:-1].isfinite().all())


# x of less than a piece per lane, of whole pieces, and of a partial last one; a wavefront's rows across two experts; 2 to 16 keys per lane
@pytest.mark.parametrize("T,k,E,H,I", [(1, 1, 1, 128, 128), (1, 8, 128, 2048, 128), (3, 2, 5, 1024, 128), (2, 3, 130, 1152, 128), (4, 64, 65, 256, 128),
                                       (1, 4, 300, 2176, 128), (2, 5, 1024, 4096, 128), (16, 8, 40, 512, 256)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_routing_and_gate_up(dev, dt, T, k, E, H, I):
    from mi355x_qlinear import capi, ops
    g = torch.Generator().manual_seed(T + k + E + H)
    x, gw = (torch.randn(T, H, generator=g)).to(dt), (torch.randn(1, H, generator=g) * 0.05).to(dt)
    logits = (torch.randn(T, E, generator=g) * 2).round().to(dt)             # many ties
    few = min(E, 12)                                                         # distinct matrices: the stack repeats them
    w, ws, wd = _fp8(few, 2 * I, H, g=g)
    at = torch.arange(E) % few
    sw, sws, swd = _fp8(2 * I, H, g=g)
    d = [t.to(dev) for t in (x, logits, gw, w[at], ws[at], sw, sws)]
    gu = torch.full((T * k + T, 2 * I), 7.0, dtype=dt, device=dev)
    ids, tw, gate = torch.full((T, k), -1, dtype=torch.int32, device=dev), torch.empty(T, k, dtype=dt, device=dev), torch.empty(T, device=dev)
    capi.call("mi_moe_gate_up_topk_fp8_block", d[0], *[capi.ptr(t) for t in d], *[capi.ptr(t) for t in (gu, ids, tw, gate)], T, k, E, H, I,
              capi.act_dtype(d[0]))
    ids2, tw2, gate2 = torch.empty_like(ids), torch.empty_like(tw), torch.empty_like(gate)
    ops.esimd_moe_topk(d[1], tw2, ids2, T, gate=(d[0], d[2], gate2))
    assert torch.equal(ids, ids2) and torch.equal(tw, tw2) and torch.equal(gate, gate2)
    eps = 2.0 ** -11 if dt == torch.float16 else 2.0 ** -8
    for r in range(T * k + T):
        t, m = (r // k, wd[at[int(ids[r // k, r % k])]]) if r < T * k else (r - T * k, swd)
        ref, scale = m.double() @ x[t].double(), m.double().abs() @ x[t].double().abs()
        assert bool(((gu[r].cpu().double() - ref).abs() <= eps * ref.abs() + 2.0 ** -18 * scale).all())
    p = capi.ptr(gu)
    assert getattr(capi.lib(), "mi_moe_gate_up_topk_fp8_block")(*[p] * 11, T, k, E, 4224, I, 0, None) == -4


def test_a_hidden_size_too_long_for_one_launch(dev):
    """H above 4096: the operator selects the experts in a launch of its own."""
    import custom_esimd_kernels_vllm  # noqa: F401
    T, k, E, H, I = 2, 2, 4, 4224, 128
    g = torch.Generator().manual_seed(4)
    x, logits, gate = torch.randn(T, H, generator=g).half(), torch.randn(T, E, generator=g).half(), (torch.randn(1, H, generator=g) * 0.01).half()
    w13, s13, _ = _fp8(E, 2 * I, H, g=g)
    w2, s2, _ = _fp8(E, H, I, g=g)
    sw13, ss13, _ = _fp8(2 * I, H, g=g)
    sw2, ss2, _ = _fp8(H, I, g=g)
    ref = O.moe_forward_full(x, logits, w13, s13, sw13, ss13, w2, s2, sw2, ss2, gate, k)
    f8 = lambda t: t.view(torch.float8_e4m3fn).to(dev)
    out = torch.empty(T, H, dtype=torch.float16, device=dev)
    torch.ops.moe_ops.moe_forward_full_fp8_block(x.to(dev), logits.to(dev), out, f8(w13), s13.to(dev), f8(sw13), ss13.to(dev), f8(w2),
                                                 s2.to(dev), f8(sw2), ss2.to(dev), gate.to(dev), k, 1, E)
    assert ((out.cpu().float() - ref).abs().mean() / ref.abs().mean()).item() < 3e-3


def test_a_token_too_long_for_one_launch(dev):
    """(top_k + 1) I activations above 64 KiB: the entry refuses, and the operator runs the down rows and their sum apart."""
    import custom_esimd_kernels_vllm  # noqa: F401
    from mi355x_qlinear import capi
    T, k, E, H, I = 2, 8, 9, 128, 3712
    g = torch.Generator().manual_seed(3)
    x, logits, gate = torch.randn(T, H, generator=g).half(), torch.randn(T, E, generator=g).half(), (torch.randn(1, H, generator=g) * 0.05).half()
    w13, s13, _ = _fp8(E, 2 * I, H, g=g)
    w2, s2, _ = _fp8(E, H, I, g=g)
    sw13, ss13, _ = _fp8(2 * I, H, g=g)
    sw2, ss2, _ = _fp8(H, I, g=g)
    ref = O.moe_forward_full(x, logits, w13, s13, sw13, ss13, w2, s2, sw2, ss2, gate, k)
    f8 = lambda t: t.view(torch.float8_e4m3fn).to(dev)
    out = torch.empty(T, H, dtype=torch.float16, device=dev)
    torch.ops.moe_ops.moe_forward_full_fp8_block(x.to(dev), logits.to(dev), out, f8(w13), s13.to(dev), f8(sw13), ss13.to(dev), f8(w2),
                                                 s2.to(dev), f8(sw2), ss2.to(dev), gate.to(dev), k, 1, E)
    assert ((out.cpu().float() - ref).abs().mean() / ref.abs().mean()).item() < 3e-3
    p = capi.ptr(out)
    assert getattr(capi.lib(), "mi_moe_down_sum_fp8_block")(p, p, p, p, p, p, p, p, p, T, k, E, H, I, 0, None) == -4


@pytest.mark.parametrize("T,k,E", [(13, 8, 16), (16, 8, 128), (97, 1, 8)])     # 104, 128 and 97 pairs
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_pairs_past_the_line_are_rounded_once_between_the_projections(dev, dt, T, k, E):
    """Above 96 (token, route) pairs the operator's routed part (the shared expert's gate is 0 here) has the error of 64-bit math with the routing
    weights, SiLU(gate) x up and the output rounded, and not the 1.3 times that of gate_up rows rounded as well."""
    import custom_esimd_kernels_vllm  # noqa: F401
    H, I = 512, 256
    g = torch.Generator().manual_seed(T + E)
    x, logits, gw = torch.randn(T, H, generator=g).to(dt), (torch.randn(T, E, generator=g) * 0.4).to(dt), torch.zeros(1, H).to(dt)
    x[:, 0], gw[0, 0] = 8.0, -32.0                          # sigmoid(-256) = 0 in fp32
    w13, s13, d13 = _fp8(E, 2 * I, H, g=g)
    w2, s2, d2 = _fp8(E, H, I, g=g)
    sw13, ss13, _ = _fp8(2 * I, H, g=g)
    sw2, ss2, _ = _fp8(H, I, g=g)
    f8 = lambda t: t.view(torch.float8_e4m3fn).to(dev)
    out = torch.empty(T, H, dtype=dt, device=dev)
    torch.ops.moe_ops.moe_forward_full_fp8_block(x.to(dev), logits.to(dev), out, f8(w13), s13.to(dev), f8(sw13), ss13.to(dev), f8(w2),
                                                 s2.to(dev), f8(sw2), ss2.to(dev), gw.to(dev), k, 1, E)
    top = torch.argsort(logits.double(), dim=1, descending=True, stable=True)[:, :k]
    tw = torch.softmax(logits.double().gather(1, top), 1)
    exact, once, twice = (torch.zeros(T, H, dtype=torch.float64) for _ in range(3))
    rnd, same = (lambda v: v.to(dt).double()), (lambda v: v)
    for t in range(T):
        for j in range(k):
            gu = d13[top[t, j]].double() @ x[t].double()
            for o, r_gu, r in ((exact, same, same), (once, same, rnd), (twice, rnd, rnd)):
                a, b = r_gu(gu[:I]), r_gu(gu[I:])
                o[t] += r(tw[t, j]) * (d2[top[t, j]].double() @ r(a / (1 + torch.exp(-a)) * b))
    err = lambda o: float((o - exact).norm() / exact.norm())
    got, lo, hi = err(out.cpu().double()), err(rnd(once)), err(rnd(twice))
    assert got < (lo + hi) / 2, (got, lo, hi)
