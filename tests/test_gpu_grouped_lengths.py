"""Grouped tiled GEMM: an M-tile of 1 .. 16 live 16-row blocks runs the K loop of the smallest length that covers them."""
import ctypes
import math

import pytest
import torch

from oracle import qlinear_oracle as O
from test_gpu_moe import TOL, _grouped_ref

pytestmark = pytest.mark.gpu
COUNTS = [16 * b - b % 3 for b in range(1, 17)] + [256 + 80]          # a full tile and one of five blocks


@pytest.mark.parametrize("dt,fuse", [(torch.float16, False), (torch.bfloat16, True)])
def test_fp8_experts(dev, dt, fuse):
    import custom_esimd_kernels_vllm as v
    E, N, K, total = len(COUNTS), 384, 256, sum(COUNTS)
    g = torch.Generator().manual_seed(3)
    st = torch.zeros(E + 1, dtype=torch.int32)
    st[1:] = torch.tensor(COUNTS).cumsum(0)
    x = (torch.randn(total, K, generator=g) * 0.5).to(dt)
    w8, ws = O.fp8_quantize_block(torch.randn(E, N, K, generator=g) * 0.05)
    out = torch.full((total, N // 2 if fuse else N), float("nan"), dtype=dt, device=dev)
    v.moe_gemm_fp8_block(x.to(dev), None, None, w8.to(dev), ws.to(dev), st.to(dev), out, N, K, E, fuse)
    ref = _grouped_ref(x, O.fp8_dequant_block(w8, ws, out_dtype=dt), COUNTS)
    if fuse:
        ref = torch.nn.functional.silu(ref[:, :N // 2]) * ref[:, N // 2:]
    o = out.cpu()
    assert torch.isfinite(o.float()).all()
    for at, n in zip(st.tolist(), COUNTS):
        assert O.max_rel_err(o[at:at + n], ref[at:at + n]) < TOL      # the bound of the other shapes' tests


@pytest.mark.parametrize("K,offset", [(256, 0), (384, 0), (128, 1), (640, 3)])   # odd numbers of 128-wide pairs; scales on a 2-byte boundary
@pytest.mark.parametrize("fmt", [2, 5, 6])
def test_gguf_experts(dev, fmt, K, offset):
    """Against the chunk kernel: the same weights, fp32 sums in another order (2^-11 of the result in norm, the fp16 rounding)."""
    from mi355x_qlinear import capi
    torch.manual_seed(fmt)
    E, N, total = len(COUNTS), 264, sum(COUNTS)
    rows, at = [], 0
    for e, n in enumerate(COUNTS):
        rows += [[e, at + t, min(64, n - t)] for t in range(0, n, 64)]
        at += n
    u8 = lambda *s: torch.randint(0, 256, s, dtype=torch.uint8, device=dev)
    h = lambda *s: (torch.rand(math.prod(s) + offset, device=dev) * 0.01).half()[offset:].view(*s)
    ql, sc = [u8(E, N, K // 2)], [h(E, N, K // (16 if fmt == 6 else 32))]
    mn = [h(E, N, K // 32)] if fmt != 6 else None
    qh = [u8(E, N, K // (8 if fmt == 5 else 4))] if fmt != 2 else None
    x, chunks = torch.randn(total, K, device=dev).half(), torch.tensor(rows, dtype=torch.int32, device=dev)
    arr = lambda t: capi.ptr_array(t) if t is not None else None
    need = ctypes.c_longlong(0)
    assert capi.lib().mi_moe_gguf_grouped_tiled_workspace(len(rows), K, ctypes.byref(need)) == 0
    ws = torch.empty(need.value, dtype=torch.uint8, device=dev)
    outs = [torch.full((total, N), float("nan"), dtype=torch.float16, device=dev) for _ in range(2)]
    for o, name, tail in ((outs[0], "mi_moe_gguf_grouped", (0,)),
                          (outs[1], "mi_moe_gguf_grouped_tiled_ws", (capi.ptr(ws), need.value))):
        capi.call(name, x, fmt, capi.ptr(x), total, None, 1, arr(ql), arr(qh), arr(sc), arr(mn), capi.ptr(o), N, total,
                  capi.ptr(chunks), len(rows), E, N, K, *tail)
    at = 0
    for n in COUNTS:
        a, b = (o[at:at + n].float() for o in outs)
        assert float((a - b).norm() / a.norm()) < 2.0 ** -11
        at += n
