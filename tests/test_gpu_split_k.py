"""Prefill on few tiles: the K range of a tile goes to several workgroups, whose fp32 sums a second launch adds."""
import ctypes

import pytest
import torch

from oracle import qlinear_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def v(dev):
    import custom_esimd_kernels_vllm
    return custom_esimd_kernels_vllm


def _call(v, kind, dt, x, w, out):
    if kind == "int4":
        v.esimd_gemm_int4_pgrp_zp(x, *w, out)
    elif kind == "fp8_channel":
        v.esimd_gemv_fp8_pern(x, *w, out, out.shape[1], x.shape[1])
    else:
        v.esimd_gemm_fp8_blockscale(x, *w, out)


@pytest.mark.parametrize("kind", ["int4", "fp8_channel", "fp8_block"])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [(65, 136, 1152),       # slices of unequal length
                                   (129, 257, 640),       # one row in the last row tile, odd N (element-wise stores)
                                   (128, 96, 4096), (200, 1000, 2048), (70, 40, 128),
                                   (1001, 105, 1024), (640, 104, 1152)])      # rows that 256 would pad alike, and 128 take
def test_one_hot_rows_and_random_rows(v, dev, kind, dt, M, N, K):
    """One 1.0 per row returns the dequantized weights value for value (each k is in exactly one slice; the other
    slices add zeros); random rows agree with the oracle."""
    if kind == "int4":
        x, *w = O.make_int4_case(M, K, N, seed=M + K, act_dtype=dt, asym=True)
        wd = O.int4_dequant(w[0], w[1], out_dtype=dt, zp=w[2])
    elif kind == "fp8_channel":
        x, *w = O.make_fp8_pern_case(M, K, N, seed=M + K, act_dtype=dt)
        wd = O.fp8_dequant_per_channel(*w)
    else:
        x, w8, s = O.make_fp8_block_case(M, K, -(-N // 128) * 128, seed=M + K, act_dtype=dt)
        w, wd = [w8[:N].contiguous(), s], O.fp8_dequant_block(w8, s, out_dtype=dt)[:N]   # the kernel's 16-bit weight
    from mi355x_qlinear import capi
    need, one = ctypes.c_longlong(0), ctypes.c_longlong(0)
    assert capi.lib().mi_gemm_tiled_workspace_split(M, N, K, ctypes.byref(need)) == 0
    assert capi.lib().mi_gemm_tiled_workspace(M, K, ctypes.byref(one)) == 0
    assert need.value > one.value or K < 640              # the shapes do split (K = 128 is a single pair of steps)
    wdev = [t.to(dev) for t in w]
    out = torch.empty(M, N, dtype=dt, device=dev)
    ks = (5 + 29 * torch.arange(M)) % K
    hot = torch.zeros(M, K, dtype=dt)
    hot[torch.arange(M), ks] = 1.0
    _call(v, kind, dt, hot.to(dev), wdev, out)
    assert torch.equal(out.cpu().float(), wd.to(dt)[:, ks].t().float())
    _call(v, kind, dt, x.to(dev), wdev, out)
    assert O.max_rel_err(out.cpu(), O.matmul_ref(x, wd)) < 1e-2


def test_workspace_without_room_for_the_sums_runs_in_one_piece(v, dev):
    """The C entry accepts the smaller workspace of mi_gemm_tiled_workspace, as before, and differs from the split
    launch by the order of fp32 sums only: at most one rounding step of the output type where a sum sits on the border."""
    from mi355x_qlinear import capi
    M, N, K = 100, 264, 2048
    x, w8, s = O.make_fp8_pern_case(M, K, N, seed=3, act_dtype=torch.float16)
    xd, wd, sd = x.to(dev), w8.to(dev), s.to(dev)
    outs = []
    for name, args in (("mi_gemm_tiled_workspace", (M, K)), ("mi_gemm_tiled_workspace_split", (M, N, K))):
        need = ctypes.c_longlong(0)
        assert getattr(capi.lib(), name)(*args, ctypes.byref(need)) == 0
        ws = torch.empty(need.value, dtype=torch.uint8, device=dev)
        out = torch.empty(M, N, dtype=torch.float16, device=dev)
        capi.call("mi_gemm_fp8_tiled_ws", xd, capi.ptr(xd), capi.ptr(wd), capi.ptr(sd), 0, 0, capi.ptr(out), capi.ptr(ws),
                  need.value, M, N, K, 0)
        outs.append(out.cpu().float())
    ref = O.matmul_ref(x, O.fp8_dequant_per_channel(w8, s))
    assert all(O.max_rel_err(o, ref) < 1e-2 for o in outs)
    assert float(((outs[0] - outs[1]).norm() / outs[0].norm())) < 2.0 ** -11      # rms of one fp16 rounding each: 2^-12.8


@pytest.mark.parametrize("kind", ["int4", "fp8"])
def test_a_shorter_prompt_captured_after_the_longest(v, dev, kind):
    """The C entries that keep their own scratch: the K slices' sums can make a problem of few tiles need more than a
    larger one.  A stream warmed up on the larger (one piece, exactly the re-tiled activations) captures the smaller in
    one piece; with a workspace for the sums the result differs by their order only."""
    from mi355x_qlinear import capi
    M, K, N, wide = 2048, 8192, 512, 4608                 # 4608: 256-row tiles, one piece; 512: split
    sizes = []
    for n in (wide, N):
        need = ctypes.c_longlong(0)
        assert capi.lib().mi_gemm_tiled_workspace_split(M, n, K, ctypes.byref(need)) == 0
        sizes.append(need.value)
    assert sizes[1] > sizes[0] == M * K * 2 == 1 << 25      # the scratch grows in powers of two
    g = torch.Generator(device=dev).manual_seed(1)
    x = torch.randn(M, K, generator=g, device=dev).half()
    if kind == "int4":
        w = torch.randint(0, 256, (wide, K // 2), dtype=torch.uint8, generator=g, device=dev)
        s = (torch.rand(wide, K // 128, generator=g, device=dev) * 0.01).half()
        tail = lambda n: ("mi_gemm_int4", [capi.ptr(s), None], [M, n, K, 0])
        ws_tail = ("mi_gemm_int4_ws", [capi.ptr(s), None])
    else:
        w = torch.randn(wide, K, generator=g, device=dev).to(torch.float8_e4m3fn)
        s = torch.rand(wide, generator=g, device=dev) * 0.01
        tail = lambda n: ("mi_gemm_fp8_pern", [capi.ptr(s)], [M, n, K, 0, 0])
        ws_tail = ("mi_gemm_fp8_tiled_ws", [capi.ptr(s), 0, 0])
    out = torch.zeros(M, wide, dtype=torch.float16, device=dev)

    def call(n):
        name, operands, sizes_ = tail(n)
        capi.call(name, x, capi.ptr(x), capi.ptr(w), *operands, capi.ptr(out), *sizes_)

    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        call(wide)
        stream.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            call(N)
    ws, want = torch.empty(sizes[1], dtype=torch.uint8, device=dev), torch.empty(M, N, dtype=torch.float16, device=dev)
    capi.call(ws_tail[0], x, capi.ptr(x), capi.ptr(w), *ws_tail[1], capi.ptr(want), capi.ptr(ws), sizes[1], M, N, K, 0)
    for _ in range(3):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        got = out.view(-1)[:M * N].view(M, N).float()
        assert float((got - want.float()).norm() / want.float().norm()) < 2.0 ** -11
