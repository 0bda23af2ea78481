"""Tiled GEMM below the size of 256-row tiles of 160 and more columns: every tile shape of the rule for one K slice, at
its edges, on every weight format that takes it; and the K slices on 256 x 64 and 128 x 128.  The library says which tile a problem runs on."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import qlinear_oracle as O
from test_capi_cpu import _tile
from test_gpu_gguf import _dequant_oracle, _gemv, _raw_case, _repack_oracle, _t
from test_gpu_split_k import _call
from test_gpu_tile_columns import FMT, _hot, _is_weights

pytestmark = pytest.mark.gpu


def _weights(kind, dt, M, K, N):
    if kind == "int4":
        x, *w = O.make_int4_case(M, K, N, seed=M + K, act_dtype=dt, asym=True)
        return x, w, O.int4_dequant(w[0], w[1], out_dtype=dt, zp=w[2])
    if kind == "fp8_channel":
        x, *w = O.make_fp8_pern_case(M, K, N, seed=M + K, act_dtype=dt)
        return x, w, O.fp8_dequant_per_channel(*w)
    if kind == "fp8_tensor":
        x, w8, _ = O.make_fp8_pern_case(M, K, N, seed=M + K, act_dtype=dt)
        s = torch.tensor([0.0173])
        return x, [w8, s], O.fp8_dequant_per_tensor(w8, s)
    if kind == "fp8_block":
        x, w8, s = O.make_fp8_block_case(M, K, -(-N // 128) * 128, seed=M + K, act_dtype=dt)
        return x, [w8[:N].contiguous(), s], O.fp8_dequant_block(w8, s, out_dtype=dt)[:N]
    if kind == "q4_k":
        x, raw = O.make_q4k_case(M, K, N, seed=M + K)
        rep = O.q4k_repack(raw)
        return x, [torch.from_numpy(a) for a in rep], torch.from_numpy(O.q4k_dequant(*rep)).float()
    rep = _repack_oracle(kind, _raw_case(kind, N, K, seed=N))
    wd = torch.from_numpy(_dequant_oracle(kind, rep).astype(np.float32))
    return torch.randn(M, K, generator=torch.Generator().manual_seed(N)).half(), [_t(a) for a in rep], wd


def _run(kind, dt, x, w, out):
    import custom_esimd_kernels_sglang as s
    import custom_esimd_kernels_vllm as v
    if kind == "q4_k":
        s.esimd_gemv_q4_k(x, *w, out)
    elif kind.startswith("q") and x.shape[0] > 128:
        _gemv(s, kind, x, w, out)
    elif kind.startswith("q"):                        # up to 128 rows the operator may stream the weights instead
        from mi355x_qlinear import capi
        (M, K), N, need = x.shape, out.shape[1], ctypes.c_longlong(0)
        assert capi.lib().mi_gemm_tiled_workspace_split(M, N, K, ctypes.byref(need)) == 0
        ws = torch.empty(need.value, dtype=torch.uint8, device=x.device)
        ql, qh, sc, mn = (w[0], w[1] if len(w) > 2 else None, w[min(len(w) - 1, 2)], w[3] if len(w) > 3 else None)
        capi.call("mi_gemm_gguf_tiled_ws", x, FMT[kind], capi.ptr(x), capi.ptr(ql), capi.ptr(qh), capi.ptr(sc), capi.ptr(mn),
                  capi.ptr(out), capi.ptr(ws), need.value, M, N, K)
    elif kind == "fp8_tensor":
        v.esimd_gemm_fp8_pert(x, *w, out)
    else:
        _call(v, kind, dt, x, w, out)


FORMATS = [("int4", torch.float16), ("int4", torch.bfloat16), ("fp8_block", torch.float16), ("fp8_block", torch.bfloat16)] + \
          [(k, torch.float16) for k in ("q4_k", "q4_0", "q8_0", "q5_k", "q6_k")]
UNSCALED = [("fp8_channel", torch.float16), ("fp8_channel", torch.bfloat16), ("fp8_tensor", torch.bfloat16)]      # one conversion: a line of its own
KINDS = FORMATS + UNSCALED


def _check(kind, dt, M, N, K, dev):
    x, w, wd = _weights(kind, dt, M, K, N)
    wdev = [t.to(dev) for t in w]
    out = torch.full((M, N), float("nan"), dtype=dt, device=dev)
    hot, ks = _hot(M, K, dt)
    _run(kind, dt, hot.to(dev), wdev, out)
    assert _is_weights(out.cpu(), kind, dt, w, wd, ks)                    # one 1.0 per row
    _run(kind, dt, x.to(dev), wdev, out)
    assert O.max_rel_err(out.cpu(), O.matmul_ref(x, wd)) < 1e-2           # the bound of the other tile shapes' tests


# first and last rows and columns of a tile, odd N (element-wise stores); K = 512 is one slice here
SHAPES = [(k, d, M, N, t) for k, d in FORMATS for M, N, t in (
    (129, 3009, (128, 64)), (300, 968, (128, 64)), (192, 8264, (192, 64)), (190, 8257, (192, 64)), (385, 4160, (192, 64)),
    (256, 8208, (256, 48)), (193, 8257, (256, 48)), (255, 12296, (256, 64)), (300, 8300, (128, 128)),
    (65, 16415, (128, 96)), (128, 16416, (128, 96)), (110, 16417, (128, 96)))]
SHAPES += [(k, d, M, N, t) for k, d in UNSCALED for M, N, t in (
    (129, 3009, (128, 64)), (300, 968, (128, 64)), (192, 12352, (192, 64)), (191, 12353, (192, 64)),
    (1153, 2417, (256, 48)), (1153, 2448, (256, 48)), (385, 6145, (256, 64)), (255, 12296, (256, 64)), (300, 8300, (128, 128)),
    (257, 8063, (128, 96)), (128, 16416, (128, 96)), (110, 16417, (128, 96)))]


@pytest.mark.parametrize("kind,dt,M,N,tile", SHAPES)
def test_every_tile_of_one_slice(dev, kind, dt, M, N, tile):
    assert _tile(FMT[kind], M, N, 512) == (*tile, 1)
    _check(kind, dt, M, N, 512, dev)


@pytest.mark.parametrize("kind,dt", KINDS)
@pytest.mark.parametrize("M,N,rows", [(129, 1000, 256), (256, 1001, 256), (1023, 40, 256), (300, 520, 128), (1001, 105, 128)])
def test_slices(dev, kind, dt, M, N, rows):
    tile = _tile(FMT[kind], M, N, 2048)
    assert tile[0] == rows and tile[2] > 1
    _check(kind, dt, M, N, 2048, dev)


@pytest.mark.parametrize("N", [11008, 14001, 17000, 20001])           # 256-row tiles of 160, 192, 224, 256 columns
def test_q5k_scales_on_a_two_byte_boundary(dev, N):
    """The large tiles load 128 k of a row's scales and mins at once: the same bits where the tensors start off an 8-byte boundary."""
    import custom_esimd_kernels_sglang as s
    M, K = 520, 1024
    torch.manual_seed(N)
    w = [torch.randint(0, 256, (N, K // d), dtype=torch.uint8, device=dev) for d in (2, 8)]
    sc, mn = ((torch.rand(N, K // 32, device=dev) * 0.01).half() for _ in range(2))
    off = lambda t: torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape)
    x = torch.randn(M, K, device=dev).half()
    outs = [torch.empty(M, N, dtype=torch.float16, device=dev) for _ in range(2)]
    s.esimd_gemv_q5_k(x, *w, sc, mn, outs[0])
    s.esimd_gemv_q5_k(x, *w, off(sc), off(mn), outs[1])
    assert torch.equal(*outs)
