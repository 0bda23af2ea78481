"""Tiled GEMM on problems of one K slice whose tiles of 96 columns fit one round of the CUs, and the 256-row tiles of the
GGUF formats."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import qlinear_oracle as O
from test_gpu_gguf import _dequant_oracle, _gemv, _raw_case, _repack_oracle, _t
from test_gpu_split_k import _call

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def v(dev):
    import custom_esimd_kernels_vllm
    return custom_esimd_kernels_vllm


def _hot(M, K, dt):
    ks = (5 + 29 * torch.arange(M)) % K
    hot = torch.zeros(M, K, dtype=dt)
    hot[torch.arange(M), ks] = 1.0
    return hot, ks


def _tile(M, N, K):
    """(rows, columns) of the tile on two wavefront columns for a problem of one K slice; None where K is split.  Below 256
    rows' worth of tiles the launch may prefer a taller, narrower one (test_gpu_tall_tiles.py)."""
    from mi355x_qlinear import capi
    one, split = ctypes.c_longlong(0), ctypes.c_longlong(0)
    assert capi.lib().mi_gemm_tiled_workspace(M, K, ctypes.byref(one)) == 0
    assert capi.lib().mi_gemm_tiled_workspace_split(M, N, K, ctypes.byref(split)) == 0
    if split.value != one.value:
        return None
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    rows = -(-M // 256)
    if M <= 128 or rows * -(-N // 256) * 2 <= cus:
        return 128, 96 if -(-M // 128) * -(-N // 96) <= cus else 128
    return 256, min((256, 224, 192, 160), key=lambda c: -(-(rows * -(-N // c)) // cus) * (c + 48))   # the first of equals


# up to K = 256 a problem is one slice; 95 / 96 / 97: an edge inside, at and behind a tile's last column; 1001: element-wise stores
@pytest.mark.parametrize("kind", ["int4", "fp8_channel", "fp8_block"])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [(65, 95, 128), (128, 96, 256), (129, 97, 256), (257, 1000, 128), (70, 1001, 256),
                                   (128, 24576, 128), (128, 24584, 128)])      # 256 tiles: the last of the rule; 128 columns
def test_one_hot_and_random_rows(v, dev, kind, dt, M, N, K):
    assert _tile(M, N, K) == (128, 128 if N == 24584 else 96)
    if kind == "int4":
        x, *w = O.make_int4_case(M, K, N, seed=M + K, act_dtype=dt, asym=True)
        wd = O.int4_dequant(w[0], w[1], out_dtype=dt, zp=w[2])
    elif kind == "fp8_channel":
        x, *w = O.make_fp8_pern_case(M, K, N, seed=M + K, act_dtype=dt)
        wd = O.fp8_dequant_per_channel(*w)
    else:
        x, w8, s = O.make_fp8_block_case(M, K, -(-N // 128) * 128, seed=M + K, act_dtype=dt)
        w, wd = [w8[:N].contiguous(), s], O.fp8_dequant_block(w8, s, out_dtype=dt)[:N]
    wdev = [t.to(dev) for t in w]
    out = torch.empty(M, N, dtype=dt, device=dev)
    hot, ks = _hot(M, K, dt)
    _call(v, kind, dt, hot.to(dev), wdev, out)
    assert torch.equal(out.cpu().float(), wd.to(dt)[:, ks].t().float())
    _call(v, kind, dt, x.to(dev), wdev, out)
    assert O.max_rel_err(out.cpu(), O.matmul_ref(x, wd)) < 1e-2          # the bound of the other tile shapes' tests


# at K = 512 these stay in one slice; the last four fill the chip with 256-row tiles, a last one of 8 rows
@pytest.mark.parametrize("kind", ["q4_0", "q8_0", "q5_k", "q6_k"])
@pytest.mark.parametrize("M,N,tile", [(300, 960, (128, 96)), (300, 1001, (128, 96)), (300, 9000, (128, 128)), (520, 11008, (256, 160)),
                                      (520, 14001, (256, 192)), (520, 17000, (256, 224)), (520, 20001, (256, 256))])
def test_gguf_one_hot_rows(dev, kind, M, N, tile):
    import custom_esimd_kernels_sglang as s
    K = 512
    assert _tile(M, N, K) == tile
    rep = _repack_oracle(kind, _raw_case(kind, N, K, seed=N))
    wd = torch.from_numpy(_dequant_oracle(kind, rep).astype(np.float32))
    x, ks = _hot(M, K, torch.float16)
    out = torch.empty(M, N, dtype=torch.float16, device=dev)
    _gemv(s, kind, x.to(dev), [_t(a).to(dev) for a in rep], out)
    assert torch.equal(out.cpu().float(), wd[:, ks].t())
