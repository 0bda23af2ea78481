"""Tiled GEMM on tiles of 96 columns (problems of one K slice whose tiles of 96 columns fit one round of the CUs)."""
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


# up to K = 256 a problem is one slice; 95 / 96 / 97: an edge inside, at and behind a tile's last column; 1001: element-wise stores
@pytest.mark.parametrize("kind", ["int4", "fp8_channel", "fp8_block"])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [(65, 95, 128), (128, 96, 256), (129, 97, 256), (257, 1000, 128), (70, 1001, 256),
                                   (128, 24576, 128), (128, 24584, 128)])      # 256 tiles: the last of the rule; 128 columns
def test_one_hot_and_random_rows(v, dev, kind, dt, M, N, K):
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


# outputs of this size stay in one slice at K = 512
@pytest.mark.parametrize("kind", ["q4_0", "q8_0", "q5_k", "q6_k"])
@pytest.mark.parametrize("M,N", [(300, 960), (300, 1001)])
def test_gguf_one_hot_rows(dev, kind, M, N):
    import custom_esimd_kernels_sglang as s
    K = 512
    rep = _repack_oracle(kind, _raw_case(kind, N, K, seed=N))
    wd = torch.from_numpy(_dequant_oracle(kind, rep).astype(np.float32))
    x, ks = _hot(M, K, torch.float16)
    out = torch.empty(M, N, dtype=torch.float16, device=dev)
    _gemv(s, kind, x.to(dev), [_t(a).to(dev) for a in rep], out)
    assert torch.equal(out.cpu().float(), wd[:, ks].t())
