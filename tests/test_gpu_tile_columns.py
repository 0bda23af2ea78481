"""Tiled GEMM on problems of one K slice: small ones, the edges of 96 columns, and the 256-row tiles of the GGUF formats.
The library says which tile a problem runs on."""
import numpy as np
import pytest
import torch

from oracle import qlinear_oracle as O
from test_capi_cpu import _tile
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


def _is_weights(got, kind, dt, w, wd, ks):
    """The result of the one-hot rows is the weights, value for value."""
    same = got == wd.to(dt)[:, ks].t()
    if kind in ("fp8_channel", "fp8_tensor") and dt == torch.float16:
        # sum x scale is rounded to fp16 at once or after an fp32 rounding, as the compiler fuses the two: either is a right answer
        exact = O.e4m3_decode(w[0])[:, ks].double().numpy() * w[1].double().reshape(-1, 1).numpy()
        same |= got == torch.from_numpy(exact.astype(np.float16)).t()
    return bool(same.all())


FMT = {"int4": 0, "fp8_channel": 1, "fp8_tensor": 1, "q4_k": 2, "q4_0": 3, "q8_0": 4, "q5_k": 5, "q6_k": 6, "fp8_block": 7}


# up to K = 256 a problem is one slice; 16415 / 16416 / 16417: an edge inside, at and behind the last of 96 columns; odd: element-wise stores
@pytest.mark.parametrize("kind", ["int4", "fp8_channel", "fp8_block"])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,columns", [
    (65, 95, 128, 64), (128, 96, 256, 64), (129, 97, 256, 64), (257, 1000, 128, 64), (70, 1001, 256, 64),
    (65, 16415, 128, 96), (128, 16416, 256, 96), (66, 16417, 128, 96),
    (128, 24576, 128, 96), (128, 24584, 128, 128)])      # 256 tiles of 96: the last of one round
def test_one_hot_and_random_rows(v, dev, kind, dt, M, N, K, columns):
    assert _tile(FMT[kind], M, N, K) == (128, columns, 1)
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
    assert _is_weights(out.cpu(), kind, dt, w, wd, ks)
    _call(v, kind, dt, x.to(dev), wdev, out)
    assert O.max_rel_err(out.cpu(), O.matmul_ref(x, wd)) < 1e-2          # the bound of the other tile shapes' tests


# at K = 512 these stay in one slice; the last four fill the chip with 256-row tiles, a last one of 8 rows
@pytest.mark.parametrize("kind", ["q4_0", "q8_0", "q5_k", "q6_k"])
@pytest.mark.parametrize("M,N,tile", [(300, 960, (128, 64)), (300, 1001, (128, 64)), (300, 9000, (128, 128)), (520, 11008, (256, 160)),
                                      (520, 14001, (256, 192)), (520, 17000, (256, 224)), (520, 20001, (256, 256))])
def test_gguf_one_hot_rows(dev, kind, M, N, tile):
    import custom_esimd_kernels_sglang as s
    K = 512
    assert _tile(FMT[kind], M, N, K) == (*tile, 1)
    rep = _repack_oracle(kind, _raw_case(kind, N, K, seed=N))
    wd = torch.from_numpy(_dequant_oracle(kind, rep).astype(np.float32))
    x, ks = _hot(M, K, torch.float16)
    out = torch.empty(M, N, dtype=torch.float16, device=dev)
    _gemv(s, kind, x.to(dev), [_t(a).to(dev) for a in rep], out)
    assert torch.equal(out.cpu().float(), wd[:, ks].t())
