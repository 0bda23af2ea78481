"""Tiled GEMM: a row's scales of 128 k are fetched in one piece (4 to 16 bytes) into a table in LDS.  The operators take them at
any address that their type allows, so operands one element off every wider alignment give the bits of aligned ones; the
row lengths leave one table, an odd number of them and more than both places hold."""
import pytest
import torch

from oracle import qlinear_oracle as O
from test_gpu_gguf import _gemv, _raw_case, _repack_oracle, _t

pytestmark = pytest.mark.gpu


def _off(t):
    """The same values one element behind an aligned address."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    view = buf[1:].view(t.shape)
    view.copy_(t)
    return view


@pytest.mark.parametrize("M,N", [(70, 97), (300, 960), (520, 11008)])      # in slices / narrow tiles, and 256 rows x 160 columns
@pytest.mark.parametrize("kind,K", [("q4_0", 128), ("q4_0", 384), ("q8_0", 128), ("q8_0", 640), ("q4_k", 256), ("q4_k", 768),
                                    ("q5_k", 512), ("q6_k", 512), ("q6_k", 1536)])
def test_gguf_scales_off_alignment(dev, kind, K, M, N):
    import custom_esimd_kernels_sglang as s
    if kind == "q4_k":
        ops = [_t(a).to(dev) for a in O.q4k_repack(O.make_q4k_case(1, K, N, seed=N + K)[1])]
    else:
        ops = [_t(a).to(dev) for a in _repack_oracle(kind, _raw_case(kind, N, K, seed=N + K))]
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(K)).half().to(dev)
    outs = []
    for move in (lambda t: t, _off):
        out = torch.empty(M, N, dtype=torch.float16, device=dev)
        _gemv(s, kind, x, [move(t) if t.dtype == torch.float16 else t for t in ops], out)
        outs.append(out)
    assert outs[0].isfinite().all() and torch.equal(*outs)


@pytest.mark.parametrize("M,N", [(70, 97), (300, 960), (520, 11008)])
@pytest.mark.parametrize("K", [128, 384, 1024])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_int4_and_block_fp8_scales_off_alignment(dev, dt, K, M, N):
    import custom_esimd_kernels_vllm as v
    g = torch.Generator().manual_seed(M + K)
    x = torch.randn(M, K, generator=g).to(dt).to(dev)
    nib = torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, generator=g).to(dev)
    sc, zp = (torch.rand(N, K // 128, generator=g) * 0.02).half().to(dev), torch.randint(0, 16, (N, K // 128), dtype=torch.uint8, generator=g).to(dev)
    w8 = (torch.randn(N, K, generator=g)).to(torch.float8_e4m3fn).to(dev)
    bs = torch.rand(-(-N // 128), K // 128, generator=g).to(dev)
    outs = []
    for move in (lambda t: t, _off):
        a, b = (torch.empty(M, N, dtype=dt, device=dev) for _ in range(2))
        v.esimd_gemm_int4_pgrp_zp(x, nib, move(sc), move(zp), a)
        v.esimd_gemm_fp8_blockscale(x, w8, move(bs), b)
        outs.append((a, b))
    assert all(torch.equal(p, q) and p.isfinite().all() for p, q in zip(*outs))
