"""Experts with 250 to 312 rows on average: rows at the tile's edges (16-row blocks, wavefronts of 4 and fewer of them, a second tile of one
row) and columns that leave a partial last tile, against fp32 math; tiles of 256 rows whatever the average."""
import ctypes

import pytest
import torch

from oracle import qlinear_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts", [[320, 257, 321, 150], [304, 305, 0, 391], [250, 250, 250, 250], [312, 312, 312, 312], [1, 640, 272, 335]])
@pytest.mark.parametrize("H,I", [(256, 128), (640, 384)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_experts_at_a_tiles_edge(dev, dt, H, I, counts):
    import custom_esimd_kernels_vllm as v
    E, T = len(counts), sum(counts)
    assert 250 * E <= T <= 312 * E
    g = torch.Generator().manual_seed(T + H + counts[0])
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(T, generator=g)]
    logits = torch.zeros(T, E).scatter_(1, ids[:, None], 8.0).to(dt)        # top 1: the weight is 1
    x = torch.randn(T, H, generator=g).to(dt)
    w13, s13 = O.fp8_quantize_block(torch.randn(E, 2 * I, H, generator=g) * 0.05)
    w2, s2 = O.fp8_quantize_block(torch.randn(E, H, I, generator=g) * 0.05)
    out = torch.empty(T, H, dtype=dt, device=dev)
    f8 = lambda t: t.view(torch.float8_e4m3fn).to(dev)
    v.moe_forward_fp8_block(x.to(dev), logits.to(dev), f8(w13), s13.to(dev), f8(w2), s2.to(dev), out, 1, False)
    ref = torch.empty(T, H)
    d13, d2 = O.fp8_dequant_block(w13, s13).float(), O.fp8_dequant_block(w2, s2).float()
    for e in range(E):
        gu = x[ids == e].float() @ d13[e].t()
        ref[ids == e] = (torch.nn.functional.silu(gu[:, :I]) * gu[:, I:]) @ d2[e].t()
    err = (out.cpu().float() - ref).norm(dim=1) / ref.norm(dim=1)           # per row: a wrong or missing row shows
    # the weights', the intermediate's and the output's roundings, each 2^-9 (bf16) / 2^-12 (fp16) in norm, four times that
    assert err.max().item() < (0.0176 if dt == torch.bfloat16 else 0.0027)


@pytest.mark.parametrize("counts", [[250], [257, 250], [300] * 3, [321, 250, 256], [700, 1, 90]])     # 250 to 300 rows on average, and 264
def test_tiles_have_256_rows(dev, counts):
    """The table of M-tiles that a launch leaves in its workspace (their number stands in the last 256 bytes): taller tiles in a range
    of averages were slower on most sizes and counts."""
    from mi355x_qlinear import capi
    E, T, H, I = len(counts), sum(counts), 256, 128
    start = torch.tensor([0] + counts).cumsum(0).to(torch.int32).to(dev)
    x, y = torch.randn(T, H, device=dev).half(), torch.empty(T, I, dtype=torch.float16, device=dev)
    w, s = torch.zeros(E, I, H, dtype=torch.uint8, device=dev), torch.ones(E, I // 128, H // 128, device=dev)
    need = ctypes.c_longlong(0)
    assert capi.lib().mi_moe_gemm_fp8_tiled_workspace(T, E, H, ctypes.byref(need)) == 0
    ws = torch.zeros(need.value, dtype=torch.uint8, device=dev)
    capi.call("mi_moe_gemm_fp8_tiled_ws", x, capi.ptr(x), None, 1, capi.ptr(w), capi.ptr(s), 0, capi.ptr(start), capi.ptr(y), None, None,
              T, T, E, I, H, 0, 0, capi.ptr(ws), need.value)
    assert int(ws[-256:].view(torch.int32)[0]) == sum(-(-c // 256) for c in counts)
