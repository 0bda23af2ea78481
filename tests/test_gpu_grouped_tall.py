"""Experts with 250 to 312 rows on average run on tiles of 320 rows x 192 columns: rows at the tile's edges (16-row blocks, wavefronts
of 5, 4 and fewer of them, a second tile of one row) and columns that leave a partial last tile, against fp32 math."""
import pytest
import torch

from oracle import qlinear_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts", [[320, 257, 321, 150], [304, 305, 0, 391], [250, 250, 250, 250], [312, 312, 312, 312], [1, 640, 272, 335]])
@pytest.mark.parametrize("H,I", [(256, 128), (640, 384)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_tall_tiles(dev, dt, H, I, counts):
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
