"""Tile table of a grouped GGUF chunk list: one byte per chunk in LDS, up to the longest list that the workspace allows."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 1024, 1025, 65536, 65537, 131071])     # one chunk a thread, two, 64 KiB of LDS and above, the most
def test_runs_across_threads_match_the_chunk_kernel(dev, n):
    """Runs of full chunks that straddle the threads' shares in a list of skipped chunks, against the chunk kernel on the live ones
    alone: the same weights, fp32 sums in another order (2^-11 of the result in norm, the fp16 rounding)."""
    from mi355x_qlinear import capi
    E, N, K, per = 3, 72, 128, -(-n // 1024)
    torch.manual_seed(n)
    starts = sorted({0, max(0, min(n - 7, 3 * per - 3)), max(0, min(n - 7, 200 * per - 1)), max(0, n - 7)})
    rows, live, at = [[0, 0, 0]] * n, [], 0
    for e, i0 in enumerate(starts):
        for i in range(i0, min(i0 + 6, starts[e + 1] if e + 1 < len(starts) else n)):
            rows[i] = [e % E, at, 64 if i < i0 + 5 else 17]
            live.append(rows[i])
            at += rows[i][2]
    ql = [torch.randint(0, 256, (E, N, K // 2), dtype=torch.uint8, device=dev)]
    qh = [torch.randint(0, 256, (E, N, K // 4), dtype=torch.uint8, device=dev)]
    sc = [(torch.rand(E, N, K // 16, device=dev) * 0.01).half()]
    x = torch.randn(at, K, device=dev).half()
    lists = [torch.tensor(r, dtype=torch.int32, device=dev) for r in (live, rows)]
    need = ctypes.c_longlong(0)
    assert capi.lib().mi_moe_gguf_grouped_tiled_workspace(n, K, ctypes.byref(need)) == 0
    ws = torch.empty(need.value, dtype=torch.uint8, device=dev)
    outs = [torch.full((at, N), float("nan"), dtype=torch.float16, device=dev) for _ in range(2)]
    arr = lambda t: capi.ptr_array(t) if t is not None else None
    for o, c, name, tail in ((outs[0], lists[0], "mi_moe_gguf_grouped", (0,)),
                             (outs[1], lists[1], "mi_moe_gguf_grouped_tiled_ws", (capi.ptr(ws), need.value))):
        capi.call(name, x, 6, capi.ptr(x), at, None, 1, arr(ql), arr(qh), arr(sc), None, capi.ptr(o), N, at,
                  capi.ptr(c), c.size(0), E, N, K, *tail)
    a, b = (o.float() for o in outs)
    assert float((a - b).norm() / a.norm()) < 2.0 ** -11
