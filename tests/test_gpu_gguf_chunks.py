"""Grouped GGUF MoE GEMMs on merged chunks (the tiled route of prompts) against the chunk kernel, on chunk lists
that do and do not merge."""
import ctypes

import pytest
import torch

from oracle import qlinear_oracle as O
from test_gpu_gguf import TOL, _down_stack, _q4k_expert_stacks

pytestmark = pytest.mark.gpu


def _lists(total, E):
    g = torch.Generator().manual_seed(total)
    merged, at = [], 0
    for e in range(E):                                  # an expert's rows in full chunks and a remainder; some experts without rows
        n = 0 if e % 5 == 4 else int(torch.randint(1, 2 * total // E, (1,), generator=g))
        n = min(n, total - at)
        merged += [[e, at + t, min(64, n - t)] for t in range(0, n, 64)]
        at += n
    odd = [[e, t0, min(n, 37)] for e, t0, n in merged]  # gaps: nothing merges
    odd += [[E, 0, 5], [-1, 0, 5], [0, -3, 5], [0, total, 5], [1, 3, 0]]       # skipped
    over = [[0, total - 10, 64], [1, 0, 200], [1, 64, 64], [2, 200, 64], [2, 264, 64], [3, 328, 20]]   # past the end; only 64 rows count
    return {"merged": merged, "odd": odd, "over": over, "reversed": merged[::-1]}


@pytest.mark.parametrize("which", ["merged", "odd", "over", "reversed"])
@pytest.mark.parametrize("fmt", [2, 5, 6])
@pytest.mark.parametrize("K,N", [(128, 40), (768, 264), (384, 257)])
def test_merged_chunks_match_the_chunk_kernel(dev, fmt, which, K, N):
    """Rows that no chunk names stay untouched; the others agree up to the order of the fp32 sums (weights and their
    roundings are the same): an fp16 step where a sum sits on the border, 2^-11 of the row's size at most."""
    from mi355x_qlinear import capi
    torch.manual_seed(K + N)
    E, total, nmat = 6, 700, 2 if fmt == 2 else 1
    u8 = lambda *s: torch.randint(0, 256, s, dtype=torch.uint8, device=dev)
    h = lambda *s: (torch.rand(*s, device=dev) * 0.01).half()
    per = 16 if fmt == 6 else 32
    ql, sc = [u8(E, N, K // 2) for _ in range(nmat)], [h(E, N, K // per) for _ in range(nmat)]
    mn = [h(E, N, K // 32) for _ in range(nmat)] if fmt != 6 else None
    qh = [u8(E, N, K // (8 if fmt == 5 else 4))] if fmt != 2 else None
    x = torch.randn(300, K, device=dev).half()
    ids = torch.randint(-2, 303, (total,), dtype=torch.int32, device=dev)       # some outside x: rows of zeros
    chunks = torch.tensor(_lists(total, E)[which], dtype=torch.int32, device=dev)
    arr = lambda t: capi.ptr_array(t) if t is not None else None
    outs = [torch.full((total, nmat * N), 7.0, dtype=torch.float16, device=dev) for _ in range(2)]
    need = ctypes.c_longlong(0)
    assert capi.lib().mi_moe_gguf_grouped_tiled_workspace(len(chunks), K, ctypes.byref(need)) == 0
    ws = torch.empty(need.value, dtype=torch.uint8, device=dev)
    for o, name, tail in ((outs[0], "mi_moe_gguf_grouped", (0,)),
                          (outs[1], "mi_moe_gguf_grouped_tiled_ws", (capi.ptr(ws), need.value))):
        capi.call(name, x, fmt, capi.ptr(x), x.shape[0], capi.ptr(ids), nmat, arr(ql), arr(qh), arr(sc), arr(mn), capi.ptr(o),
                  nmat * N, total, capi.ptr(chunks), len(chunks), E, N, K, *tail)
    a, b = (o.float() for o in outs)
    assert torch.equal(a == 7.0, b == 7.0)
    assert float((a - b).abs().max()) <= 2.0 ** -10 * float(a.abs().max())
    assert float((a - b).norm() / a.norm()) < 2.0 ** -11


def test_many_chunks_and_no_token_list(dev):
    """More chunks than the table kernel has threads; x in place of a gathered copy."""
    from mi355x_qlinear import capi
    E, N, K = 7, 64, 128
    sizes = [64, 64, 64, 64, 64, 10]
    chunks, at = [], 0
    for i in range(3000):
        n = sizes[i % 6]
        chunks.append([i // 6 % E, at, n])
        at += n
    x = torch.randn(at, K, device=dev).half()
    ql = torch.randint(0, 256, (E, N, K // 2), dtype=torch.uint8, device=dev)
    sc, mn = ((torch.rand(E, N, K // 32, device=dev) * 0.01).half() for _ in range(2))
    c = torch.tensor(chunks, dtype=torch.int32, device=dev)
    need = ctypes.c_longlong(0)
    assert capi.lib().mi_moe_gguf_grouped_tiled_workspace(len(c), K, ctypes.byref(need)) == 0
    ws = torch.empty(need.value, dtype=torch.uint8, device=dev)
    outs = [torch.zeros(at, N, dtype=torch.float16, device=dev) for _ in range(2)]
    for o, name, tail in ((outs[0], "mi_moe_gguf_grouped", (0,)),
                          (outs[1], "mi_moe_gguf_grouped_tiled_ws", (capi.ptr(ws), need.value))):
        capi.call(name, x, 2, capi.ptr(x), at, None, 1, capi.ptr_array([ql]), None, capi.ptr_array([sc]), capi.ptr_array([mn]),
                  capi.ptr(o), N, at, capi.ptr(c), len(c), E, N, K, *tail)
    a, b = (o.float() for o in outs)
    assert float((a - b).norm() / a.norm()) < 2.0 ** -11


def _record(monkeypatch):
    """Names of the C entries that the operators call from here on."""
    from mi355x_qlinear import capi
    inner, names = capi.call, []
    monkeypatch.setattr(capi, "call", lambda name, *a: names.append(name) or inner(name, *a))
    return names


@pytest.mark.parametrize("rows,E,per,n_list,want", [
    (1200, 6, 200, None, "mi_moe_gguf_grouped"),             # few experts, small matrices: the tiles would fill a few CUs
    (6144, 2, 3072, None, "mi_moe_gguf_grouped_tiled_ws"),
    (6144, 2, 3072, 6, "mi_moe_gguf_grouped")])              # a buffer of the largest size, a handful of chunks
def test_which_kernel_the_module_takes(dev, monkeypatch, rows, E, per, n_list, want):
    from custom_esimd_kernels_sglang import moe_grouped_gguf_xpu as mg
    H, I = 384, 1536
    u8 = lambda *s: torch.randint(0, 256, s, dtype=torch.uint8, device=dev)
    h = lambda *s: (torch.rand(*s, device=dev) * 0.01).half()
    gate, up = [(u8(E, I, H // 2), h(E, I, H // 32), h(E, I, H // 32)) for _ in range(2)]
    chunks = torch.tensor([[e, e * per + t, min(64, per - t)] for e in range(E) for t in range(0, per, 64)][:n_list],
                          dtype=torch.int32, device=dev)
    x = torch.randn(rows, H, device=dev).half()
    names = _record(monkeypatch)
    mg.moe_up_q4k_ggemv(x, *gate, *up, torch.zeros(rows, 2 * I, dtype=torch.float16, device=dev), chunks, H, I)
    assert names == [want]


def _sorted_rows(counts):
    """Chunk list of experts with `counts` rows each, and the expert of every row."""
    chunks, of, at = [], [], 0
    for e, n in enumerate(counts):
        chunks += [[e, at + t, min(64, n - t)] for t in range(0, n, 64)]
        of += [e] * n
        at += n
    return torch.tensor(chunks, dtype=torch.int32), torch.tensor(of)


@pytest.mark.parametrize("kind", ["q4_k", "q5_k", "q6_k"])
def test_module_on_merged_chunks_against_the_oracle(dev, monkeypatch, kind):
    """The module's own call of the tiled route (operands, workspace, decoding of the stacks): one-hot rows return the
    experts' dequantized weights value for value, random rows agree with the oracle's product.  One expert ends in a full
    tile, one in a tile of 1 row, one has no rows, and the last rows of the buffer belong to no chunk."""
    from custom_esimd_kernels_sglang import moe_grouped_gguf_xpu as mg
    E, K, N = 4, 384, 1536
    counts = (2048, 0, 1793, 2200)
    chunks, of = _sorted_rows(counts)
    rows, total = len(of), len(of) + 40
    g = torch.Generator().manual_seed(3)
    if kind == "q4_k":
        tokens = 900
        ids = torch.randint(0, tokens, (total,), generator=g).to(torch.int32)
        reps, deq = _q4k_expert_stacks(E, N, K, (71, 72), torch.arange(E), dev)
        run = lambda x, out: mg.moe_up_q4k_ggemv(x, *reps[0], *reps[1], out, chunks.to(dev), K, N, ids.to(dev))
        weights = torch.cat(deq, 1)                       # [E, 2 N, K]
    else:
        tokens, ids = total, torch.arange(total)
        stack, weights = _down_stack(kind, E, N, K, 73, torch.arange(E), dev)
        fn = mg.moe_down_q5k_ggemv if kind == "q5_k" else mg.moe_down_q6k_ggemv
        run = lambda x, out: fn(x, *stack, out, chunks.to(dev), K, N)
    names = _record(monkeypatch)
    hot = torch.zeros(tokens, K, dtype=torch.float16)
    ks = (3 + 37 * torch.arange(tokens)) % K
    hot[torch.arange(tokens), ks] = 1.0
    out = torch.full((total, weights.shape[1]), 7.0, dtype=torch.float16, device=dev)
    run(hot.to(dev), out)
    got = out.cpu().float()
    assert torch.equal(got[:rows], weights[of, :, ks[ids[:rows].long()]]) and bool((got[rows:] == 7.0).all())
    x = (torch.randn(tokens, K, generator=g) * 0.1).half()
    run(x.to(dev), out)
    xs = x.float()[ids[:rows].long()]
    want = torch.cat([xs[of == e] @ weights[e].t() for e in range(E)])
    assert O.max_rel_err(out.cpu()[:rows], want) < TOL
    assert names == ["mi_moe_gguf_grouped_tiled_ws"] * 2
    # in a graph: the same bits on every replay
    eager, stream, graph = out.clone(), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    xd, cd, idd = x.to(dev), chunks.to(dev), ids.to(dev)
    if kind == "q4_k":
        again = lambda: mg.moe_up_q4k_ggemv(xd, *reps[0], *reps[1], out, cd, K, N, idd)
    else:
        again = lambda: fn(xd, *stack, out, cd, K, N)
    torch.cuda.synchronize()
    with torch.cuda.stream(stream), torch.cuda.graph(graph, stream=stream):
        again()
    for _ in range(3):
        out[:rows].fill_(float("nan"))
        junk = torch.randn(256, 256, device=dev) @ torch.randn(256, 256, device=dev)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        del junk
        assert torch.equal(out.view(torch.int16), eager.view(torch.int16))
    # activations that are not 16-byte aligned stay on the chunk kernel
    del names[:]
    shifted = torch.empty(tokens * K + 4, dtype=torch.float16, device=dev)[4:].view(tokens, K)
    shifted.copy_(xd)
    assert shifted.data_ptr() % 16 == 8
    run(shifted, out)
    assert names == ["mi_moe_gguf_grouped"]
    assert O.max_rel_err(out.cpu()[:rows], want) < TOL
