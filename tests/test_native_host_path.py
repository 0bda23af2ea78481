"""The native host path of the hot operators against their Python implementations (mi355x_checked::<name>): the same
schema, the same results bit for bit over the forms that both accept, the same refusals."""
import pytest
import torch

from mi355x_qlinear import ops as _ops

_V, _S = torch.ops.custom_esimd_kernels_vllm, torch.ops.custom_esimd_kernels_sglang


def test_every_native_operator_has_its_python_implementation():
    assert len(_ops._CHECKED) == 25
    for ns, names in _ops._DEFINED.items():
        for name in names:
            if name in _ops._CHECKED:
                own = getattr(getattr(torch.ops, ns), name).default._schema
                other = getattr(torch.ops.mi355x_checked, name).default._schema
                assert str(own).split("::", 1)[1] == str(other).split("::", 1)[1]
                assert torch._C._dispatch_has_kernel_for_dispatch_key(f"mi355x_checked::{name}", "CUDA")


def _u8(*s):
    return torch.randint(0, 256, s, dtype=torch.uint8, device="cuda")


def _h(*s):
    return (torch.rand(*s, device="cuda") * 0.01 + 0.005).half()


def _args(name, M, K, N, dt):
    """(arguments, index of the output) of one call."""
    x = torch.randn(M, K, device="cuda").to(dt)
    o = torch.empty(M, N, device="cuda", dtype=dt)
    f8 = (torch.randn(N, K, device="cuda") * 4).to(torch.float8_e4m3fn)
    one = torch.full((1,), 0.01, device="cuda")
    if name == "esimd_gemv_fp8_pern":
        return [x, f8, torch.rand(N, device="cuda") * 0.01, o, N, K], 3
    if name.startswith("esimd_gemv_fp8_pern_fused"):
        n = int(name[-1])
        sc = [_h(N) for _ in range(n)]
        return [x] + [a for i in range(n) for a in (f8, sc[i], o if i == 0 else torch.empty_like(o), N)] + [K], 3
    if "blockscale" in name:
        bs = torch.rand(-(-N // 128), K // 128, device="cuda") * 0.01
        more = [f8.view(torch.uint8), bs, torch.empty_like(o)] if name.endswith("fused2") else []
        return [x, f8, bs, o] + more + [128, 128], 3
    if "resadd" in name:
        K1 = K
        xs = [torch.randn(1, K1, device="cuda").to(dt) for _ in range(3)]
        w = [_u8(N, K // 2), _h(N, K // 128)] if "int4" in name else [f8, one]
        return xs[:2] + [xs[2].view(-1)] + w + [torch.empty(1, N, device="cuda", dtype=dt), torch.empty_like(xs[0]), 1e-6], 5
    if "fp8_pert" in name:
        n = int(name[-1]) if "fused" in name else 1
        return [x] + [a for i in range(n) for a in (f8, one, o if i == 0 else torch.empty_like(o))], 3
    if "int4" in name:
        w, sc = _u8(N, K // 2), _h(N, K // 128)
        if name.endswith("_zp"):
            return [x, w, sc, _u8(N, K // 128) & 15, o], 4
        more = [w, sc, torch.empty_like(o)] if name.endswith("fused2") else []
        return [x.view(1, M, K), w.view(torch.int32), sc, o] + more, 3      # 3-D input, int32 view of the weight
    if name == "esimd_gemv_q4_k":
        return [x, _u8(N, K // 2), _h(N, K // 32), _h(N, K // 32), o], 4
    if "q4_0" in name:
        return [x, _u8(N, K // 2), _h(N, K // 32), o], 3
    if "q8_0" in name:
        return [x, _u8(N, K).view(torch.int8), _h(N, K // 32), o], 3
    if "q5_k" in name:
        return [x, _u8(N, K // 2), _u8(N, K // 8), _h(N, K // 32), _h(N, K // 32), o], 5
    return [x, _u8(N, K // 2), _u8(N, K // 4), _h(N, K // 16), o], 4


_LINEAR = sorted(n for n in _ops._CHECKED if not n.startswith("moe_"))


def _own(name):
    return getattr(_V, name) if name in _ops._DEFINED["custom_esimd_kernels_vllm"] else getattr(_S, name)


@pytest.mark.gpu
@pytest.mark.parametrize("name", _LINEAR)
def test_same_results_and_same_refusals(dev, name):
    checked = getattr(torch.ops.mi355x_checked, name)
    for dt in (torch.float16, torch.bfloat16):
        if dt == torch.bfloat16 and "_q" in name and "_k" in name or dt == torch.bfloat16 and ("q4_0" in name or "q8_0" in name):
            continue                                      # GGUF formats run in fp16
        for M, K, N in ((1, 512, 40), (3, 1024, 257), (65, 512, 136), (130, 1024, 264)):
            torch.manual_seed(M + N)
            args, at = _args(name, M, K, N, dt)
            clone = [a.clone() if torch.is_tensor(a) else a for a in args]
            assert _own(name)(*args) is args[at] and checked(*clone) is clone[at]
            for a, b in zip(args, clone):                 # outputs, and the residual that the norm updates
                assert not torch.is_tensor(a) or torch.equal(a.reshape(-1).view(torch.uint8), b.reshape(-1).view(torch.uint8))
    args, at = _args(name, 2, 512, 24, torch.float16)
    bad = [(0, args[0].cpu()), (0, args[0].double()), (1, args[1][..., :-1]), (at, args[at].float()),
           (at, torch.empty(3, 7, dtype=torch.float16, device=dev))]
    for i, v in bad:
        broken = list(args)
        broken[i] = v
        said = []
        for op in (_own(name), checked):
            with pytest.raises((RuntimeError, NotImplementedError)) as e:
                op(*broken)
            said.append(str(e.value).split("\n")[0])
        if i or v.is_cuda:
            assert said[0] == said[1]


@pytest.mark.gpu
@pytest.mark.parametrize("M", [2, 70])                  # weight-streaming and tiled kernel
def test_a_strided_scale_is_read_with_its_stride(dev, M):
    """Accepted although not as the kernels want it: per-channel scales that are views with a stride."""
    args, at = _args("esimd_gemv_fp8_pern", M, 512, 24, torch.float16)
    want = _V.esimd_gemv_fp8_pern(*args).clone()
    assert float(want.abs().max()) > 0
    wide = torch.stack([args[2], args[2] + 1.0], 1)      # the other column holds other scales
    args[2] = wide[:, 0]
    assert not args[2].is_contiguous()
    assert torch.equal(_V.esimd_gemv_fp8_pern(*args), want)
    two, at = _args("esimd_gemv_fp8_pern_fused2", M, 512, 24, torch.float16)
    want = [_V.esimd_gemv_fp8_pern_fused2(*two).clone(), two[7].clone()]
    two[6] = torch.stack([two[6], two[6] + 1.0], 1)[:, 0]
    assert torch.equal(_V.esimd_gemv_fp8_pern_fused2(*two), want[0]) and torch.equal(two[7], want[1])


@pytest.mark.gpu
@pytest.mark.parametrize("name,M,N,K,tiled", [
    ("esimd_gemm_q4_0", 70, 264, 3072, False), ("esimd_gemm_q4_0", 70, 264, 3200, True),
    ("esimd_gemv_q8_0_m", 70, 264, 2048, False), ("esimd_gemv_q8_0_m", 70, 264, 2176, True),
    ("esimd_gemv_q5_k", 97, 264, 1024, False), ("esimd_gemv_q5_k", 96, 264, 1024, True),
    ("esimd_gemv_q6_k_m", 97, 2056, 3072, False), ("esimd_gemv_q6_k_m", 96, 2056, 3072, True)])
def test_both_host_paths_take_the_same_route(dev, monkeypatch, name, M, N, K, tiled):
    """Either side of the lines between streaming and tiled kernels (their sums differ in order, so equal bits are
    the same route), and the route is the expected one."""
    torch.manual_seed(K)
    args, at = _args(name, M, K, N, torch.float16)
    other = list(args)
    other[at] = torch.empty_like(args[at])
    _own(name)(*args)
    inner, entries = _ops.capi.call, []
    monkeypatch.setattr(_ops.capi, "call", lambda entry, *a: entries.append(entry) or inner(entry, *a))
    getattr(torch.ops.mi355x_checked, name)(*other)
    assert torch.equal(args[at], other[at])
    assert (entries == ["mi_gemm_gguf_tiled_ws"]) == tiled and len(entries) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 3, 12, 13])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_moe_decode_is_the_same(dev, T, dt):
    """Both sides of the largest batch with one GEMV per route (96 pairs)."""
    torch.manual_seed(T)
    E, k, H, I = 16, 8, 256, 128
    f8 = lambda *s: (torch.randn(*s, device=dev) * 4).to(torch.float8_e4m3fn)
    sc = lambda *s: torch.rand(*s, device=dev) * 0.01
    x, logits = torch.randn(T, H, device=dev).to(dt), torch.randn(T, E, device=dev).to(dt)
    w = [f8(E, 2 * I, H), sc(E, 2 * I // 128, H // 128), f8(2 * I, H), sc(2 * I // 128, H // 128), f8(E, H, I),
         sc(E, H // 128, I // 128), f8(H, I), sc(H // 128, I // 128), torch.randn(1, H, device=dev).to(dt)]
    outs = [torch.empty_like(x) for _ in range(2)]
    for op, o in zip((torch.ops.moe_ops, torch.ops.mi355x_checked), outs):
        assert op.moe_forward_full_fp8_block(x, logits, o, *w, k, 1, E) is o
    assert torch.equal(outs[0], outs[1])


@pytest.mark.gpu
@pytest.mark.parametrize("T,k,E,H,I,plan", [(1, 8, 16, 256, 128, 7), (2, 8, 8, 256, 1024, 3), (8, 1, 8, 256, 128, 5), (64, 1, 8, 256, 128, 1),
                                            (97, 1, 8, 256, 128, 0)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_moe_decode_launches_the_plan(dev, monkeypatch, T, k, E, H, I, plan, dt):
    """Each choice of mi_moe_decode_plan: both host paths give the same bits, the entries are the plan's, the result is the oracle's."""
    from oracle import qlinear_oracle as O
    g = torch.Generator().manual_seed(T + k)
    x, logits, gw = torch.randn(T, H, generator=g).to(dt), torch.randn(T, E, generator=g).to(dt), (torch.randn(1, H, generator=g) * 0.1).to(dt)
    w = [t for s in ((E, 2 * I, H), (2 * I, H), (E, H, I), (H, I)) for t in O.fp8_quantize_block(torch.randn(*s, generator=g) * 0.1)]
    want = O.moe_forward_full(x, logits, *w, gw, k)
    args = [t.view(torch.float8_e4m3fn).to(dev) if t.dtype == torch.uint8 else t.to(dev) for t in w] + [gw.to(dev)]
    x, logits = x.to(dev), logits.to(dev)
    outs = [torch.empty_like(x) for _ in range(2)]
    torch.ops.moe_ops.moe_forward_full_fp8_block(x, logits, outs[0], *args, k, 1, E)
    inner, entries = _ops.capi.call, []
    monkeypatch.setattr(_ops.capi, "call", lambda entry, *a: entries.append(entry) or inner(entry, *a))
    torch.ops.mi355x_checked.moe_forward_full_fp8_block(x, logits, outs[1], *args, k, 1, E)
    assert torch.equal(*outs)
    gate_up = ["mi_moe_gate_up_topk_fp8_block"] if plan & 2 else ["mi_moe_topk", "mi_moe_gemv_fp8_block_routed"]
    down = ["mi_moe_down_sum_fp8_block"] if plan & 4 else ["mi_moe_gemv_fp8_block_routed", "mi_moe_combine_shared"]
    assert entries == gate_up + down if plan else "mi_moe_sort" in entries
    mean_rel = float((outs[0].cpu().float() - want).abs().mean() / want.abs().mean())
    assert mean_rel < (3e-3 if dt == torch.float16 else 1e-2)               # the bars of the operator's test


def _refused(dev):
    """(Python building block of the operator, call) where the checks pass and the C entry refuses the size before it
    launches anything: K of no whole granule, and an expert row longer than the LDS holds."""
    h = lambda *s: torch.zeros(*s, dtype=torch.float16, device=dev)
    f8 = lambda *s: torch.zeros(*s, dtype=torch.uint8, device=dev)
    one = torch.ones(1, device=dev)
    H = 40960
    moe = [h(1, H), h(1, 2), h(1, H), f8(2, 256, H), torch.ones(2, 2, H // 128, device=dev), f8(256, H),
           torch.ones(2, H // 128, device=dev), f8(2, H, 128), torch.ones(2, H // 128, 1, device=dev), f8(H, 128),
           torch.ones(H // 128, 1, device=dev), h(1, H), 1, 1, 2]
    return {"esimd_gemv_fp8_pern": ("_fp8_pern_multi", lambda: _V.esimd_gemv_fp8_pern(h(1, 48), f8(8, 48), h(8), h(1, 8), 8, 48)),
            "esimd_gemv_fp8_pert": ("_fp8_pert_multi", lambda: _V.esimd_gemv_fp8_pert(h(1, 48), f8(8, 48), one, h(1, 8))),
            "esimd_resadd_norm_gemv_fp8_pert": ("_norm_gemv", lambda: _V.esimd_resadd_norm_gemv_fp8_pert(
                h(1, 24), h(1, 24), h(24), f8(8, 24), one, h(1, 8), h(1, 24), 1e-6)),
            "moe_forward_full_fp8_block": ("esimd_moe_topk", lambda: torch.ops.moe_ops.moe_forward_full_fp8_block(*moe))}


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["esimd_gemv_fp8_pern", "esimd_gemv_fp8_pert", "esimd_resadd_norm_gemv_fp8_pert",
                                  "moe_forward_full_fp8_block"])
def test_a_status_is_raised_and_the_call_not_run_again(dev, monkeypatch, name):
    block, call = _refused(dev)[name]
    inner, again = getattr(_ops, block), []
    monkeypatch.setattr(_ops, block, lambda *a, **k: again.append(1) or inner(*a, **k))
    with pytest.raises(RuntimeError, match="failed: unsupported shape or divisibility"):
        call()
    assert not again


@pytest.mark.gpu
def test_a_pending_error_does_not_add_to_the_residual_twice(dev):
    """An error that something else left on the thread is what the status of the next launch reports: the operator
    raises it, as its Python implementation does, and has added x to the residual once."""
    import ctypes
    with open("/proc/self/maps") as f:
        hip = ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64.so" in line))
    args, _ = _args("esimd_resadd_norm_gemv_fp8_pert", 1, 512, 40, torch.float16)
    want = args[1] + args[0]
    torch.cuda.synchronize()
    assert hip.hipSetDevice(1 << 20) != 0                 # no such device: refused on the host
    with pytest.raises(RuntimeError, match="mi_norm_gemv_scaled failed: kernel launch failed"):
        _V.esimd_resadd_norm_gemv_fp8_pert(*args)
    torch.cuda.synchronize()
    assert torch.equal(args[1], want)
