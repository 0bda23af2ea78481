"""CPU-only checks of the boundary: the shared library loads, exports every
symbol include/mi355x_qlinear.h declares, the torch.ops schemas carry the
reference's names and argument order, and there is no silent CPU fallback."""
import ctypes
import os

import pytest
import torch

import mi355x_qlinear  # noqa: F401
from mi355x_qlinear import capi


def test_library_exports_every_declared_symbol():
    protos = capi.parse_header()
    assert len(protos) >= 14
    handle = ctypes.CDLL(capi.LIB_PATH)
    for name in protos:
        assert hasattr(handle, name), name
    # and the loader wires argtypes for all of them
    lib = capi.lib()
    for name, types in protos.items():
        assert getattr(lib, name).argtypes == types


def test_moe_tiled_workspace_sizes_and_argument_errors():
    """Host-side answers of the grouped tiled GEMM entry points (no launch): the workspace of the expert MLP
    holds the single GEMM's (re-tiled x + tables) plus the re-tiled intermediate; limits and bad arguments
    come back as error codes before anything is enqueued."""
    lib = capi.lib()
    one, mlp = ctypes.c_longlong(0), ctypes.c_longlong(0)
    total, E, H, I = 32768, 128, 2048, 768
    assert lib.mi_moe_gemm_fp8_tiled_workspace(total, E, H, ctypes.byref(one)) == 0
    assert lib.mi_moe_mlp_fp8_tiled_workspace(total, E, H, I, ctypes.byref(mlp)) == 0
    blocks = total // 16 + E
    assert one.value >= blocks * 16 * H * 2 and one.value % 256 == 0
    assert mlp.value == one.value + (blocks * 16 * I * 2 + 255) // 256 * 256
    # re-tiled activations of 2 GiB or more: the tiled route does not apply (the size is still reported)
    assert lib.mi_moe_mlp_fp8_tiled_workspace(1 << 19, E, 4096, I, ctypes.byref(mlp)) == -2 and mlp.value > (1 << 31)
    assert lib.mi_moe_mlp_fp8_tiled_workspace(total, 1025, H, I, ctypes.byref(mlp)) == -2      # more than 1024 experts
    assert lib.mi_moe_mlp_fp8_tiled_workspace(total, E, H, I, None) == -1
    # the call itself: null pointers, unknown activation, sizes off the 128 grid, short workspace
    ok = ctypes.c_void_p(256)                      # never dereferenced: every case below returns before a launch
    args = lambda **kw: [kw.get("a", ok), None, kw.get("div", 1), ok, ok, ok, ok, kw.get("spe", 0), ok, ok, None, None, 64,
                         4096, 8, kw.get("H", 256), kw.get("I", 128), kw.get("act", 1), kw.get("dt", 1), kw.get("ws", ok),
                         ctypes.c_longlong(kw.get("wsb", 1 << 40)), None]
    f = lib.mi_moe_mlp_fp8_tiled_ws
    assert f(*args(a=None)) == -1
    assert f(*args(act=0)) == -1 and f(*args(act=3)) == -1 and f(*args(dt=2)) == -1 and f(*args(spe=3)) == -1
    assert f(*args(div=0)) == -1
    assert f(*args(H=200)) == -2 and f(*args(I=100)) == -2
    assert f(*args(ws=None)) == -1 and f(*args(wsb=1024)) == -1


def test_moe_gguf_grouped_argument_errors():
    """mi_moe_gguf_grouped answers bad arguments and sizes beyond its 32-bit addressing with error codes, and
    empty inputs with success, before anything is enqueued."""
    lib = capi.lib()
    ok = ctypes.c_void_p(256)                      # never dereferenced: every case below returns before a launch
    arr = (ctypes.c_void_p * 2)(256, 256)
    none2 = (ctypes.c_void_p * 2)(None, None)

    def f(**kw):
        return lib.mi_moe_gguf_grouped(kw.get("fmt", 2), kw.get("x", ok), kw.get("x_rows", 64), None, kw.get("nmat", 2),
                                       kw.get("ql", arr), kw.get("qh", None), kw.get("sc", arr), kw.get("mn", arr),
                                       kw.get("out", ok), ctypes.c_longlong(kw.get("stride", 1024)), kw.get("rows", 64),
                                       kw.get("chunks", ok), kw.get("n", 4), 8, kw.get("N", 512), kw.get("K", 2048), 0,
                                       None)
    assert f(x=None) == -1 and f(out=None) == -1 and f(chunks=None) == -1 and f(ql=None) == -1 and f(sc=None) == -1
    assert f(fmt=3) == -1 and f(fmt=7) == -1 and f(nmat=0) == -1 and f(nmat=3) == -1
    assert f(mn=None) == -1 and f(mn=none2) == -1 and f(ql=none2) == -1          # Q4_K needs mins
    assert f(fmt=5) == -1 and f(fmt=6) == -1                                     # Q5_K / Q6_K need the high bits
    assert f(fmt=6, qh=none2) == -1
    assert f(K=2040) == -2 and f(K=0) == -2 and f(stride=1023) == -2 and f(rows=-1) == -2 and f(n=-1) == -2
    assert f(N=1 << 20, stride=1 << 22) == -2                                    # N K beyond 2^31
    assert f(x_rows=1 << 19) == -2                                               # x beyond 2 GiB
    assert f(n=0) == 0 and f(rows=0) == 0 and f(x_rows=0) == 0 and f(N=0, stride=0) == 0


@pytest.mark.parametrize("M,N,K,split", [
    (128, 4096, 4096, True), (100, 5120, 5120, True), (129, 5120, 5120, True), (1024, 2048, 6144, True), (70, 1024, 1024, True),
    (256, 4936, 1280, False), (320, 2760, 1024, False), (256, 2568, 768, False), (65, 9584, 1024, False), (160, 5120, 1024, False),
    (256, 5688, 1536, False), (64, 4096, 4096, False), (2048, 14336, 4096, False)])
def test_k_is_split_where_it_was_measured_faster(M, N, K, split):
    """Few tiles and a long K: slices.  Short K: one piece (measured 12 to 28 % ahead of slices there)."""
    lib = capi.lib()
    one, need = ctypes.c_longlong(-1), ctypes.c_longlong(-1)
    assert lib.mi_gemm_tiled_workspace(M, K, ctypes.byref(one)) == 0
    assert lib.mi_gemm_tiled_workspace_split(M, N, K, ctypes.byref(need)) == 0
    assert (need.value > one.value) == split and need.value >= one.value


def test_rows_beyond_64_of_gguf_weights_take_the_measured_route():
    """mi_gemm_gguf_tiled_pays: one rule for both host paths; either side of its lines, and sizes it does not take."""
    lib = capi.lib()

    def pays(fmt, M, N, K):
        p = ctypes.c_int(-1)
        rc = lib.mi_gemm_gguf_tiled_pays(fmt, M, N, K, ctypes.byref(p))
        return p.value if rc == 0 else rc
    q4k, q40, q80, q5k, q6k = 2, 3, 4, 5, 6
    for fmt in (q40, q80, q5k, q6k):
        assert pays(fmt, 64, 14336, 14336) == 0 and pays(fmt, 129, 4096, 1024) == 1 and pays(fmt, 65, 10240, 14336) == 1
        assert pays(fmt, 200, 4096, 96) == 0 and pays(fmt, 200, 1 << 20, 4096) == 0 and pays(fmt, 1 << 20, 256, 4096) == 0
        assert pays(fmt, 200, 0, 4096) == 0
    assert pays(q4k, 65, 4096, 1024) == 1 and pays(q4k, 64, 4096, 1024) == 0 and pays(q4k, 65, 4096, 1056) == 0
    assert pays(q40, 128, 1024, 3072) == 0 and pays(q40, 128, 1024, 3200) == 1
    assert pays(q40, 96, 4096, 4096) == 0 and pays(q40, 97, 4096, 4096) == 1
    assert pays(q80, 128, 1024, 2048) == 0 and pays(q80, 128, 1024, 2176) == 1
    assert pays(q80, 80, 4096, 3072) == 0 and pays(q80, 80, 4104, 3072) == 1 and pays(q80, 80, 4096, 3200) == 1
    for fmt in (q5k, q6k):
        assert pays(fmt, 96, 4096, 2560) == 0 and pays(fmt, 96, 4096, 3072) == 1 and pays(fmt, 97, 4096, 3072) == 0
        assert pays(fmt, 97, 1024, 1024) == 0 and pays(fmt, 96, 1024, 1024) == 1 and pays(fmt, 112, 1024, 1536) == 1
        assert pays(fmt, 128, 8192, 1536) == 0 and pays(fmt, 128, 8200, 1536) == 1 and pays(fmt, 200, 512, 1152) == 0
    assert pays(7, 200, 512, 512) == -1 and pays(1, 200, 512, 512) == -1 and pays(q80, 1, 1, 0) == -2
    assert lib.mi_gemm_gguf_tiled_pays(q80, 200, 512, 512, None) == -1


def test_merged_chunks_argument_errors():
    """The tiled entry refuses what the chunk kernel refuses, whichever of the two a call would take."""
    lib = capi.lib()
    ok, arr = ctypes.c_void_p(256), (ctypes.c_void_p * 2)(256, 256)

    def f(**kw):
        return lib.mi_moe_gguf_grouped_tiled_ws(kw.get("fmt", 2), ok, kw.get("x_rows", 64), None, kw.get("nmat", 2), arr,
                                                kw.get("qh", None), arr, kw.get("mn", arr), ok, ctypes.c_longlong(kw.get("stride", 1024)),
                                                64, ok, kw.get("n", 4), 8, kw.get("N", 512), kw.get("K", 2048), kw.get("ws", ok),
                                                ctypes.c_longlong(kw.get("wsb", 0)), None)
    assert f(fmt=3) == -1 and f(nmat=0) == -1 and f(mn=None) == -1 and f(fmt=5, nmat=1) == -1 and f(fmt=6, nmat=2, qh=arr) == -1
    assert f(K=2080) == -2 and f(stride=1023) == -2 and f(n=-1) == -2 and f(n=1 << 14) == -2
    assert f(N=1 << 20, stride=1 << 22) == -2                                    # N K beyond 2^31
    assert f(x_rows=1 << 19) == -2                                               # x beyond 2 GiB
    assert f() == -1 and f(ws=None, wsb=1 << 30) == -1                           # workspace too small / missing
    assert f(n=0) == 0 and f(x_rows=0) == 0 and f(N=0, stride=0) == 0


def test_merged_chunks_are_expected_where_they_were_measured_faster():
    """mi_moe_gguf_grouped_tiled_pays decides from the length of the chunk list, not from the rows of the caller's
    buffer alone; geometries where either kernel was measured ahead by 8 % and more."""
    lib = capi.lib()

    def pays(fmt, n, rows, E, N, K, nmat=None):
        p = ctypes.c_int(-1)
        rc = lib.mi_moe_gguf_grouped_tiled_pays(fmt, (2 if fmt == 2 else 1) if nmat is None else nmat, n, rows, E, N, K, ctypes.byref(p))
        return p.value if rc == 0 else rc
    for case in ((2, 314, 16384, 128, 768, 2048), (6, 314, 16384, 128, 2048, 768), (5, 231, 9216, 128, 2048, 768),
                 (2, 513, 24576, 256, 512, 2048), (5, 80, 4096, 32, 2048, 1024), (2, 68, 4096, 8, 1536, 4096)):
        assert pays(*case) == 1, case
    for case in ((2, 20, 1024, 8, 512, 1024), (2, 32, 1536, 16, 768, 2048), (2, 128, 7680, 128, 768, 2048),
                 (2, 328, 15360, 256, 512, 2048), (6, 16, 1024, 8, 1024, 512), (6, 5, 240, 4, 2048, 768)):
        assert pays(*case) == 0, case
    # a buffer of the largest size: 64 tokens' chunks stay, a list of full chunks does not
    assert pays(2, 126, 16384, 128, 768, 2048) == 0 and pays(6, 126, 16384, 128, 2048, 768) == 0
    assert pays(2, 314, 32768, 128, 768, 2048) == 1
    assert pays(2, 7680, 7680, 128, 768, 2048) == 0                              # one-row chunks: nothing merges
    assert pays(2, 314, 16384, 128, 768, 2080) == 0 and pays(2, 200000, 12800000, 8, 768, 2048) == 0    # sizes it does not take
    assert pays(2, 0, 16384, 128, 768, 2048) == 0 and pays(2, 314, 16384, 128, 0, 2048) == 0
    assert pays(6, 314, 16384, 128, 2048, 768, nmat=2) == 0
    assert pays(3, 4, 64, 8, 64, 128) == -1 and pays(2, 4, 64, 0, 64, 128) == -1 and pays(2, -1, 64, 8, 64, 128) == -2
    assert lib.mi_moe_gguf_grouped_tiled_pays(2, 2, 4, 64, 8, 64, 128, None) == -1


@pytest.mark.parametrize("case, tiles", [((6, 16, 576, 8, 4096, 2048), 1), ((5, 14, 569, 8, 4096, 2048), 1), ((6, 78, 3578, 60, 2560, 1536), 1),
                                         ((6, 39, 1908, 32, 2048, 1024), 1), ((5, 136, 3003, 128, 2048, 768), 0),
                                         ((6, 256, 8192, 256, 2048, 512), 0), ((5, 32, 1536, 32, 2048, 1024), 0)])
def test_down_launches_either_side_of_the_line(case, tiles):
    """Down launches near the line of mi_moe_gguf_grouped_tiled_pays, where either kernel was measured ahead by 9 % and more."""
    p = ctypes.c_int(-1)
    fmt, n, rows, E, N, K = case
    assert capi.lib().mi_moe_gguf_grouped_tiled_pays(fmt, 1, n, rows, E, N, K, ctypes.byref(p)) == 0 and p.value == tiles


# (T, top k, E, H, I): us of the step with mi_moe_topk and a row GEMV for gate_up / the selecting launch, a row GEMV and a sum for down / the summing launch
@pytest.mark.parametrize("case, plan", [((1, 8, 128, 2048, 768), 7),        # 20.3 -> 16.8, -> 18.2
                                        ((12, 8, 128, 2048, 768), 7),       # 119 -> 103, -> 108
                                        ((8, 8, 8, 2048, 768), 5),          # 60 -> 65, -> 52
                                        ((32, 1, 8, 4096, 1536), 1),        # 123 -> 166, -> 205
                                        ((64, 1, 8, 4096, 512), 1),         # 130 -> 151, -> 268
                                        ((1, 1, 8, 4096, 1536), 7),         # 18.9 -> 15.9, -> 17.8
                                        ((2, 3, 8, 2176, 2048), 3),         # 26.1 -> 26.5, -> 27.6
                                        ((2, 1, 8, 4096, 8192), 3),         # 63 -> 65, -> 68
                                        ((1, 32, 512, 1024, 512), 5),       # 33 -> 41, -> 33.5
                                        ((96, 1, 8, 4096, 512), 1), ((97, 1, 8, 4096, 512), 0), ((12, 8, 16, 256, 128), 7), ((13, 8, 16, 256, 128), 0),
                                        ((1, 8, 9, 4224, 128), 5), ((1, 8, 9, 128, 3712), 3), ((1, 65, 70, 256, 128), 1), ((1, 2, 1025, 256, 128), 1)])
def test_decode_step_launches_what_was_measured_faster(case, plan):
    """Either side of the lines of mi_moe_decode_plan: 1 = a GEMV per route, 2 = selection in the gate_up launch, 4 = sum in the down launch."""
    p = ctypes.c_int(-1)
    assert capi.lib().mi_moe_decode_plan(*case, ctypes.byref(p)) == 0 and p.value == plan
    assert capi.lib().mi_moe_decode_plan(*case, None) == -1 and capi.lib().mi_moe_decode_plan(-1, *case[1:], ctypes.byref(p)) == -2


def test_moe_grouped_module_matches_the_reference_binding():
    """Names, argument order and defaults of the pybind module the patched SGLang imports
    (S/csrc/moe_grouped/moe_grouped_entry.sycl:108-127, sglang_for_multi_arc.patch:2114)."""
    import inspect
    from custom_esimd_kernels_sglang import moe_grouped_gguf_xpu as mg
    want = {
        "moe_up_q4k_ggemv": ["expert_states", "gate_ql", "gate_sc", "gate_mn", "up_ql", "up_sc", "up_mn", "gate_buf",
                             "chunks", "hidden_size", "intermediate_size", "tok_ids", "smallm"],
        "moe_down_q5k_ggemv": ["intermediate", "w_ql", "w_qh", "w_scale", "w_min", "expert_output", "chunks",
                               "intermediate_size", "hidden_size", "smallm"],
        "moe_down_q6k_ggemv": ["intermediate", "w_ql", "w_qh", "w_scale", "expert_output", "chunks",
                               "intermediate_size", "hidden_size", "smallm"],
    }
    for name, params in want.items():
        sig = inspect.signature(getattr(mg, name))
        assert list(sig.parameters) == params, name
        assert sig.parameters["smallm"].default is False
    # argument checks run before the library is touched
    z = torch.zeros(1, 4, dtype=torch.float16)
    with pytest.raises(RuntimeError, match=r"chunks \[num_chunks,3\]"):
        mg.moe_up_q4k_ggemv(z, z, z, z, z, z, z, z, torch.zeros(2, 2, dtype=torch.int32), 4, 4)


def test_header_pointer_and_scalar_mapping():
    p = capi.parse_header()
    assert p["mi_gemm_fp8_pern"] == [ctypes.c_void_p] * 4 + [ctypes.c_int] * 5 + [ctypes.c_void_p]
    assert p["mi_decode_e4m3"][2] is ctypes.c_longlong


import json

import custom_esimd_kernels_sglang  # noqa: F401,E402  (importing the packages registers every namespace)
import custom_esimd_kernels_vllm  # noqa: F401,E402

_GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "reference_schemas.json")
with open(_GOLDEN) as _f:
    REFERENCE_OPS = json.load(_f)["ops"]          # every m.def(...) of the reference's two kernel packages

# Reference operators this package does not register, by reason.  Everything else in the fixture
# must be registered with the reference's argument names, types and return type.
UNBUILT_NAMESPACES = {
    "eagle_ops": "speculative-decoding / GDN / paged-attention kernels: not quantized-linear work",
    "sgl_esimd_attn": "attention",
    "moe_int4_ops": "INT4 MoE family: outside the configurations of this path",
}
UNBUILT_OPS = {
    "custom_esimd_kernels_vllm::esimd_gdn_conv_fused": "GDN convolution",
    "custom_esimd_kernels_vllm::esimd_gdn_conv_fused_seq": "GDN convolution",
    "custom_esimd_kernels_vllm::esimd_gdn_conv_fused_seq_spec": "GDN convolution",
    "custom_esimd_kernels_sglang::esimd_gdn_conv_fused": "GDN convolution",
    "custom_esimd_kernels_sglang::esimd_gdn_conv_fused_seq": "GDN convolution",
    "custom_esimd_kernels_vllm::esimd_qkv_split_norm_rope": "RoPE",
    "custom_esimd_kernels_vllm::esimd_qkv_split_norm_rope_v": "RoPE",
    "custom_esimd_kernels_sglang::esimd_qkv_split_norm_rope": "RoPE",
    "custom_esimd_kernels_vllm::esimd_sdpa_prefill_dpas": "attention",
    "custom_esimd_kernels_vllm::esimd_moe_gemm_fp8": "E5M2 weights (per-N scales); no caller in the patches",
    "custom_esimd_kernels_vllm::esimd_moe_gemm_fp8_pert": "E5M2 weights (per-tensor scale); no caller in the patches",
    "custom_esimd_kernels_sglang::esimd_moe_gemm_fp8": "E5M2 weights",
    "custom_esimd_kernels_sglang::esimd_moe_gemm_fp8_pert": "E5M2 weights",
    "moe_ops::moe_forward_full_silu_routed_e5m2": "E5M2 weights",
    "moe_ops::moe_up_forward": "staged K-major op: the fused forms (moe_forward_full / _v2) are built instead",
    "moe_ops::moe_down_forward": "staged K-major op",
    "moe_ops::moe_forward_fused": "staged K-major op",
    "moe_int4_prefill_ops::moe_prefill_accumulate_forward_v2": "INT4 MoE prefill",
    "moe_int4_prefill_ops::moe_prefill_accumulate_permuted_forward_v2": "INT4 MoE prefill",
    "moe_int4_prefill_ops::moe_prefill_down_forward_v2": "INT4 MoE prefill",
    "moe_int4_prefill_ops::moe_prefill_full_int4": "INT4 MoE prefill",
    "moe_int4_prefill_ops::moe_prefill_scatter_x_forward": "INT4 MoE prefill",
    "moe_int4_prefill_ops::moe_prefill_silu_mul_forward": "INT4 MoE prefill",
    "moe_int4_prefill_ops::moe_prefill_up_forward_v2": "INT4 MoE prefill",
}


def _is_unbuilt(qual):
    return qual in UNBUILT_OPS or qual.split("::")[0] in UNBUILT_NAMESPACES


def _registered(qual):
    ns, name = qual.split("::")
    try:
        return getattr(getattr(torch.ops, ns), name).default
    except (AttributeError, RuntimeError):
        return None


def _parsed(op, args, ret):
    """The reference's schema through torch's own parser -> ([type, name] per argument, return types)."""
    sch = torch._C.parse_schema(f"{op}({', '.join(t + ' ' + n for t, n in args)}) -> {ret}")
    return [[str(a.type), a.name] for a in sch.arguments], [str(r.type) for r in sch.returns]


BUILT = sorted(q for q in REFERENCE_OPS if not _is_unbuilt(q))


def test_reference_schema_fixture_is_whole():
    # 154 operators in the reference's two packages; what is not registered here is listed above
    assert len(REFERENCE_OPS) == 154 and len(BUILT) == 97
    for q in REFERENCE_OPS:
        assert (_registered(q) is None) == _is_unbuilt(q), q


@pytest.mark.parametrize("qual", BUILT)
def test_schema_matches_reference(qual):
    """Argument names, argument types and the return type of every registered operator equal the
    reference's m.def(...) string (either package's, where the two differ)."""
    op = _registered(qual)
    assert op is not None, f"{qual} is not registered"
    got_args = [[str(a.type), a.name] for a in op._schema.arguments]
    got_ret = [str(r.type) for r in op._schema.returns]
    e = REFERENCE_OPS[qual]
    variants = [(e["args"], e["returns"])] + [(v["args"], v["returns"]) for v in e.get("variants", [])]
    want = [_parsed(e["op"], args, ret) for args, ret in variants]
    assert (got_args, got_ret) in want, f"{qual}: registered {got_args} -> {got_ret}, reference {want}"


def _meta_value(arg):
    t = str(arg.type)
    if t == "Tensor":
        return torch.empty(4, 8, device="meta", dtype=torch.float16)
    if t == "Optional[Tensor]":
        return None
    if t == "List[Tensor]":
        return [torch.empty(4, 8, device="meta", dtype=torch.float16)]
    if t == "int":
        return 1
    if t == "float":
        return 1.0
    if t == "bool":
        return False
    if t == "str":
        return ""
    raise AssertionError(f"no meta stand-in for argument type {t}")


def _all_registered_ops():
    """Every operator of the five namespaces this package defines, reference-named or sibling."""
    out = []
    from mi355x_qlinear import ops as _ops
    for ns in sorted(_ops._DEFINED):
        for name in sorted(_ops._DEFINED[ns]):
            out.append(f"{ns}::{name}")
    return out


@pytest.mark.parametrize("qual", _all_registered_ops())
def test_every_op_has_a_meta_kernel(qual):
    """vllm/patches/vllm_for_multi_arc.patch:2793-2937 registers a fake per operator; here every
    operator carries a Meta kernel, so tracing with meta / fake tensors never reaches the library:
    the call returns the pre-allocated output it aliases (or nothing) without touching data."""
    op = _registered(qual)
    args = [_meta_value(a) for a in op._schema.arguments]
    r = op(*args)
    rets = op._schema.returns
    if not rets:
        assert r is None
    else:
        if len(rets) == 1 and str(rets[0].type) == "List[Tensor]":
            rs = list(r)
        else:
            rs = r if isinstance(r, (tuple, list)) else (r,)
            assert len(rs) == len(rets)
        for v in rs:
            assert v is None or (isinstance(v, torch.Tensor) and v.device.type == "meta")


def test_fake_tensor_tracing_of_one_op_per_family():
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode():
        x = torch.empty(1, 128, dtype=torch.float16, device="cuda")
        w = torch.empty(16, 64, dtype=torch.uint8, device="cuda")
        s = torch.empty(16, 1, dtype=torch.float16, device="cuda")
        out = torch.empty(1, 16, dtype=torch.float16, device="cuda")
        r = torch.ops.custom_esimd_kernels_vllm.esimd_gemv_int4(x, w, s, out)
        assert r.shape == (1, 16) and r.dtype == torch.float16
        w8 = torch.empty(16, 128, dtype=torch.float8_e4m3fn, device="cuda")
        r = torch.ops.custom_esimd_kernels_vllm.esimd_gemv_fp8_pern(x, w8, torch.empty(16, device="cuda"), out, 16, 128)
        assert r.shape == (1, 16)


def test_extension_module_stand_ins_import():
    """The patched callers import the reference's compiled extension modules by name for their
    registration side effect (vllm/patches/vllm_for_multi_arc.patch:8218,
    sglang/patches/sglang_for_multi_arc.patch:1181, :1414); each stand-in resolves its ops."""
    import custom_esimd_kernels_vllm.moe_int4_prefill_ops as a
    import custom_esimd_kernels_vllm.moe_ops as b
    from custom_esimd_kernels_sglang import moe_fp8_prefill_ops as c
    from custom_esimd_kernels_sglang import moe_ops as d
    assert a.moe_prefill_gather_forward_v2 is not None and b.moe_forward_full_v2 is not None
    assert c.moe_prefill_full_fp8 is not None and d.moe_forward_full_silu_routed_sglang is not None
    with pytest.raises(AttributeError):
        d.moe_forward_full_silu_routed_e5m2          # not built: the caller's try / except falls back


def test_no_cpu_fallback():
    x = torch.zeros(1, 128, dtype=torch.float16)
    w = torch.zeros(16, 64, dtype=torch.uint8)
    s = torch.zeros(16, 1, dtype=torch.float16)
    out = torch.zeros(1, 16, dtype=torch.float16)
    with pytest.raises((RuntimeError, NotImplementedError)):
        torch.ops.custom_esimd_kernels_vllm.esimd_gemv_int4(x, w, s, out)


def test_host_tensors_are_refused_before_any_launch():
    """A host address handed to a kernel would be a GPU memory fault rather than an error code: the pointer
    helpers refuse tensors that are not on a ROCm device."""
    t = torch.zeros(4, dtype=torch.int32)
    with pytest.raises(RuntimeError, match="must live on a ROCm device"):
        capi.ptr(t)
    with pytest.raises(RuntimeError, match="must live on a ROCm device"):
        capi.ptr_array([None, t])
    assert capi.ptr(None) is None


def test_meta_kernels_trace():
    x = torch.zeros(1, 128, dtype=torch.float16, device="meta")
    w = torch.zeros(16, 64, dtype=torch.uint8, device="meta")
    s = torch.zeros(16, 1, dtype=torch.float16, device="meta")
    out = torch.zeros(1, 16, dtype=torch.float16, device="meta")
    r = torch.ops.custom_esimd_kernels_vllm.esimd_gemv_int4(x, w, s, out)
    assert r.shape == (1, 16)


def test_missing_library_fails_loudly(monkeypatch):
    monkeypatch.setattr(capi, "_lib", None)
    monkeypatch.setattr(capi, "LIB_PATH", os.path.join(os.path.dirname(capi.LIB_PATH), "nope.so"))
    with pytest.raises(ImportError):
        capi.lib()


# ---- names the reference's patched callers read from the kernel packages ----
_NAMES = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "esimd_import_names.json")
with open(_NAMES) as _f:
    IMPORT_NAMES = json.load(_f)     # made by tests/golden/make_esimd_import_names.py from the patch text

# Guarded reads (getattr default / try-except around the import) of names this package lacks: the
# caller falls back, which is the intended behaviour for kernels outside the quantized-linear path.
ABSENT_BY_DESIGN = {
    "sglang_decode_attn", "eagle_page_attn_decode_temp_size", "custom_esimd_kernels_prefill_dpas",
    ("custom_esimd_kernels_sglang", "esimd_gdn_conv_fused_seq"),
    ("custom_esimd_kernels_sglang", "esimd_qkv_split_norm_rope"),
}


def _resolve(pkg_name, module, name):
    import importlib
    mod = importlib.import_module(pkg_name + ("." + module if module else ""))
    return mod if name is None else getattr(mod, name)


def test_esimd_utils_handle_reads_resolve():
    """The patched vLLM's esimd_utils.py binds ~25 names off `import custom_esimd_kernels_vllm as
    _esimd` at import time (vllm/patches/vllm_for_multi_arc.patch:3119-3224); one missing name is an
    AttributeError that takes the whole model-executor import down."""
    reads = IMPORT_NAMES["esimd_utils_reads"]
    assert len(reads) >= 28
    for r in reads:
        obj = _resolve("custom_esimd_kernels_vllm", r["module"], r["name"])
        assert callable(obj), r


def test_patch_import_sites_resolve():
    """Every `from custom_esimd_kernels_{vllm,sglang}[.module] import name` of the two patches: an
    unguarded site must resolve; a guarded one resolves or is absent by design (the caller falls back)."""
    sites = IMPORT_NAMES["imports"]
    assert len(sites) >= 32
    for s in sites:
        for name in (s["names"] or [None]):
            key = name if name is not None else s["module"]
            try:
                _resolve(s["package"], s["module"], name)
                found = True
            except (ImportError, AttributeError):
                found = False
            if s["guarded"]:
                assert found or key in ABSENT_BY_DESIGN or (s["package"], key) in ABSENT_BY_DESIGN, s
            else:
                assert found, s


def test_sglang_package_exports_what_the_library_registers():
    """The reference's SGLang package re-exports a fixed list of wrapper names
    (S/python/custom_esimd_kernels_sglang/__init__.py:69-147); every one of them that this library registers
    under torch.ops.custom_esimd_kernels_sglang must also be an attribute of the package — the patched GGUF path
    looks names up on the package, not on torch.ops (`_imp_kernels`, sglang_for_multi_arc.patch:2077-2140) —
    and every name that lookup takes must resolve there."""
    import custom_esimd_kernels_sglang as s
    ns = torch.ops.custom_esimd_kernels_sglang
    exports = IMPORT_NAMES["sglang_package_exports"]
    assert len(exports) >= 60
    registered = [n for n in exports if hasattr(ns, n)]
    assert len(registered) >= 30
    guarded_elsewhere = {"esimd_qkv_split_norm_rope", "esimd_gdn_conv_fused", "esimd_gdn_conv_fused_seq"}
    for n in registered:
        if n in guarded_elsewhere:
            continue                                  # raising placeholders of the vLLM namespace: must stay absent here
        assert callable(getattr(s, n, None)), n
    for n in IMPORT_NAMES["imp_kernels_names"]:
        assert callable(getattr(s, n, None)), n
    # the MoE batch helpers of torch.ops.moe_ops that the list names and this library registers
    import custom_esimd_kernels_vllm as v
    for n, op in (("moe_router_forward", "moe_router_forward"), ("moe_batch_topk", "moe_topk"),
                  ("moe_accumulate", "moe_accumulate"), ("moe_forward_full", "moe_forward_full")):
        assert n in exports and hasattr(torch.ops.moe_ops, op)
        assert callable(getattr(s, n, None)) and callable(getattr(v, n, None)), n


def test_names_outside_the_path_raise_when_called():
    import custom_esimd_kernels_vllm as v
    import custom_esimd_kernels_sglang as s
    for fn, switch in ((v.esimd_qkv_split_norm_rope, "DISABLE_ESIMD_QKV"),
                       (v.esimd_gdn_conv_fused, "DISABLE_ESIMD_GDN_CONV"),
                       (v.esimd_gdn_conv_fused_seq, "DISABLE_ESIMD_GDN_CONV"),
                       (v.eagle_ops.page_attn_decode, "DISABLE_ESIMD_PA"),
                       (s.eagle_page_attn_decode, "attention backend")):
        with pytest.raises(RuntimeError, match=switch):
            fn(torch.zeros(1))
    # guarded sglang sites must keep falling back: no placeholder may shadow them
    assert not hasattr(s, "esimd_gdn_conv_fused_seq") and not hasattr(s, "esimd_qkv_split_norm_rope")


def _tile(fmt, M, N, K):
    """(rows, columns, slices) that the dense tiled GEMM launches; fmt as in mi_gemm_tiled_shape."""
    out = [ctypes.c_int(0) for _ in range(3)]
    assert capi.lib().mi_gemm_tiled_shape(fmt, M, N, K, *map(ctypes.byref, out)) == 0
    return tuple(v.value for v in out)


def test_k_slices_take_the_tile_that_was_measured_ahead():
    """256 x 64 reads twice the rows of x per workgroup: behind 128 x 128 where x is large beside the weights and a slice short."""
    int4, fp8, q4_k, q4_0, q8_0, q5_k, block = 0, 1, 2, 3, 4, 5, 7
    for fmt, M, N, K in ((q4_0, 1002, 224, 2048), (fp8, 1189, 528, 8192), (block, 1268, 504, 6144), (q8_0, 997, 224, 2048),
                         (q4_0, 961, 392, 2688), (int4, 1234, 336, 4992), (fp8, 898, 344, 3712), (q4_0, 5352, 280, 6144),
                         (int4, 904, 520, 3072), (q4_k, 966, 520, 3072), (block, 904, 520, 3072), (fp8, 501, 960, 3072)):
        assert _tile(fmt, M, N, K)[:2] == (128, 128) and _tile(fmt, M, N, K)[2] > 1, (fmt, M, N, K)
    for fmt, M, N, K in ((q5_k, 145, 7384, 2560), (int4, 387, 1720, 5120), (block, 978, 1720, 6144), (q8_0, 150, 3504, 7552),
                         (q5_k, 1231, 64, 1024), (q8_0, 1955, 192, 2304), (fp8, 488, 1936, 8064), (q4_k, 196, 1400, 4096)):
        assert _tile(fmt, M, N, K)[:2] == (256, 64) and _tile(fmt, M, N, K)[2] > 1, (fmt, M, N, K)
    assert _tile(q5_k, 300, 7384, 2560)[:2] != (256, 64)                 # a third row tile of 128: 256 would pad


def test_tile_query_refuses_what_the_launch_refuses():
    v = [ctypes.c_int(0) for _ in range(3)]
    q = lambda *a: capi.lib().mi_gemm_tiled_shape(*a, *map(ctypes.byref, v))
    assert q(8, 100, 100, 128) == q(-1, 100, 100, 128) == capi.lib().mi_gemm_tiled_shape(0, 100, 100, 128, None, None, None) != 0
    assert q(0, 100, 100, 64) == q(0, 0, 100, 128) == -2
