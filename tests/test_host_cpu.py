"""Host-side checks that need no GPU: the C ABI library loads and exports every
symbol include/xq.h declares; module construction, state names/dtypes/shapes and
error behaviour match the reference's QLoRA modules; nothing runs on CPU tensors."""

import ctypes
import os
import re

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_library_exports_every_declared_symbol():
    from xorl_amd import _C

    hdr = open(os.path.join(ROOT, "include", "xq.h")).read()
    declared = set(re.findall(r"\b(xq_[a-z0-9_]+)\s*\(", hdr))
    assert declared, "no declarations found"
    L = ctypes.CDLL(_C.LIB_PATH)
    for name in sorted(declared):
        assert hasattr(L, name), f"{name} declared in xq.h but not exported"
    assert declared == set(_C.EXPORTS)
    assert b"gfx950" in _C.lib().xq_version()


def test_product_never_imports_the_oracle():
    for base, _, files in os.walk(os.path.join(ROOT, "xorl_amd")):
        for f in files:
            if f.endswith((".py", ".hip", ".h")):
                src = open(os.path.join(base, f)).read()
                assert "oracle" not in src.replace("oracle's", ""), f"{f} mentions the oracle package"


def test_dense_module_state_matches_reference_contract():
    from xorl_amd.qlora import BlockFP8QLoRALinear, Int4QLoRALinear, NF4QLoRALinear, NvFP4QLoRALinear, QLoRALinear

    with pytest.raises(TypeError):
        QLoRALinear(8, 8)
    m = BlockFP8QLoRALinear(576, 384, r=16, lora_alpha=32)      # 576: partial edge tile of scales
    assert m.packed_weight_f32.dtype == torch.float32 and tuple(m.packed_weight_f32.shape) == (384, 144)
    assert not m.packed_weight_f32.requires_grad
    assert m.weight_block_scales.dtype == torch.uint8 and tuple(m.weight_block_scales.shape) == (3, 5 * 4)
    assert m.lora_A.dtype == torch.float32 and tuple(m.lora_A.shape) == (16, 576)
    assert tuple(m.lora_B.shape) == (384, 16) and torch.count_nonzero(m.lora_B) == 0
    assert m.weight is None and m.bias is None and m.scaling == 2.0
    assert m.quant_format == "block_fp8" and m.quant_group_size == 128
    assert m.adapter_gradient_producer_family == "module_managed" and m.fsdp_requires_full_precision
    assert set(m.get_quantized_state_dict()) == {"packed_weight_f32", "weight_block_scales"}
    assert set(m.get_lora_state_dict()) == {"lora_A", "lora_B"}
    n = NvFP4QLoRALinear(64, 32)
    assert tuple(n.packed_weight_f32.shape) == (32, 8) and tuple(n.weight_global_scale.shape) == (4,)
    assert tuple(n.weight_block_scales.shape) == (32, 16)
    i4 = Int4QLoRALinear(256, 32)
    assert tuple(i4.weight_scales.shape) == (32, 4) and i4._scale_dtypes["weight_scales"] == torch.bfloat16
    n4 = NF4QLoRALinear(256, 32)
    assert n4.quant_group_size == 64 and tuple(n4.packed_weight_f32.shape) == (32, 32)
    assert tuple(n4.weight_scales.shape) == (32, 16) and n4._scale_dtypes["weight_scales"] == torch.float32
    with pytest.raises(NotImplementedError):
        n4._load_prequantized(lambda k: None)
    with pytest.raises(ValueError):
        m.set_runtime_lora_config(17, 1)


def test_from_module_roundtrip_and_model_dtype_move():
    from xorl_amd.qlora import QLoRALinear

    lin = torch.nn.Linear(256, 128, bias=True)
    for fmt in ("block_fp8", "nvfp4", "int4", "nf4"):
        q = QLoRALinear.from_module(lin, r=8, lora_alpha=16, quant_format=fmt)
        assert q.quant_format == fmt and torch.equal(q.bias, lin.bias)
        packed = q.packed_weight_f32.detach().clone()
        q.to(torch.bfloat16)                              # must not touch packed bytes / fp32 masters
        assert q.packed_weight_f32.dtype == torch.float32
        assert torch.equal(q.packed_weight_f32.detach().view(torch.int32), packed.view(torch.int32))   # bytes, NaN-safe
        assert q.lora_A.dtype == torch.float32
        assert q._read_packed_weight_uint8().dtype == torch.uint8
        q.packed_weight_f32.data = q.packed_weight_f32.data.to(torch.bfloat16)
        with pytest.raises(RuntimeError, match="expected float32"):
            q._read_packed_weight_uint8()
    with pytest.raises(ValueError):
        QLoRALinear.from_module(lin, quant_format="mxfp4")


def test_from_quantized_and_delta_weight():
    from xorl_amd import quantize as Q
    from xorl_amd.qlora import QLoRALinear

    w = torch.randn(128, 256) * 0.02
    fp8, s = Q.block_fp8_quantize_gkn(w)
    q = QLoRALinear.from_quantized(fp8, weight_block_scales=s, in_features=256, out_features=128, r=4, lora_alpha=8,
                                   quant_format="block_fp8")
    assert q._is_prequantized and q._scale_dtypes["weight_block_scales"] == torch.float32
    assert torch.equal(q._read_packed_weight_uint8().reshape(128, 256), fp8.view(torch.uint8))
    with torch.no_grad():
        q.lora_B.normal_()
    d = q.get_delta_weight()
    assert torch.allclose(d, (q.lora_B @ q.lora_A) * 2.0)


def test_no_cpu_fallback():
    from xorl_amd import quantize as Q
    from xorl_amd.qlora import BlockFP8QLoRALinear

    m = BlockFP8QLoRALinear(128, 64)
    with pytest.raises((RuntimeError, NotImplementedError)):
        m(torch.zeros(2, 128, dtype=torch.bfloat16))
    with pytest.raises(RuntimeError):
        Q.block_fp8_dequantize_gkn(torch.zeros(128, 128).to(torch.float8_e4m3fn), torch.ones(1, 1))


def test_moe_module_state_matches_reference_contract():
    from xorl_amd.qlora import BlockFP8QLoRAMoeExperts, NvFP4QLoRAMoeExperts, QLoRAMoeExperts

    with pytest.raises(TypeError):
        QLoRAMoeExperts(2, 2, 64, 64)
    m = BlockFP8QLoRAMoeExperts(4, 4, 128, 256, r=8, lora_alpha=16)
    shapes = {n: tuple(p.shape) for n, p in m.named_parameters()}
    assert shapes == {"gate_proj_lora_A": (1, 256, 8), "gate_proj_lora_B": (4, 8, 128),
                      "up_proj_lora_A": (1, 256, 8), "up_proj_lora_B": (4, 8, 128),
                      "down_proj_lora_A": (4, 128, 8), "down_proj_lora_B": (1, 8, 256)}
    assert m._skip_fsdp and m._qlora_expected_skip_keys == {"gate_proj", "up_proj", "down_proj"}
    assert m.gated and m.hidden_act == "silu" and m.hidden_dim == 256 and m.swiglu_limit == 0.0
    m.load_weights(torch.randn(4, 256, 128) * 0.02, torch.randn(4, 256, 128) * 0.02, torch.randn(4, 128, 256) * 0.02)
    assert m.gate_packed.dtype == torch.uint8 and tuple(m.gate_packed.shape) == (4, 256, 128)
    assert tuple(m.down_block_scales.shape) == (4, 1, 2 * 4)
    n = NvFP4QLoRAMoeExperts(4, 4, 128, 256, hybrid_shared=False, target_modules=["down_proj"])
    assert [k for k, _ in n.named_parameters()] == ["down_proj_lora_A", "down_proj_lora_B"]
    assert tuple(n.gate_proj_lora_A.shape) == (4, 256, 16) and not n.gate_proj_lora_A.requires_grad
    with pytest.raises(ValueError):
        BlockFP8QLoRAMoeExperts(4, 4, 128, 256, target_modules=["q_proj"])
    with pytest.raises(ValueError):
        BlockFP8QLoRAMoeExperts(2, 4, 128, 256)          # expert parallel shards are out of scope


@pytest.mark.parametrize("M,steps", [(1, 32), (16, 32), (17, 16), (32, 16), (33, 8), (64, 8)])
def test_skinny_plan_holds_any_contraction(M, steps):
    """A K split of the streaming forward keeps at most `steps` 128-element steps of x in LDS, so a contraction of K needs at
    least K / 128 / steps splits, each with an fp32 partial sum in the workspace -- also beyond 64 of them."""
    from xorl_amd import _C

    N = 1024
    for splits in (1, 63, 64, 65, 100):
        for K in (128 * steps * splits - 128, 128 * steps * splits, 128 * steps * splits + 128):
            if K >= 1024:
                need = -(-K // (128 * steps)) * M * N * 4 + K // 128 * M * 16 * 4
                assert _C.lib().xq_linear_workspace_bytes(M, N, K, 16) >= need, (M, K)


def test_workspace_holds_an_image_only_where_the_format_uses_one():
    """Several forwards in one call know their weights, the _fmt queries the format: room for a decoded weight (two bytes an element)
    is asked for 4-bit weights from 640 rows on and for block-fp8 ones from 6144 on; without a format it is the largest of all."""
    from xorl_amd import _C

    L, N, K = _C.lib(), 12288, 4096
    image = 2 * N * K
    for M in (639, 640, 2048, 6143, 6144, 8192):
        sizes = {}
        for fmt, code in _C.FORMATS.items():
            sizes[fmt] = s = [L.xq_linear_workspace_bytes_fmt(code, M, N, K, 16), L.xq_linear_fwd_swiglu_workspace_bytes_fmt(code, M, N, K, 16) - 2 * M * N,
                              L.xq_mlp_workspace_bytes_fmt(code, M, K, N, 16, 0), L.xq_mlp_infer_workspace_bytes_fmt(code, M, K, N, 16) - 6 * M * N]
            w = _C.XqWeight()
            w.format, w.rows, w.cols, w.num_experts = code, N, K, 1
            job = _C.XqLinearJob(ctypes.pointer(w), None, None, 16, 1.0, None, None, N)
            s.append(L.xq_linear_fwd_multi_workspace_bytes(ctypes.byref(job), 1, M))
            for b in s:
                assert (b >= image) == (M >= (6144 if fmt == "block_fp8" else 640)), (fmt, M, s)
            bwd = L.xq_mlp_workspace_bytes_fmt(code, M, K, N, 16, 1)
            assert bwd <= L.xq_mlp_workspace_bytes(M, K, N, 16, 1)
            sizes[fmt].append(bwd)
        any_fmt = [L.xq_linear_workspace_bytes(M, N, K, 16), L.xq_linear_fwd_swiglu_workspace_bytes(M, N, K, 16) - 2 * M * N,
                   L.xq_mlp_workspace_bytes(M, K, N, 16, 0), L.xq_mlp_infer_workspace_bytes(M, K, N, 16) - 6 * M * N]
        assert any_fmt == [max(s[i] for s in sizes.values()) for i in range(4)]
        assert L.xq_mlp_workspace_bytes(M, K, N, 16, 1) == max(s[5] for s in sizes.values())


def test_build_refuses_scratch_under_hand_counted_reads():
    """Kernels that read LDS from inline assembly may not spill; the build reads that from the compiler's remarks."""
    from xorl_amd.csrc import build as b

    guarded = b.asm_read_kernels()
    assert {"gemm_dec_kernel", "gemm_dtl16_kernel"} <= set(guarded)
    tag = " [-Rpass-analysis=kernel-resource-usage]"

    def output(name, scratch):
        lines = ["In file included from a.hip:2:"]
        for what in (f"Function Name: {name}", "    VGPRs: 256", f"    ScratchSize [bytes/lane]: {scratch}", "    VGPRs Spill: 0"):
            lines += [f"a.h:9:1: remark: {what}{tag}", "    9 | __global__ void", "      | ^"]
        return "\n".join(lines)

    dec, other = "_ZN2xq15gemm_dec_kernelILb0ELi8ELi5EEEvNS_8G256ArgsE", "_ZN2xq14lowrank_kernelILi1EEEvi"
    text = "\n".join([output(other, 128), output(dec, 0), "In file included from a.hip:3:", "b.h:1:1: warning: unused", "    1 | int x;", "      | ^"])
    remarks, rest = b._split_remarks(text)
    assert rest.splitlines() == ["In file included from a.hip:3:", "b.h:1:1: warning: unused", "    1 | int x;", "      | ^"]
    b.check_scratch(remarks, guarded)
    with pytest.raises(RuntimeError, match="gemm_dec_kernel"):
        b.check_scratch(b._split_remarks(output(other, 0) + "\n" + output(dec, 80))[0], guarded)


def test_build_finds_every_kernel_that_reads_lds_from_assembly():
    """Whatever a kernel's attributes and parameters; a __global__ function whose name is not found stops the build."""
    from xorl_amd.csrc import build as b

    assert {"gemm_bank_kernel", "gemm_dec_kernel", "gemm_dtl16_kernel"} <= set(b.asm_read_kernels())
    text = """// a __global__ void in a comment
    template <bool A> __global__ void __launch_bounds__(256, 2) one_kernel(std::conditional_t<A, Pair, Args> args) {}
    static __global__ void __launch_bounds__(Geo<int>::nt()) two_kernel(const float* __restrict__ p,
                                                                        int n) {}
    __global__ __launch_bounds__(64) void three_kernel() {}"""
    assert b.kernels_in(text) == ["one_kernel", "two_kernel", "three_kernel"]
    with pytest.raises(RuntimeError, match="not found"):
        b.kernels_in(text + " extern \"C\" __global__ auto four_kernel() -> void {}")


def test_build_refuses_m0_beside_loads_that_take_it():
    """gemm_bank_kernel writes M0 in one assembly statement and loads with it in others: nothing of the compiler's may touch it."""
    from xorl_amd.csrc import build as b

    guarded = b.asm_m0_kernels()
    assert guarded == ["gemm_bank_kernel"]

    def listing(name, line):
        return f"""{name}:                ; @{name}
; %bb.0:
\t;;#ASMSTART
\ts_mov_b32 m0, s7
\ts_nop 0
\t;;#ASMEND
\tv_add_u32_e32 v1, s4, v0              ; not m0
{line}
\t;;#ASMSTART
\tglobal_load_lds_dwordx4 v1, s[8:9] offset:1024
\t;;#ASMEND
\ts_endpgm
.Lfunc_end0:
\t.size\t{name}, .Lfunc_end0-{name}
"""
    bank, other = "_ZN2xq16gemm_bank_kernelILi2ELb1ELb1EEEvNS_8G256ArgsE", "_ZN2xq14lowrank_kernelILi1EEEvi"
    b.check_m0(listing(other, "\ts_mov_b32 m0, -1") + listing(bank, "\tv_mov_b32_e32 v2, 0"), guarded)
    with pytest.raises(RuntimeError, match="m0, s3"):
        b.check_m0(listing(other, "") + listing(bank, "\ts_mov_b32 m0, s3"), guarded)


@pytest.mark.parametrize("K,near", [(1152, 2), (2048, 1)])     # a depth of the streaming kernels and one of the one-launch kernels (to 16 rows)
def test_rows_of_x_far_apart_leave_the_streaming_kernels(K, near):
    """Their addresses within eight rows are 32 bits wide: 2 * 7 * ldx bytes and a row's 128 at most.  One row has no pitch."""
    from tests.util_cases import skinny_route

    route = lambda M, ldx: skinny_route("int4", 512, K, M, ldx)[0]
    for M in (1, 2, 3, 8, 9, 16, 17, 64):
        here = near if M <= 16 else 2
        assert route(M, K) == here and route(M, (1 << 28) - 8) == here, M
        for ldx in (1 << 28, 306783384, 1 << 30, 1 << 31, 1 << 33):
            want = here if M == 1 or here == 1 else 0
            assert route(M, ldx) == want, (M, ldx)
    assert 2 * 7 * ((1 << 28) - 8) + 128 < 1 << 32
    assert route(65, K) == 0


def test_streaming_plans_know_the_storage():
    """What a storage allows (int4 with fp32 scales holds two row tiles) and what its codes cost (nf4's are looked up) decide its own K
    splits, and every workspace holds the sums of the plan with the most."""
    from tests.util_cases import skinny_route
    from xorl_amd import _C

    assert skinny_route("int4", 4096, 12288, 64, 12288, _C.XQ_SCALE_F32)[1:] == (2, 2) != skinny_route("int4", 4096, 12288, 64, 12288)[1:]
    assert skinny_route("nf4", 12288, 8192, 64, 8192)[1:] != skinny_route("int4", 12288, 8192, 64, 8192)[1:]
    for N, K in ((1024, 1024), (4096, 4096), (4096, 12288), (13056, 4992), (16384, 2048)):
        for M in (1, 17, 33, 64):
            for fmt, sdt, most in (("int4", None, 8), ("int4", _C.XQ_SCALE_F32, 2), ("nvfp4", _C.XQ_SCALE_F32, 2), ("nf4", None, 8), ("block_fp8", None, 8)):
                where, splits, tiles = skinny_route(fmt, N, K, M, K, sdt)
                assert 1 <= tiles <= most if where == 2 else where == 1, (fmt, sdt, N, K, M)
                assert _C.lib().xq_linear_workspace_bytes_fmt(_C.FORMATS[fmt], M, N, K, 16) >= splits * M * N * 4 + (K // 128) * M * 16 * 4
    assert [_C.lib().xq_linear_workspace_bytes(0, 1024, K, 16) > 0 for K in (64, 128, 4096)] == [True] * 3      # (no rows, no plan)


def test_banks_get_the_tiles_of_the_kernel_that_takes_them():
    """128 x 256 tiles, and their rule, are gemm_bank_kernel's: a bank, a contraction or a switch that keeps a launch off that kernel leaves it the
    rule of the 256 x 256 tiles, from 400 rows an expert on (block-fp8: 100)."""
    from tests.util_cases import bank_route
    from xorl_amd import _C

    E, H, I = 128, 2048, 768
    per = (8, 64, 200, 500)
    routes = lambda fmt, K=H, **kw: [bank_route(fmt, E, K, I, n * E, True, joint=True, **kw) for n in per]
    assert routes("nvfp4") == ["half"] * 4 and routes("block_fp8") == ["half"] * 4
    assert routes("nvfp4", scale_dtype=_C.XQ_SCALE_F32) == ["128", "128", "128", "256"] == routes("nf4")
    assert routes("nvfp4", kept=True) == ["128", "128", "128", "256"]
    assert routes("block_fp8", kept=True) == ["128", "128", "half", "half"]
    assert routes("block_fp8", K=128) == ["128", "128", "256", "256"]          # two K-steps
    assert routes("nvfp4", K=128) == ["128", "128", "128", "256"]
    try:
        _C.check(_C.lib().xq_set_fp8_direct_tiles(0))
        assert routes("block_fp8") == ["128", "128", "256", "256"]
        assert routes("nvfp4") == ["half"] * 4                              # (the switch is block-fp8's)
    finally:
        _C.check(_C.lib().xq_set_fp8_direct_tiles(1))
    # 640 columns are no whole tiles of 256: two banks side by side take small ones where one alone does ((4 + 64) 640 / 256 tiles, of 256)
    assert bank_route("nvfp4", E, H, 640, 64 * E, True) == "half"
    assert bank_route("nvfp4", E, H, 640, 4 * E, True) == bank_route("nvfp4", E, H, 640, 4 * E, True, joint=True) == "128"


@pytest.mark.parametrize("M,joint", [(1000, True), (300, False)])
@pytest.mark.parametrize("field", ["su_gate_up", "su_down"])
def test_mlp_forward_refuses_misaligned_intermediates(M, joint, field):
    """Before anything is launched, whether gate and up share a launch or not (a call that reaches the device would not fail by this message)."""
    import ctypes

    from tests.util_cases import gate_up_joint
    from xorl_amd import _C

    H, I, r = 320, 9280, 8
    assert gate_up_joint(M, H, I) == joint

    def weight(n, k):
        w = _C.XqWeight()
        w.format, w.layout, w.rows, w.cols, w.num_experts, w.group, w.scale_dtype = _C.FORMATS["block_fp8"], _C.XQ_LAYOUT_FLAT, n, k, 1, 128, _C.XQ_SCALE_F32
        w.packed = w.scales = 4096
        return w
    ws = [weight(I, H), weight(I, H), weight(H, I)]
    lora, S = _C.XqMlpLora(), _C.XqMlpSaved()
    for p in range(3):
        lora.A[p] = lora.B[p] = 4096
    lora.dtype, lora.r, lora.scaling = _C.XQ_DT_F32, r, 1.0
    S.gate_up = S.h = S.su_gate_up = S.su_down = 4096
    setattr(S, field, 4096 + 8)
    L = _C.lib()
    with pytest.raises(_C.XqError, match="su_gate_up and su_down .* 16-byte aligned"):
        _C.check(L.xq_mlp_fwd(*(ctypes.byref(w) for w in ws), ctypes.byref(lora), 4096, H, M, 4096, H, ctypes.byref(S), 4096,
                              L.xq_mlp_workspace_bytes(M, H, I, r, 0), None))


def test_bank_tile_tests_reach_the_kernel():
    """The shapes of tests/test_gpu_moe.py::test_bank_tiles_vs_fp32 in both directions (three, four, seven and 130 K-steps forward: the last loads
    block scales twice)."""
    from tests.util_cases import bank_route

    counts = [128, 0, 1, 127, 129, 16, 113, 300, 0, 240] * 8
    for K, N in ((192, 320), (256, 832), (448, 768), (8320, 256)):
        here = counts + [0, 300] * 100 if K == 192 else counts
        for fmt in ("block_fp8", "nvfp4"):
            assert [bank_route(fmt, len(here), K, N, sum(here), fwd) for fwd in (True, False)] == ["half", "half"], (fmt, K, N)


def test_saved_of_a_routed_forward_is_as_callers_built_it():
    """xq_grouped_saved is filled by callers (thirteen words): a library that reads further reads what they never wrote.  Which forward is meant
    is said by the entry point."""
    import ctypes
    import os
    import subprocess

    from xorl_amd import _C

    assert ctypes.sizeof(_C.XqGroupedSaved) == 13 * 8
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    code = '#include "xq.h"\n_Static_assert(sizeof(xq_grouped_saved) == 13 * 8, "grown");\n'
    subprocess.run(["gcc", "-x", "c", "-fsyntax-only", "-I", os.path.join(root, "include"), "-"], input=code, text=True, check=True)
    assert [hasattr(_C.lib(), f"xq_grouped_fwd{kind}_ids") for kind in ("", "_eval", "_infer")] == [True] * 3
