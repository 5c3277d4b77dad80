"""Host-side mirror of the reference's operator interface: names, defaults, validation and error convention.
Runs without a GPU (nothing is launched)."""

import inspect

import pytest
import torch


def test_public_names_match_the_reference_package():
    import nkilib.core.moe.moe_cte as m

    # src/nkilib_src/nkilib/core/moe/moe_cte/__init__.py:17-36
    for n in ("moe_cte", "MoECTESpec", "MoECTEImplementation", "ShardOnBlockConfig", "ShardOnIConfig",
              "QuantizationConfig", "BlockShardStrategy", "SkipMode"):
        assert hasattr(m, n)
    assert [e.name for e in m.MoECTEImplementation] == [
        "shard_on_block", "shard_on_i", "shard_on_i_hybrid", "shard_on_i_dropping", "shard_on_block_mx",
        "shard_on_i_mx", "shard_on_i_mx_hybrid"]
    assert [e.value for e in m.MoECTEImplementation] == list(range(7))
    from nkilib.core.utils.common_types import ActFnType, ExpertAffinityScaleMode, NormType, QuantizationType

    assert ActFnType.SiLU.value == 0 and ActFnType.Swish.value == 3
    assert ExpertAffinityScaleMode.POST_SCALE.value == 1 and ExpertAffinityScaleMode.PRE_SCALE_DELAYED.value == 3
    assert NormType.RMS_NORM.value == 1 and QuantizationType.ROW.value == 2 and QuantizationType.STATIC.value == 1


def test_moe_cte_signature_is_the_reference_signature_plus_one_keyword():
    from nkilib.core.moe.moe_cte import moe_cte

    params = list(inspect.signature(moe_cte).parameters)
    # src/nkilib_src/nkilib/core/moe/moe_cte/moe_cte.py:253-277
    ref = ["hidden_states", "expert_affinities_masked", "gate_up_proj_weight", "down_proj_weight",
           "token_position_to_id", "block_to_expert", "block_size", "spec", "conditions", "gate_and_up_proj_bias",
           "down_proj_bias", "quantization_config", "gate_up_activations_T", "down_activations",
           "activation_function", "skip_dma", "compute_dtype", "is_tensor_update_accumulating",
           "expert_affinities_scaling_mode", "gate_clamp_upper_limit", "gate_clamp_lower_limit",
           "up_clamp_upper_limit", "up_clamp_lower_limit"]
    assert params[: len(ref)] == ref
    assert params[len(ref):] == ["hidden_states_scale"]
    assert moe_cte[2] is moe_cte  # kernel[lnc](...) launch syntax is accepted
    sig = inspect.signature(moe_cte)
    assert sig.parameters["is_tensor_update_accumulating"].default is True
    assert sig.parameters["expert_affinities_scaling_mode"].default.name == "POST_SCALE"


def test_spec_defaults():
    from nkilib.core.moe.moe_cte import (BlockShardStrategy, MoECTEImplementation, MoECTESpec, ShardOnBlockConfig,
                                         ShardOnIConfig)

    s = MoECTESpec(MoECTEImplementation.shard_on_block_mx)
    assert isinstance(s.shard_on_block, ShardOnBlockConfig) and s.shard_on_I is None
    assert s.shard_on_block.n_dynamic_blocks == 55 and s.shard_on_block.n_static_blocks == -1
    assert s.shard_on_block.block_sharding_strategy == BlockShardStrategy.PING_PONG
    s = MoECTESpec(MoECTEImplementation.shard_on_i_hybrid)
    assert isinstance(s.shard_on_I, ShardOnIConfig) and s.shard_on_I.num_static_block is None


def test_rmsnorm_args_validation():
    from nkilib.core.rmsnorm import RmsNormQuantKernelArgs, rmsnorm_quant_kernel
    from nkilib.core.utils.common_types import NormType, QuantizationType

    a = RmsNormQuantKernelArgs()
    assert a.lower_bound == 0.0 and a.eps == 1e-6 and a.is_row_quant() and a.needs_rms_normalization()
    with pytest.raises(AssertionError, match="NCC_INKI016"):
        RmsNormQuantKernelArgs(quantization_type=QuantizationType.MX)
    with pytest.raises(AssertionError):
        RmsNormQuantKernelArgs(norm_type=NormType.LAYER_NORM)
    with pytest.raises(AssertionError):
        RmsNormQuantKernelArgs(lower_bound=-1.0)
    # shape rules of the reference (rmsnorm_quant.py:174-262), raised before anything touches a device
    with pytest.raises(AssertionError, match="Rank of hidden"):
        rmsnorm_quant_kernel(torch.zeros(8), torch.zeros(8), a)
    with pytest.raises(AssertionError, match="exceeds maximum"):
        rmsnorm_quant_kernel(torch.zeros(1, 2, 16385), torch.zeros(16385), a)
    with pytest.raises(AssertionError, match="ln_w vector length"):
        rmsnorm_quant_kernel(torch.zeros(1, 2, 64), torch.zeros(32), a)
    with pytest.raises(AssertionError, match="input_dequant_scale must be provided"):
        rmsnorm_quant_kernel(torch.zeros(1, 2, 64), torch.zeros(64),
                             RmsNormQuantKernelArgs(quantization_type=QuantizationType.STATIC))


def test_no_cpu_fallback():
    """CPU tensors are rejected loudly; nothing silently computes on the host."""
    from nkilib._native import NativeLibraryError
    from nkilib.core.moe.moe_cte import MoECTEImplementation, MoECTESpec, moe_cte
    from nkilib.core.rmsnorm import RmsNormQuantKernelArgs, rmsnorm_quant_kernel

    with pytest.raises(NativeLibraryError, match="no CPU path"):
        rmsnorm_quant_kernel(torch.zeros(1, 2, 64, dtype=torch.bfloat16), torch.zeros(64, dtype=torch.bfloat16),
                             RmsNormQuantKernelArgs())
    with pytest.raises(NativeLibraryError, match="no CPU path"):
        moe_cte(torch.zeros(9, 64, dtype=torch.bfloat16), torch.zeros(18, 1, dtype=torch.bfloat16),
                torch.zeros(2, 64, 2, 32, dtype=torch.bfloat16), torch.zeros(2, 32, 64, dtype=torch.bfloat16),
                torch.zeros(16, dtype=torch.int32), torch.zeros(2, dtype=torch.int32), 8,
                MoECTESpec(MoECTEImplementation.shard_on_block))


def test_mx_shard_on_i_entry_points_validate_like_the_reference():
    """blockwise_mm_shard_intermediate_mx[_hybrid] exist under the reference's import path, refuse PRE_SCALE with the
    reference's message (bwmm_shard_on_I_mx.py:914-915) and are what the shard_on_i_mx enum members dispatch to."""
    from nkilib.core.moe.moe_cte import MoECTEImplementation, MoECTESpec, moe_cte
    from nkilib.core.moe.moe_cte.bwmm_shard_on_I_mx import (blockwise_mm_shard_intermediate_mx,
                                                            blockwise_mm_shard_intermediate_mx_hybrid)
    from nkilib.core.utils.common_types import ExpertAffinityScaleMode

    z = torch.zeros(1)
    with pytest.raises(AssertionError, match="PRE_SCALE mode not implemented"):
        blockwise_mm_shard_intermediate_mx[2](z, z, z, z, z, z, block_size=256)  # the default mode is PRE_SCALE
    with pytest.raises(AssertionError, match="conditions is required"):
        blockwise_mm_shard_intermediate_mx_hybrid(None, z, z, z, z, z, z, block_size=256)
    with pytest.raises(AssertionError, match="PRE_SCALE mode not implemented"):
        moe_cte(z, z, z, z, z, z, 256, MoECTESpec(MoECTEImplementation.shard_on_i_mx),
                expert_affinities_scaling_mode=ExpertAffinityScaleMode.PRE_SCALE)
    with pytest.raises(AssertionError, match="gate_up_proj_scale and down_proj_scale are required"):
        moe_cte(z, z, z, z, z, z, 256, MoECTESpec(MoECTEImplementation.shard_on_i_mx_hybrid), conditions=z)


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    from nkilib import _native as nv

    monkeypatch.setattr(nv, "_lib", None)
    monkeypatch.setattr(nv, "LIB_PATH", str(tmp_path / "absent.so"))
    with pytest.raises(nv.NativeLibraryError, match="no CPU fallback"):
        nv.lib()


def test_bench_refuses_more_than_one_gpu():
    """bench.py measures one GPU: --gpus N with N > 1 exits with a message that says so (before touching a GPU)."""
    import os
    import subprocess
    import sys

    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    res = subprocess.run([sys.executable, os.path.join(root, "bench.py"), "--gpus", "2"], capture_output=True, text=True,
                         timeout=120)
    assert res.returncode != 0
    assert "one GPU" in res.stderr and res.stdout.strip() == ""


@pytest.mark.parametrize("stage,fmt,H,I,E,k,T,few", [
    # MX gate/up: up to four experts, one round of half tiles, the start of the second
    (1, "e4m3", 7168, 2048, 256, 8, 1, True), (1, "e4m3", 7168, 2048, 256, 8, 2, False),
    (1, "e4m3", 7168, 2048, 256, 8, 32, False), (1, "e5m2", 5120, 1536, 64, 4, 2, True),
    (1, "e4m3", 4096, 14336, 8, 2, 2, True), (1, "e4m3", 4096, 14336, 8, 2, 5, False),
    (1, "e4m3", 7168, 2048, 8, 2, 32, True), (1, "e4m3", 7168, 2048, 8, 2, 33, False),
    # 4-bit weights: these had been sent to the kernel that takes up to twice as long
    (1, "e2m1", 7168, 2048, 256, 8, 2, False), (1, "e2m1", 7168, 2048, 256, 8, 4, False),
    (1, "e2m1", 4096, 2048, 128, 8, 8, False), (1, "e2m1", 3072, 1536, 32, 4, 1, True),
    (1, "e2m1", 4096, 14336, 8, 2, 2, True), (1, "e2m1", 4096, 14336, 8, 2, 4, False),
    (1, "e2m1", 512, 512, 8, 2, 8, True), (1, "e2m1", 512, 512, 8, 2, 9, False),
    (2, "e2m1", 4096, 2048, 128, 8, 32, True), (2, "e2m1", 4096, 2048, 128, 8, 48, False),
    (2, "e2m1", 3072, 1536, 32, 4, 64, True), (2, "e2m1", 3072, 1536, 32, 4, 65, False),
    (2, "e4m3", 7168, 2048, 256, 8, 32, True), (2, "e4m3", 7168, 2048, 256, 8, 33, False),
    # dense kinds
    (1, "bf16", 7168, 2048, 64, 8, 16, True), (1, "bf16", 7168, 2048, 64, 8, 32, False),
    (1, "bf16", 4096, 2048, 64, 4, 32, True), (1, "bf16", 7168, 512, 64, 4, 32, True),
    (1, "bf16", 1024, 768, 60, 4, 64, True), (2, "bf16", 7168, 2048, 64, 8, 64, True),
    (1, "row8", 4096, 2048, 64, 4, 32, True), (1, "row8", 512, 512, 8, 2, 33, False),
    (2, "row8", 7168, 2048, 32, 4, 64, True), (2, "row8", 7168, 2048, 32, 4, 65, False),
    (1, "bf16", 512, 1024, 8, 2, 256, True), (1, "bf16", 512, 1024, 8, 2, 257, False),
    (2, "bf16", 4096, 1024, 8, 2, 256, False),
])
def test_few_rows_rule(stage, fmt, H, I, E, k, T, few):
    """mx_rows_fits (csrc/bwmm_rows.hip) at sizes where both kernels were timed."""
    from nkilib.core.moe.moe_cte import get_n_blocks

    assert _rows_fit(stage, fmt, H, I, E, get_n_blocks(T, k, E, 128), 128, T) is few


@pytest.mark.parametrize("H,I,E,N,B,few", [
    (512, 1024, 8, 1, 256, True), (2048, 1024, 8, 7, 128, True), (2048, 1024, 8, 4, 256, True),
    (1024, 1024, 32, 16, 256, False), (4096, 512, 32, 31, 256, False), (512, 512, 32, 31, 64, True),
])
def test_few_rows_rule_of_a_table_with_fewer_blocks_than_experts(H, I, E, N, B, few):
    """Such a table may hold whole blocks: many chunks of 256 rows are no launch of few rows."""
    assert _rows_fit(1, "bf16", H, I, E, N, B, 256) is few


def _rows_fit(stage, fmt, H, I, E, N, B, rows):
    import ctypes

    from nkilib import _native as nv

    class RowsCall(ctypes.Structure):  # (csrc/bwmm.hpp)
        _fields_ = [(n, ctypes.c_int64) for n in ("rows", "H", "E", "N", "B", "col_tiles", "max_chunks")]

    f = getattr(nv.lib(), "_ZN3moe12mx_rows_fitsEiiRKNS_8RowsCallE")
    f.restype, f.argtypes = ctypes.c_bool, [ctypes.c_int, ctypes.c_int, ctypes.POINTER(RowsCall)]
    tiles = (I + 127) // 128 if stage == 1 else H // 256
    c = RowsCall(rows, H, E, N, B, tiles, N * ((B + 255) // 256))
    return bool(f(stage, ("e4m3", "e5m2", "e2m1", "row8", "bf16").index(fmt), ctypes.byref(c)))


@pytest.mark.parametrize("N,B,I,per_block", [
    (15, 512, 2048, (64, 32)), (2000, 128, 14336, (448, 8)),  # a workgroup per 64 columns, per 16 rows
    (1 << 18, 2, 2048, (4, 1)), (37500, 4, 14336, (27, 1)),   # past a million of them
    ((1 << 24) - 1, 1, 8, (1, 1)),
])
def test_checkpoint_padding_grids_fit_a_launch(N, B, I, per_block):
    """ckpt_grid (csrc/combine.hip): each of the two launches stays below 2^32 threads of 256 to a workgroup."""
    import ctypes

    from nkilib import _native as nv

    class CkptGrid(ctypes.Structure):
        _fields_ = [(n, ctypes.c_int64) for n in ("n_gu", "y_gu", "n_dn", "y_dn")]

    f = nv.lib()._ZN3moe9ckpt_gridElllbb
    f.restype, f.argtypes = CkptGrid, [ctypes.c_int64] * 3 + [ctypes.c_bool] * 2
    g = f(N, B, 2 * I, True, True)
    assert (g.y_gu, g.y_dn) == per_block and (g.n_gu, g.n_dn) == (N * g.y_gu, N * g.y_dn)
    assert max(g.n_gu, g.n_dn) * 256 < 1 << 32
    assert (f(N, B, 2 * I, False, True).n_gu, f(N, B, 2 * I, True, False).n_dn) == (0, 0)


def _build_module():
    import importlib.util
    import os

    path = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nki-library_amd", "build.py")
    spec = importlib.util.spec_from_file_location("moe_build", path)
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    return build


_LOAD = ["s_add_u32 m0, s33, 0xf000", "s_nop 0", "buffer_load_dwordx4 v186, s[60:63], s10 offen lds"]
_MFMA = "v_mfma_f32_16x16x32_bf16 a[0:3], v[8:11], v[12:15], a[0:3]"


@pytest.mark.parametrize("code,ok", [
    (["v_accvgpr_write_b32 a0, 0", "v_accvgpr_read_b32 v5, a3", _MFMA, *_LOAD], True),
    (["v_accvgpr_write_b32 a0, v7", *_LOAD], False),             # a spill into an accumulation register
    (["ds_read_b64 a[4:5], v7", *_LOAD], False),                 # a load into one
    (["v_readfirstlane_b32 s10, v3", "s_nop 1", *_LOAD], False),
    (["v_add_co_u32_e64 v3, s[10:11], v4, v5", *_LOAD], False),
    (["v_readfirstlane_b32 s10, v3", "s_nop 0", "s_nop 0", "s_nop 0", "s_nop 0", "s_nop 0", *_LOAD], True),
    (["v_perm_b32 v9, v3, v4, v5", _MFMA, *_LOAD], False),       # its operand, just written
    (["v_perm_b32 v16, v3, v4, v5", _MFMA, *_LOAD], True),
    (["v_perm_b32 v9, v3, v4, v5", "s_nop 1", _MFMA, *_LOAD], True),
    ([_MFMA], False),                                            # no load of the K loop at all
])
def test_check_of_the_compiled_tile_loops(code, ok):
    """build.check_tile_lines on listings that keep and break what the tile loops rely on."""
    build = _build_module()
    if ok:
        build.check_tile_lines(code, "listing")
    else:
        with pytest.raises(RuntimeError):
            build.check_tile_lines(code, "listing")


def test_build_without_the_listing_tools(tmp_path, monkeypatch):
    """Where LLVM's binary tools are absent the build goes on and says so."""
    monkeypatch.setenv("ROCM_PATH", str(tmp_path))
    build = _build_module()
    assert "not checked" in build.check_tile_code("x.o")
