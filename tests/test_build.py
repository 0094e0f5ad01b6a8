"""What a build is refused for."""
import pytest

from litinfer_amd.kernels import build

NAME = "_Z21gemm_bf16_tile_kernelILi256EEvv"
GOOD = """
{name}: ; @{name}
	v_mov_b32_e32 v0, 0
	v_accvgpr_write_b32 a0, 0
	v_mfma_f32_16x16x32_bf16 a[0:3], v[8:11], v[8:11], 0
.LBB0_1:
	ds_read_b128 v[12:15], v1
	v_add_u32_e32 v2, 64, v2
	s_waitcnt lgkmcnt(0)
	v_mfma_f32_16x16x32_bf16 a[0:3], v[12:15], v[16:19], a[0:3]
	s_cbranch_scc1 .LBB0_1
	s_nop 15
	s_nop 15
	v_accvgpr_read_b32 v0, a0
	s_endpgm
	.amdhsa_kernel {name}
		.amdhsa_private_segment_fixed_size 0
	.end_amdhsa_kernel
""".format(name=NAME)


def test_the_assembly_of_the_tiles_in_pieces_is_looked_through():
    assert build.tile_kernel_faults(GOOD) == []
    loop = "	s_waitcnt lgkmcnt(0)\n"
    for line, what in (("	v_accvgpr_read_b32 v9, a2\n", "a sum moves"), ("	v_accvgpr_mov_b32 a4, a0\n", "a sum moves"), ("	ds_write_b32 v1, a3\n", "a sum moves"),
                       ("	scratch_store_dword off, v3, off\n", "scratch"), ("	v_mov_b32_e32 v13, v40\n", "an operand written right before"),
                       ("	v_mov_b64_e32 v[18:19], v[40:41]\n", "an operand written right before")):
        faults = build.tile_kernel_faults(GOOD.replace(loop, loop + line))
        assert faults and all(NAME in f for f in faults) and what in faults[0], line
    assert "scratch" in build.tile_kernel_faults(GOOD.replace("fixed_size 0", "fixed_size 16"))[0]
    assert "no wait" in build.tile_kernel_faults(GOOD.replace("	s_nop 15\n", "", 1))[0]
    assert build.tile_kernel_faults(GOOD.replace("gemm_bf16_tile", "gemm_bf16_dma")) and build.tile_kernel_faults(GOOD.replace("	.end_amdhsa_kernel\n", ""))


def test_a_library_whose_assembly_is_not_sound_is_not_built(monkeypatch, tmp_path):
    try:
        build._hipcc()
    except build.KernelBuildError:
        pytest.skip("no compiler")
    (tmp_path / "csrc").mkdir()
    (tmp_path / "lib").mkdir()
    (tmp_path / "csrc" / "gemm.hip").write_text("#include <hip/hip_runtime.h>\n__global__ void k(float* x) { x[threadIdx.x] = 1.f; }\n")
    monkeypatch.setattr(build, "CSRC", tmp_path / "csrc")
    monkeypatch.setattr(build, "_writable_dir", lambda: tmp_path / "lib")
    with pytest.raises(build.KernelBuildError, match="not sound"):
        build.compile_module("gemm", verbose=False)
    assert list((tmp_path / "lib").iterdir()) == []
    seen = []
    monkeypatch.setitem(build.CHECKS, "gemm", lambda assembly: seen.append(assembly) or [])
    assert build.compile_module("gemm", verbose=False).exists() and len(seen) == 1 and "s_endpgm" in seen[0]
