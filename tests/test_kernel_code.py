"""What the compiler makes of a kernel's inner loop, read from its assembly (gfx950, built here from source)."""
import os
import re
import shutil
import subprocess

import pytest

from vipera_rs_amd.ops import build


@pytest.fixture(scope="module")
def gemm_generic_code(tmp_path_factory):
    if not shutil.which("hipcc") and not os.path.exists("/opt/rocm/bin/hipcc"):
        pytest.skip("needs hipcc")
    out = str(tmp_path_factory.mktemp("code") / "gemm_generic.s")
    flags = [flag for flag in build.HIP_FLAGS if flag not in ("-shared", "-fPIC")]
    subprocess.run([build._hipcc(), *flags, "--cuda-device-only", "-S", os.path.join(build._CSRC, "kernels", "gemm_generic.hip"), "-o", out],
                   check=True, capture_output=True)
    code = {}
    for name, body in re.findall(r"^(_ZN\S*gemm_matrix_kernel\S*):[^\n]*\n(.*?)\.Lfunc_end", open(out).read(), re.S | re.M):
        types, units, vector = re.search(r"gemm_matrix_kernelI(.*?)Lb\dELi(\d)ELb(\d)E", name).groups()
        code[name] = (types.startswith("ff"), int(units), vector == "1", body)      # both operands 32-bit, how K is cut, wide loads
    assert {units for _, units, _, _ in code.values()} == {0, 1, 4}
    return code


def test_the_32_bit_product_keeps_its_sums_in_place_from_step_to_step(gemm_generic_code):
    """No move between the two register files in the basic blocks that hold the matrix instructions: a product of 2,048 x
    37,888 x 3,584 takes half as long again with them."""
    for name, (_, _, _, body) in gemm_generic_code.items():
        blocks = [b for b in re.split(r"^(?:\.LBB|\s+s_cbranch|; %bb)[^\n]*\n", body, flags=re.M) if "v_mfma" in b]
        assert blocks and not any("v_accvgpr" in b for b in blocks), name


def test_whole_steps_of_an_odd_k_are_read_in_wide_loads(gemm_generic_code):
    """Rows off 16-byte boundaries: a load a number is for a row's last step only (2,001 x 9,942 x 7,950: 6.3 ms with one
    everywhere, 3.6 ms)."""
    for name, (both_32_bit, _, wide, body) in gemm_generic_code.items():
        if both_32_bit and not wide:
            assert body.count("global_load_dwordx4") >= 2, name


@pytest.fixture(scope="module")
def gemm_bf16_code(tmp_path_factory):
    """The instructions of each kernel of the built library, by its name."""
    tools = os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(build._hipcc()))), "llvm", "bin")
    if not os.path.exists(os.path.join(tools, "clang-offload-bundler")):
        pytest.skip("needs ROCm's binary tools")
    folder = tmp_path_factory.mktemp("library")
    bundle, code = str(folder / "bundle"), str(folder / "code")
    library = build.library_path("gemm_bf16") or build.compile_module("gemm_bf16")
    for command in (["llvm-objcopy", f"--dump-section=.hip_fatbin={bundle}", library, os.devnull],
                    ["clang-offload-bundler", "--unbundle", "--type=o", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--input={bundle}", f"--output={code}"]):
        subprocess.run([os.path.join(tools, command[0]), *command[1:]], check=True, capture_output=True)
    text = subprocess.run([os.path.join(tools, "llvm-objdump"), "-d", "--no-show-raw-insn", code], check=True, capture_output=True, text=True).stdout
    return dict(re.findall(r"^[0-9a-f]+ <(_ZN\S+)>:\n(.*?)(?=^\s*$|\Z)", text, re.S | re.M))


def test_a_tile_with_as_many_stages_of_both_operands_works_out_one_place_a_step(gemm_bf16_code):
    """Where the next step's rows lie is one choice of two (``s_cselect``) for what is read and one for what is asked for; with a
    choice for each operand the 64x64 tiles that add K's ranges themselves took 8 to 10 % longer (512 x 2,048 x 2,048)."""
    loops = 0
    for name, body in gemm_bf16_code.items():
        found = re.search(r"gemm_tile_direct_kernelI(?:Li\d+E){4}(?:f|DF16b)Lb\dELb\dELi(\d)ELb\dELi(\d)E", name)
        if not found or found[1] != found[2]:
            continue
        for block in re.split(r"^\ts_c?branch\S*[^\n]*\n", body, flags=re.M):
            if "v_mfma" in block and re.search(r"buffer_load_dwordx4 .* lds", block):
                loops += 1
                assert block.count("s_cselect") <= 2, name
    assert loops >= 20
