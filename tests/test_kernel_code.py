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
