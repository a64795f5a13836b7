"""What the compiler makes of the library's device helpers, without a GPU (hipcc cross-compiles)."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lrqk_amd", "csrc")
HIPCC = os.environ.get("HIPCC") or shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")

# the accumulator starts with the value of a later operand: a column, the vector, a column known to be zero
ROW_DOT = """
#include "common.hpp"
#include "small_inverse.hpp"
using namespace lrqk;
__global__ void dot16(const float* in, float* out) {
  float col[16];
  for (int i = 0; i < 16; ++i) col[i] = ZERO == i ? 0.0f : in[64 * i + threadIdx.x];
  const float x = in[2048 + threadIdx.x];
  out[threadIdx.x] = START;
}
"""


def _asm(tmp_path, source, *defines):
    src, out = tmp_path / "probe.hip", tmp_path / "probe.s"
    src.write_text(source)
    subprocess.run([HIPCC, "-O3", "-std=c++17", "--offload-arch=gfx950", "--cuda-device-only", "-S", "-I", CSRC,
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", *defines, str(src), "-o", str(out)],
                   check=True, capture_output=True, timeout=300)
    return out.read_text()


@pytest.mark.parametrize("start,zero", [("row_dot16(x, col, col[5])", -1), ("row_dot16(x, col, x)", -1),
                                        ("row_dot16(x, col)", 3)])
def test_row_dot_accumulator_has_a_register_of_its_own(tmp_path, start, zero):
    """Sixteen instructions add to the accumulator and read the operands: it may share a register with none of them, whatever
    values they have."""
    asm = _asm(tmp_path, ROW_DOT, f"-DSTART={start}", f"-DZERO={zero}")
    steps = re.findall(r"v_fmac_f32_dpp (v\d+), (v\d+), (v\d+) row_newbcast", asm)
    assert len(steps) == 16
    assert len({acc for acc, _, _ in steps}) == 1
    acc = steps[0][0]
    assert all(acc not in (x, c) for _, x, c in steps), steps


LIB = os.path.join(os.path.dirname(CSRC), "liblrqk_hip.so")


@pytest.mark.skipif(not os.path.exists(LIB) or not shutil.which("nm"), reason="needs the built library and nm")
def test_gram_pass_is_compiled_for_the_rows_that_reach_it():
    """The factor update's pass on 16-byte pieces: fp32 rows of 32, 64 and 128 elements and bf16 rows of 64 (8, 16, 32 and 8
    pieces).  bf16 rows of 128 have a pass of their own, and those of 256 need more LDS than the pass has."""
    names = subprocess.run(["nm", "-C", LIB], check=True, capture_output=True, text=True).stdout
    assert set(re.findall(r"lrqk::als_gram_vec_kernel<([^>]*)>", names)) == {
        "float, 8", "float, 16", "float, 32", "lrqk::bf16_t, 8"}
