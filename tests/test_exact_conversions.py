"""The exponential of the exact functions (csrc/tt06_exact.hpp) on the compiled
code of a small kernel."""
import os
import subprocess

import pytest

from cardioid_amd import build as B

KERNEL = """
#include "tt06_exact.hpp"
__global__ void k_ex(const cdh::TT06ExactConst *E, const double *x, double *y)
{
   y[threadIdx.x] = cdh::ExactMath<const cdh::TT06ExactConst>{E}.ex(x[threadIdx.x]);
}
"""


def test_exponent_conversion_is_defined_for_every_argument(tmp_path):
    """At a clamped voltage of +-1e7 the exponent of a squared argument reaches
    6e11, and NaN goes through: the conversion to an integer must not be the
    language's, whose result is undefined there."""
    try:
        hipcc = B.hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    src, out = tmp_path / "k.hip", tmp_path / "k.ll"
    src.write_text(KERNEL)
    flags = [f for f in B.COMMON if f not in ("-fPIC", "-fopenmp")]
    subprocess.run([hipcc, *flags, "-ffp-contract=off", "-I", B.CSRC, "-S", "-emit-llvm",
                    "--cuda-device-only", str(src), "-o", str(out)], check=True,
                   capture_output=True, cwd=os.path.dirname(B.CSRC))
    code = out.read_text()
    assert "k_ex" in code and "llvm.ldexp" in code
    assert "fptosi" not in code and "fptoui" not in code
