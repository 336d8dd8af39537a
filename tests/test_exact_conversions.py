"""The exponential of the exact functions (csrc/tt06_exact.hpp) on the compiled
code of a small kernel."""
from native_lib import device_code

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
    code = device_code(KERNEL, tmp_path, "-emit-llvm", "-ffp-contract=off")
    assert "k_ex" in code and "llvm.ldexp" in code
    assert "fptosi" not in code and "fptoui" not in code
