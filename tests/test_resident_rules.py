"""The rules of the resident form that need no device (csrc/resident_rules.hpp),
by the library's own functions."""
import pytest

import native_lib


@pytest.fixture(scope="module")
def shim():
    try:
        return native_lib.shim()
    except Exception as e:      # no library built, no compiler
        pytest.skip(f"no shim: {e}")


def test_only_a_launch_too_large_or_unsupported_falls_back(shim):
    """hip_runtime_api.h: 720 cooperative launch too large, 801 not supported;
    an invalid value, no memory, a sticky fault and the rest are errors."""
    refused = {e for e in range(1200) if shim.shim_resident_refused(e)}
    assert refused == {720, 801}
