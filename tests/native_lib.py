"""ctypes bindings to tests/native/libshim.so: the library's C++ parts that no
C entry point shows."""
import ctypes as C
import os
import subprocess

import pytest

from cardioid_amd import build as B
from cardioid_amd import hip

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native")
PATH = os.path.join(HERE, "libshim.so")
_shim = None


def build():
    subprocess.run(["make", "-s", "-C", HERE], check=True)


def shim():
    global _shim
    if _shim is None:
        hip.lib()
        if not os.path.exists(PATH):
            build()
        _shim = C.CDLL(PATH)
    return _shim


def check(rc):
    assert rc == 0, hip.lib().cdh_last_error()


def device_code(source, tmp_path, *flags):
    """The device code of a small HIP source that includes the library's
    headers, compiled with the library's flags, as text."""
    try:
        hipcc = B.hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    src, out = tmp_path / "k.hip", tmp_path / "k.s"
    src.write_text(source)
    common = [f for f in B.COMMON if f not in ("-fPIC", "-fopenmp")]
    subprocess.run([hipcc, *common, *flags, "-I", B.CSRC, "-S", "--cuda-device-only", str(src),
                    "-o", str(out)], check=True, capture_output=True)
    return out.read_text()
