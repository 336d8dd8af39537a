"""ctypes bindings to tests/native/libshim.so: the library's C++ parts that no
C entry point shows."""
import ctypes as C
import os
import subprocess

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
