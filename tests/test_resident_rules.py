"""The resident form's rules that need no device (csrc/resident_rules.hpp) by
the library's own functions, and the code of its wait."""
import ctypes as C

import numpy as np
import pytest

import native_lib
from test_tile_links import NODES


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


@pytest.mark.parametrize("dims,dens,seed", [((1, 1, 1), 1.0, 0), ((64, 1, 1), 1.0, 0),
                                            ((1, 1, 130), 1.0, 0), ((7, 8, 9), 1.0, 0),
                                            ((3, 5, 200), 1.0, 0), ((200, 5, 3), 0.8, 1),
                                            ((4, 90, 4), 0.6, 2), ((20, 21, 22), 0.15, 3),
                                            ((20, 21, 22), 0.9, 4), ((6, 6, 65), 0.02, 5)])
def test_tile_ranges_hold_every_neighbour(shim, dims, dens, seed):
    """The ranges that the kernel's own function finds hold every tile that
    owns a neighbour of one of the tile's cells, and whom a tile reads waits
    for it too, so that no tile writes the box a neighbour still reads."""
    t = np.random.default_rng(seed).random(dims) < dens
    if not t.any():
        t[0, 0, 0] = True
    x, y, z = np.nonzero(t)                       # box order: z fastest
    plane, row = (dims[1] + 2) * (dims[2] + 2), dims[2] + 2
    bi = ((x + 1) * plane + (y + 1) * row + (z + 1)).astype(np.int64)
    ntile = (bi.size + 63) // 64
    out = np.zeros((ntile, 3, 2), np.int32)
    shim.shim_tile_ranges(C.c_int64(bi.size), bi.ctypes.data_as(C.c_void_p), C.c_int64(plane),
                          C.c_int64(row), out.ctypes.data_as(C.c_void_p))
    assert (out[..., 0] >= 0).all() and (out[..., 0] <= out[..., 1]).all() and out.max() <= ntile
    tile_of = {int(b): k // 64 for k, b in enumerate(bi)}
    for k, b in enumerate(bi):
        for dx, dy, dz in NODES:
            n = tile_of.get(int(b + dx * plane + dy * row + dz))
            if n is not None:
                assert any(f <= n < e for f, e in out[k // 64]), (k, n)
                assert any(f <= k // 64 < e for f, e in out[n]), (k, n)


WAIT = """
#include "engine_resident.hpp"
__global__ void k_wait(cdh::ResidentArgs r, const uint32_t *lk, uint32_t target, int *out)
{
   bool bail = false;
   cdh::resident_wait(r, lk, threadIdx.x, target, bail);
   out[0] = bail;
}
"""


def test_the_bound_of_a_wait_is_no_time_of_day(tmp_path):
    """A clock goes on while a process is held off the chip, for which a wait
    must not fail: it reads none and counts its polls."""
    code = native_lib.device_code(WAIT, tmp_path)
    assert "k_wait" in code and "global_load" in code
    assert "s_memrealtime" not in code and "s_memtime" not in code
