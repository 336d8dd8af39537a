"""A resident tile's wait past its bound: the error, and what follows it.  The
first tile is made to wait for a flag that nobody advances, so that the
kernel's own bound ends the wait and every launch exits."""
import time

import numpy as np
import pytest

import native_lib
from cardioid_amd import hip
from test_gpu_resident import make, results, slab

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
POLLS = 1_000_000                 # some 0.16 s


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    hip.lib()
    yield


def stuck(mode, s):
    """A batch holding slab s (its id) whose resident runs time out."""
    b = make([s], mode, False)
    i = b.add(s)
    b.run(8)
    b.sync()
    assert b.resident()["steps"] == 8
    native_lib.check(native_lib.shim().shim_resident_stuck(b.h, POLLS))
    return b, i


# few tiles: six wavefronts to a tile, 1,024 steps a launch; many: one, 256 steps
SIZES = [("mixed_fused", (9, 10, 11), 1024), ("fp64_fma", (5, 6, 70), 1024),
         ("fp64_fused", (40, 42, 44), 256), ("mixed_fused", (40, 42, 44), 256)]


@pytest.mark.parametrize("mode,dims,launch", SIZES)
def test_later_launches_do_not_wait_again(mode, dims, launch):
    took = []
    for launches in (1, 10):
        b, _ = stuck(mode, slab(*dims))
        t = time.perf_counter()
        with pytest.raises(hip.CardioidHipError, match="waited past its bound"):
            b.run(launches * launch)
            b.sync()
        took.append(time.perf_counter() - t)
        print(f"{launches} launches, the first times out: {took[-1]:.3f} s, "
              f"{took[-1] / POLLS * 1e6:.3f} us a poll", flush=True)
        b.close()
    assert took[1] < 3 * took[0], took


def test_a_timed_run_is_an_error_too():
    """It used to return a time for states that are not valid."""
    b, _ = stuck("mixed_fused", slab(9, 10, 11))
    with pytest.raises(hip.CardioidHipError, match="waited past its bound"):
        b.run_timed(40)
    b.close()


@pytest.mark.parametrize("mode,dims", [("mixed_fused", (9, 10, 11)), ("fp64_fma", (40, 42, 44))])
def test_the_engine_goes_on_once_the_slab_is_replaced(mode, dims):
    """The failure belongs to the slabs that took part: they stay an error
    until they leave, and what is added after runs as in a fresh engine."""
    s, t = slab(*dims, phi=-30.0), slab(*dims, phi=15.0)
    b, i = stuck(mode, s)
    b.run(40)
    for call in (b.sync, lambda: b.vm(i), lambda: b.state(i), lambda: b.run(40),
                 lambda: b.run_timed(40), b.sync):
        with pytest.raises(hip.CardioidHipError, match="waited past its bound"):
            call()
    b.remove(i)
    b.sync()
    i = b.add(t)
    steps = b.resident()["steps"]
    b.run(300)
    got = results(b, [i])
    assert b.resident()["steps"] == steps + 300
    b.close()
    fresh = make([t], mode, False)
    j = fresh.add(t)
    fresh.run(300)
    for a, r in zip(got, results(fresh, [j])):
        assert np.array_equal(a, r)
    fresh.close()


def test_a_slab_added_behind_the_failing_run_is_not_lost():
    """Replaced without a sync in between: the new slab took no part."""
    s, t = slab(9, 10, 11), slab(6, 7, 8, phi=15.0)
    b, i = stuck("mixed_fused", s)
    b.run(40)
    time.sleep(1.0)                    # the launch has failed by now
    b.remove(i)
    i = b.add(t)
    b.run(100)
    got = results(b, [i])
    b.close()
    fresh = make([t], "mixed_fused", False)
    j = fresh.add(t)
    fresh.run(100)
    for a, r in zip(got, results(fresh, [j])):
        assert np.array_equal(a, r)
    fresh.close()
