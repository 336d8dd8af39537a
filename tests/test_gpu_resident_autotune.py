"""The autotune and the resident form."""
import numpy as np
import pytest

from cardioid_amd import hip
from test_gpu_resident import make, slab

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    hip.lib()
    yield


@pytest.mark.parametrize("chosen", [False, True])
def test_a_batch_too_large_leaves_the_form_as_it_was(chosen):
    """A form that was not timed is not chosen: on stays on, and off behind a
    chosen launch stays off for the slabs that fit later."""
    big, small = slab(4, 8, 2 * 6145), slab(9, 10, 11)
    b = make([big, small], "mixed_fused", chosen)
    i = b.add(big)
    b.run(8)
    b.autotune(2)
    assert b.resident() == {"on": not chosen, "steps": 0, "tiles": 0}
    b.remove(i)
    b.add(small)
    b.run(16)
    assert b.resident()["steps"] == (0 if chosen else 16)
    b.close()


def test_the_resident_form_is_timed_like_the_launches():
    """Warmed up and the better of two timings, as each launch; where it is the
    fastest, best_ms is its time and no row's."""
    s = slab(9, 10, 11)
    b = make([s], "mixed_fused", True)
    i = b.add(s)
    vm = b.vm(i)
    best, rows = b.autotune(5)
    assert b.resident() == {"on": True, "steps": 2 * (8 + 256), "tiles": 1024}
    assert best < min(r[4] for r in rows)
    assert np.array_equal(b.vm(i), vm) and b.slab_info(i)["loop"] == 0
    b.close()
