"""Which form a run takes (cdh_batch_get_resident, cdh_sim_get_resident): the
kernel at each edge of what the chip holds, and the switch."""
import numpy as np
import pytest

from cardioid_amd import hip, workloads as W
from test_gpu_resident import DT, make, results, slab

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    hip.lib()
    yield


F64 = [(1, 768), (768, 768), (769, 1024), (1024, 1024), (1025, 3072), (3072, 3072)]
FITS = F64 + [(3073, 4096), (4096, 4096), (4097, 0)]
MIXED = [(1, 1024), (1024, 1024), (1025, 4096), (4096, 4096), (4097, 6144), (6144, 6144),
         (6145, 0)]


@pytest.mark.parametrize("mode,exact,edges", [("fp64_fused", False, FITS), ("fp64_fma", False, FITS),
                                              ("mixed_fused", False, MIXED),
                                              ("fp64_fused", True, F64 + [(3073, 0)])])
def test_kernel_at_the_edges_of_what_the_chip_holds(mode, exact, edges):
    """Tiles on one MI355X (256 CUs) and how many the kernel that runs them
    holds (0: the step kernels)."""
    assert torch.cuda.get_device_properties(0).multi_processor_count == 256
    for ntile, holds in edges:
        print(mode, "exact" if exact else "fits", ntile, "tiles", flush=True)
        s = slab(4, 8, 2 * ntile)
        b = make([s], mode, False, exact, sensors=0)
        b.add(s)
        assert b.resident() == {"on": True, "steps": 0, "tiles": 0}
        b.run(7)                       # too few to be worth a cooperative launch
        assert b.resident()["steps"] == 0
        b.run(16)
        b.sync()
        assert b.resident() == {"on": True, "steps": 16 if holds else 0, "tiles": holds}
        b.close()


@pytest.mark.parametrize("mode", ["fp64_fma", "mixed_fused"])
def test_switch(mode):
    """A chosen launch turns the form off, set_resident on again; the results
    are the same, and the launch stays for the runs that do not fit."""
    s = slab(9, 10, 11, holes=0.2)
    got = []
    for choose, on, steps in ((False, None, 80), (False, False, 0), (True, None, 0),
                              (True, True, 80)):
        b = make([s], mode, choose)
        i = b.add(s)
        if on is not None:
            b.set_resident(on)
        b.run(80)
        assert b.resident()["steps"] == steps
        assert b.resident()["on"] == (steps > 0)
        if choose:
            assert b.launch()[:2] == (3, 64)
        got.append(results(b, [i]))
        b.close()
    for k in range(1, 4):
        for a, r in zip(got[0], got[k]):
            assert np.array_equal(a, r)


def test_simulation():
    a = W.fibre_slab(6, 7, 8, 20.0)
    st = [W.box_stimulus(xMax=2, nx=6, ny=7, nz=8)]

    def sim(**kw):
        return hip.Simulation(a, ["midCellML"], DT, W.DIFFUSION_SCALE, st, **kw)

    vm = []
    for variant, on, steps in ((0, None, 40), (3, None, 0), (3, True, 40), (0, False, 0)):
        s = sim(mode="fp64_fma", variant=variant)
        if on is not None:
            s.set_resident(on)
        s.run(40)
        assert s.resident()["steps"] == steps
        vm.append(s.vm())
        s.close()
    for v in vm[1:]:
        assert np.array_equal(v, vm[0])
    s = sim(mode="fp64_unfused")
    s.run(40)
    assert s.resident() == {"on": False, "steps": 0, "tiles": 0}
    s.set_resident(False)
    with pytest.raises(hip.CardioidHipError):
        s.set_resident(True)
    s.close()
