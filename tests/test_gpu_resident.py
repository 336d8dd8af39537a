"""The resident kernels (csrc/engine_resident.hpp) against the step kernels,
bit for bit: Vm, states, activation and APD90 times, counts, range record and
clock.  A launch chosen with set_launch runs the step kernels; the default
runs of 8 steps and more are resident where the tiles fit the chip (3,072
tiles, for the fits also 4,096 at four wavefronts per SIMD; mixed 6,144)."""
import numpy as np
import pytest

from cardioid_amd import hip, workloads as W

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
DT = 0.02


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    hip.lib()
    yield


def make(slabs, mode, chosen, exact=False, sensors=3):
    ext = [s.extent() for s in slabs]
    b = hip.Batch(DT, sum(e[0] for e in ext), sum(e[1] for e in ext), slab_capacity=len(slabs),
                  mode=mode, sensors=sensors, exact_functions=exact, jhTauSmooth=int(exact))
    if chosen:
        b.set_launch(3, 64)
    return b


def slab(nx, ny, nz, phi=20.0, vm_max=100.0, holes=0.0, seed=0, dur=1.0):
    a = W.fibre_slab(nx, ny, nz, phi)
    if holes:
        keep = np.random.default_rng(seed).random(a.ncell) >= holes
        a = W.Anatomy(nx, ny, nz, a.dx, a.dy, a.dz, a.gid[keep], a.celltype[keep], a.sigma[keep])
    st = [W.box_stimulus(xMax=3, nx=nx, ny=ny, nz=nz, duration=dur),
          W.box_stimulus(zMax=2, nx=nx, ny=ny, nz=nz, tStart=1.5, duration=0.4, vStim=-30.0)]
    return hip.Slab(a, ["midCellML"], W.DIFFUSION_SCALE, st, scales=(0.7, 0.9, 1.0),
                    vm_max=vm_max)


def results(b, ids):
    out = []
    for i in ids:
        out += [b.vm(i), b.state(i), *b.activation(i), b.t90(i), np.array(b.sensor_counts(i)),
                b.sensors(i)[0]]
        r, info = b.range_report(i), b.slab_info(i)
        out.append(np.array([info["time"], info["loop"], r["count"] if r else 0]))
    return out


def compare(slabs, mode, runs, exact=False):
    got = []
    for chosen in (False, True):
        b = make(slabs, mode, chosen, exact)
        ids = [b.add(s) for s in slabs]
        for n in runs:
            print(mode, "step kernels" if chosen else "resident", [s.ncell for s in slabs], n,
                  flush=True)
            b.run(n)
        got.append(results(b, ids))
        b.close()
    for a, r in zip(*got):
        assert np.array_equal(a, r)
    return got[0]


KINDS = [("fp64_fused", False), ("fp64_fma", False), ("mixed_fused", False), ("fp64_fused", True)]


@pytest.mark.parametrize("mode,exact", KINDS)
@pytest.mark.parametrize("dims,holes", [((1, 1, 1), 0.0), ((2, 4, 8), 0.0), ((5, 13, 1), 0.0),
                                        ((9, 10, 11), 0.3), ((3, 5, 130), 0.0), ((70, 3, 2), 0.1)])
def test_small_slabs_equal_the_step_kernels(mode, exact, dims, holes):
    """From one cell and one whole tile on; odd chunks (both box parities),
    chunks too short for the resident form in between, and more steps than
    one launch takes."""
    s = slab(*dims, holes=holes, vm_max=20.0)
    out = compare([s], mode, (17, 3, 8, 301), exact)
    assert np.ptp(out[0]) >= 0 and np.isfinite(out[0]).all()


@pytest.mark.parametrize("mode,ntile", [("fp64_fused", 3072), ("fp64_fused", 3073),
                                        ("fp64_fma", 4096), ("mixed_fused", 4096),
                                        ("mixed_fused", 4097), ("mixed_fused", 5120),
                                        ("mixed_fused", 5184), ("mixed_fused", 6144),
                                        ("mixed_fused", 6145)])
def test_tiles_at_the_edges_of_what_the_chip_holds(mode, ntile):
    """64 x ntile cells in one slab: the last that fits each kernel, and the
    first that does not."""
    compare([slab(ntile // 64 if ntile % 64 == 0 else ntile, 64 if ntile % 64 == 0 else 8,
                  64 if ntile % 64 == 0 else 8)], mode, (40,))


@pytest.mark.parametrize("mode,exact", KINDS)
@pytest.mark.parametrize("ntile", [767, 769, 1024, 1025])
def test_tiles_at_the_edges_of_six_wavefronts_to_a_tile(mode, exact, ntile):
    """The last tiles that fit six wavefronts each (768 at 80 registers, 1,024
    at 64), and the first that do not; the last tile ragged."""
    nz = 64 * ntile // 32
    compare([slab(4, 8, nz, holes=0.0)], mode, (16, 31), exact)
    a = slab(2, 16, nz + 1 if ntile % 2 else nz - 1)
    compare([a], mode, (33,), exact)


@pytest.mark.parametrize("mode", ["fp64_fma", "mixed_fused"])
def test_slabs_come_and_go(mode):
    """Several slabs with clocks of their own; one leaves (the tiles then are
    a list with a hole) and a smaller one takes its place."""
    s = [slab(9, 10, 11, 5.0), slab(20, 6, 7, -40.0, holes=0.2), slab(4, 4, 40, 80.0),
         slab(6, 7, 8, 33.0)]
    got = []
    for chosen in (False, True):
        b = make(s, mode, chosen)
        ids = [b.add(x) for x in s[:3]]
        b.run(33)
        b.remove(ids[1])
        b.run(20)
        ids[1] = b.add(s[3])
        b.run(50)
        b.run(21)
        got.append(results(b, ids))
        b.close()
    for a, r in zip(*got):
        assert np.array_equal(a, r)


@pytest.mark.parametrize("mode", ["fp64_fma", "mixed_fused"])
def test_apd90_over_a_whole_beat(mode):
    """25,000 steps of a tiny slab: activation, Vmax and t90 of every cell."""
    out = compare([slab(4, 5, 6)], mode, (20000,))
    assert (out[5] > 0).all()


def test_autotune_leaves_the_state_alone():
    s = slab(12, 13, 14)
    got = []
    for tune in (False, True):
        b = make([s], "fp64_fma", False)
        ids = [b.add(s)]
        b.run(31)
        if tune:
            best, rows = b.autotune(5)
            assert best > 0 and len(rows) == 18
        b.run(64)
        got.append(results(b, ids))
        b.close()
    for a, r in zip(*got):
        assert np.array_equal(a, r)


@pytest.mark.parametrize("mode", ["fp64_fma", "mixed_fused"])
@pytest.mark.parametrize("dims", [(3, 4, 5), (100, 90, 60)])
def test_results_come_in_the_callers_order(mode, dims):
    """The device's gather into the caller's order, short rows and rows of
    several pieces (540,000 cells): cells given in a shuffled order read back
    as the same anatomy's in box order, and the order is the slab's own where
    two share the engine."""
    nx, ny, nz = dims
    a = W.fibre_slab(nx, ny, nz, 30.0)
    p = np.random.default_rng(1).permutation(a.ncell)
    shuffled = W.Anatomy(nx, ny, nz, a.dx, a.dy, a.dz, a.gid[p], a.celltype[p], a.sigma[p])
    st = [W.box_stimulus(xMax=2, nx=nx, ny=ny, nz=nz)]
    slabs = [hip.Slab(x, ["epiCellML"], W.DIFFUSION_SCALE, st, gate_tail_rule=False)
             for x in (a, shuffled)]
    b = make(slabs, mode, False)
    ids = [b.add(s) for s in slabs]
    b.run(120)
    first, second = ([b.vm(i), b.state(i), *b.activation(i), b.t90(i)] for i in ids)
    b.close()
    assert np.ptp(first[0]) > 1.0
    if mode == "mixed_fused":        # compact weights are alike: the same tiles
        assert np.array_equal(first[0][p], second[0])
    for x, y in zip(first, second):
        assert np.array_equal(x[..., p], y)


@pytest.mark.parametrize("mode,nz", [("fp64_fused", 1400), ("fp64_fma", 4000), ("mixed_fused", 4000)])
def test_range_record_is_the_earliest_steps(mode, nz):
    """Cells leave the range at six places along a slab, each a step later
    than the last, in an order unlike the tiles': the record is the first
    step's, and the next record that of the steps after the first is read."""
    nx, ny = 4, 8
    a = W.fibre_slab(nx, ny, nz, 0.0)
    z = [nz * f // 16 for f in (9, 3, 14, 1, 12, 6)]
    st = [W.box_stimulus(zMin=p, zMax=p + 4, nx=nx, ny=ny, nz=nz, tStart=1.0 + k * DT,
                         duration=0.5, vStim=-45.0) for k, p in enumerate(z)]
    s = hip.Slab(a, ["midCellML"], W.DIFFUSION_SCALE, st, vm_max=-84.0)
    got = []
    for chosen in (False, True):
        b = make([s], mode, chosen)
        i = b.add(s)
        b.run(80)
        first = b.range_report(i)
        b.run(30)
        got.append((first, b.range_report(i)))
        b.close()
    for r, want in zip(*got):
        assert r["count"] == want["count"] and r["loop"] == want["loop"]
        assert r["V"] > -84.0
    first, cell = got[0][0], got[0][0]["cell"]
    assert z[0] < cell // (nx * ny) < z[0] + 4, first


def test_results_of_a_slab_longer_than_one_gather():
    """Rows of more cells than one gather takes (2,097,152), in the caller's
    (shuffled) order.  The exact functions: their gates do not depend on a
    cell's place, as the fits' loop bounds do."""
    nx, ny, nz = 128, 128, 130
    a = W.fibre_slab(nx, ny, nz, 10.0)
    order = np.random.default_rng(3).permutation(a.ncell)
    b = W.Anatomy(nx, ny, nz, a.dx, a.dy, a.dz, a.gid[order], a.celltype[order], a.sigma[order])
    got = []
    for an in (a, b):
        st = [W.box_stimulus(xMax=4, nx=nx, ny=ny, nz=nz)]
        sim = hip.Simulation(an, ["endoCellML"], DT, W.DIFFUSION_SCALE, st, mode="fp64_fused", sensors=3,
                             exact_functions=True, jhTauSmooth=1)
        sim.run(60)
        got.append([sim.vm(), *sim.activation(), sim.t90(), *sim.state()])
        sim.close()
    for x, y in zip(*got):
        assert np.array_equal(x[order], y)
    assert np.unique(got[0][0]).size > 4


@pytest.mark.parametrize("modes", [("fp64_fma", "fp64_fma"), ("mixed_fused", "fp64_fused")])
def test_engines_side_by_side(modes):
    """Two engines that each fill the chip, queued on their own streams from
    two threads: their resident launches follow one another, and each one's
    results are those it has alone."""
    import threading
    s = [slab(50, 60, 63, 5.0), slab(48, 56, 70, -40.0, holes=0.1)]
    alone = []
    for k in range(2):
        b = make([s[k]], modes[k], False)
        i = b.add(s[k])
        b.run(530)
        alone.append(results(b, [i]))
        b.close()
    bs = [make([s[k]], modes[k], False) for k in range(2)]
    ids = [b.add(x) for b, x in zip(bs, s)]

    def work(k):
        for n in (300, 9, 221):
            bs[k].run(n)
        bs[k].sync()

    t = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for x in t:
        x.start()
    for x in t:
        x.join()
    for k in range(2):
        for a, r in zip(alone[k], results(bs[k], [ids[k]])):
            assert np.array_equal(a, r)
        bs[k].close()
