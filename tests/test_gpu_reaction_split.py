"""The drop-in reaction's form for few tiles (k_tt06_calc_split_f64) against
the one for many, bit for bit: the same cells as an object of their own and at
the head of a larger object (cell counts in whole twelves, so that the v2 gate
loops treat them alike), through a scattered index and without one."""
import ctypes as C

import numpy as np
import pytest

from cardioid_amd import hip

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
DT = 0.02


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    hip.lib()
    yield


def calc(n, V, st, exact, index, nongate_only=False):
    """Two calls; (dVm of both, states)."""
    L = hip.lib()
    l, m, c = hip.read_fit_file().packed()
    p = hip.TT06Params(dt=DT, tolerance=0.0 if exact else 1e-4, mod=1, fastGate=1, fastNonGate=0,
                       fit_l=hip.ptr(l, hip.ip), fit_m=hip.ptr(m, hip.ip), fit_coef=hip.ptr(c),
                       celltype=hip.standard_celltype("midRRG"), s_kr=0.4, s_cal=0.9, s_na=1.0)
    h = C.c_void_p()
    hip.check(L.cdh_tt06_create(C.byref(p), n, C.byref(h)), "create")
    P = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
    try:
        hip.check(L.cdh_tt06_set_state(h, hip.ptr(np.ascontiguousarray(st[:, :n]).reshape(-1))),
                  "set_state")
        order = np.random.default_rng(3).permutation(n).astype(np.int32) if index else np.arange(n)
        full = np.empty(n)
        full[order] = V[:n]
        d_i = torch.from_numpy(order.astype(np.int32)).cuda()
        d_v = torch.from_numpy(full).cuda()
        out = []
        for k in range(2):
            d = torch.full((n,), float("nan"), dtype=torch.float64, device="cuda")
            if nongate_only:
                rc = L.cdh_tt06_update_nongate(h, DT, P(d_i) if index else None, n, P(d_v), P(d),
                                               None)
            else:
                rc = L.cdh_tt06_calc(h, DT, P(d_i) if index else None, n, P(d_v), None, P(d), None)
            hip.check(rc, "calc")
            torch.cuda.synchronize()
            out.append(d.cpu().numpy()[order])
        got = np.zeros(19 * n)
        hip.check(L.cdh_tt06_get_state(h, hip.ptr(got)), "get_state")
    finally:
        L.cdh_tt06_destroy(h)
    return out, got.reshape(19, n)


@pytest.mark.parametrize("exact,limit", [(False, 1536), (True, 1280)])
@pytest.mark.parametrize("index", [False, True])
@pytest.mark.parametrize("nongate_only", [False, True])
def test_few_tiles_equal_many(exact, limit, index, nongate_only):
    big = 64 * limit + 1200
    rng = np.random.default_rng(11)
    V = rng.uniform(-90.0, 40.0, big)
    ct = hip.standard_celltype("midRRG")
    st = np.repeat(np.array(ct.state0[:])[:, None], big, 1) * rng.uniform(0.9, 1.1, (19, big))
    st[1] = -138.0 * rng.uniform(0.95, 1.05, big) * 0.016404 * 96485.3415 / 0.185 + V
    want_d, want_s = calc(big, V, st, exact, index, nongate_only)
    for n in (12, 60, 72, 1200, 64 * limit // 12 * 12):
        print("split reaction", "exact" if exact else "fits", n, index, nongate_only, flush=True)
        d, s = calc(n, V, st, exact, index, nongate_only)
        for k in range(2):
            assert np.isfinite(d[k]).all()
            assert np.array_equal(d[k], want_d[k][:n])
        assert np.array_equal(s, want_s[:, :n])


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("name", ["endoCellML", "midCellML"])
def test_gates_far_outside_the_range(exact, name):
    """The quotients and exponentials written out for the gates, where their
    operands overflow, vanish or are not numbers: infinite and NaN where the
    oracle's are.  With the fits bit for bit the oracle's; with the exact
    functions within the few ulps (1e-12) of the other comparisons."""
    import oracle_lib as OL
    V = np.array([0.0, 15.0, -40.0, 1e3, 5e3, 2e4, 1.6e5, 1e6, 2e7, 1e9, 1e20, np.inf, 1e-200,
                  -1.0, -90.0, -1e3, -5e3, -7.5e3, -2e4, -1.6e5, -1e6, -2e7, -1e9, -1e20, -np.inf,
                  np.nan] + list(np.linspace(-700.0, 700.0, 38)))
    n = V.size
    ct = OL.celltype(name)
    st, vm = np.zeros(19 * n), np.zeros(n)
    OL.oracle().ora_tt06_init_state(C.byref(ct), n, OL.ptr(st), n, OL.ptr(vm))
    fs = hip.read_fit_file()
    l, m, c = fs.packed()
    p = hip.TT06Params(dt=DT, tolerance=0.0 if exact else 1e-4, mod=1, fastGate=int(not exact),
                       fastNonGate=0, fit_l=hip.ptr(l, hip.ip), fit_m=hip.ptr(m, hip.ip),
                       fit_coef=hip.ptr(c), celltype=hip.standard_celltype(name), s_kr=1.0,
                       s_cal=1.0, s_na=1.0)
    h = C.c_void_p()
    hip.check(hip.lib().cdh_tt06_create(C.byref(p), n, C.byref(h)), "create")
    try:
        hip.check(hip.lib().cdh_tt06_set_state(h, hip.ptr(st)), "set_state")
        d_v = torch.from_numpy(V).cuda()
        d = torch.zeros_like(d_v)
        hip.check(hip.lib().cdh_tt06_calc(h, DT, None, n, C.c_void_p(d_v.data_ptr()), None,
                                          C.c_void_p(d.data_ptr()), None), "calc")
        torch.cuda.synchronize()
        got = np.zeros(19 * n)
        hip.check(hip.lib().cdh_tt06_get_state(h, hip.ptr(got)), "get_state")
    finally:
        hip.lib().cdh_tt06_destroy(h)
    if exact:
        OL.oracle().ora_tt06_gates_exact(DT, ct.s_switch, 1, n, OL.ptr(V), OL.ptr(st), n)
    else:
        ofs = OL.make_fitset(fs, DT)
        OL.oracle().ora_tt06_gates_v2(C.byref(ofs), ct.s_switch, n, OL.ptr(V), OL.ptr(st), n)
    for q in range(7, 19):
        a, b = got.reshape(19, n)[q], st.reshape(19, n)[q]
        where = (name, q, [(v, x, y) for v, x, y in zip(V, a, b)
                           if not (x == y or (np.isnan(x) and np.isnan(y)))][:6])
        if exact:
            assert np.array_equal(np.isnan(a), np.isnan(b)), where
            with np.errstate(invalid="ignore"):
                ok = (a == b) | np.isnan(a) | (np.abs(a - b) <= 1e-12 * np.abs(b))
            assert ok.all(), where
        else:
            assert np.array_equal(a, b, equal_nan=True), where
