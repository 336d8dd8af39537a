"""cdh_tt06_update_nongate (the pdr loop's updateNonGate): the seven other
states and dVm as the whole update gives them, every gate as it was."""
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


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("index", [False, True])
def test_gates_stay_and_the_rest_is_the_whole_updates(exact, index):
    """Sizes of both forms of the kernel and of its last tile: five wavefronts
    to a tile up to 98,304 cells (81,920 with the exact functions), one above."""
    L = hip.lib()
    l, m, c = hip.read_fit_file().packed()
    p = hip.TT06Params(dt=DT, tolerance=0.0 if exact else 1e-4, mod=1, fastGate=1, fastNonGate=0,
                       fit_l=hip.ptr(l, hip.ip), fit_m=hip.ptr(m, hip.ip), fit_coef=hip.ptr(c),
                       celltype=hip.standard_celltype("epiCellML"), s_kr=0.4, s_cal=0.9, s_na=1.0)
    s0 = np.array(p.celltype.state0[:])
    P = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
    for n in (1, 63, 64, 65, 1000, 81920, 98304, 98305, 130001):
        print("nongate", "exact" if exact else "fits", n, flush=True)
        rng = np.random.default_rng(n)
        V = rng.uniform(-90.0, 40.0, n)
        st = np.repeat(s0[:, None], n, 1) * rng.uniform(0.9, 1.1, (19, n))
        st[1] = -138.0 * rng.uniform(0.95, 1.05, n) * 0.016404 * 96485.3415 / 0.185 + V
        order = rng.permutation(n).astype(np.int32) if index else np.arange(n, dtype=np.int32)
        full = np.empty(n)
        full[order] = V
        d_i, d_v = torch.from_numpy(order).cuda(), torch.from_numpy(full).cuda()
        got = {}
        for name in ("calc", "nongate"):
            h = C.c_void_p()
            hip.check(L.cdh_tt06_create(C.byref(p), n, C.byref(h)), "create")
            hip.check(L.cdh_tt06_set_state(h, hip.ptr(np.ascontiguousarray(st).reshape(-1))), "set")
            d = torch.full((n,), float("nan"), dtype=torch.float64, device="cuda")
            ix = P(d_i) if index else None
            if name == "calc":
                hip.check(L.cdh_tt06_calc(h, DT, ix, n, P(d_v), None, P(d), None), name)
            else:
                hip.check(L.cdh_tt06_update_nongate(h, DT, ix, n, P(d_v), P(d), None), name)
            torch.cuda.synchronize()
            out = np.zeros(19 * n)
            hip.check(L.cdh_tt06_get_state(h, hip.ptr(out)), "get")
            L.cdh_tt06_destroy(h)
            got[name] = (d.cpu().numpy(), out.reshape(19, n))
        assert np.isfinite(got["calc"][0]).all()
        assert np.array_equal(got["nongate"][0], got["calc"][0])
        assert np.array_equal(got["nongate"][1][:7], got["calc"][1][:7])
        assert np.array_equal(got["nongate"][1][7:], st[7:])
        if n > 12:
            assert not np.array_equal(got["calc"][1][7:], st[7:])
