"""The right-hand side on host arrays that are pinned already (the state, the result, both, or one array
for both), on any number of CPUs: bit for bit the result of ordinary arrays, ghost cells of the
result untouched."""
import ctypes as C
import os

import numpy as np
import pytest

from oracle.oracle import Geom

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[1, 2, None])
def cpus(request):
    whole = os.sched_getaffinity(0)
    if request.param:
        os.sched_setaffinity(0, sorted(whole)[:request.param])
    yield request.param
    os.sched_setaffinity(0, whole)


@pytest.mark.parametrize("n", [(5, 7, 3), (33, 31, 30), (60, 58, 57)])
def test_pinned_arrays(engine, oracle, cpus, n):
    import granite_amd as ga
    from hipmem import _check, _hip

    L, held = _hip(), []
    L.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
    L.hipHostFree.argtypes = [C.c_void_p]

    def array(a, pinned):
        if not pinned:
            return a.copy()
        q = C.c_void_p()
        _check(L.hipHostMalloc(C.byref(q), a.nbytes, 0), "hipHostMalloc")
        held.append(q)
        b = np.ctypeslib.as_array(C.cast(q, C.POINTER(C.c_double)), shape=a.shape)
        b[...] = a
        return b

    g = Geom(n, 4, (-1.0, -1.1, -0.9), (1.0, 0.9, 1.2))
    u = oracle.add_noise(g, oracle.init_bl(g, [1.0], [[0.1, 0.2, 0.3]]), 5, 1e-3, range(22))
    geom, p = ga.GridBlock(0, 0, g.n, g.lo, g.hi, g.ng).geom(), ga.CCZ4Params().c()
    dp = C.POINTER(C.c_double)

    def rhs(a, r):
        engine.check(engine.lib.gr_ccz4_rhs(engine.handle, C.byref(geom), C.byref(p), 22, a.ctypes.data_as(dp),
                                            r.ctypes.data_as(dp), None, None, None, None))

    I = g.interior()
    want = np.full_like(u, 7.25)
    rhs(u, want)
    assert np.isfinite(want[I]).all()
    for u_pinned, r_pinned in ((True, False), (False, True), (True, True)):
        print(f"[gpu] host rhs {n} pinned {u_pinned} {r_pinned} cpus {cpus}", flush=True)
        a, r = array(u, u_pinned), array(np.full_like(u, 7.25), r_pinned)
        rhs(a, r)
        assert np.array_equal(r, want) and np.array_equal(a, u)
    a = array(u, True)  # in place
    rhs(a, a)
    assert np.array_equal(a[I], want[I])
    a[I] = u[I]
    assert np.array_equal(a, u)
    for q in held:
        _check(L.hipHostFree(q), "hipHostFree")
