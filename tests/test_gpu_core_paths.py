"""The device-array entry points of the force chain: the one-element route, which stays on the device, against the
element-mapped route (one element mapped to block 0 gives the same numbers), against the route for pairs in another
order, and against the CPU oracle; what is refused stays refused, with nothing written.

Bounds: 1e-12 of the array's largest value for U and E, 1e-10 for forces and virials, as for the golden vectors.
"""
import ctypes

import numpy as np
import pytest

from conftest import relerr
from test_gpu_dropin_paths import TOL_F, TOL_U, _pairs, _sna

pytestmark = pytest.mark.gpu

D, I = ctypes.c_double, ctypes.c_int  # noqa: E741


def _fn(lib, name, shape):
    f = getattr(lib.cdll, "mdp_hip" + name)
    f.restype = None
    f.argtypes = [{"p": ctypes.c_void_p, "d": D, "i": I}[c] for c in shape]
    return f


@pytest.fixture(scope="module")
def gpu():
    import mdp_amd
    return mdp_amd.library()


def _chain(lib, s, p, chem=0, order=None, aii=None):
    from mdp_amd.devarray import DevArray
    P, N, iu, J = p["ijnum"], p["n"], s.idxu_max, s.twojmax
    order = np.arange(P) if order is None else order
    q = {k: np.ascontiguousarray(p[k][order]) for k in ("ai", "aj", "ti", "tj")}
    if aii is not None:
        q["ai"] = aii
    q["rij"] = np.ascontiguousarray(p["rij"].reshape(-1, 3)[order].ravel())
    q.update(rp=s.rootpqarray, wj=s.wjelem, rad=s.radelem, cg=s.cglist, bz=s.bzero, c=s.coeffelem, map=s.map,
             type=p["atomtype"], il=p["ilist"], Ur=np.full(N * iu, 0.01), Ui=np.full(N * iu, -0.02),
             Yr=np.zeros(N * iu), Yi=np.zeros(N * iu), e=np.full(N, 0.5), f=np.full(3 * N, 0.25), v=np.full(6 * N, -0.5))
    d = {k: DevArray.from_numpy(a) for k, a in q.items()}
    a = lambda *n: [d[k].ptr for k in n]  # noqa: E731
    _fn(lib, "SnapComputeUi", "pppppp" "ddd" "ppppp" "iiiiii")(
        *a("Ur", "Ui", "rp", "rij", "wj", "rad"), s.rmin0, s.rfac0, s.rcutfac, None, *a("map", "ai", "ti", "tj"), J, iu, N,
        P, s.switchflag, chem)
    _fn(lib, "AddWself2Ui", "ppd" "pppp" "iiiiii")(*a("Ur", "Ui"), s.wself, None, *a("type", "map", "ai"), 0, chem, iu, 1, J,
                                                   N)
    _fn(lib, "SnapComputeEi", "pppppppppppp" "iiiiiiiiii")(
        *a("e", "Ur", "Ui", "cg", "bz", "c", "il", "map", "type"), None, None, None, J, s.idxb_max, iu, 1, s.ncoeffall,
        s.bnormflag, 1, 0, 0, N)
    _fn(lib, "SnapComputeYi", "pppppppppppp" "iiiiiiii")(
        *a("Yr", "Yi", "Ur", "Ui", "cg", "c", "map", "type"), None, None, None, None, J, s.idxb_max, iu, s.idxz_max, 1,
        s.ncoeffall, s.bnormflag, N)
    _fn(lib, "SnapComputeFi", "pppppppp" "ddd" "ppppppp" "iiiiiii")(
        *a("f", "v", "Yr", "Yi", "rp", "rij", "wj", "rad"), s.rmin0, s.rfac0, s.rcutfac, None,
        *a("map", "ai", "ai", "aj", "ti", "tj"), J, iu, N, N, P, s.switchflag, chem)
    return {k: d[k].numpy() for k in ("Ur", "Ui", "e", "Yr", "Yi", "f", "v")}


@pytest.mark.parametrize("J,N,P,bnorm", [(2, 1, 1, 0), (4, 63, 800, 1), (6, 65, 257, 0), (8, 130, 3000, 0)])
def test_one_element_route(gpu, oracle, J, N, P, bnorm):
    import mdp_amd
    s, p = _sna(gpu, J, 0, bnorm), _pairs(N, P, 1, J + N)
    a = _chain(gpu, s, p)
    mdp_amd.check("device chain")
    mapped = _chain(gpu, s, p, chem=1)
    shuffled = _chain(gpu, s, p, order=np.random.default_rng(3).permutation(P))
    mdp_amd.check("device chain, other routes")
    for k in a:
        assert relerr(a[k], mapped[k]) < TOL_F, k
        assert relerr(a[k], shuffled[k]) < TOL_F, k
    so, iu = _sna(oracle, J, 0, bnorm), s.idxu_max
    Ur, Ui, e, f, v = np.full(N * iu, 0.01), np.full(N * iu, -0.02), np.full(N, 0.5), np.full(3 * N, 0.25), np.zeros(6 * N)
    Yr, Yi = np.zeros(N * iu), np.zeros(N * iu)
    oracle.cpuSnapComputeUi(Ur, Ui, so.rootpqarray, p["rij"], so.wjelem, so.radelem, so.rmin0, so.rfac0, so.rcutfac, so.map,
                            p["ai"], p["ti"], p["tj"], J, iu, N, P, 1, 0)
    oracle.cpuAddWself2Ui(Ur, Ui, so.wself, so.idxu_block, p["atomtype"], so.map, 0, 0, iu, 1, J, N)
    oracle.cpuSnapComputeEi(e, Ur, Ui, so.cglist, so.bzero, so.coeffelem, p["ilist"], so.map, p["atomtype"], so.idxb,
                            so.idxcg_block, so.idxu_block, J, so.idxb_max, iu, 1, so.ncoeffall, bnorm, 1, 0, 0, N)
    oracle.cpuSnapComputeYi(Yr, Yi, Ur, Ui, so.cglist, so.coeffelem, so.map, p["atomtype"], so.idxz, so.idxb_block,
                            so.idxu_block, so.idxcg_block, J, so.idxb_max, iu, so.idxz_max, 1, so.ncoeffall, bnorm, 0, N)
    oracle.cpuSnapComputeFi(f, v, Yr, Yi, so.rootpqarray, p["rij"], so.wjelem, so.radelem, so.rmin0, so.rfac0, so.rcutfac,
                            so.map, p["ai"], p["ai"], p["aj"], p["ti"], p["tj"], J, iu, N, N, P, 1, 0)
    for k, b, tol in (("Ur", Ur, TOL_U), ("Ui", Ui, TOL_U), ("e", e, TOL_U), ("Yr", Yr, TOL_U), ("f", f, TOL_F)):
        assert relerr(a[k], b) < tol, k
    # half of each pair's virial on either atom: the same total
    assert relerr((a["v"] + 0.5).reshape(6, N).sum(1), v.reshape(N, 6).sum(0)) < TOL_F


@pytest.mark.parametrize("bad", [-1, 20])
def test_centres_out_of_range_are_refused(gpu, bad):
    import mdp_amd
    s, p = _sna(gpu, 4), _pairs(20, 300, 1, 1)
    from mdp_amd.devarray import DevArray
    ai = p["ai"].copy()
    ai[0 if bad < 0 else -1] = bad
    d = {k: DevArray.from_numpy(v) for k, v in dict(rp=s.rootpqarray, rij=p["rij"], wj=s.wjelem, rad=s.radelem, map=s.map,
                                                    ai=ai, ti=p["ti"], tj=p["tj"], U=np.full(20 * s.idxu_max, 0.75)).items()}
    a = lambda *n: [d[k].ptr for k in n]  # noqa: E731
    _fn(gpu, "SnapComputeUi", "pppppp" "ddd" "ppppp" "iiiiii")(
        *a("U", "U", "rp", "rij", "wj", "rad"), s.rmin0, s.rfac0, s.rcutfac, None, *a("map", "ai", "ti", "tj"), 4, s.idxu_max,
        20, 300, 1, 0)
    assert "out of range" in mdp_amd.last_error()
    assert np.all(d["U"].numpy() == 0.75)


def test_forces_on_atoms_out_of_range_are_refused(gpu):
    import mdp_amd
    from mdp_amd.devarray import DevArray
    s, p = _sna(gpu, 4), _pairs(20, 300, 1, 1)
    aj = p["aj"].copy()
    aj[17] = 20
    n = 20 * s.idxu_max
    d = {k: DevArray.from_numpy(v) for k, v in dict(rp=s.rootpqarray, rij=p["rij"], wj=s.wjelem, rad=s.radelem, map=s.map,
                                                    ai=p["ai"], aj=aj, ti=p["ti"], tj=p["tj"], Y=np.ones(n),
                                                    f=np.full(60, 0.75), v=np.full(120, 0.75)).items()}
    a = lambda *k: [d[x].ptr for x in k]  # noqa: E731
    _fn(gpu, "SnapComputeFi", "pppppppp" "ddd" "ppppppp" "iiiiiii")(
        *a("f", "v", "Y", "Y", "rp", "rij", "wj", "rad"), s.rmin0, s.rfac0, s.rcutfac, None,
        *a("map", "ai", "ai", "aj", "ti", "tj"), 4, s.idxu_max, 20, 20, 300, 1, 0)
    assert "not below anum" in mdp_amd.last_error()
    assert np.all(d["f"].numpy() == 0.75) and np.all(d["v"].numpy() == 0.75)


@pytest.mark.parametrize("route", ["device", "device, elements", "host"])
@pytest.mark.parametrize("array,value", [("ai", -1), ("aj", -2147483648), ("aii", -1), ("aii", 20)])
def test_negative_and_centre_indices_of_forces_are_refused(gpu, route, array, value):
    """20 atoms; the device arrays also through the element-mapped route, and the host arrays.  Nothing is written."""
    import mdp_amd
    from mdp_amd.devarray import DevArray
    s, p = _sna(gpu, 4), _pairs(20, 300, 1, 1)
    q = dict(aii=p["ai"].copy(), ai=p["ai"].copy(), aj=p["aj"].copy(), ti=p["ti"], tj=p["tj"])
    q[array][150] = value
    y, f, v = np.ones(20 * s.idxu_max), np.full(60, 0.75), np.full(120, 0.75)
    print(route, array, value, flush=True)
    if route == "host":
        gpu.cpuSnapComputeFi(f, v, y, y, s.rootpqarray, p["rij"], s.wjelem, s.radelem, s.rmin0, s.rfac0, s.rcutfac, s.map,
                             q["aii"], q["ai"], q["aj"], q["ti"], q["tj"], 4, s.idxu_max, 20, 20, 300, 1, 0)
        message = mdp_amd.last_error()
    else:
        d = {k: DevArray.from_numpy(a) for k, a in dict(q, rp=s.rootpqarray, rij=p["rij"], wj=s.wjelem, rad=s.radelem,
                                                        map=s.map, Y=y, f=f, v=v).items()}
        a = lambda *k: [d[x].ptr for x in k]  # noqa: E731
        _fn(gpu, "SnapComputeFi", "pppppppp" "ddd" "ppppppp" "iiiiiii")(
            *a("f", "v", "Y", "Y", "rp", "rij", "wj", "rad"), s.rmin0, s.rfac0, s.rcutfac, None,
            *a("map", "aii", "ai", "aj", "ti", "tj"), 4, s.idxu_max, 20, 20, 300, 1, int("elements" in route))
        message = mdp_amd.last_error()
        f, v = d["f"].numpy(), d["v"].numpy()
    assert ("centre index out of range" if array == "aii" else "negative pair atom index") in message
    assert np.all(f == 0.75) and np.all(v == 0.75)


@pytest.mark.parametrize("call", ["AddWself2Ui", "Cumsum", "SnapTallyForceFull", "VirialPairTally"])
def test_waits_for_the_callers_default_stream(gpu, call):
    """Outputs cleared, and for Cumsum inputs, by memsets that still wait on the default stream behind 48 GB of others when the
    call is made: it sees what they leave.  (Were it to run before them, sums would be lost or start from the old values.)"""
    import mdp_amd
    from mdp_amd.devarray import DevArray
    c = gpu.cdll
    c.hipMemsetAsync.argtypes, c.hipMemsetAsync.restype = [ctypes.c_void_p, I, ctypes.c_size_t, ctypes.c_void_p], I
    clear = lambda d: c.hipMemsetAsync(d.ptr, 0, d.nbytes, None)  # noqa: E731
    n, J = 1000, 4
    s = _sna(gpu, J)
    ones = lambda m, t=np.float64: DevArray.from_numpy(np.ones(m, t))  # noqa: E731
    big = DevArray(1 << 30)
    i, force = np.arange(n, dtype=np.int32), np.arange(3.0 * n)
    ai, aj, fij, ty, mp = (DevArray.from_numpy(a) for a in (i, (i + 1) % n, force, np.ones(n, np.int32), s.map))
    U, V, f, v, count, total = (ones(m, t) for m, t in ((n * s.idxu_max, float), (n * s.idxu_max, float), (3 * n, float),
                                                        (6 * n, float), (n, np.int32), (n + 1, np.int32)))
    work = {"AddWself2Ui": ("ppd" "pppp" "iiiiii", (U.ptr, V.ptr, 3.0, None, ty.ptr, mp.ptr, ai.ptr, 0, 0, s.idxu_max, 1, J, n)),
            "Cumsum": ("ppppi", (total.ptr, count.ptr, None, None, n + 1)),
            "SnapTallyForceFull": ("pppppi", (f.ptr, fij.ptr, ai.ptr, aj.ptr, None, n)),
            "VirialPairTally": ("pppdpiii", (v.ptr, fij.ptr, fij.ptr, 2.0, ai.ptr, 3, n, n))}
    shape, args = work[call]
    fn = _fn(gpu, call, shape)
    print(call, flush=True)
    for _ in range(6):
        assert c.hipMemsetAsync(big.ptr, 1, big.nbytes, None) == 0
    for d in (U, V, f, v, count):
        assert clear(d) == 0
    fn(*args)
    mdp_amd.check(call)
    if call == "AddWself2Ui":
        assert U.numpy().sum() == 3.0 * n * sum(j + 1 for j in range(J + 1)) and not V.numpy().any()
    elif call == "Cumsum":
        assert not total.numpy().any()
    elif call == "SnapTallyForceFull":
        assert np.array_equal(f.numpy(), force - np.roll(force, 3))
    else:
        x, y, z = force.reshape(n, 3).T
        assert np.array_equal(v.numpy().reshape(6, n), 2.0 * np.array([x * x, y * y, z * z, x * y, x * z, y * z]))
