"""The drop-in entry points at the sizes where their kernels change shape: odd atom counts and the counts around a
wave and around the switch between the two compute_yi splits, atoms without pairs, one and two elements, a caller's own
coupling table (which must leave the kernels that carry the library's), and the derivative rows that the per-pair U
recursion leaves unwritten.

Bounds: 1e-12 of the array's largest value for U, Z, B, Y and E, 1e-10 for forces, virials and dB/dr, as for the golden
vectors; sums over pairs in another order lose a few eps of the sum of magnitudes, far below that.
"""
import numpy as np
import pytest

from conftest import relerr
from mdp_amd import lattice, snapcpp

pytestmark = pytest.mark.gpu

TOL_U = 1e-12
TOL_F = 1e-10


@pytest.fixture(scope="module")
def gpu():
    import mdp_amd
    return mdp_amd.library()


def _sna(lib, J, chem=0, bnorm=0, wselfall=0, quad=0, seed=3):
    nt = 2 if chem else 1
    param = [nt, J, 4.6, 0.99363, 0.0, 1, 1, quad, chem, bnorm, wselfall]
    rad, w = ([0.5, 0.45], [1.0, 0.9]) if chem else ([0.5], [1.0])
    s0 = snapcpp.initsna(lib, param, rad, w)
    coeff = np.random.default_rng(seed).normal(size=nt * s0.ncoeffall)
    return snapcpp.initsna(lib, param, rad, w, coeff)


def _pairs(N, P, nt, seed):
    """P pairs in the order of their centre atoms, some atoms without any; distances well inside the cutoffs"""
    rng = np.random.default_rng(seed)
    ai = np.sort(rng.integers(0, N, P)).astype(np.int32)
    r = rng.normal(size=(P, 3))
    r *= (rng.uniform(1.5, 4.0, P) / np.linalg.norm(r, axis=1))[:, None]
    t = rng.integers(1, nt + 1, N).astype(np.int32)
    aj = rng.integers(0, N, P).astype(np.int32)
    return dict(rij=np.ascontiguousarray(r.ravel()), ai=ai, aj=aj, ti=t[ai], tj=t[aj], atomtype=t,
                ilist=np.arange(N, dtype=np.int32), n=N, ijnum=P)


def _u_y(lib, s, p, cg=None, own_u=True):
    N, iu, ne = p["n"], s.idxu_max, s.nelements
    Ur, Ui = np.full(N * iu * ne, 0.01), np.full(N * iu * ne, -0.02)
    lib.cpuSnapComputeUi(Ur, Ui, s.rootpqarray, p["rij"], s.wjelem, s.radelem, s.rmin0, s.rfac0, s.rcutfac, s.map,
                         p["ai"], p["ti"], p["tj"], s.twojmax, iu, N, p["ijnum"], s.switchflag, s.chemflag)
    lib.cpuAddWself2Ui(Ur, Ui, s.wself, s.idxu_block, p["atomtype"], s.map, s.wselfallflag, s.chemflag, iu, ne,
                       s.twojmax, N)
    if not own_u:   # one entry behind the middle of the last layer is not the mirror image of its partner
        Ui.reshape(iu * ne, N)[iu - 1, N - 1] += 0.5
    cg = s.cglist if cg is None else cg
    e = np.zeros(N)
    lib.cpuSnapComputeEi(e, Ur, Ui, cg, s.bzero, s.coeffelem, p["ilist"], s.map, p["atomtype"], s.idxb,
                         s.idxcg_block, s.idxu_block, s.twojmax, s.idxb_max, iu, ne, s.ncoeffall, s.bnormflag,
                         s.bzeroflag, s.wselfallflag, s.chemflag, N)
    b = np.zeros(N * s.idxb_max * ne ** 3)
    lib.cpuSnapComputeBi(b, Ur, Ui, cg, s.bzero, s.idxb, s.idxcg_block, s.idxu_block, s.idxz_block, s.twojmax,
                         s.idxb_max, iu, s.idxz_max, ne, s.bnormflag, s.bzeroflag, s.wselfallflag, N)
    Yr, Yi = np.zeros(N * iu * ne), np.zeros(N * iu * ne)
    lib.cpuSnapComputeYi(Yr, Yi, Ur, Ui, cg, s.coeffelem, s.map, p["atomtype"], s.idxz, s.idxb_block, s.idxu_block,
                         s.idxcg_block, s.twojmax, s.idxb_max, iu, s.idxz_max, ne, s.ncoeffall, s.bnormflag,
                         s.chemflag, N)
    return dict(Ur=Ur, Ui=Ui, e=e, b=b, Yr=Yr, Yi=Yi)


@pytest.mark.parametrize("J,N,P,chem,bnorm,wselfall", [
    (2, 1, 0, 0, 0, 0), (2, 1, 3, 0, 0, 0), (2, 65, 400, 0, 1, 0), (4, 63, 900, 0, 0, 1), (4, 8191, 9000, 0, 0, 0),
    (4, 8257, 9000, 0, 0, 0), (6, 129, 2500, 0, 1, 0), (6, 65, 300, 1, 0, 0), (8, 64, 1500, 0, 0, 0),
    (8, 5057, 6000, 0, 0, 0), (8, 5185, 6000, 0, 1, 0), (8, 9, 40, 1, 1, 1)])
def test_u_b_e_y(gpu, oracle, J, N, P, chem, bnorm, wselfall):
    import mdp_amd
    p = _pairs(N, P, 2 if chem else 1, 7 * J + N)
    a = _u_y(gpu, _sna(gpu, J, chem, bnorm, wselfall), p)
    mdp_amd.check("u, b, e, y")
    o = _u_y(oracle, _sna(oracle, J, chem, bnorm, wselfall), p)
    for k in ("Ur", "Ui", "b", "e", "Yr", "Yi"):
        assert relerr(a[k], o[k]) < TOL_U, k


@pytest.mark.parametrize("J", [2, 4, 6, 8])
def test_a_callers_coupling_table_is_used(gpu, oracle, J):
    """A table that differs from the library's in one entry that every atom's terms use has to show in B, E and Y."""
    p = _pairs(33, 500, 1, J)
    s, so = _sna(gpu, J), _sna(oracle, J)
    cg = s.cglist.copy()
    cg[0] += 0.25
    a, o, own = _u_y(gpu, s, p, cg), _u_y(oracle, so, p, cg), _u_y(gpu, s, p)
    for k in ("b", "e", "Yr", "Yi"):
        assert relerr(a[k], o[k]) < TOL_U, k
    assert relerr(a["e"], own["e"]) > 1e-6


@pytest.mark.parametrize("J", [2, 4, 6, 8])
def test_a_callers_u_is_read_whole(gpu, oracle, J):
    """U that is not its own mirror image: B, E and Y have to read the entries behind the middle of each layer."""
    p = _pairs(33, 500, 1, J)
    s, so = _sna(gpu, J), _sna(oracle, J)
    a, o, own = _u_y(gpu, s, p, own_u=False), _u_y(oracle, so, p, own_u=False), _u_y(gpu, s, p)
    for k in ("b", "e", "Yr", "Yi"):
        assert relerr(a[k], o[k]) < TOL_U, k
    assert relerr(a["Yi"], own["Yi"]) > 1e-6


@pytest.mark.parametrize("J,P", [(2, 1), (4, 63), (6, 65), (8, 129), (2, 200001)])
def test_uij_rows(gpu, oracle, J, P):
    """U and dU of every pair; the derivative rows that are not written keep what they held."""
    p = _pairs(5, P, 1, 11 + P)
    out = []
    for lib in (gpu, oracle):
        s = _sna(lib, J)
        n = s.idxu_max * P
        ur, ui, du, dv = np.zeros(n), np.zeros(n), np.full(3 * n, 0.125), np.full(3 * n, -0.375)
        lib.cpuComputeUij(ur, ui, du, dv, s.rootpqarray, p["rij"], s.wjelem, s.radelem, s.rmin0, s.rfac0, s.rcutfac,
                          s.idxu_block, p["ti"], p["tj"], J, s.idxu_max, P, 1)
        out.append((ur, ui, du, dv))
    for a, b in zip(*out):
        assert relerr(a, b) < TOL_F
    for a, b, base in ((out[0][2], out[1][2], 0.125), (out[0][3], out[1][3], -0.375)):
        kept = b == base
        assert kept.any() and np.array_equal(a[kept], b[kept])


@pytest.mark.parametrize("J,N,P,chem,bnorm,quad", [
    (2, 3, 70, 0, 0, 0), (4, 31, 9001, 0, 0, 0), (6, 65, 700, 0, 1, 0), (8, 7, 100, 0, 0, 0), (4, 12, 200, 1, 0, 0),
    (4, 5, 130, 0, 0, 1)])
def test_descriptors(gpu, oracle, J, N, P, chem, bnorm, quad):
    import mdp_amd
    p = _pairs(N, P, 2 if chem else 1, 5 * J + P)
    a = snapcpp.snapdescriptors_pairs(gpu, _sna(gpu, J, chem, bnorm, 0, quad), p)
    mdp_amd.check("descriptors")
    o = snapcpp.snapdescriptors_pairs(oracle, _sna(oracle, J, chem, bnorm, 0, quad), p)
    for k in range(3):
        assert relerr(a[k], o[k]) < TOL_F, k
    for k in ("Ur", "Ui", "zr", "zi", "blist", "dblist"):
        assert relerr(a[3][k], o[3][k]) < TOL_F, k


@pytest.mark.parametrize("N,P,order", [(1, 1, "sorted"), (3, 64, "sorted"), (40, 65, "sorted"), (2, 300, "sorted"),
                                       (7, 1000, "shuffled"), (900, 1000, "alternating")])
def test_force_sums_over_runs_of_a_centre(gpu, oracle, N, P, order):
    """fatom and vatom, added into what they held, for runs that end inside a wave, at its edge and at every pair."""
    p = _pairs(N, P, 1, N + P)
    if order == "shuffled":
        perm = np.random.default_rng(2).permutation(P)
    elif order == "alternating":
        perm = np.concatenate([np.arange(0, P, 2), np.arange(1, P, 2)])
    else:
        perm = np.arange(P)
    ai, aj, ti, tj = (np.ascontiguousarray(p[k][perm]) for k in ("ai", "aj", "ti", "tj"))
    rij = np.ascontiguousarray(p["rij"].reshape(-1, 3)[perm].ravel())
    out = []
    for lib in (gpu, oracle):
        s = _sna(lib, 4)
        y = np.random.default_rng(1).normal(size=(2, N * s.idxu_max))
        f, v = np.full(3 * N, 0.25), np.full(6 * N, -0.5)
        lib.cpuSnapComputeFi(f, v, y[0].copy(), y[1].copy(), s.rootpqarray, rij, s.wjelem, s.radelem, s.rmin0, s.rfac0,
                             s.rcutfac, s.map, ai, ai, aj, ti, tj, 4, s.idxu_max, N, N, P, 1, 0)
        out.append((f, v))
    for a, b in zip(*out):
        assert relerr(a, b) < TOL_F
