"""Training kernels of the learned surrogate against numpy in float64 on ragged pair lists: atoms without pairs,
with more pairs than a workgroup has lanes, atom counts around a workgroup's share, every descriptor count.

Sums of at most 700 products in float64: 1e-12 of the max norm.  The parameter reduction is in float32, 16 sums of
nparts/16 terms: (nparts/16 + 16) rounding errors of 2^-24 of the sum of the magnitudes.
"""
import numpy as np
import pytest

from conftest import relerr

pytestmark = pytest.mark.gpu


def _pairs(n, rng):
    cnt = rng.integers(0, 40, n)
    cnt[rng.integers(0, n, max(1, n // 7))] = 0
    cnt[n // 2] = 600
    pi = np.repeat(np.arange(n), cnt).astype(np.int32)
    pj = rng.integers(0, n, len(pi)).astype(np.int32)
    return pi, pj


@pytest.mark.parametrize("n,K", [(1, 1), (7, 5), (33, 14), (257, 16), (16384, 14), (16417, 3)])
def test_chain_rule_kernels(n, K):
    from mdp_amd import surrogate as S
    from mdp_amd.devarray import DevArray
    rng = np.random.default_rng(n + K)
    pi, pj = _pairs(n, rng)
    P = len(pi)
    g, dbdr, R, fref = rng.normal(size=(K, n)), rng.normal(size=(K, 3, P)), rng.normal(size=(n, 3)), rng.normal(size=(n, 3))
    off = lambda v: np.concatenate([[0], np.cumsum(np.bincount(v, minlength=n))]).astype(np.int32)  # noqa: E731
    c = S._lib()
    d = {k: DevArray.from_numpy(v) for k, v in dict(g=g, dbdr=dbdr, R=R, fref=fref, pi=pi, pj=pj, own=off(pi), inc=off(pj),
                                                     idx=np.argsort(pj, kind="stable").astype(np.int32)).items()}
    out = {k: DevArray.zeros(v) for k, v in dict(s=3 * P, F=3 * n, Res=3 * n, U=K * n).items()}
    S._chk(c.mdp_sur_pair_s(d["g"].ptr, d["dbdr"].ptr, d["pi"].ptr, K, n, P, out["s"].ptr, None), "pair_s")
    S._chk(c.mdp_sur_atom_f(out["s"].ptr, d["own"].ptr, d["inc"].ptr, d["idx"].ptr, P, n, d["fref"].ptr, out["F"].ptr,
                            out["Res"].ptr, None), "atom_f")
    S._chk(c.mdp_sur_u(d["R"].ptr, d["dbdr"].ptr, d["own"].ptr, d["pj"].ptr, K, n, P, 0.7, out["U"].ptr, None), "u")
    s = np.einsum("kp,kcp->cp", g[:, pi], dbdr)
    F = np.zeros((n, 3))
    np.add.at(F, pi, s.T)
    np.add.at(F, pj, -s.T)
    U = np.zeros((n, K))
    np.add.at(U, pi, 0.7 * np.einsum("pc,kcp->pk", R[pi] - R[pj], dbdr))
    assert relerr(out["s"].numpy().reshape(3, P), s) < 1e-12
    # forces cancel (exactly, for one atom): the bound is on the sum of the magnitudes, 700 terms x 2^-53
    A = np.zeros((n, 3))
    np.add.at(A, pi, np.abs(s.T))
    np.add.at(A, pj, np.abs(s.T))
    assert np.all(np.abs(out["F"].numpy().reshape(n, 3) - F) <= 1e-12 * A)
    assert np.all(np.abs(out["Res"].numpy().reshape(n, 3) - (F - fref)) <= 1e-12 * (A + np.abs(fref)))
    assert relerr(out["U"].numpy().reshape(K, n).T, U) < 1e-12


@pytest.mark.parametrize("sizes", [[1], [63, 64, 65], [250, 1, 2, 700, 0, 3]])
def test_configuration_energies(sizes):
    from mdp_amd import surrogate as S
    from mdp_amd.devarray import DevArray
    rng = np.random.default_rng(len(sizes))
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    e, ref = rng.normal(size=off[-1]), rng.normal(size=len(sizes))
    de, do, dr = DevArray.from_numpy(e), DevArray.from_numpy(off), DevArray.from_numpy(ref)
    Ec, al = DevArray.zeros(len(sizes)), DevArray.zeros(off[-1])
    S._chk(S._lib().mdp_sur_energy(de.ptr, do.ptr, dr.ptr, len(sizes), 0.3, Ec.ptr, al.ptr, None), "energy")
    E = np.array([e[off[k]:off[k + 1]].sum() for k in range(len(sizes))])
    alpha = np.concatenate([np.full(m, 0.6 * (E[k] - ref[k]) / m ** 2) for k, m in enumerate(sizes) if m])
    assert np.max(np.abs(Ec.numpy() - E)) < 1e-12
    assert relerr(al.numpy(), alpha) < 1e-12


@pytest.mark.parametrize("nparts", [1, 15, 37, 1024])
def test_parameter_gradient_reduction(nparts):
    """mdp_mlp_train's gradient is the sum of the per-wave partials it leaves behind."""
    from mdp_amd import surrogate as S
    from mdp_amd.devarray import DevArray
    rng = np.random.default_rng(nparts)
    n, nin = 3000, 14
    c = S._lib()
    m = S.Model.init(np.zeros(nin), np.ones(nin), 1.0, 0.0, seed=1)
    p, aff, q = DevArray.from_numpy(m.params), DevArray.from_numpy(m.aff), DevArray(10240, np.int16)
    X, U, al = (DevArray.from_numpy(rng.normal(size=k)) for k in (nin * n, nin * n, n))
    part, grad = DevArray.zeros(nparts * S.NPARAM, np.float32), DevArray.zeros(S.NPARAM, np.float32)
    S._chk(c.mdp_mlp_pack(p.ptr, q.ptr, None), "pack")
    S._chk(c.mdp_mlp_train(q.ptr, p.ptr, aff.ptr, nin, X.ptr, U.ptr, al.ptr, n, part.ptr, nparts, grad.ptr, None), "train")
    rows = part.numpy().reshape(nparts, S.NPARAM).astype(np.float64)
    bound = (nparts / 16 + 17) * 2.0 ** -24 * np.abs(rows).sum(0) + 1e-30
    assert np.all(np.abs(grad.numpy() - rows.sum(0)) <= bound)
