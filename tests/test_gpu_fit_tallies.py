"""Tallies and normal equations of the batched fit where their kernels change form: configurations around the
number of threads of a workgroup and above what it holds, atoms with long incoming lists, every number of 16-column
tiles of the normal equations (1 to 5), several element types.

Reference: numpy in float64 on the engine's own B, dB/dr and pair list.  Sums of m terms, m <= 200,000 here, differ by
at most m 2^-53 of the sum of the magnitudes; the orders used keep it far below the 1e-11 allowed.
"""
import numpy as np
import pytest

from mdp_amd import lattice
from mdp_amd.fit import SnapFit

pytestmark = pytest.mark.gpu


def _config(n, seed, a=3.316, types=1):
    cells = int(np.ceil((n / 2) ** (1 / 3)))
    x, box = lattice.crystal("bcc", cells, a, 0.1, seed)
    rng = np.random.default_rng(seed)
    keep = np.sort(rng.permutation(len(x))[:n])
    return np.ascontiguousarray(x[keep]), box, rng.integers(1, types + 1, n).astype(np.int32)


def _reference(fit, configs, types):
    b, db = fit.raw()
    ai, aj, rij = fit.pairs()
    out = []
    K = fit.ncoeff
    for c, (x, _, ty) in enumerate(configs):
        B, dB, sl = fit.config(c, b, db)                     # (N, K), (P, 3, K)
        i, j, r = ai[sl], aj[sl], rij[sl]
        bi, bd, bv = np.zeros((types, K)), np.zeros((3, len(x), types, K)), np.zeros((6, types, K))
        mag = np.zeros_like(bd)
        for t in range(types):
            bi[t] = B[ty == t + 1].sum(0)
            p = np.nonzero(ty[i] == t + 1)[0]
            for comp in range(3):
                np.add.at(bd[comp, :, t], i[p], dB[p, comp])
                np.add.at(bd[comp, :, t], j[p], -dB[p, comp])
                np.add.at(mag[comp, :, t], i[p], np.abs(dB[p, comp]))
                np.add.at(mag[comp, :, t], j[p], np.abs(dB[p, comp]))
            for m, (u, v) in enumerate(((0, 0), (1, 1), (2, 2), (1, 2), (0, 2), (0, 1))):
                bv[m, t] = -(r[p, u, None] * dB[p, v]).sum(0)
        out.append((bi.reshape(-1), bd.reshape(3, len(x), -1), bv.reshape(6, -1), mag.reshape(3, len(x), -1)))
    return out


@pytest.mark.parametrize("sizes,J,types", [([2, 511, 512, 513], 4, 1), ([2047, 1, 65], 2, 1), ([2100, 30], 4, 1),
                                           ([64, 40], 8, 1), ([63, 100], 6, 1), ([128, 60], 6, 2), ([70, 33], 4, 3),
                                           ([60, 95], 4, 5)])
def test_tallies_and_normal_equations(sizes, J, types):
    configs = [_config(n, 40 + k, types=types) for k, n in enumerate(sizes)]
    if sizes[0] == 64:   # tightly packed cells: more than 128 incoming pairs per atom
        configs.append(_config(54, 90, a=1.7))
    fit = SnapFit(configs, J, elemradius=(0.5, 0.47, 0.45, 0.52, 0.49)[:types],
                  elemweight=(1.0, 0.8, 0.9, 1.1, 0.7)[:types])
    fit.compute()
    ref = _reference(fit, configs, types)
    print(f"tallies {sizes} J={J} types={types}", flush=True)
    for (bi, bd, bv), (ri, rd, rv, mag) in zip(fit.descriptors(), ref):
        assert np.max(np.abs(bi - ri)) <= 1e-11 * max(np.max(np.abs(ri)), 1e-300)
        assert np.all(np.abs(bd - rd) <= 1e-11 * (mag + 1e-300))
        assert np.max(np.abs(bv - rv)) <= 1e-11 * max(np.max(np.abs(rv)), 1e-300)
    rng = np.random.default_rng(1)
    C, N = len(configs), sum(len(c[0]) for c in configs)
    e, f, s = rng.normal(size=C), rng.normal(size=(N, 3)), rng.normal(size=(C, 6))
    we, wf, ws = (rng.uniform(0.5, 2, C) for _ in range(3))
    L, h = fit.normal_equations(e, f, s, we, wf, ws)
    at = 0
    Lr, hr, Lm, hm = (np.zeros_like(v) for v in (L, h, L, h))
    for c, (ri, rd, rv, _) in enumerate(ref):
        n = len(configs[c][0])
        rows = ((ri[None], e[c:c + 1], we[c]),
                (rd.transpose(1, 0, 2).reshape(3 * n, -1), f[at:at + n].ravel(), wf[c]), (rv, s[c], ws[c]))
        for g, (a, b, w) in enumerate(rows):
            Lr[g] += w * w * a.T @ a
            hr[g] += w * w * a.T @ b
            Lm[g] += w * w * np.abs(a).T @ np.abs(a)
            hm[g] += w * w * np.abs(a).T @ np.abs(b)
        at += n
    assert np.all(np.abs(L - Lr) <= 1e-11 * (Lm + 1e-300))
    assert np.all(np.abs(h - hr) <= 1e-11 * (hm + 1e-300))
