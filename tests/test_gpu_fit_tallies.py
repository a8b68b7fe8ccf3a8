"""Tallies and normal equations of the batched fit where their kernels change form: configurations around the
number of threads of a workgroup and above what it holds, atoms with long incoming lists, every number of 16-column
tiles of the normal equations (1 to 5), several element types.

Reference: numpy in float64 on the engine's own B, dB/dr and pair list.  Sums of m terms, m <= 200,000 here, differ by
at most m 2^-53 of the sum of the magnitudes; the orders used keep it far below the 1e-11 allowed.
"""
import time

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
                                           ([2048, 2049, 30], 4, 1),
                                           ([3072, 513, 2100], 2, 1), ([3073, 40], 2, 1),
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


def _tally_time(sizes, J=8):
    """median microseconds per thousand pairs of the tallies, the energy row's normal equations with them"""
    fit = SnapFit([_config(n, 10 + k) for k, n in enumerate(sizes)], J)
    fit.compute()
    e = np.ones(len(sizes))
    t = []
    for _ in range(9):
        t0 = time.perf_counter()
        fit.normal_equations(e, None, None, e, e, e)
        t.append(time.perf_counter() - t0)
    pairs = len(fit.pairs()[0])
    fit.close()
    return 1e9 * float(np.median(t)) / pairs


def test_a_larger_configuration_does_not_slow_the_batch():
    """Configurations of 2,049 to 2,730 atoms, alone and as one of many, keep about the rate of smaller ones.  The form that
    reads dB/dr pair by pair takes six to nine times as long; twice allows for the clock."""
    small, many = _tally_time([2000] * 24), _tally_time([250] * 200)
    for sizes, rate in (([2500] * 24, small), ([2730] * 24, small), ([250] * 200 + [2500], many)):
        now = _tally_time(sizes)
        print(f"{len(sizes)} configurations, largest {max(sizes)}: {now:.2f} us per 1,000 pairs, {rate:.2f} without", flush=True)
        assert now < 2 * rate
