"""MD engine kernels whose work is split for systems too small to fill the GPU, at the sizes where the split can
go wrong: one atom, a block of 64 atoms less one and plus one, boxes with a single cell along an axis.

Neighbour lists are compared as sorted sets, bit for bit, with the oracle's brute force; energies, forces and
virials with the oracle's force chain within 1e-10 of the max norm, as in test_gpu_md.py.
"""
import numpy as np
import pytest

from mdp_amd import lattice
from test_gpu_md import RCUTFAC, _coeff, _engine, _first_step_vs_oracle, _oracle_bruteforce

pytestmark = pytest.mark.gpu


def _atoms(n, seed):
    """n atoms of a displaced BCC crystal with vacancies (n = 1: alone in its box)"""
    cells = max(1, int(np.ceil((n / 2) ** (1 / 3))))
    x, box = lattice.crystal("bcc", cells, 3.316, 0.1, seed)
    keep = np.sort(np.random.default_rng(seed).permutation(len(x))[:n])
    return np.ascontiguousarray(x[keep]), box


@pytest.mark.parametrize("n", [1, 63, 65])
@pytest.mark.parametrize("J", [2, 4, 6, 8])
def test_yi_row_workgroups_vs_oracle(oracle, monkeypatch, J, n):
    """compute_yi with a workgroup per output row (variant 208)."""
    monkeypatch.setenv("MDP_YI_VARIANT", "208")
    x, box = _atoms(n, 7 + n + J)
    md = _first_step_vs_oracle(oracle, x, box, J, 3)
    assert md.tuning()["chosen"]["compute_yi_waves"] == 208


@pytest.mark.parametrize("n", [1, 63, 65, 250])
@pytest.mark.parametrize("J", [2, 4, 6, 8])
def test_yi_classes_vs_oracle(oracle, monkeypatch, J, n):
    """compute_yi with the output rows of one j - 2 mb on a wave (variant 308)."""
    monkeypatch.setenv("MDP_YI_VARIANT", "308")
    x, box = _atoms(n, 7 + n + J)
    md = _first_step_vs_oracle(oracle, x, box, J, 3)
    assert md.tuning()["chosen"]["compute_yi_waves"] == 308


@pytest.mark.parametrize("variant", ["4", "16"])
@pytest.mark.parametrize("J,n", [(2, 1), (4, 63), (6, 65), (8, 17), (8, 250)])
def test_ui_lanes_per_atom_vs_oracle(oracle, monkeypatch, J, n, variant):
    """compute_ui with 4 or 16 lanes sharing an atom's pairs: fewer and more pairs than lanes, ragged last waves."""
    monkeypatch.setenv("MDP_UI_VARIANT", variant)
    x, box = _atoms(n, 70 + n + J)
    md = _first_step_vs_oracle(oracle, x, box, J, 5)
    assert md.tuning()["chosen"]["compute_ui"] == int(variant)


def test_neighbor_tile_of_256_lanes_identical(oracle, monkeypatch):
    """The tile kernel on 256 lanes per cell writes the lists of the L1 kernel entry for entry: ragged cells, empty
    cells, and cells whose surroundings need more than one tile."""
    rng = np.random.default_rng(6)
    x1, box1 = lattice.crystal("bcc", 9, 3.316, 0.35, 62)
    x2 = rng.uniform(0.0, 40.0, size=(400, 3))
    x3, box3 = lattice.crystal("bcc", 8, 2.75, 0.2, 63)
    for x, box in ((x1, box1), (x2, np.full(3, 40.0)), (x3, box3)):
        lists = []
        for v in ("0", "1", "2"):
            monkeypatch.setenv("MDP_NB_VARIANT", v)
            md = _engine(x, box, 4, _coeff(oracle, 4, 1))
            md.compute()
            lists.append(md.neighbors())
            md.close()
        for other in lists[1:]:
            for a, b in zip(lists[0], other):
                assert np.array_equal(a, b)


@pytest.mark.parametrize("cells", [(1, 1, 1), (1, 4, 5), (2, 2, 7), (4, 4, 4)])
def test_small_box_lists_vs_bruteforce(oracle, cells):
    """The small-box kernel where images are skipped: flat and long boxes, one cell along an axis."""
    x, box = lattice.crystal("bcc", cells, 3.316, 0.15, 17)
    x[0] = 0.0   # on the lower faces
    md = _engine(x, box, 4, _coeff(oracle, 4, 1))
    md.compute()
    off, nj, ns = md.neighbors()
    o2, j2, s2 = _oracle_bruteforce(oracle, x, box, RCUTFAC + 0.3)
    for i in range(len(x)):
        a = sorted(zip(nj[off[i]:off[i + 1]].tolist(), map(tuple, ns[off[i]:off[i + 1]].tolist())))
        b = sorted(zip(j2[o2[i]:o2[i + 1]].tolist(), map(tuple, s2[o2[i]:o2[i + 1]].tolist())))
        assert a == b, i


@pytest.mark.parametrize("n,J,types,zbl", [(5, 4, 1, True), (250, 6, 2, False), (16000, 2, 1, False), (18522, 2, 2, False),
                                           (18522, 2, 1, True)])
def test_pair_list_blocks_vs_oracle(oracle, n, J, types, zbl):
    """The pair list in blocks of 16 atoms (up to 16,384) and of 64, with gaps at the blocks' ends: pair count,
    energies, forces and virials, also with two types and the ZBL term."""
    from conftest import relerr
    from mdp_amd import snapcpp
    from mdp_amd.md import SnapMD
    if n == 5:
        x, box = lattice.crystal("bcc", 2, 3.316, 0.1, 3)
        x = np.ascontiguousarray(x[:5])
    else:
        x, box = lattice.crystal("bcc", round((n / 2) ** (1 / 3)), 3.316, 0.1, 3) if n != 250 else _atoms(250, 9)
    n = len(x)
    ty = np.random.default_rng(2).integers(1, types + 1, n).astype(np.int32)
    rad, wt = [0.5, 0.48][:types], [1.0, 0.9][:types]
    param = [types, J, RCUTFAC, 0.99363, 0, 1, 1, 0, 0, 0, 0]
    coeff = np.tile(_coeff(oracle, J, 4), types)
    md = SnapMD(x, box, ty, J, coeff, rad, wt, [180.95] * types)
    s = snapcpp.initsna(oracle, param, rad, wt, coeff)
    B = np.diag(box)
    p = snapcpp.pairs_from_box(x, ty, B[0], B[1], B[2], [1, 1, 1], s)
    e, f, w = snapcpp.snappotential_pairs(oracle, s, p)
    if zbl:
        import zbl_oracle
        md.set_zbl()
        g, d, v = zbl_oracle.bind(oracle.cdll)
        z = snapcpp.initsna(oracle, [1, 2, 4.8, 0.99363, 0, 1, 1, 0, 0, 0, 0], [0.5], [1.0])
        q = snapcpp.pairs_from_box(x, np.ones(n, np.int32), B[0], B[1], B[2], [1, 1, 1], z)   # all pairs within 4.8 A
        P, rij, ai = q["ijnum"], np.ascontiguousarray(q["rij"].ravel()), np.ascontiguousarray(q["ai"], np.int32)
        u, ux, ez, fz, wz = np.zeros(P), np.zeros(3 * P), np.zeros(n), np.zeros(3 * n), np.zeros(6 * n)
        g(u, ux, rij, zbl_oracle.TA_MU, P)
        d(ez, fz, u, ux, ai, P, 3)
        v(wz, ux, rij, -0.5, ai, 3, n, P)
        e, f, w = e + ez, f - fz.reshape(n, 3), w + wz.reshape(6, n).T
    md.compute()
    st = md.state()
    assert md.stats()["pairs"] == p["ijnum"]
    assert relerr(st["eatom"], e) < 1e-10
    assert relerr(st["f"], f) < 1e-10
    assert relerr(st["vatom"], w) < 1e-10


@pytest.mark.parametrize("n", [128, 9826])
@pytest.mark.parametrize("nvt", [False, True])
def test_steps_one_by_one_and_in_a_run(oracle, n, nvt):
    """Twelve steps in one run, where a step's first half goes with the end of the step before, against twelve runs of
    one step, where it is a launch of its own: the same arithmetic, so to rounding of the last place along the
    trajectory.  9,826 atoms are above the one-workgroup thermostat."""
    x, box = lattice.crystal("bcc", round((n / 2) ** (1 / 3)), 3.316, 0.05, 8)
    v = lattice.maxwell_boltzmann(len(x), 180.95, 300.0, seed=4)
    out = []
    for chunks in ([12], [1] * 12):
        md = _engine(x, box, 2, _coeff(oracle, 2, 3), v=v)
        if nvt:
            md.set_nvt(300.0, 500.0, 0.05, endstep=50, mtchain=4, nc_tchain=2)
        md.compute()
        for c in chunks:
            md.run(c)
        st = md.state()
        out.append([st[k] for k in ("x", "v", "f", "eatom", "vatom")] + ([np.concatenate([np.ravel(a) for a in md.nvt_state().values()])] if nvt else []))
    for a, b in zip(*out):
        assert np.max(np.abs(a - b)) <= 1e-12 * np.max(np.abs(b))
