"""Copies between host arrays and the device through pinned chunks: several threads at once, each with a system of its own;
arrays below and above a piece of 2 MB (87,381 atoms), above a batch of pieces (16 MB) and, positions and velocities together,
above all chunks of a set (32 MB); every byte as it was."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from mdp_amd import lattice
from test_gpu_md import _engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,threads", [((3, 3, 3), 4), ((16, 16, 17), 4), ((40, 30, 31), 4), ((43, 32, 32), 4),
                                           ((71, 71, 72), 2)])
def test_states_of_several_threads(cells, threads):
    x, box = lattice.crystal("bcc", cells, 3.316, 0.02, 1)
    n = len(x)
    engines = [_engine(x, box, 2, lattice.snap_coefficients(5, seed=1)) for _ in range(threads)]

    def one(k):
        rng = np.random.default_rng(k)
        same = True
        for _ in range(4):
            y = rng.uniform(0, 1, (n, 3)) * box
            v = rng.normal(size=(n, 3))
            engines[k].set_state(y, v)
            s = engines[k].state()
            same = same and np.array_equal(s["x"], y) and np.array_equal(s["v"], v)
        return same

    with ThreadPoolExecutor(threads) as ex:
        assert all(ex.map(one, range(threads)))
