"""Copies between host arrays and the device through the shared pinned chunks: several threads at once, each with a
system of its own, sizes on both sides of the pieces the copies are cut into; every byte as it was."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from mdp_amd import lattice
from test_gpu_md import _engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [(3, 3, 3), (16, 16, 17), (40, 30, 31)])
def test_states_of_several_threads(cells):
    x, box = lattice.crystal("bcc", cells, 3.316, 0.02, 1)
    n = len(x)
    engines = [_engine(x, box, 2, lattice.snap_coefficients(5, seed=1)) for _ in range(4)]

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

    with ThreadPoolExecutor(4) as ex:
        assert all(ex.map(one, range(4)))
