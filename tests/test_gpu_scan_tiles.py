"""Cell offsets of grids at the edges of the scan's tiles (4,096 cells, sums of
up to 32 tiles formed by every block itself, of more by a launch before it),
with cell counts that are no multiple of four, against numpy; and again after
the particles have moved, from counts cleared by the build before."""
import numpy as np
import pytest

from particlesolver_amd import System, capi, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [1, 3, 4095, 4096, 4097, 8194, 32 * 4096 - 1, 32 * 4096, 32 * 4096 + 1, 33 * 4096 + 2])
def test_offsets(gpu_available, cells):
    rng = np.random.default_rng(cells)
    n, cell = 3000, 0.25
    p = scenes.pbf_params((0.0, 0.0, 0.0), (cells * cell, cell, cell), cell, cell / 4.0, 2, n, 96)
    assert list(p.grid) == [cells, 1, 1]
    p.gravity[:] = (0.0, 0.0, 0.0)
    # half of the particles in few cells, among them the first and the last
    crowd = rng.choice(np.unique([0, cells // 2, cells - 1, min(cells - 1, 4095), min(cells - 1, 4096)]), n)
    at = np.where(rng.random(n) < 0.5, crowd, rng.integers(0, cells, n))
    pos = np.full((n, 3), 0.125, np.float32)
    pos[:, 0] = (at + 0.5) * cell
    with System(p) as g:
        g.add_particles(pos, np.tile(np.float32([cell, 0.0, 0.0]), (n, 1)))
        for step in range(3):
            g.predict(1.0 if step else 0.0)     # from the second on one cell further
            g.build_grid()
            index, key, off = g.grid()
            want = np.minimum(at + (1 if step else 0), cells - 1)
            assert np.array_equal(key, np.sort(want))
            assert np.array_equal(off, np.searchsorted(np.sort(want), np.arange(cells + 1)))
            assert np.array_equal(index, np.lexsort((np.arange(n), want)))
