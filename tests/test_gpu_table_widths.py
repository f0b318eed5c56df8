"""Staged neighbour tables (16-bit entries, eight to 16 bytes, the first chunks
of each lane loaded ahead of the rest) against the FP32 oracle, bit for bit, at
the widths where they can go wrong: a particle's share of one chunk pair or an
odd number of chunks, rows that end inside a chunk, at the last preloaded chunk
(32 entries) and well past it, and tables cut off at max_neighbors."""
import pytest

from particlesolver_amd import System, scenes
from oracle import load_scene
from test_gpu_parity import assert_bitexact, staged_compare

pytestmark = pytest.mark.gpu


# h = 2 spacings: about 28 neighbours; 3 spacings: about 100
@pytest.mark.parametrize("h,max_neighbors", [(0.2, 4), (0.2, 20), (0.2, 32), (0.2, 36), (0.3, 100), (0.3, 128)])
def test_table_widths(gpu_available, h, max_neighbors):
    sc = scenes.dam_break(64, 8, 16, h=h, max_neighbors=max_neighbors)
    ref = load_scene(sc, "f32")
    with System(sc.params) as g:
        sc.load_into(g)
        for s in (g, ref):
            s.predict(sc.dt)
            s.build_grid()
            s.find_neighbors()
        assert g.status().staged_units > 0
        gn, gt = g.neighbors()
        rn, rt = ref.neighbors()
        assert_bitexact(gn, rn, "neighbour counts")
        for k in range(max_neighbors):
            used = rn > k
            assert_bitexact(gt[used, k], rt[used, k], "entry %d" % k)
    staged_compare(sc, 2)
