"""The staged neighbour build's plan (a unit's stencil intervals merged into
slot segments) and its two searches, one lane a particle and, for up to 32
units, four lanes a particle, against the FP32 oracle, bit for bit: units of
one grid row, of several whose stencils overlap, and of more than the plan
takes (which keep global slots); last units of one and of few particles; 32
units and 33; lists longer than a lane collects; a table cut off at
max_neighbors; particles outside the grid."""
import numpy as np
import pytest

from particlesolver_amd import System, scenes
from oracle import load_scene
from test_gpu_parity import assert_bitexact, staged_compare

pytestmark = pytest.mark.gpu


def check_tables(sc):
    ref = load_scene(sc, "f32")
    with System(sc.params) as g:
        sc.load_into(g)
        for s in (g, ref):
            s.predict(sc.dt)
            s.build_grid()
            s.find_neighbors()
        gn, gt = g.neighbors()
        rn, rt = ref.neighbors()
        assert_bitexact(gn, rn, "neighbour counts")
        used = np.arange(sc.params.max_neighbors)[None, :] < rn[:, None]
        assert_bitexact(np.where(used, gt, 0), np.where(used, rt, 0), "neighbour table")
        st = g.status()
        assert st.flags == ref.status().flags and st.max_neighbors == ref.status().max_neighbors
        return st


@pytest.mark.parametrize("dims,h,max_neighbors", [
    ((1, 1, 1), 0.2, 64), ((257, 1, 1), 0.2, 64), ((4, 40, 4), 0.2, 64), ((12, 9, 13), 0.2, 64),
    ((16, 8, 64), 0.2, 64), ((16, 8, 65), 0.2, 64), ((30, 20, 30), 0.2, 64), ((20, 12, 20), 0.4, 320),
    ((20, 12, 20), 0.4, 100), ((40, 20, 40), 0.4, 320)])
def test_plans_and_searches(gpu_available, dims, h, max_neighbors):
    check_tables(scenes.dam_break(*dims, h=h, max_neighbors=max_neighbors))


@pytest.mark.parametrize("n", [600, 8192, 8193, 20000])
def test_cloud_with_clamped_cells(gpu_available, n):
    """uniform random positions, a quarter of them outside the grid"""
    sc = scenes.dam_break(2, 2, 2, max_neighbors=128)
    rng = np.random.default_rng(n)
    box = 0.2 * np.ceil((n / 8.0) ** (1.0 / 3.0))
    sc.params.grid[:] = [int(round(box / 0.2))] * 3
    sc.params.max_particles = n
    pos = (rng.uniform(-0.05, 1.05, (n, 3)) * box).astype(np.float32)
    big = scenes.Scene(sc.params, pos, np.ones(n, np.float32), np.zeros(n, np.int32),
                       np.full(n, sc.rest_density[0], np.float32), sc.dt)
    st = check_tables(big)
    assert st.staged_units > 0


def test_split_search_trajectory(gpu_available):
    staged_compare(scenes.dam_break(20, 9, 19, max_neighbors=64), 3)
