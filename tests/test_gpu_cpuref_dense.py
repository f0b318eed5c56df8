"""The CPU-reference mode's neighbour lists where they can go wrong, against
ref2d's FP32 build, bit for bit: more neighbours than a list holds (64) and
than two lists, fewer particles than one tile and counts that end inside one,
coincident particles, fluid and gas objects together."""
import numpy as np
import pytest

from particlesolver_amd import System, scenes
from oracle import load_ref2d
from test_gpu_parity import assert_bitexact

pytestmark = pytest.mark.gpu


def block(nx, ny, spacing, x0, y0, seed):
    p = scenes.fluid_block(nx, ny, 1, spacing, (x0, y0, 0.0), 0.2 * spacing, seed)
    p[:, 2] = 0.0
    return p


@pytest.mark.parametrize("nx,ny,spacing", [(3, 2, 0.5), (13, 5, 0.6), (20, 15, 0.3), (27, 19, 0.2), (24, 43, 0.45)])
def test_neighbour_lists_bitexact(gpu_available, nx, ny, spacing):
    a = block(nx, ny, spacing, -nx * spacing, 0.1, 11)
    b = block(nx, ny, spacing, 0.0, 0.1, 12)
    c = block(nx, ny, spacing, -0.5 * nx * spacing, ny * spacing + 0.2, 13)
    if len(b) > 8:
        b[5] = b[7]
    n = len(a) + len(b) + len(c)
    half = nx * spacing + 1.0
    p = scenes.cpu_reference_params((-half, 0.0, -1.0), (half, 100.0, 1.0), 0.25, 2.0, 3, n)
    sc = scenes.FluidObjectsScene(p, [(a, 1.0), (c, 0.75, "open gas"), (b, 2.5)], 0.01)
    ref = load_ref2d(sc, "f32")
    with System(p) as g:
        sc.load_into(g)
        for step in range(3):
            g.step(sc.dt, 1)
            ref.step(np.float32(sc.dt), 1)
            assert_bitexact(g.positions(), ref.positions(), "positions after step %d" % step)
            assert_bitexact(g.velocities(), ref.velocities(), "velocities after step %d" % step)
