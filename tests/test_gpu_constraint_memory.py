"""What contact walkers and links cost in device memory on a handle of large
capacity: a rank and a result per particle of the capacity for each kind that
the scene has (20 bytes), and lists of the walkers or linked particles there
are, grown as more are added.  Results over the growth against the FP32 oracle."""
import ctypes

import numpy as np
import pytest

from particlesolver_amd import System, capi, scenes
from oracle import load_scene
from test_gpu_parity import assert_bitexact

pytestmark = pytest.mark.gpu

CAPACITY = 1 << 22
# hipMalloc's granularity (2 MiB an allocation, five of them) and the small lists
SLACK = 16 << 20


def free_bytes():
    hip = ctypes.CDLL("libamdhip64.so.7")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipDeviceSynchronize() == 0
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("walkers,links,per_particle", [(True, False, 20), (False, True, 20), (True, True, 40)])
def test_memory_by_kind(gpu_available, walkers, links, per_particle):
    sc = scenes.dam_break(8, 4, 8, max_neighbors=32)
    p = sc.params.copy()
    p.max_particles = CAPACITY
    with System(p) as g:
        sc.load_into(g)
        g.step(sc.dt, 1)  # the runtime's own buffers
        before = free_bytes()
        n = 100
        pos = np.full((n, 3), 0.1, np.float32)
        pos[:, 0] += 0.01 * np.arange(n, dtype=np.float32)
        phase = np.full(n, capi.PHASE_CLOTH if walkers else capi.PHASE_GAS, np.int32)
        first = g.add_particles(pos, None, np.ones(n, np.float32), phase, np.ones(n, np.float32))
        if links:
            i = first + np.arange(n - 1, dtype=np.uint32)
            g.add_distance_constraints(np.stack([i, i + 1], 1), np.full(n - 1, 0.1, np.float32))
        took = before - free_bytes()
        print("walkers %s links %s: %.1f MiB" % (walkers, links, took / 2**20), flush=True)
        assert took <= per_particle * CAPACITY + SLACK
        g.step(sc.dt, 1)


def test_lists_grow_between_steps(gpu_available):
    rng = np.random.default_rng(11)
    sc = scenes.dam_break(6, 4, 6, max_neighbors=96, iterations=2)
    sc.params = sc.params.copy()
    sc.params.max_particles = 600
    ref = load_scene(sc, "f32")
    with System(sc.params) as g:
        sc.load_into(g)
        for n in (1, 2, 3, 10, 60):
            pos = rng.uniform(0.05, 0.9, (n, 3)).astype(np.float32)
            first = g.n
            for s in (g, ref):
                s.add_particles(pos, None, np.ones(n, np.float32), np.full(n, capi.PHASE_CLOTH, np.int32),
                                np.ones(n, np.float32))
            pairs = [(first + k, (first + k + 1) if k + 1 < n else 0) for k in range(n)]
            for s in (g, ref):
                s.add_distance_constraints(np.array(pairs, np.uint32), np.full(n, 0.08, np.float32))
                for _ in range(18):
                    s.step(sc.dt, 1)
            assert_bitexact(g.positions(), ref.positions(), "positions with %d more" % n)
            assert_bitexact(g.velocities(), ref.velocities(), "velocities with %d more" % n)
