"""Contacts, distance constraints and shape matching as blocks of their own
beside the fluid's multipliers, against the FP32 oracle, bit for bit, where
they can go wrong: walkers, linked particles and bodies at the edges of their
blocks (64, 128 and 8 of them; one; none), lists of links past four and none,
partners with w = 0, contacts in more chunks than four lanes take at once and
more than a list holds, and constraints added to a scene that has run
without."""
import numpy as np
import pytest

from particlesolver_amd import System, capi, scenes
from oracle import load_scene
from test_gpu_parity import assert_bitexact, staged_compare

pytestmark = pytest.mark.gpu


def crowd(walkers, linked, bodies, seed=0x5EED0D01):
    """A fluid block with `walkers` moving CLOTH and SOLID particles (three of
    each body's in a body phase), `linked` particles that share links, and
    four static ones, all strewn over the block."""
    rng = np.random.default_rng(seed)
    sc = scenes.dam_break(8, 5, 7, max_neighbors=96, iterations=2, seed=seed)
    nf, nb = sc.n, 3 * bodies
    ns = 4
    gas = max(linked - walkers, 0)                      # linked, but not walking
    extra = walkers + gas + ns + nb
    pos = np.concatenate([sc.pos, rng.uniform((0.02, 0.02, 0.02), (0.78, 0.6, 0.68), (extra, 3)).astype(np.float32)])
    n = nf + extra
    w = np.ones(n, np.float32)
    ph = np.zeros(n, np.int32)
    ph[nf:nf + walkers] = np.where(np.arange(walkers) % 3 == 0, capi.PHASE_SOLID, capi.PHASE_CLOTH)
    w[nf:nf + walkers] = rng.choice([1.0, 0.5, 2.0], walkers)
    ph[nf + walkers:nf + walkers + gas] = capi.PHASE_GAS
    st = nf + walkers + gas
    ph[st:st + ns] = capi.PHASE_SOLID
    w[st:st + ns] = 0.0
    ph[st + ns:] = capi.PHASE_RIGID + np.arange(nb) // 3
    p = sc.params.copy()
    p.max_particles = n
    r0 = np.full(n, sc.rest_density[0], np.float32)
    out = scenes.Scene(p, pos, w, ph, r0, sc.dt, name="crowd")
    if linked > 1:
        a = nf + np.arange(linked)
        pairs = [(a[k], a[k + 1]) for k in range(linked - 1)]
        # the first has eight links more, one particle a static partner
        pairs += [(a[0], a[k]) for k in range(2, min(linked, 10))] + [(a[linked // 2], st), (st + 1, a[1])]
        m = len(pairs)
        out.distance = (np.array(pairs, np.uint32), rng.uniform(0.05, 0.2, m).astype(np.float32),
                        rng.uniform(0.1, 1.0, m).astype(np.float32))
        out.pins = (np.array([a[0]], np.uint32), pos[a[0]][None])
    out.bodies = [(np.arange(st + ns + 3 * k, st + ns + 3 * k + 3), 0.5) for k in range(bodies)]
    return out


def unstaged(sc):
    sc.params = sc.params.copy()
    sc.params.flags |= capi.PS_FLAG_NO_LDS_STAGING
    return sc


@pytest.mark.parametrize("staged", [True, False])
@pytest.mark.parametrize("walkers,linked,bodies", [(1, 0, 0), (64, 64, 1), (65, 129, 0), (0, 2, 8), (63, 128, 9),
                                                   (0, 0, 1)])
def test_block_edges(gpu_available, walkers, linked, bodies, staged):
    sc = crowd(walkers, linked, bodies)
    staged_compare(sc if staged else unstaged(sc), 2)


@pytest.mark.parametrize("staged", [True, False])
@pytest.mark.parametrize("spacing", [0.035, 0.025])     # about 100 and 270 contacts a particle
def test_many_contacts(gpu_available, spacing, staged):
    rng = np.random.default_rng(7)
    m = 9
    g = np.stack(np.meshgrid(*(np.arange(m) * spacing,) * 3, indexing="ij"), -1).reshape(-1, 3)
    pos = (g + rng.uniform(-0.1, 0.1, g.shape) * spacing + 1.0).astype(np.float32)
    n = len(pos)
    p = scenes.pbf_params((0.0, 0.0, 0.0), (3.0, 3.0, 3.0), 0.12, 0.05, 2, n, 480)
    ph = np.where(np.arange(n) % 5 == 0, capi.PHASE_CLOTH, capi.PHASE_SOLID).astype(np.int32)
    w = rng.choice([1.0, 0.5, 0.0], n, p=[0.6, 0.3, 0.1]).astype(np.float32)
    sc = scenes.Scene(p, pos, w, ph, np.ones(n, np.float32), 1e-3)
    staged_compare(sc if staged else unstaged(sc), 1)


def test_constraints_added_later(gpu_available):
    ref = load_scene(crowd(40, 0, 0), "f32")
    bare = crowd(40, 0, 0)
    n, dt = bare.n, bare.dt
    pairs = np.array([(n - 10, n - 9), (n - 9, 3), (5, 6)], np.uint32)
    with System(bare.params) as g:
        bare.load_into(g)

        def both(call):
            call(g)
            call(ref)
            for s in (g, ref):
                s.step(dt, 2)
            assert_bitexact(g.positions(), ref.positions(), "positions")

        both(lambda s: None)
        both(lambda s: s.add_distance_constraints(pairs, np.full(3, 0.08, np.float32), np.full(3, 0.7, np.float32)))
        both(lambda s: s.add_point_constraints(np.array([2], np.uint32), bare.pos[2:3]))
        both(lambda s: s.add_distance_constraints(pairs[:1] - 1, np.full(1, 0.09, np.float32)))
