"""ps_step on a small scene replays graphs after a number of equal calls (one
per arrangement its buffers rotate through).  Against the FP32 oracle, bit for
bit, over enough calls that every arrangement is captured and replayed several
times, with eager work (other step lengths, another dt, changed parameters, a
graph of ps_step_graph, velocities set, export) between."""
import numpy as np
import pytest

from particlesolver_amd import System, capi, scenes
from oracle import load_ref2d, load_scene
from test_gpu_parity import assert_bitexact

pytestmark = pytest.mark.gpu


def same(g, ref, what):
    assert_bitexact(g.positions(), ref.positions(), what + " positions")
    assert_bitexact(g.velocities(), ref.velocities(), what + " velocities")


@pytest.mark.parametrize("iterations,substeps", [(4, 1), (3, 1), (3, 2), (2, 3)])
def test_replayed_steps_bitexact(gpu_available, iterations, substeps):
    sc = scenes.dam_break(10, 8, 9, iterations=iterations, max_neighbors=64)
    ref = load_scene(sc, "f32")
    with System(sc.params) as g, capi.DeviceBuffer(16 * sc.n) as buf:
        sc.load_into(g)
        for call in range(44):
            g.step(sc.dt, substeps)
            ref.step(sc.dt, substeps)
            if call % 5 == 0:
                g.export_device(capi.PS_FIELD_POSITIONS, buf.ptr)
                g.synchronize()
                assert_bitexact(buf.numpy(np.float32, (sc.n, 4))[:, :3], ref.positions(), "export after %d" % call)
        same(g, ref, "replayed")
        assert g.status().substeps == 44 * substeps and g.status().iterations == 44 * substeps * iterations


def test_eager_work_between_replays(gpu_available):
    sc = scenes.rope_over_fluid()
    ref = load_scene(sc, "f32")
    with System(sc.params) as g:
        sc.load_into(g)

        def both(call):
            call(g)
            call(ref)

        for block in range(3):
            for _ in range(26):
                both(lambda s: s.step(sc.dt, 1))
            same(g, ref, "block %d" % block)
            both(lambda s: s.step(sc.dt, 2))          # another length starts over
            both(lambda s: s.step(0.75 * sc.dt, 1))   # and another dt
            g.step_graph(sc.dt, 12)
            ref.step(sc.dt, 12)
            both(lambda s: s.step(sc.dt, 1))          # the buffers no longer as the graph left them
            g.step_graph(sc.dt, 12)
            ref.step(sc.dt, 12)
            same(g, ref, "block %d, after other calls" % block)
            for s in (g, ref):
                s.begin(sc.dt)
                for _ in range(sc.params.iterations):
                    s.iterate()
                s.end()
            same(g, ref, "block %d, after single stages" % block)
        p = sc.params.copy()
        p.gravity[:] = (1.0, -5.0, 0.0)
        for _ in range(20):
            both(lambda s: s.step(sc.dt, 1))
        g.set_params(p)
        ref.set_params(p)
        for _ in range(24):
            both(lambda s: s.step(sc.dt, 1))
        same(g, ref, "after set_params")


def test_two_handles_and_the_2d_solver(gpu_available):
    sc = scenes.reference_two_fluids()
    refs = [load_ref2d(sc, "f32"), load_ref2d(sc, "f32")]
    with System(sc.params) as a, System(sc.params) as b:
        for s in (a, b):
            sc.load_into(s)
        for call in range(40):
            a.step(sc.dt, 1)
            refs[0].step(sc.dt, 1)
            if call % 2:
                b.step(sc.dt, 2)
                refs[1].step(sc.dt, 2)
        same(a, refs[0], "first handle")
        same(b, refs[1], "second handle")


@pytest.mark.parametrize("change", ["dt", "length", "params", "tuning", "graph"])
def test_graphs_let_go_of_while_a_replay_runs(gpu_available, change):
    """A replayed call is followed at once, with no wait, by one that lets go
    of the graphs, and the next capture destroys them."""
    sc = scenes.dam_break(14, 12, 13, max_neighbors=64)
    ref = load_scene(sc, "f32")
    with System(sc.params) as g:
        sc.load_into(g)
        for block in range(10):
            dt, sub = sc.dt, 1
            if change == "dt":
                dt = sc.dt * (1.0 if block % 2 else 0.75)
            if change == "length":
                sub = 1 + block % 2
            for _ in range(21):
                g.step(dt, sub)
                ref.step(dt, sub)
            if change == "params":
                g.set_params(sc.params)
            if change == "tuning":
                g.set_tuning({"lambda": 64 * (1 + block % 4)})
            if change == "graph":
                g.step_graph(0.5 * sc.dt, 4)
                ref.step(0.5 * sc.dt, 4)
        same(g, ref, change)
        g.synchronize()
        g.step(sc.dt, 1)
        ref.step(sc.dt, 1)
        same(g, ref, change + ", after a wait")
