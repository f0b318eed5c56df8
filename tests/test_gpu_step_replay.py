"""ps_step on a small scene replays graphs after a number of equal calls (one
per arrangement its buffers rotate through).  Against the FP32 oracle, bit for
bit, over enough calls that every arrangement is captured and replayed several
times, with eager work (other step lengths, another dt, changed parameters, a
graph of ps_step_graph, velocities set, export) between; the library's count of
replayed calls says that they were."""
import ctypes
import threading

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
        assert g.step_replays()[0] > 0 and g.step_replays()[1] == 44 - 16


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
            assert g.step_replays()[0] > 0 and g.step_replays()[1] == 10 * (block + 1)
            both(lambda s: s.step(sc.dt, 2))          # another length starts over
            assert g.step_replays() == (0, 10 * (block + 1))
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
        assert g.step_replays()[0] > 0
        g.set_params(p)
        ref.set_params(p)
        assert g.step_replays()[0] == 0
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
        assert a.step_replays()[1] == 40 - 16 and b.step_replays()[1] == 20 - 16


def replay_bitexact(sc, calls, substeps=1):
    ref = load_scene(sc, "f32")
    with System(sc.params) as g:
        sc.load_into(g)
        for _ in range(calls):
            g.step(sc.dt, substeps)
            ref.step(sc.dt, substeps)
        same(g, ref, "%d calls" % calls)
        assert g.status().flags == ref.status().flags
        return g.step_replays()


@pytest.mark.parametrize("flags", [0, capi.PS_FLAG_NO_LDS_STAGING, capi.PS_FLAG_REBUILD_EVERY_ITERATION,
                                   capi.PS_FLAG_SLEEPING])
@pytest.mark.parametrize("iterations", [3, 4])
def test_bodies_and_contacts_replayed(gpu_available, flags, iterations):
    """Cloth and rigid cubes (whose rotations carry over from one replay to
    the next) falling on two fluids."""
    sc = scenes.mixed(cloth_n=16, cubes=(2, 1, 2), fluid=(8, 6, 6), box=(5.0, 8.0, 5.0), iterations=iterations)
    sc.params = sc.params.copy()
    sc.params.flags |= flags
    graphs, replayed = replay_bitexact(sc, 48)
    assert graphs > 0 and replayed == 48 - 16


@pytest.mark.parametrize("dims,replays", [((64, 16, 64), True), ((65537, 1, 1), False)])
def test_largest_replayed_scene(gpu_available, dims, replays):
    sc = scenes.dam_break(*dims, max_neighbors=64, iterations=2)
    graphs, replayed = replay_bitexact(sc, 22)
    assert (graphs > 0, replayed) == ((True, 6) if replays else (False, 0))


def test_batch_replayed(gpu_available):
    b = scenes.ensemble(nscenes=3, nmin=300, nmax=2500)
    with System(b.params, b.descs) as g, System(b.params, b.descs) as ref:
        b.load_into(g)
        b.load_into(ref)
        for _ in range(40):
            g.step(b.dt, 1)
            ref.begin(b.dt)
            for _ in range(b.params.iterations):
                ref.iterate()
            ref.end()
        same(g, ref, "batch")
        assert g.step_replays()[1] == 24 and ref.step_replays() == (0, 0)


def test_threads_step_while_another_allocates_and_waits(gpu_available):
    """Handles in threads of their own reach their captures while the main
    thread allocates, frees and waits for the device."""
    sc = scenes.dam_break(12, 10, 11, max_neighbors=64)
    ref = load_scene(sc, "f32")
    for _ in range(60):
        ref.step(sc.dt, 1)
    hip = ctypes.CDLL("libamdhip64.so.7")
    handles, failures = [System(sc.params) for _ in range(4)], []

    def work(g):
        try:
            for _ in range(60):
                g.step(sc.dt, 1)
            g.synchronize()
        except Exception as e:
            failures.append(e)

    try:
        for g in handles:
            sc.load_into(g)
        threads = [threading.Thread(target=work, args=(g,)) for g in handles]
        for t in threads:
            t.start()
        rounds = 0
        while any(t.is_alive() for t in threads) or rounds < 20:
            p = ctypes.c_void_p()
            assert hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(1 << 20)) == 0
            assert hip.hipDeviceSynchronize() == 0
            assert hip.hipFree(p) == 0
            rounds += 1
        for t in threads:
            t.join()
        assert not failures, failures
        for g in handles:
            same(g, ref, "a thread's handle")
            assert g.step_replays()[1] == 60 - 16
    finally:
        for g in handles:
            g.close()


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


def test_graphs_of_a_process_are_bounded(gpu_available):
    """More handles than the process's 1,024 step graphs go round: the last
    ones launch, and capture once others have closed."""
    sc = scenes.dam_break(3, 2, 2, max_neighbors=32)
    ref = load_scene(sc, "f32")
    handles = []
    try:
        for _ in range(300):
            handles.append(System(sc.params))
            sc.load_into(handles[-1])
            for _ in range(24):
                handles[-1].step(sc.dt, 1)
        held = [g.step_replays()[0] for g in handles]
        assert sum(held) == 1024 and held[0] > 0 and held[-1] == 0, held
        ref.step(sc.dt, 24)
        for g in (handles[0], handles[-1]):
            same(g, ref, "24 calls")
        for g in handles[:10]:
            g.close()
        for _ in range(8):
            handles[-1].step(sc.dt, 1)
        ref.step(sc.dt, 8)
        same(handles[-1], ref, "32 calls")
        assert handles[-1].step_replays()[0] > 0
    finally:
        for g in handles:
            g.close()
