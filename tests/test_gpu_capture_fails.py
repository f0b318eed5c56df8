"""A graph capture that fails (the runtime refuses to begin it, or to
instantiate the graph) costs ps_step nothing but the replay: the call launches
its substeps, equal calls after it do not try again, and the handle's timing
stays on.  ps_step_graph reports the failure.  In a child process whose
runtime calls fail: a library of the two functions is put before the runtime's."""
import subprocess
import sys
import os

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

REFUSE = {
    "instantiate": "int tries; int hipGraphInstantiate(void *a, void *b, void *c, char *d, unsigned long e)"
                   " { tries++; return 2; }",
    "begin": "int tries; int hipStreamBeginCapture(void *a, int mode) { tries++; return 900; }",
}

CHILD = r"""
import ctypes, sys
sys.path.insert(0, %(root)r)
refuse = ctypes.CDLL(%(lib)r, mode=ctypes.RTLD_GLOBAL)
tries = ctypes.c_int.in_dll(refuse, "tries")
import numpy as np
from particlesolver_amd import System, capi, scenes

sc = scenes.rope_over_fluid()
with System(sc.params) as g, System(sc.params) as staged:
    sc.load_into(g)
    sc.load_into(staged)

    def by_stages():
        staged.begin(sc.dt)
        for _ in range(sc.params.iterations):
            staged.iterate()
        staged.end()

    def same(what):
        for a, b in ((g.positions(), staged.positions()), (g.velocities(), staged.velocities())):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), what

    for call in range(40):
        g.step(sc.dt, 1)
        by_stages()
    same("after 40 equal calls")
    assert tries.value == 1, tries.value
    assert g.status().substeps == 40
    # a changed scene may be captured again: it tries once more
    g.set_params(sc.params)
    for call in range(24):
        g.step(sc.dt, 1)
        by_stages()
    same("after set_params")
    assert tries.value == 2, tries.value
    g.timing(["predict_hash"])
    try:
        g.step_graph(sc.dt, 12)
        raise SystemExit("ps_step_graph did not report the failure")
    except capi.PsError as e:
        print("ps_step_graph:", e)
    g.step(sc.dt, 1)
    by_stages()
    same("after ps_step_graph")
    g.synchronize()
    ms, launches = g.timing_read()["predict_hash"]
    assert launches == 1, launches
print("child ok")
"""


@pytest.mark.parametrize("call", sorted(REFUSE))
def test_step_goes_on_when_a_capture_fails(gpu_available, tmp_path, call):
    src, lib = tmp_path / "refuse.c", tmp_path / "librefuse.so"
    src.write_text(REFUSE[call] + "\n")
    subprocess.run(["gcc", "-shared", "-fPIC", str(src), "-o", str(lib)], check=True)
    r = subprocess.run([sys.executable, "-c", CHILD % {"root": ROOT, "lib": str(lib)}], capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0 and "child ok" in r.stdout, r.stdout + r.stderr
