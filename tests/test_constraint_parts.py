"""The counts and launches of the constraint blocks (ps_blocks.hpp), compiled
for the host: every walker, linked particle and body has its lanes up to the
largest scenes (2^30 particles), where their threads are past 2^32, and no
launch is."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "particlesolver_amd", "csrc")

PROBE = r"""
#include <cstdio>
#include <cstdlib>
#include "ps_blocks.hpp"
int main(int, char **v)
{
    const uint32_t nwalk = strtoul(v[1], 0, 0), nlink = strtoul(v[2], 0, 0), nbody = strtoul(v[3], 0, 0);
    const uint32_t fluid = strtoul(v[4], 0, 0), threads = strtoul(v[5], 0, 0);
    const ps::ConParts p = ps::con_parts(nwalk, nlink, nbody, threads);
    printf("%u %u %u\n", p.walks, p.links, p.all);
    for (uint32_t first = 0, k = 0; k < 100; k++) {
        const ps::ConLaunch l = ps::con_launch(p.all, first, fluid, threads);
        printf("%u %u %d\n", first, l.blocks, l.last ? 1 : 0);
        if (l.last) break;
        first += l.blocks;
    }
}
"""


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    d = tmp_path_factory.mktemp("con")
    (d / "probe.cpp").write_text(PROBE)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I" + CSRC, str(d / "probe.cpp"), "-o", str(d / "probe")],
                   check=True)

    def run(*args):
        out = subprocess.run([str(d / "probe")] + [str(a) for a in args], check=True, capture_output=True, text=True)
        rows = [[int(x) for x in line.split()] for line in out.stdout.splitlines()]
        return rows[0], rows[1:]

    return run


@pytest.mark.parametrize("threads", [64, 256, 512])
@pytest.mark.parametrize("nwalk,nlink,nbody", [
    (0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1), (63, 129, 9), (50000, 16384, 3125),
    (1 << 29, 0, 0), ((1 << 29) + 1, 0, 0), (1 << 30, 1 << 30, 1 << 29), (0, 1 << 30, 0), (0, 0, 1 << 26),
    (1 << 30, 0, 1 << 29)])
def test_parts_cover_and_launches_fit(probe, nwalk, nlink, nbody, threads):
    n = max(2 * nbody, nwalk, nlink, 1)
    fluid = -(-n // 256) if threads == 512 else -(-n // threads)
    (walks, links, total), launches = probe(nwalk, nlink, nbody, fluid, threads)
    assert walks == -(-8 * nwalk // threads) and links == -(-4 * nlink // threads)
    bodies = -(-64 * nbody // threads)
    assert total == -(-(walks + links + bodies) // 8) * 8
    at = 0
    for k, (first, blocks, last) in enumerate(launches):
        assert first == at and blocks % 8 == 0
        assert last or blocks > 0
        assert (blocks + (fluid if last else 0)) * threads < 1 << 32
        assert last == (k == len(launches) - 1)
        at += blocks
    assert at == total
    if total + fluid < (1 << 32) // threads - 8:
        assert len(launches) == 1
