"""The bench's byte model of the kernels that read the neighbour table: an
entry counts 2 bytes in a staged unit and 4 in any other, and what the model
says a launch cannot do without is no more than the counted traffic of the
dam break."""
import os
import re
import types

import pytest

import bench

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("staged,units,want", [(0, 0, 4.0), (0, 8, 4.0), (8, 8, 2.0), (6, 8, 2.5)])
def test_entry_bytes(staged, units, want):
    assert bench.entry_bytes(types.SimpleNamespace(staged_units=staged, units=units)) == want


@pytest.mark.parametrize("kernel", sorted(bench.ALGO_BYTES))
def test_model_against_counted_traffic(kernel):
    text = open(os.path.join(ROOT, "profiles", "traffic_dam_break_1M.md")).read()
    n, k = re.search(r"N = (\d+) particles, mean neighbour-table length K = (\d+\.\d+)", text).groups()
    traffic = float(re.search(r"^\| %s \|[^|]+\|[^|]+\| ([\d.]+) \|" % kernel, text, re.M).group(1)) * 1e6
    # every unit of the dam break is staged
    model = bench.ALGO_BYTES[kernel](float(k), 2.0) * int(n)
    assert model <= traffic
    assert bench.ALGO_BYTES[kernel](float(k), 4.0) - bench.ALGO_BYTES[kernel](float(k), 2.0) == \
        pytest.approx(2.0 * float(k))
