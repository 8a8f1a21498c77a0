"""bench.py's words per node against the recorded HBM traffic."""
import json
import os
import sys

import pytest

ROOT = os.path.abspath(os.path.join(os.path.dirname(__file__), ".."))
sys.path.insert(0, ROOT)
import bench  # noqa: E402

L2_BYTES = 8 * (4 << 20)  # eight XCDs

with open(os.path.join(ROOT, "profiles", "traffic.json")) as f:
    TRAFFIC = json.load(f)


@pytest.mark.parametrize("family", sorted(bench.WORDS))
def test_words_are_moved(family):
    """A family's words are a floor of what its launches move: the measured
    bytes are no fewer, but for what one L2 can keep from a launch's reads or
    hold of its writes."""
    assert TRAFFIC["workload"] == bench.workload_name(bench.HEADLINE_DIMS)
    n1 = bench.HEADLINE_DIMS[0] * bench.HEADLINE_DIMS[1] * bench.HEADLINE_DIMS[2]
    moved = TRAFFIC["families"][f"{family}@1"]["hbm_bytes_per_launch"]
    assert moved >= bench.level_words(family, 1) * 8 * n1 - L2_BYTES
