"""bench.py's roofline figures: what a launch must move, and the byte-counter
profiles of the headline workload that go with it."""
import os
import sys

import pytest

ROOT = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..")
sys.path.insert(0, ROOT)


@pytest.mark.parametrize("regions", [False, True])
def test_headline_has_a_measured_traffic_profile(regions):
    import bench
    from seidart_amd import configs
    problems = configs.batched_layered(nt=60)
    alg = bench.algorithmic_bytes(problems, [len(p.shots) for p in problems], 4)
    got = bench.measured_traffic(regions, alg)
    # the counters see at least what a launch must move, and less than that
    # many bytes per step of the launch (two steps, five on regions)
    assert got is not None and alg < got < (5 if regions else 2) * alg
    assert bench.measured_traffic(regions, alg + 1) is None
