"""The benchmark prices a launch of JOR sweeps by what the case takes: two sweeps where
the library has the pair for it, one where it refuses the pair's entry."""
import sys
from pathlib import Path

import impact_hip as ih

sys.path.insert(0, str(Path(__file__).resolve().parent.parent))
import bench  # noqa: E402


class Case:
    def __init__(self, takes):
        self.takes = takes

    def bench_kernel(self, name, launches):
        if name not in self.takes:
            raise ih.IHError(f"unknown kernel '{name}'")
        return 1.0


def test_sweeps_per_launch():
    c = Case(("jor", "jor_f32", "jor_pair"))
    assert bench.sweeps_per_launch(ih, c, "jor_pair") == 2
    assert bench.sweeps_per_launch(ih, c, "jor_pair_f32") == 1
