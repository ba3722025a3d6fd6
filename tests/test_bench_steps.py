"""bench.py's timed steps: K steps are K gradient shots, in batches."""
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))


@pytest.mark.parametrize("steps,S,positions", [(20, 16, 16), (5, 16, 16), (16, 8, 16), (1, 16, 16), (9, 4, 4), (0, 16, 16)])
def test_steps_are_shots(steps, S, positions):
    import bench
    b = bench.batches_of(steps, S, positions)
    assert sum(len(ids) for ids in b) == steps and all(len(ids) == S for ids in b[:-1])
    assert [i for ids in b for i in ids] == [n % positions for n in range(steps)]
    assert all(len(set(ids)) == len(ids) for ids in b)
