"""Worlds whose LDS layout lies at the 160 KB a workgroup can have: what fits is accepted, launches
and gives the results of the same world at its usual capacities; what doesn't is refused."""

import numpy as np
import pytest

import metalrobo as mr
from test_mlp_world import chain_world, run


@pytest.mark.gpu
def test_sample_capture_at_a_large_constraint_capacity(gpu):
    """The learned instance holds 36 bytes of LDS a constraint beside the chain workload's 28 KB, so
    sample capture fits up to about 3,800 constraints."""
    model, cfg = chain_world()
    _, plain = run(model, cfg, 2)
    big = chain_world(constraint_capacity=3800)[1]
    w, got = run(model, big, 2, setup=lambda w: w.set_mlp_capture(True))
    for a, b in zip(got, plain):
        assert np.array_equal(np.ascontiguousarray(a).view(np.uint8), np.ascontiguousarray(b).view(np.uint8))
    over = mr.World(model, chain_world(constraint_capacity=4096)[1])
    with pytest.raises(Exception, match="160 KiB"):
        over.set_mlp_capture(True)
