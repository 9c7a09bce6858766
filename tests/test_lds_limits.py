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


def largest_accepted(overrides):
    lo, hi = 256, 4097
    while hi - lo > 1:
        mid = (lo + hi) // 2
        try:
            mr.World(*chain_world(constraint_capacity=mid, **overrides)).close()
            lo = mid
        except mr.MetalRoboError as err:
            assert "bytes of LDS" in str(err), err
            hi = mid
    return lo


@pytest.mark.gpu
@pytest.mark.parametrize("hybrid", [False, True])
def test_the_largest_accepted_capacity_launches(gpu, hybrid):
    """The relaxed Jacobi solver takes 40 bytes of LDS a constraint. The kernels' own 160 bytes count too:
    a layout that only just fits must still launch, and one step more must have been refused."""
    overrides = dict(solver=mr.MR_SOLVER_RELAXED_JACOBI)
    if hybrid:
        overrides.update(ccd_mode=1, max_ccd_events=4, max_ccd_iterations=16, ccd_distance_tolerance=1e-3,
                         ccd_time_tolerance=1e-5, ccd_minimum_advance=1e-5)
    most = largest_accepted(overrides)
    assert 256 < most < 4096
    w, got = run(*chain_world(constraint_capacity=most, **overrides), 2)
    lds = w.layout().lds_bytes_per_environment
    assert 160 * 1024 - 160 - 56 < lds <= 160 * 1024 - 160
    _, plain = run(*chain_world(**overrides), 2)
    for a, b in zip(got, plain):
        assert np.array_equal(np.ascontiguousarray(a).view(np.uint8), np.ascontiguousarray(b).view(np.uint8))
