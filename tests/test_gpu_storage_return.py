"""Checkpointed runs of different lengths on one region: what a short run kept (inner stage
states, stress slots) gives way to a longer one's store, and the longer one's to the next, so
that every run has the storage plan of a fresh region.  Most of the device memory is held by a
tensor, so that a plan takes some 40 GB: 128^3 takes 84 MB a state, 0.25 GB a held step and
0.8 GB for the stress slots of a step, of which the first run then keeps some but not all."""
import gc

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BUDGET = 40 << 30
STEPS = (24, 110, 24, 300, 110)      # all held, all held, all held, some held, all held


def _region(c):
    from magudi_amd.solver import Region
    R = Region(c)
    R.set_march_tile(16)
    R.set_z_chunk(32)
    return R


def _fill(c, regions):
    """A tensor that leaves BUDGET to plan with beside `regions` regions and the reserve."""
    import torch
    gc.collect()
    torch.cuda.empty_cache()
    free, total = torch.cuda.mem_get_info()
    state = 40 * c.npoints
    own = 40 * state                           # a region's other arrays, generously
    reserve = max(8 << 30, total // 32)
    hold = free - reserve - regions * own - BUDGET
    if hold < 0:
        pytest.skip("needs 60 GB of device memory")
    return torch.empty(hold, dtype=torch.uint8, device="cuda")


def _run(R, c, nsteps, q0):
    from magudi_amd.solver import Solver
    R.states[0].conservedVariables = q0
    S = Solver(R, dt=c.dt, nsteps=nsteps, save_interval=10)
    S.runForwardCheckpointed()
    J = R.terminalKineticEnergy()
    S.runAdjointCheckpointed(terminal=True, want_gradient=False)
    return R.checkpoint_plan, J[0], R.states[0].adjointVariables


def test_plans_of_one_region_equal_a_fresh_regions():
    import torch
    from magudi_amd import cases
    c = cases.kolmogorov3d(n=128, nsteps=24)
    q0 = c.initial_state()
    filler = _fill(c, 1)
    try:
        R = _region(c)
        once = [_run(R, c, n, q0) for n in STEPS]
        R.close()
        for n, (plan, J, lam) in zip(STEPS, once):
            F = _region(c)
            fresh = _run(F, c, n, q0)
            F.close()
            print(f"storage: {n} steps, plan {plan}, fresh {fresh[0]}", flush=True)
            assert plan["mode"] == fresh[0]["mode"] == "step store"
            # the last held step or two may come and go with what else the device holds
            assert abs(plan["held"] - fresh[0]["held"]) <= (0 if n < 300 else 2)
            assert plan["held"] == n if n < 300 else 0 < plan["held"] < n
            assert J == fresh[1] and np.array_equal(lam, fresh[2])
        F = _region(c)
        F.set_step_store(1)
        F.set_window_cache(0)                  # no step held, no slots kept
        bare = _run(F, c, STEPS[0], q0)
        F.close()
        assert bare[0]["held"] == 0
        assert bare[1] == once[0][1] and np.array_equal(bare[2], once[0][2])
    finally:
        del filler
        torch.cuda.empty_cache()


def test_two_regions_in_turn_keep_their_storage():
    """Each region's run leaves the other's storage as it is: after the first run of each, runs in
    turn allocate nothing."""
    import torch
    from magudi_amd import cases
    c = cases.kolmogorov3d(n=128, nsteps=24)
    q0 = c.initial_state()
    filler = _fill(c, 2)
    try:
        A, B = _region(c), _region(c)
        first = [_run(R, c, 24, q0) for R in (A, B)]
        free = []
        for turn in range(3):
            for R in (A, B):
                plan, J, lam = _run(R, c, 24, q0)
                assert plan["held"] == 24 and J == first[0][1] and np.array_equal(lam, first[0][2])
                free.append(torch.cuda.mem_get_info()[0])
        print(f"storage in turn: free {free}", flush=True)
        assert len(set(free)) == 1
        A.close()
        B.close()
    finally:
        del filler
        torch.cuda.empty_cache()


def test_other_allocations_leave_the_storage_as_it_is():
    """3 GB that the process takes after a region's first run, far less than the reserve is for:
    the next runs keep that run's storage and allocate nothing."""
    import torch
    from magudi_amd import cases
    c = cases.kolmogorov3d(n=128, nsteps=300)
    q0 = c.initial_state()
    filler = _fill(c, 1)
    later = None
    try:
        R = _region(c)
        first = _run(R, c, 300, q0)
        assert 0 < first[0]["held"] < 300
        later = torch.empty(3 << 30, dtype=torch.uint8, device="cuda")
        free = torch.cuda.mem_get_info()[0]
        for _ in range(2):
            plan, J, lam = _run(R, c, 300, q0)
            print(f"storage beside 3 GB more: {plan} after {first[0]}", flush=True)
            assert plan == first[0] and torch.cuda.mem_get_info()[0] == free
            assert J == first[1] and np.array_equal(lam, first[2])
        R.close()
    finally:
        del filler, later
        torch.cuda.empty_cache()
