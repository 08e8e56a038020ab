"""The stress slots that the forward pass keeps for the adjoint pass (3-D viscous marches): the
adjoint state with every step's slots kept and with none (the held steps limited by the caller,
so that steps are computed again), on repeated runs of one region, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,instances", [((32, 16, 16), 1), ((33, 20, 35), 2), ((16, 48, 9), 1)])
def test_kept_stress_changes_nothing(shape, instances):
    from magudi_amd.solver import Region, Solver
    from test_gpu_parity import periodic_box, perturbed
    c = periodic_box(shape, dissipation=False)
    nsteps, K = 5, 2
    q0 = [perturbed(c, 7 + k) for k in range(instances)]
    lamT = np.random.default_rng(8).standard_normal((instances, c.nv, c.npoints))
    out = []
    for cache in (-1, 1, 0):
        print(f"stress cache: {shape} cache={cache}", flush=True)
        R = Region(c, n_instances=instances)
        R.set_window_cache(cache)
        R.set_step_store(1)
        S = Solver(R, dt=c.dt, nsteps=nsteps, save_interval=K)
        for rep in range(2):
            for k in range(instances):
                R.states[k].conservedVariables = q0[k]
            S.runForwardCheckpointed()
            assert R.checkpoint_plan["mode"] == "step store"
            for back in range(2):              # two marches back over one forward run
                for k in range(instances):
                    R.states[k].adjointVariables = lamT[k]
                S.runAdjointCheckpointed(terminal=True, want_gradient=False)
                out.append([R.states[k].adjointVariables for k in range(instances)])
    assert all(np.all(np.isfinite(x)) and np.abs(x).max() > 1.0 for x in out[0])
    for o in out[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(out[0], o))
