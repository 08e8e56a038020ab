"""The 1-D kernels that run whole RK4 steps against the generic kernels: both form every sum in
the same order, so states and gradients agree bit for bit; J and the sensitivity are summed in
another order (rounding only: 1e-13).  Lines shorter than one work-group's piece, pieces that
hold an end of the line in their halo, both ends, one point more than a piece (96 points at four
steps per launch), step counts that no launch divides, every kind of patch that the kernels
take, and each way of keeping the forward states."""
import dataclasses

import numpy as np
import pytest

from magudi_amd import cases

pytestmark = pytest.mark.gpu


def line(n, periodic, composite=False, dissipation=True):
    """A wave on an uneven line (even where periodic) with every patch type of the 1-D path."""
    c = cases.periodic_wave_1d(n=n, nsteps=7, save_interval=3)
    P = cases.Patch
    x = c.coords[0]
    patches = [P("target", cases.COST_TARGET, 0, (3, n - 4, 1, -1, 1, -1)),
               P("control", cases.ACTUATOR, 0, (2, n // 2, 1, -1, 1, -1)),
               P("forcing", cases.KOLMOGOROV, 0, (5, n // 3 + 6, 1, 1, 1, 1), (1.0, 0.05, 0, 0))]
    if not periodic:
        x = x + 0.2 / n * np.sin(9.0 * x)
        patches += [P("far.E", cases.FAR_FIELD, 1, (1, 1, 1, -1, 1, -1), (1.0, 0.0, 0, 0)),
                    P("far.W", cases.FAR_FIELD, -1, (-1, -1, 1, -1, 1, -1), (0.7, 0.0, 0, 0)),
                    P("sponge.E", cases.SPONGE, 1, (1, 9, 1, -1, 1, -1), (0.2, 2.0, 0, 0)),
                    P("sponge.W", cases.SPONGE, -1, (-6, -1, 1, -1, 1, -1), (0.3, 2.0, 0, 0))]
    return dataclasses.replace(
        c, coords=x[None, :].copy(), patches=patches, composite_dissipation=composite,
        dissipation=dissipation, periodicity=c.periodicity if periodic else (0, 0, 0),
        sources=[cases.Source((0.3, 0.0, 0.0), 1e-2, 0.7, 0.1),
                 cases.Source((0.8, 0.0, 0.0), 2e-2, 0.2, 0.05)],
        target_mollifier=0.5 + 0.1 * np.cos(5 * x), control_mollifier=0.3 + 0.1 * np.sin(7 * x))


def runs(c, plain, instances=2, **opts):
    """Everything a forward run, a checkpointed run and its adjoint return; twice."""
    from magudi_amd.solver import Region, Solver
    R = Region(c, n_instances=instances, force_plain=plain)
    if "step" in opts:
        R.set_step_store(opts["step"])
        R.set_window_cache(opts["cache"])
    rng = np.random.default_rng(3)
    ctl = np.stack([a * rng.standard_normal((4 * c.nsteps, R.n_actuator)) for a in np.linspace(0.0, 2e-2, instances)])
    q0 = c.initial_state()
    S = Solver(R, dt=c.dt, nsteps=c.nsteps, save_interval=c.save_interval)
    exact, sums = [], []
    for _ in range(2):
        for k in range(instances):
            R.states[k].conservedVariables = q0
        sums.append(S.runForward(control=ctl))
        exact += [R.states[k].conservedVariables for k in range(0, instances, 1 + instances // 8)]
        for k in range(instances):
            R.states[k].conservedVariables = q0
        sums.append(S.runForwardCheckpointed(control=ctl))
        exact += [R.states[k].conservedVariables for k in range(0, instances, 1 + instances // 8)]
        sens, grad = S.runAdjointCheckpointed()
        sums.append(sens)
        exact += [grad] + [R.states[k].adjointVariables for k in range(0, instances, 1 + instances // 8)]
    return exact, np.array(sums)


def same(c, **opts):
    (xa, sa), (xb, sb) = runs(c, False, **opts), runs(c, True, **opts)
    for a, b in zip(xa, xb):
        assert np.all(np.isfinite(b))
        assert np.array_equal(a, b)
    assert np.allclose(sa, sb, rtol=1e-13, atol=0.0)
    assert np.all(sb[:3] > 0.0) and np.array_equal(sa[:3], sa[3:])


@pytest.mark.parametrize("n", [25, 96, 97, 113, 192, 389])
@pytest.mark.parametrize("periodic", [True, False])
def test_line_runs_match_generic(n, periodic):
    print(f"line1d: n={n} periodic={periodic}", flush=True)
    same(line(n, periodic))


@pytest.mark.parametrize("periodic", [True, False])
def test_many_lines_take_one_step_per_launch(periodic):
    same(line(193, periodic), instances=330)       # 990 pieces of a four-step launch


@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("composite,dissipation", [(True, True), (False, False)])
def test_line_dissipation_options(periodic, composite, dissipation):
    same(line(130, periodic, composite, dissipation))


@pytest.mark.parametrize("step,cache", [(0, 0), (0, 1), (0, -1), (1, 0), (1, 1), (1, -1)])
def test_line_storage_modes(step, cache):
    same(line(130, False), step=step, cache=cache)


def test_stage_calls_match_whole_steps():
    """A step driven stage by stage (generic kernels) gives the whole run's state, and every
    stage state served from the checkpointed run is the one it passed through."""
    from magudi_amd.solver import Region, RK4Integrator, Solver, UniformCheckpointer
    c = line(130, False)
    R = Region(c)
    R.set_step_store(1)
    R.set_window_cache(1)
    q0 = c.initial_state()
    ti, states, time = RK4Integrator(), {(0, 4): q0}, 0.0
    R.states[0].conservedVariables = q0
    for ts in range(1, c.nsteps + 1):
        for i in range(1, 5):
            if i in (2, 4):
                time = time + c.dt / 2.0
            ti.substepForward(R, time, c.dt, ts, i)
            states[(ts, i)] = R.states[0].conservedVariables
    R.states[0].conservedVariables = q0
    Solver(R, dt=c.dt, nsteps=c.nsteps, save_interval=c.save_interval).runForwardCheckpointed()
    for key in sorted(states, reverse=True):
        UniformCheckpointer().migrateTo(R, *key)
        assert np.array_equal(R.states[0].conservedVariables, states[key]), key


def test_graph_replays_match_eager_runs():
    from magudi_amd.solver import Region, Solver
    c = line(130, False)
    R = Region(c, n_instances=2)
    S = Solver(R, dt=c.dt, nsteps=c.nsteps, save_interval=c.save_interval)
    rng = np.random.default_rng(5)
    out = {False: [], True: []}
    for graph in (False, True):
        rng = np.random.default_rng(5)
        for _ in range(3):
            ctl = 1e-2 * rng.standard_normal((2, 4 * c.nsteps, R.n_actuator))
            for k in range(2):
                R.states[k].conservedVariables = c.initial_state()
            sens, grad, J = S.runAdjoint(control=ctl, use_graph=graph)
            lam = R.states[1].adjointVariables
            for k in range(2):
                R.states[k].conservedVariables = c.initial_state()
            out[graph] += [sens, grad, J, lam, S.runForward(control=ctl, use_graph=graph),
                           R.states[1].conservedVariables]
    for a, b in zip(out[False], out[True]):
        assert np.array_equal(a, b)
