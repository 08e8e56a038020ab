"""Work units of the 3-D marches fixed by option, over the shapes that the autotuner may choose:
z chunks of 1, 2, 3, 4, 8, 10 and 16 planes (shorter than the stencil's reach, no divisors of the
grid, longer than it), 16- and 32-wide tiles on sizes that are no multiple of either.  Forward and
adjoint run and rhs equal the per-operator kernels' bit for bit; the shape reported is the one set.
Grids that are OVERLAP-periodic (the last grid line repeats the first) likewise."""
import dataclasses

import numpy as np
import pytest

from magudi_amd import capi, cases
from magudi_amd.capi import MagudiError
from test_gpu_march_sizes import _plain
from test_gpu_parity import inviscid_box, periodic_box, perturbed

pytestmark = pytest.mark.gpu


def _run(case, instances, q0, lamT, units=None):
    from magudi_amd.solver import Region, Solver
    R = Region(case, n_instances=instances)
    if units:
        R.set_march_tile(units[0])
        R.set_z_chunk(units[1])
    for k in range(instances):
        R.states[k].conservedVariables = q0 + 1e-3 * k
    S = Solver(R, dt=case.dt, nsteps=3, save_interval=2)
    S.runForwardCheckpointed()
    qT = [s.conservedVariables for s in R.states]
    S.runAdjointCheckpointed(terminal=lamT, want_gradient=False)
    if units:
        assert R.march_units == (units, units)
        assert (R.march_tile, R.z_chunk) == units
    return qT + [s.adjointVariables for s in R.states]


@pytest.mark.parametrize("shape,instances", [((33, 20, 35), 2), ((50, 16, 21), 1)])
def test_every_unit_shape(shape, instances):
    c = periodic_box(shape, dissipation=False)
    q0 = perturbed(c, 63)
    lamT = np.random.default_rng(64).standard_normal((instances, c.nv, c.npoints))
    ref = _run(_plain(c), instances, q0, lamT)
    for width in (16, 32):
        for chunk in (1, 2, 3, 4, 8, 10, 16, 32, 64):
            print(f"march units: {shape} x {instances} tile {width} chunk {chunk}", flush=True)
            out = _run(c, instances, q0, lamT, (width, chunk))
            assert all(np.array_equal(a, b) for a, b in zip(out, ref)), (width, chunk)


def test_units_of_one_dimension_fixed():
    """One of tile width and z chunk fixed, the other tuned."""
    from magudi_amd.solver import Region, Solver
    c = periodic_box((33, 20, 35), dissipation=False)
    for width, chunk in ((0, 10), (32, 0), (0, 0)):
        R = Region(c)
        R.set_march_tile(width)
        R.set_z_chunk(chunk)
        R.states[0].conservedVariables = c.initial_state()
        Solver(R, dt=c.dt, nsteps=1, save_interval=1).runForward()
        for (w, z), (ws, zs) in zip(R.march_units, R.march_shape):
            assert w in ((16, 32) if width == 0 else (width,))
            assert z == chunk if chunk else 2 <= z <= 128
            assert (ws, zs) == (w, max(z, 32))


@pytest.mark.parametrize("option,value", [(capi.OPT_Z_CHUNK, -1), (capi.OPT_Z_CHUNK, 1025),
                                          (capi.OPT_MARCH_TILE, 8), (capi.OPT_MARCH_TILE, 64)])
def test_units_out_of_range(option, value):
    from magudi_amd.solver import Region
    R = Region(periodic_box((16, 16, 16), dissipation=False))
    with pytest.raises(MagudiError):
        capi.check(capi.lib().mgd_region_set_option(R.handle, option, value))


@pytest.mark.parametrize("overlap", [(1, 1, 1), (0, 0, 1), (1, 0, 0)])
@pytest.mark.parametrize("kind", ["viscous", "inviscid"])
def test_rhs_on_overlap_grids(overlap, kind):
    from magudi_amd.solver import Region
    c = (inviscid_box if kind == "inviscid" else lambda s: periodic_box(s, dissipation=False))((33, 17, 25))
    c = dataclasses.replace(c, periodicity=tuple(cases.OVERLAP if o else cases.PLANE for o in overlap))
    q = perturbed(c, 65)
    lam = np.random.default_rng(66).standard_normal((c.nv, c.npoints))
    for mode in (1, -1):
        ref = None
        for case, units in ((_plain(c), None), (c, (16, 32)), (c, (32, 3)), (c, (16, 64))):
            R = Region(case)
            if units:
                R.set_march_tile(units[0])
                R.set_z_chunk(units[1])
            R.states[0].conservedVariables = q
            R.states[0].adjointVariables = lam
            R.updateAdjointForcing(no_adjoint_forcing=True)
            R.computeRhs(mode, time=0.3, forcing_factor=0.5)
            out = R.states[0].rightHandSide
            assert np.all(np.isfinite(out))
            if ref is None:
                ref = out
            else:
                assert np.array_equal(out, ref), (mode, units)


@pytest.mark.parametrize("shape", [(33, 20, 35), (32, 16, 40)])
@pytest.mark.parametrize("kind", ["viscous", "inviscid", "sponge"])
def test_autotuner_leaves_the_adjoint_state(shape, kind):
    """An adjoint state put before a region's first call, which is when the tuner runs, is the one
    that this call marches back, or leaves as it is."""
    from magudi_amd.solver import Region, RK4Integrator, Solver
    c = inviscid_box(shape) if kind == "inviscid" else periodic_box(shape, dissipation=False)
    if kind == "sponge":
        c = _plain(c)
    q = perturbed(c, 67)
    lam = np.random.default_rng(68).standard_normal((c.nv, c.npoints))
    out = []
    for fixed in (True, False):
        R = Region(c)
        if fixed:
            R.set_march_tile(16)
            R.set_z_chunk(32)
        R.states[0].conservedVariables = q
        R.states[0].adjointVariables = lam
        R.updateAdjointForcing(no_adjoint_forcing=True)
        RK4Integrator().substepAdjoint(R, 0.0, c.dt, 1, 4)
        out.append(R.states[0].adjointVariables)
    assert np.array_equal(out[0], out[1]) and not np.array_equal(out[0], lam)
    R = Region(c)
    R.states[0].conservedVariables = q
    R.states[0].adjointVariables = lam
    Solver(R, dt=c.dt, nsteps=1, save_interval=1).runForward()
    assert np.array_equal(R.states[0].adjointVariables, lam)
