"""The 3-D marches on grids that are no multiple of their tiles: partial tiles in x and y
(the threads beyond them double a point), partial z chunks, chunks shorter than the stencil's
reach and the smallest grids they take.  A sponge of amount 0 adds nothing but sends the rhs
to the per-operator kernels; the two must agree bit for bit (same operations in the same
order), and with the oracle to the rhs tolerance (1e-13 max-norm relative)."""
import dataclasses

import numpy as np
import pytest

import oracle_bind as ob
from magudi_amd import cases
from test_gpu_parity import RHS_TOL, inviscid_box, maxrel, periodic_box, perturbed

pytestmark = pytest.mark.gpu

SIZES = [(9, 9, 9), (9, 33, 11), (31, 17, 34), (50, 16, 21), (100, 30, 9), (33, 47, 35)]


def _plain(c):
    return dataclasses.replace(c, patches=list(c.patches) + [
        cases.Patch("sponge.E", cases.SPONGE, 1, (1, 4, 1, -1, 1, -1), (0.0, 2.0, 0, 0))])


@pytest.mark.parametrize("shape", SIZES)
@pytest.mark.parametrize("kind", ["power", "constant", "inviscid"])
def test_rhs_on_any_size(shape, kind):
    from magudi_amd.solver import Region
    c = inviscid_box(shape) if kind == "inviscid" else periodic_box(shape, dissipation=False)
    if kind == "constant":
        c.power_law = 0.0
    q = perturbed(c, 61)
    lam = np.random.default_rng(62).standard_normal((c.nv, c.npoints))
    O = ob.Region(c)
    for mode in (1, -1):
        out = []
        for case in (c, _plain(c)):
            R = Region(case)
            R.states[0].conservedVariables = q
            R.states[0].adjointVariables = lam
            R.updateAdjointForcing(no_adjoint_forcing=True)
            R.computeRhs(mode, time=0.3, forcing_factor=0.5)
            out.append(R.states[0].rightHandSide)
        assert np.array_equal(out[0], out[1]), (mode, maxrel(out[0], out[1]))
        ref = O.rhs(1, q, time=0.3) if mode == 1 else O.rhs(-1, q, lam, aforcing=None, factor=0.5)
        assert maxrel(out[0], ref) < RHS_TOL, (mode, maxrel(out[0], ref))


@pytest.mark.parametrize("shape,instances", [((33, 20, 35), 2), ((18, 40, 70), 1)])
def test_runs_on_any_size(shape, instances):
    """Forward + adjoint run over partial tiles and chunks: the tuned shape, chunks of 32 and
    128 planes on 16-wide tiles and the per-operator kernels, bit for bit."""
    from magudi_amd.solver import Region, Solver
    c = periodic_box(shape, dissipation=False)
    q0 = perturbed(c, 63)
    lamT = np.random.default_rng(64).standard_normal((instances, c.nv, c.npoints))
    out = []
    for case, zc in ((c, 0), (c, 32), (c, 128), (_plain(c), 0)):
        R = Region(case, n_instances=instances)
        if zc:
            R.set_march_tile(16)
            R.set_z_chunk(zc)
        for k in range(instances):
            R.states[k].conservedVariables = q0 + 1e-3 * k
        S = Solver(R, dt=c.dt, nsteps=3, save_interval=2)
        S.runForwardCheckpointed()
        qT = [s.conservedVariables for s in R.states]
        S.runAdjointCheckpointed(terminal=lamT, want_gradient=False)
        out.append((qT, [s.adjointVariables for s in R.states]))
    for qT, lam in out[1:]:
        for k in range(instances):
            assert np.array_equal(qT[k], out[0][0][k]), k
            assert np.array_equal(lam[k], out[0][1][k]), k
