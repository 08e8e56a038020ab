"""The 3-D forward march and the gradient pass with 64-bit offsets, which grids of 2^29 - 1024
points and more take by themselves, here asked for on small grids with partial tiles and chunks:
rhs, forward and adjoint run equal those with 32-bit offsets bit for bit."""
import numpy as np
import pytest

from magudi_amd import capi
from test_gpu_parity import inviscid_box, periodic_box, perturbed

pytestmark = pytest.mark.gpu


def _wide(R, on):
    capi.check(capi.lib().mgd_region_set_option(R.handle, capi.OPT_WIDE_OFFSETS, int(on)))


@pytest.mark.parametrize("shape,instances", [((33, 20, 35), 2), ((9, 33, 11), 1), ((64, 32, 40), 1)])
@pytest.mark.parametrize("kind", ["power", "constant", "inviscid", "dissipation"])
def test_wide_offsets_change_nothing(shape, instances, kind):
    from magudi_amd.solver import Region, Solver
    c = inviscid_box(shape) if kind == "inviscid" else periodic_box(shape, dissipation=kind == "dissipation")
    if kind == "constant":
        c.power_law = 0.0
    q0 = perturbed(c, 71)
    lamT = np.random.default_rng(72).standard_normal((instances, c.nv, c.npoints))
    ref = None
    for wide, width, chunk in ((0, 16, 32), (1, 16, 32), (1, 32, 3), (1, 32, 64)):
        print(f"wide offsets: {shape} x {instances} {kind} wide={wide} {width} x {chunk}", flush=True)
        R = Region(c, n_instances=instances)
        R.set_march_tile(width)
        R.set_z_chunk(chunk)
        _wide(R, wide)
        for k in range(instances):
            R.states[k].conservedVariables = q0 + 1e-3 * k
        R.computeRhs(1, time=0.3)
        out = [s.rightHandSide for s in R.states]
        S = Solver(R, dt=c.dt, nsteps=2, save_interval=2)
        S.runForward()
        out += [s.conservedVariables for s in R.states]
        S.runForwardCheckpointed()
        S.runAdjointCheckpointed(terminal=lamT, want_gradient=False)
        out += [s.conservedVariables for s in R.states] + [s.adjointVariables for s in R.states]
        if ref is None:
            ref = out
        assert all(np.array_equal(a, b) for a, b in zip(out, ref)), (wide, width, chunk)
