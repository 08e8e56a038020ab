"""The fused 2-D stage kernels at the places where a tile, a patch or a table can go wrong:
grids whose tiles are the smallest and the largest of a shape (12, 13, 16, 32 points and one
more), far fields too deep or too many for the terms formed ahead, sponges that overlap, several
sources, a periodic direction, the composite dissipation.  rhs of both modes against the generic
kernels and the oracle; both form the same sums of some fifty terms of order one, in another
order for the adjoint dissipation, so 1e-13 of the largest value is a few hundred roundings."""
import dataclasses

import numpy as np
import pytest

import oracle_bind as ob
from magudi_amd import cases

pytestmark = pytest.mark.gpu


def maxrel(a, b):
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


def monopole(nx, ny, composite=False, patches=(), sources=(), periodicity=(0, 0, 0)):
    """The monopole of an nx x ny grid of uneven spacing, with extra patches and sources."""
    c = cases.acoustic_monopole(n=41, nsteps=1, composite=composite)
    x = np.linspace(-14.0, 14.0, nx) + 0.1 * np.sin(np.linspace(0.0, 3.0, nx))
    y = np.linspace(-11.0, 11.0, ny) + 0.1 * np.sin(np.linspace(0.0, 5.0, ny))
    if periodicity[0]:
        x = np.linspace(-14.0, 14.0, nx)
    X, Y = np.meshgrid(x, y, indexing="xy")
    r = np.hypot(X, Y).ravel()
    keep = [p for p in c.patches if not p.name.startswith(("target", "control"))
            and not (periodicity[0] and abs(p.normal_dir) == 1)]
    keep += [cases.Patch("targetRegion", cases.COST_TARGET, 0, (2, nx - 3, 2, ny - 3, 1, -1)),
             cases.Patch("controlRegion", cases.ACTUATOR, 0, (4, 9, 3, 10, 1, -1))]
    period = (x[-1] - x[0] + (x[1] - x[0]), 0.0, 0.0)
    return dataclasses.replace(
        c, n=(nx, ny, 1), coords=np.stack([X.ravel(), Y.ravel()]), patches=keep + list(patches),
        sources=c.sources + list(sources), target=cases.quiescent_state(2, nx * ny),
        target_mollifier=0.5 + 0.1 * np.cos(r), control_mollifier=0.3 + 0.1 * np.sin(r),
        periodicity=periodicity, periodic_length=period if periodicity[0] else (0.0, 0.0, 0.0))


FAR = [cases.Patch("deep.E", cases.FAR_FIELD, 1, (1, 5, 1, -1, 1, -1), (0.7, 0.0, 0, 0)),
       cases.Patch("strip.S", cases.FAR_FIELD, 2, (3, -4, 2, 3, 1, -1), (0.4, 0.0, 0, 0))]
MORE = [cases.Patch("sponge.S2", cases.SPONGE, 2, (1, -1, 1, 6, 1, -1), (0.3, 2.0, 0, 0)),
        cases.Patch("forcing", cases.KOLMOGOROV, 0, (5, 12, 3, 9, 1, 1), (1.0, 0.05, 0, 0))]
SRC = [cases.Source((3.0, -2.0, 0.0), 2e-2, 0.05, 2.0), cases.Source((-4.0, 5.0, 0.0), 1e-2, 0.02, 0.4)]

CASES = {
    "25x26": lambda: monopole(25, 26),
    "33x64": lambda: monopole(33, 64),
    "65x32_composite": lambda: monopole(65, 32, composite=True),
    "40x29_far_sponges_sources": lambda: monopole(40, 29, patches=FAR + MORE, sources=SRC),
    "96x31_far_composite": lambda: monopole(96, 31, composite=True, patches=FAR, sources=SRC),
    "49x25_plane_x": lambda: monopole(49, 25, periodicity=(cases.PLANE, 0, 0)),
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("mode", [1, -1])
def test_rhs_matches_generic_and_oracle(name, mode):
    from magudi_amd.solver import Region
    c = CASES[name]()
    rng = np.random.default_rng(17)
    q = c.target + 0.05 * rng.standard_normal((c.nv, c.npoints))
    q[0] = np.abs(q[0]) + 0.2
    lam = rng.standard_normal((c.nv, c.npoints))
    outs = []
    for shape in (-2, 0, 2, 4, 5):         # -2: the generic kernels
        print(f"stage2d: {name} mode={mode} shape={shape}", flush=True)
        R = Region(c, force_plain=True) if shape == -2 else Region(c, tile_shape=shape)
        if R.tile_shape != max(shape, -1):     # edge tiles of fewer than 12 points: generic
            continue
        R.states[0].conservedVariables = q
        R.states[0].adjointVariables = lam
        ctl = np.linspace(-1.0, 1.0, R.n_actuator)
        if mode == 1:
            R.computeRhs(1, time=2.3, control=ctl)
        else:
            R.updateAdjointForcing()
            R.computeRhs(-1, forcing_factor=0.5)
        outs.append(R.states[0].rightHandSide)
    assert len(outs) >= 2
    O = ob.Region(c)
    if mode == 1:
        ref = O.rhs(1, q, time=2.3, control=ctl)
    else:
        ref = O.rhs(-1, q, lam, aforcing=O.adjoint_forcing(q), factor=0.5)
    assert np.all(np.isfinite(ref))
    assert maxrel(outs[0], ref) < 1e-13
    assert maxrel(outs[1], ref) < 1e-13
    for o in outs[2:]:
        assert np.array_equal(o, outs[1])
