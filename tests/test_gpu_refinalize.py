"""A region that has run -- eagerly, from a captured graph and as a member of a merged group --
and is then given another source, a sponge and another target state and finalized again must run
as a fresh region of that case does, bit for bit: nothing laid out or captured for the earlier
runs (group tiling, tile records, stage tables, graphs) is used again."""
import ctypes as C
import dataclasses

import numpy as np
import pytest

from magudi_amd import capi, cases
from magudi_amd.capi import check, dptr

pytestmark = pytest.mark.gpu

SOURCES = [cases.Source((1.0, -2.0, 0.0), 3e-2, 0.2, 1.0, 0.4),
           cases.Source((-3.0, 2.0, 0.0), 2e-2, 0.1, 2.0, 0.1)]


def _before(kind):
    if kind == "wave":
        c = cases.periodic_wave_1d(n=300, nsteps=6, save_interval=2)
        sponge = cases.Patch("sponge.I", cases.SPONGE, 1, (40, 90, 1, 1, 1, 1), (0.3, 2.0, 0, 0))
    else:
        c = cases.acoustic_monopole(n=61, nsteps=6, save_interval=2)
        c.dt = 0.2
        sponge = cases.Patch("sponge.I", cases.SPONGE, -1, (21, 38, 12, 50, 1, -1), (0.3, 2.0, 0, 0))
    return c, sponge


def _after(c, sponge):
    target = np.array(c.target) if c.target is not None else cases.quiescent_state(c.nd, c.npoints, c.gamma)
    target[-1] *= 1.0 + 1e-3 * np.sin(np.arange(c.npoints) / 50.0)
    return dataclasses.replace(c, patches=list(c.patches) + [sponge],
                               sources=list(c.sources) + SOURCES, target=target)


def _change(R, c2, sponge):
    pd = capi.PatchDesc()
    pd.type, pd.normal_dir = sponge.type, sponge.normal_dir
    for i in range(6):
        pd.extent[i] = sponge.extent[i]
    for i, v in enumerate(sponge.params):
        pd.p[i] = v
    check(capi.lib().mgd_region_add_patch(R.handle, C.byref(pd)))
    check(capi.lib().mgd_region_set_field(R.handle, capi.FIELD_TARGET_STATE,
                                          dptr(np.ascontiguousarray(c2.target))))
    for s in SOURCES:
        loc = np.array(s.location, dtype=np.float64)
        check(capi.lib().mgd_region_add_source(R.handle, dptr(loc), s.amplitude, s.frequency,
                                               s.radius, s.phase))
    check(capi.lib().mgd_region_finalize(R.handle))


def _runs(R, q0):
    """Forward and adjoint run, eager and from a graph (captured, then replayed)."""
    from magudi_amd.solver import Solver
    S = Solver(R)
    out = []
    for graph in (False, True, True):
        R.states[0].conservedVariables = q0
        J = S.runForward(use_graph=graph)
        q = R.states[0].conservedVariables
        R.states[0].conservedVariables = q0
        s, g, Ja = S.runAdjoint(use_graph=graph)
        lam = R.states[0].adjointVariables
        out.append((J, q, s, Ja, lam) + (() if g is None else (g,)))
    return out


@pytest.mark.parametrize("kind", ["monopole", "wave"])
def test_runs_after_another_finalize(kind):
    from magudi_amd.solver import Region
    c, sponge = _before(kind)
    c2 = _after(c, sponge)
    q0 = np.array(c.initial_state())
    q0[0] += 1e-2 * np.cos(np.arange(c.npoints) / 7.0)
    R = Region(c)
    first = _runs(R, q0)
    _change(R, c2, sponge)
    again = _runs(R, q0)
    fresh = _runs(Region(c2), q0)
    assert not np.array_equal(first[0][1], fresh[0][1])
    for o in again + fresh[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(o, fresh[0]))


def test_merged_run_after_another_finalize():
    from magudi_amd.group import RegionGroup
    c, sponge = _before("monopole")
    other = cases.acoustic_monopole(n=45, nsteps=c.nsteps, save_interval=c.save_interval)
    other.dt = c.dt
    c2 = _after(c, sponge)
    G, F = RegionGroup([c, other]), RegionGroup([c2, other])
    F.regions[0].states[0].initialCondition = c.initial_state()   # the target differs, not the start
    G.restart()
    first = G.run_adjoint_merged()
    _change(G.regions[0], c2, sponge)
    G.restart()
    again = G.run_adjoint_merged()
    F.restart()
    fresh = F.run_adjoint_merged()
    assert not np.array_equal(first[0][1], fresh[0][1])
    for o, f in zip(again, fresh):
        assert all(np.array_equal(a, b) for a, b in zip(o, f))
