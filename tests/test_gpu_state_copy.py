"""States copied to the host through the pinned ring: sizes on both sides of the least one that
takes it (4 MiB), of one ring (32 MiB) and odd remainders, into arrays at any address of a chunk;
bit for bit, nothing written beside them."""
import ctypes as C

import numpy as np
import pytest

from magudi_amd import capi, cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1000, 174762, 174763, 262145, 700001, 1398101, 2000003])
def test_large_state_copies(n):
    from magudi_amd.solver import Region
    c = cases.periodic_wave_1d(n=n, nsteps=1)
    R = Region(c, n_instances=2)
    rng = np.random.default_rng(n)
    q = [1.0 + rng.random((3, n)) for _ in range(2)]
    for k in range(2):
        R.states[k].conservedVariables = q[k]
    room = np.empty(3 * n + 3 * 2 ** 18)
    base = -(room.ctypes.data // 8) % 2 ** 18             # a 2 MiB boundary
    for off in (0, 1, 513, 2 ** 18 - 1, 2 ** 18 - 3):
        for k in range(2):
            room[:] = -7.0
            out = room[base + off:base + off + 3 * n]
            print(f"state copy: n={n} offset={off} instance={k}", flush=True)
            rc = capi.lib().mgd_state_get(R.handle, capi.CONSERVED, k,
                                          out.ctypes.data_as(C.POINTER(C.c_double)))
            assert rc == 0
            assert np.array_equal(out, q[k].ravel())
            assert np.all(room[:base + off] == -7.0) and np.all(room[base + off + 3 * n:] == -7.0)
