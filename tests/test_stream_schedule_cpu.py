"""The kernels' schedules at the edges of what they hold: bie_schedule_check replays them (every
element once, slots handed on in turn, a node's contributions within their 16-bit counts)."""
import ctypes

import numpy as np
import pytest

from bie_amd import _lib
from bie_amd import mesh as M


def fan(n):
    """n triangles around one node."""
    th = np.linspace(0.0, 2.0 * np.pi, n, endpoint=False)
    X = np.zeros((3, n + 1))
    X[0, 1:], X[1, 1:] = np.cos(th), np.sin(th)
    T = np.stack([np.zeros(n, dtype=np.int64), 1 + np.arange(n), 1 + (np.arange(n) + 1) % n])
    return M.Mesh3d(X, T, X.copy(), T.copy(), 3, 3)


def apart(n):
    """n triangles without a common node: every node goes straight to its column."""
    X = np.random.default_rng(n).standard_normal((3, 3 * n))
    T = np.arange(3 * n, dtype=np.int64).reshape(n, 3).T.copy()
    return M.Mesh3d(X, T, X.copy(), T.copy(), 3, 3)


@pytest.mark.parametrize("make,n,segments", [(fan, 3, 1), (fan, 300, 1), (fan, 70000, 1),
                                             (apart, 1, 1), (apart, 500, 7)])
def test_schedules_of_unusual_meshes(make, n, segments):
    hm = _lib.HostMesh(make(n))
    st = (ctypes.c_int64 * 6)()
    assert _lib.lib().bie_schedule_check(ctypes.byref(hm.struct), segments, st) == 0, \
        _lib.lib().bie_last_error()
    assert st[0] >= segments
