"""DeviceSession.pull without a device: a download that fails, at any point, leaves the solver as it
was, and one that succeeds lands whole in U whatever its size and layout."""
import ctypes as C

import numpy as np
import pytest

from quick_gpu_cfd_for_neural_network_with_converging_inputs_airfoil2d_version_amd import _native as N
from quick_gpu_cfd_for_neural_network_with_converging_inputs_airfoil2d_version_amd import euler2d as E


class Library:
    """The three calls of a pull: writes `part` of the state 0, 1, 2, ... and of the times, then returns."""

    def __init__(self, part=1.0, download=0, stats=0):
        self.part, self.download, self.stats = part, download, stats

    def ugrid_download(self, handle, u, u_len, t, dt, err, err_len):
        n = int(u_len * self.part)
        np.ctypeslib.as_array(u, (u_len,))[:n] = np.arange(n, dtype=np.float64)
        if self.part == 1.0:
            t[0], dt[0] = 0.5, 0.25
        if self.download:
            err.value = b"download dt: lost"
        return self.download

    def ugrid_implicit_stats(self, handle, info):
        return self.stats


def session(nx, ny, cases, lib):
    par = E.params2d_default()
    par.limiter = E.LIM_FIRST_ORDER
    s = E.Solver2D(nx, ny, 0.0, 1.0, 0.0, 1.0, cases, par)
    s.U[:] = -1.0
    d = E.DeviceSession.__new__(E.DeviceSession)
    d.lib, d.solver, d.handle = lib, s, C.c_void_p()
    d.meta, d._counted, d._staging = N.ugrid_meta(7, 3), (0, 0, 0, 0), None
    return s, d


@pytest.mark.parametrize("lib", [Library(0.5, 3), Library(1.0, 3), Library(1.0, 0, 1)])
def test_failed_download_leaves_the_solver(lib):
    s, d = session(20, 9, 1, lib)
    for _ in range(2):
        with pytest.raises(RuntimeError):
            d.pull()
        assert (s.U == -1.0).all() and (s.t == 0.0).all() and (s.dt == 0.0).all()
        assert (s.nsteps, s.nreject) == (0, 0)
    lib.download, lib.stats, lib.part = 0, 0, 1.0
    d.pull()
    np.testing.assert_array_equal(s.U, np.arange(s.U.size))
    assert (s.nsteps, s.nreject, s.t[0], s.dt[0]) == (7, 3, 0.5, 0.25)


@pytest.mark.parametrize("layout", ["own", "float32", "strided"])
@pytest.mark.parametrize("nx, ny, cases", [(1, 1, 1), (1020, 1019, 1), (1020, 1020, 1), (637, 501, 4)])
def test_whole_state_lands(nx, ny, cases, layout):  # below, at and above the size that is copied in parts
    s, d = session(nx, ny, cases, Library())
    if layout == "float32":
        s.U = s.U.astype(np.float32)
    elif layout == "strided":
        s.U = np.full(2 * s.U.size, -1.0)[::2]
    d.pull()
    np.testing.assert_array_equal(s.U, np.arange(s.U.size).astype(s.U.dtype))
