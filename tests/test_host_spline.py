"""The host's integration weights of the cubic spline (exc_hml_spline_weights, the transposed
recurrences) against the oracle's spline integral of every unit vector, on logarithmic and
linear meshes from the smallest (4 points) up: within 16 eps of the largest weight (both sides round a
few operations a point, and the recurrences damp them)."""
import ctypes as C

import numpy as np
import pytest


@pytest.mark.parametrize("n", [4, 5, 6, 7, 33, 200])
@pytest.mark.parametrize("mesh", ["log", "linear"])
def test_spline_weights(n, mesh):
    from exciting_amd import lapw
    from oracle import hmlint_ref as M
    lib = C.CDLL(str(lapw.LIBPATH))
    f = lib._Z22exc_hml_spline_weightsiPKdPd
    f.restype = None
    x = np.geomspace(1e-5, 2.0, n) if mesh == "log" else np.linspace(0.1, 2.0, n)
    wt = np.zeros(n)
    f(n, C.c_void_p(x.ctypes.data), C.c_void_p(wt.ctypes.data))
    ref = M.fderiv_int(x, np.eye(n))
    assert np.abs(wt - ref).max() <= 16 * 2.3e-16 * np.abs(ref).max()
