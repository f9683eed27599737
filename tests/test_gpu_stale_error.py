"""An error that an earlier HIP call of the program left behind is not taken for
one of the library's: handles are made, change their scheme and move states as
if it were not there."""
import ctypes

import numpy as np
import pytest

from imodel_amd import capi
from imodel_amd.swm import H0_GEO, Ensemble, Mesh, Swm

pytestmark = pytest.mark.gpu


@pytest.fixture
def leave_error():
    """A call that the runtime refuses (a device that is not there)."""
    capi.lib()
    paths = {ln.split()[-1] for ln in open("/proc/self/maps") if "libamdhip64" in ln}
    hip = ctypes.CDLL(sorted(p for p in paths if "torch" not in p)[0])

    def leave():
        assert hip.hipSetDevice(9999) != 0

    yield leave
    hip.hipGetLastError()


@pytest.mark.parametrize("prec", ["fp64_ref", "fp64", "fp32"])
def test_handle(prec, leave_error):
    print("[gpu-case] stale error, handle", prec, flush=True)
    m = Mesh.icos(3)
    h, u = m.spectral(1)

    def through(before):
        before()
        with Swm(m, precision=prec, dt=600.0, h_ref=H0_GEO) as s:
            before()
            s.set_scheme(pv="apvm", pvspar=0.5)
            before()
            s.set_coriolis(2, 1e-4)
            before()
            s.set_state(h, u)
            s.step(2)
            before()
            x = s.get_state()
            before()
            return x + s.tendency(h, u)

    assert all(np.array_equal(a, b) for a, b in zip(through(leave_error), through(lambda: None)))


def test_ensemble(leave_error):
    print("[gpu-case] stale error, ensemble", flush=True)
    m = Mesh.icos(3)
    h, u = m.spectral(1)
    leave_error()
    with Ensemble([m, m], [600.0, 300.0], precision="fp32", h_ref=H0_GEO) as E:
        leave_error()
        E.set_state(1, h, u)
        leave_error()
        x = E.get_state(1)
    assert np.max(np.abs(x[0] - h)) < 1e-3 and np.max(np.abs(x[1] - u)) < 1e-4
