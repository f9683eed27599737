"""h_ref is the fused handles' storage offset: a reference-order handle that is
given one evaluates the same state."""
import numpy as np
import pytest

from imodel_amd.swm import H0_GEO, Mesh, Swm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme", [{}, {"wrap": "gass18"}], ids=["trsk10", "gass18"])
def test_href_leaves_reference_handles_alone(scheme):
    print("[gpu-case] fp64_ref with h_ref", scheme, flush=True)
    m = Mesh.icos(3)
    h, u = m.spectral(8)
    got = []
    for h_ref in (0.0, H0_GEO):
        with Swm(m, precision="fp64_ref", dt=900.0, h_ref=h_ref) as s:
            s.set_scheme(**scheme)
            t = s.tendency(h, u)
            s.set_state(h, u)
            d0 = s.diagnostics()
            s.step(5)
            got.append(t + s.get_state() + (np.array(list(d0.values())), np.array(list(s.diagnostics().values()))))
    for a, b in zip(*got):
        assert np.array_equal(a, b)
