"""The FP64_REF step where one launch forms everything up to the Coriolis term
(csrc/imx_swm.hip, ref_one): meshes of few cells, the largest that takes it
(glevel 5) and the next (glevel 6), bit for bit the oracle's."""
import numpy as np
import pytest

from imodel_amd.swm import Mesh, Swm
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [{}, {"stag": "HC"}, {"pv": "apvm", "pvspar": 0.5, "k2": 1e5, "diffus": "align"}], ids=str)
@pytest.mark.parametrize("glevel", [0, 1, 4, 5, 6])
def test_steps(glevel, kw):
    print("[gpu-case] ref one launch", glevel, kw, flush=True)
    m = Mesh.icos(glevel)
    dt = 225.0
    h, u = m.spectral(12)
    ho, uo = Oracle(m.arrays, scheme=dict(kw, dt=dt)).step(h, u, dt, 5)
    with Swm(m, precision="fp64_ref", dt=dt) as s:
        s.set_scheme(**kw)
        s.set_state(h, u)
        s.step(5)
        hg, ug = s.get_state()
    assert np.all(np.isfinite(ho)) and np.all(np.isfinite(uo))
    assert np.array_equal(hg, ho) and np.array_equal(ug, uo)
