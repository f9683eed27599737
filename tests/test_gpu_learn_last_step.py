"""Training on the last corrected step: imx_learn_step leaves the state before
its last step where imx_learn_train and imx_learn_store take features from, as
imx_learn_sample does."""
import numpy as np
import pytest

from imodel_amd.learn import Learn
from imodel_amd.mlp import Mlp
from imodel_amd.swm import H0_GEO, Mesh, Swm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("steps", [1, 4, 21])  # one graph of each size; all three
def test_features_of_the_last_step(steps, prec):
    """Bound 0 keeps the plain step, so the last corrected step is the plain
    step a sample takes from the same state: the losses before training are the
    same numbers, whatever was sampled earlier."""
    print("[gpu-case] learn last step", steps, prec, flush=True)
    m = Mesh.icos(4)
    rng = np.random.default_rng(5)
    du, dh = rng.standard_normal(m.ne), rng.standard_normal(m.nv)
    loss = []
    for corrected in (True, False):
        with Swm(m, precision=prec, dt=600.0, h_ref=H0_GEO) as s:
            L = Learn(s, Mlp(seed=2), m)
            s.set_state(*m.spectral(1))
            if corrected:
                raw = L.sample(raw=True)  # another state's
                scaling = (raw.mean(0), raw.std(0) + 1e-3, 1.0, 1.0)
            L.set_scaling(*scaling)
            s.set_state(*m.spectral(2))
            if corrected:
                assert L.step(steps, 0.0) == steps
            else:
                s.step(steps - 1)
                L.sample()
            stored = Learn.reserve(L, 1), L.store(du, dh)
            assert stored[1] == 0
            loss.append(tuple(L.train(du, dh, epochs=1, lr=0.0)) + tuple(L.fit(1, 0.0, 0.0)) + s.get_state())
            L.close()
    assert loss[0][:4] == loss[1][:4]
    assert all(np.array_equal(a, b) for a, b in zip(loss[0][4:], loss[1][4:]))
