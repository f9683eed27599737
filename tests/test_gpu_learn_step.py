"""The corrected step's network kernel, which gathers and normalises its
features itself, against the sampled features put through the network that
reads rows."""
import numpy as np
import pytest

from imodel_amd.learn import Learn
from imodel_amd.mlp import Mlp
from imodel_amd.swm import H0_GEO, Mesh, Swm
from oracle import learn_oracle as lo

pytestmark = pytest.mark.gpu


# a mesh of pentagons only, a last tile with few edges, one tile a wave, several
@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("g", [0, 1, 4, 6])
def test_gathered_features(g, prec):
    """Both networks read the same BF16 inputs and differ in the order of
    layer 1's sums, so in roundings of BF16 activations (2^-9 each): 2^-8 of
    the correction's norm, 2^-6 of its largest value at any one place. The
    state's own rounding (2^-24 of u, h) is below both at these scales."""
    print("[gpu-case] corrected step", g, prec, flush=True)
    M = Mesh.icos(g)
    dt = 1800.0 / 2 ** max(0, g - 3)
    s = Swm(M, precision=prec, dt=dt, h_ref=H0_GEO)
    m = Mlp(seed=20 + g)
    L = Learn(s, m, M)
    s.set_state(*M.spectral(g))
    hn, un = s.get_state()
    raw = L.sample(raw=True)
    hp, up = s.get_state()
    mu, sig = raw.mean(0), raw.std(0)
    sig[sig < 1e-6] = 1.0
    X = (raw - mu) / sig
    Y = m.forward(X).astype(np.float64)
    F = lo.div_matrix(M.arrays) @ Y[:, 1]
    # corrections of the size of the state's own variation
    tsu, tsh = np.abs(Y[:, 0]).max() / np.abs(up).max(), np.abs(F).max() / np.ptp(hp)
    L.set_scaling(mu, sig, tsu, tsh)
    s.set_state(hn, un)
    assert L.step(1, bound=1e30) == 0
    hc, uc = s.get_state()
    for got, want in (((uc - up) * tsu, Y[:, 0]), ((hc - hp) * tsh, F)):
        d = got - want
        assert np.linalg.norm(d) <= 2 ** -8 * np.linalg.norm(want)
        assert np.abs(d).max() <= 2 ** -6 * np.abs(want).max()
