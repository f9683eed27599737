"""The fused training kernel (csrc/imx_mlp.hip) where its batches of 64 edges,
its 256 blocks and the optimiser's fragment updates can go wrong."""
import numpy as np
import pytest

from imodel_amd.mlp import Mlp
from oracle import mlp_oracle as mo

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-case]", *a, flush=True)


def data(n):
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n, 48)).astype(np.float32)
    T = rng.standard_normal((n, 2)).astype(np.float32)
    w = rng.uniform(0.5, 1.5, n).astype(np.float32) / n
    return X, T, w


@pytest.mark.parametrize("n", [1, 15, 63, 64, 65, 64 * 256, 64 * 256 + 1, 64 * 515 + 17])
def test_gradient_by_batches(n):
    """Parts of a batch, whole batches, a second and a third round of the
    blocks: every parameter block within the BF16-level bound of the
    gradient tests."""
    say("train batches", n)
    m = Mlp(seed=5)
    p = m.params().astype(np.float64)
    X, T, w = data(n)
    loss, g = m.train_step(X, T, w, apply=False)
    Lo, go = mo.loss_and_grad(p, X.astype(np.float64), T.astype(np.float64), w.astype(np.float64), emulate_bf16=True)
    assert abs(loss / Lo - 1) < 1e-2
    o = 0
    for name, s in mo.SHAPES:
        k = int(np.prod(s))
        assert np.linalg.norm(g[o:o + k] - go[o:o + k]) <= 3e-2 * np.linalg.norm(go[o:o + k]) + 1e-12, name
        o += k


def test_fragments_follow_the_parameters():
    """The optimiser writes the updated weights into the three fragment copies
    itself: a handle given the trained parameters, whose copies are packed
    from them, evaluates and differentiates bit for bit the same."""
    say("train fragments")
    X, T, w = data(1000)
    a = Mlp(seed=3)
    for _ in range(3):
        a.train_step(X, T, w, lr=1e-2, wd=1e-3)
    b = Mlp(seed=8)
    b.set_params(a.params())
    assert np.array_equal(a.forward(X), b.forward(X))
    ga, gb = (m.train_step(X, T, w, apply=False) for m in (a, b))
    assert ga[0] == gb[0] and np.array_equal(ga[1], gb[1])
