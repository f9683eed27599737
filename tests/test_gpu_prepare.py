"""Graphs of 16, 4 and 1 steps are captured when first needed; imx_swm_prepare
asks for them ahead, and the timed runs of the learned correction's evaluation
capture none."""
import numpy as np
import pytest

from imodel_amd import learn
from imodel_amd.learn import Learn, Trainer, evaluate, restriction
from imodel_amd.mlp import Mlp
from imodel_amd.swm import H0_GEO, Ensemble, Mesh, Swm

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-case]", *a, flush=True)


@pytest.mark.parametrize("prec", ["fp64_ref", "fp32"])
def test_prepare(prec):
    say("prepare", prec)
    m = Mesh.icos(3)
    h, u = m.spectral(1)
    with Swm(m, precision=prec, dt=600.0) as s:
        s.set_state(h, u)
        s.step(1)
        assert (s.prepare(1), s.prepare(0), s.prepare(21), s.prepare(21)) == (0, 0, 2, 0)
        s.set_coriolis(2, 1e-4)
        s.set_coriolis()
        assert (s.prepare(16), s.prepare(5)) == (1, 2)
        x = s.get_state()
        s.set_state(h, u)
        s.step(1)
        assert all(np.array_equal(a, b) for a, b in zip(s.get_state(), x))  # no step was run
    with Swm(m, precision=prec, dt=600.0, use_graph=False) as s:
        assert s.prepare(21) == 0


def test_prepare_of_ensembles_and_corrected_steps():
    say("prepare ensemble, learned")
    m = Mesh.icos(3)
    with Ensemble([m, m], [600.0, 300.0], precision="fp32", h_ref=H0_GEO) as E:
        assert (E.prepare(21), E.prepare(21)) == (3, 0)
    with Swm(m, precision="fp32", dt=600.0, h_ref=H0_GEO) as s:
        L = Learn(s, Mlp(seed=1), m)
        assert (L.prepare(4), L.prepare(5), L.prepare(21)) == (1, 1, 1)
        L.close()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_prepared_before_the_first_state(prec):
    """Without h_ref the first state sets the storage offset, which the captured
    steps hold: graphs captured before it are not used after it."""
    say("prepare before the first state", prec)
    m = Mesh.icos(3)
    h, u = m.spectral(2)
    got = []
    for early in (0, 5):
        with Ensemble([m, m], [600.0, 300.0], precision=prec) as E, Swm(m, precision=prec, dt=600.0) as s:
            E.prepare(early)
            s.prepare(early)
            for i in range(2):
                E.set_state(i, h, u)
            s.set_state(h, u)
            E.step(5)
            s.step(5)
            got.append(E.get_state(0) + E.get_state(1) + s.get_state())
    assert all(np.array_equal(a, b) for a, b in zip(*got))


def test_evaluation_times_no_capture(monkeypatch):
    say("evaluation")
    timed, seen = [False], []

    def sync_time(fn):
        timed[0] = True
        fn()
        timed[0] = False
        return 1.0

    for cls in (Swm, Learn):
        def step(self, nsteps, *a, of=cls.step):
            if timed[0]:
                seen.append(self.prepare(nsteps))
            return of(self, nsteps, *a)
        monkeypatch.setattr(cls, "step", step)
    monkeypatch.setattr(learn, "_sync_time", sync_time)
    tr = Trainer(gc=2, gf=4, dt_c=1800.0, log=lambda *a: None)
    m3 = Mesh.icos(3)
    with Swm(m3, precision="fp32", dt=900.0, h_ref=H0_GEO) as mid:
        evaluate(tr, 1, 21, bound=0.0,
                 mid=(mid,) + restriction(tr.fine_mesh, m3) + restriction(m3, tr.coarse_mesh))
    assert seen == [0, 0, 0]
