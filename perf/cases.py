"""The framework's workloads as timed cases: what a user's program does with
imodel_amd, through its public entry points, from the smallest call to the
largest mesh.

kind "tendency"  one right-hand side of host arrays (subroutine tendency)
     "run"       an initial state set, `steps` RK4 steps, the state read back:
                 a simulated interval between two outputs
     "ensemble"  the same for `instances` instances of mixed levels, each with
                 its own Courant-0.8 time step, advanced together
     "learned"   "run" with the per-edge network correcting every step
     "fit"       AdamW steps of that network on stored samples

Meshes and handles are made once per configuration and kept, as a program
that integrates many states keeps them. FP32 handles compute in 32 bits and
their states are returned so; FP64 handles return 64 bits. exact() restates
the paths in torch FP64 on the mesh's arrays.
"""
import math

import numpy as np
import torch

from imodel_amd.learn import Learn
from imodel_amd.mlp import Mlp
from imodel_amd.swm import ERAD_REF, GRAV, H0_GEO, OMEGA, Ensemble, Mesh, Swm, cfl_dt

SCHEMES = {  # par/swm.par option sets
    "plain": {},
    "hc": {"stag": "HC"},
    "k2": {"k2": 1e5, "diffus": "const"},
    "apvm": {"pv": "apvm", "pvspar": 0.5},
    "pxt16": {"wrap": "pxt16"},
    "gass18": {"wrap": "gass18"},
}


def cells(glevel):
    return 10 * 4 ** glevel + 2


def time_step(glevel):
    """900 s at glevel 5, halved per level (the benchmark's 112.5 s at 8);
    no longer than 1800 s."""
    return min(1800.0, 900.0 * 2.0 ** (5 - glevel))


def listed():
    def run(name, glevel, precision, steps, scheme="plain"):
        return {"name": name, "kind": "run", "glevel": glevel, "precision": precision, "scheme": scheme,
                "steps": steps}

    return [
        # one tendency call of the reference's drop-in boundary on a test mesh:
        # launches and copies are all there is
        {"name": "tendency_g3_ref", "kind": "tendency", "glevel": 3, "precision": "fp64_ref", "scheme": "plain"},
        # a simulated day of the FP64 parity configuration (glevel 5, 96 steps)
        run("day_g5_ref", 5, "fp64_ref", 96),
        # a day at the learned correction's coarse level: the plain model of it
        run("day_g6_fp32", 6, "fp32", 192),
        # the fused FP64 model, which makes the training truths
        run("run_g7_fp64", 7, "fp64", 96),
        # the benchmark: a day at glevel 8 in FP32
        run("day_g8_fp32", 8, "fp32", 768),
        # the mesh past the last-level cache
        run("run_g9_fp32", 9, "fp32", 48),
        # scheme options of par/swm.par at throughput size: PV upwinding ...
        run("apvm_g8_fp32", 8, "fp32", 96, "apvm"),
        # ... and the Perot-based methods
        run("pxt16_g7_fp32", 7, "fp32", 96, "pxt16"),
        # independent instances of mixed levels in one set of launches
        {"name": "ensemble_24", "kind": "ensemble", "instances": 24, "lowest": 4, "highest": 7,
         "precision": "fp32", "steps": 48},
        # a day of the corrected model at its configuration's level
        {"name": "learned_day_g6", "kind": "learned", "glevel": 6, "steps": 192},
        # the correction at the benchmark's size
        {"name": "learned_g8", "kind": "learned", "glevel": 8, "steps": 32},
        # training: shuffled AdamW steps over stored glevel-6 samples
        {"name": "fit_g6", "kind": "fit", "glevel": 6, "samples": 6, "steps": 24},
    ]


def draw(rng):
    kind = rng.choice(["tendency", "run", "run", "run", "run", "ensemble", "learned", "fit"])

    def count(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    if kind == "tendency":
        return {"kind": kind, "glevel": rng.randint(2, 7), "precision": rng.choice(["fp64_ref", "fp64", "fp32"]),
                "scheme": rng.choice(list(SCHEMES))}
    if kind == "run":
        g = rng.randint(3, 8)
        precision = rng.choice(["fp32", "fp32", "fp64", "fp64_ref"])
        return {"kind": kind, "glevel": g, "precision": precision,
                "scheme": rng.choice(["plain", "plain"] + list(SCHEMES)),
                "steps": count(8, min(300, 48 * 4 ** (9 - g) // {"fp32": 1, "fp64": 2, "fp64_ref": 4}[precision]))}
    if kind == "ensemble":
        lo = rng.randint(3, 5)
        return {"kind": kind, "instances": count(3, 30), "lowest": lo, "highest": rng.randint(lo, 7),
                "precision": rng.choice(["fp32", "fp64"]), "steps": count(8, 48)}
    if kind == "learned":
        g = rng.randint(4, 8)
        return {"kind": kind, "glevel": g, "steps": count(4, min(200, 24 * 4 ** (8 - g)))}
    return {"kind": kind, "glevel": rng.randint(3, 6), "samples": rng.randint(1, 8), "steps": count(4, 30)}


# ---- what a program keeps --------------------------------------------------
_meshes, _kept = {}, {}


def mesh(glevel):
    if glevel not in _meshes:
        _meshes[glevel] = Mesh.icos(glevel)
    return _meshes[glevel]


def levels(case):
    """Levels of an ensemble's instances (the same for every seed)."""
    r = np.random.default_rng(case["instances"])
    return [int(g) for g in r.integers(case["lowest"], case["highest"] + 1, size=case["instances"])]


def handle(case):
    """The step handle of a configuration (the correction's own objects are
    made per state: their scaling and stored samples belong to it)."""
    kind = case["kind"]
    if kind == "ensemble":
        key = (kind, case["instances"], case["lowest"], case["highest"], case["precision"])
        if key not in _kept:
            ms = [mesh(g) for g in levels(case)]
            _kept[key] = Ensemble(ms, [ensemble_dt(m) for m in ms], precision=case["precision"], h_ref=H0_GEO)
        return _kept[key]
    key = (case["glevel"], case.get("precision", "fp32"), case.get("scheme", "plain"))
    if key not in _kept:
        # the fused handles store h - h_ref; the reference-order ones store h
        h_ref = 0.0 if key[1] == "fp64_ref" else H0_GEO
        _kept[key] = Swm(mesh(key[0]), precision=key[1], dt=time_step(key[0]), h_ref=h_ref)
        if SCHEMES[key[2]]:
            _kept[key].set_scheme(**SCHEMES[key[2]])
    return _kept[key]


def ensemble_dt(m):
    return cfl_dt(m, np.array([80.0]))  # Courant 0.8 at 80 m/s plus the gravity wave


def sample(L, h, u):
    """Features and plain step from (h, u), and the step's increments."""
    L.swm.set_state(h, u)
    h0, u0 = L.swm.get_state()
    raw = L.sample(raw=True)
    h1, u1 = L.swm.get_state()
    return raw, u1 - u0, h1 - h0


def prepare(case, seed):
    kind, H = case["kind"], handle(case)
    state = {"case": case, "H": H}
    if kind == "ensemble":
        first = {g: mesh(g).spectral(1000 * seed + g) for g in set(levels(case))}
        # one draw per level, the wind reversed for every other instance
        state["x"] = [(first[g][0], -first[g][1] if i % 2 else first[g][1]) for i, g in enumerate(levels(case))]
        return state
    m = mesh(case["glevel"])
    state["h"], state["u"] = m.spectral(seed)
    if kind in ("learned", "fit"):
        L = state["L"] = Learn(H, Mlp(seed=seed), m)
        raw, du, dh = sample(L, state["h"], state["u"])
        # a correction of small amplitude (a network not yet trained must not
        # disturb the run), or unit-variance targets
        ts = (1e4, 1e3) if kind == "learned" else (1.0 / rms(0.1 * du), 1.0 / rms(0.1 * dh))
        state["scaling"] = (raw.mean(0), raw.std(0) + 1e-3) + ts
        L.set_scaling(*state["scaling"])
    if kind == "fit":
        # stored samples with targets the network can learn: a tenth of the
        # plain step's increments
        L.reserve(case["samples"])
        state["stored"] = []
        for k in range(case["samples"]):
            raw, du, dh = sample(L, *m.spectral(100 * seed + k))
            L.store(0.1 * du, 0.1 * dh)
            state["stored"].append((raw, 0.1 * du, 0.1 * dh))
    return state


def rms(x):
    return float(np.sqrt(np.mean(x * x)))


def out(case, h, u):
    if case.get("precision", "fp32") == "fp32":
        return h.astype(np.float32), u.astype(np.float32)
    return h, u


FIT = (5e-5, 2e-5, 1e-4, 3)  # the last rates of a schedule, weight decay, shuffle seed


def run(state):
    case, H, kind = state["case"], state["H"], state["case"]["kind"]
    if kind == "tendency":
        return out(case, *H.tendency(state["h"], state["u"]))
    if kind == "ensemble":
        for i, x in enumerate(state["x"]):
            H.set_state(i, *x)
        H.step(case["steps"])
        return [out(case, *H.get_state(i)) for i in range(len(state["x"]))]
    if kind == "fit":
        state["L"].mlp.init(1)  # a new fit: the same initial weights every pass
        state["L"].fit(case["steps"], *FIT)
        return state["L"].mlp.params()
    H.set_state(state["h"], state["u"])
    if kind == "learned":
        state["L"].step(case["steps"], 1e30)
    else:
        H.step(case["steps"])
    return out(case, *H.get_state())


def work(case):
    """Per RK4 stage the state, the RK base and the accumulators (17 passes
    over the state in a step) and the geometry no stage can do without: the
    two lengths of an edge, three kite areas, f and the area of a triangle,
    the area of a cell, and each edge's two cells. The network: 78,336
    operations per edge forward, three times that in training, on 48
    features of 16 bits."""
    kind = case["kind"]
    es = 4 if case.get("precision", "fp32") == "fp32" else 8
    total = {"bytes": 0.0, "flops": 0.0}
    for g in levels(case) if kind == "ensemble" else [case["glevel"]]:
        nv = cells(g)
        ne, nt = 3 * nv - 6, 2 * nv - 4
        geometry = es * (2 * ne + 5 * nt + nv) + 8 * ne
        flops = 250 * nv + 14 * nt + 10 * ne
        host = 2 * 8 * (nv + ne)
        if kind == "tendency":
            total["bytes"] += host + geometry
            total["flops"] += flops
            continue
        n = case["steps"]
        if kind == "fit":
            total["bytes"] += n * ne * (96 + 8 + 8)
            total["flops"] += 3.0 * n * 78336 * ne
            continue
        total["bytes"] += host + n * (4 * geometry + 17 * es * (nv + ne))
        total["flops"] += 4.0 * n * flops
        if kind == "learned":  # both states in, both corrected, 21 ids and 6 geometry features per edge
            total["bytes"] += n * (6 * es * (nv + ne) + 4 * 27 * ne)
            total["flops"] += n * 78336.0 * ne
    return total


# ---- the same in 64 bits, torch on the mesh's arrays -------------------------
_DEV = "cuda" if torch.cuda.is_available() else "cpu"


def tensor(x, dtype=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(x), device=_DEV).to(dtype)


def unit(v):
    return v / v.norm(dim=-1, keepdim=True)


def arc(a, b):
    return torch.atan2(torch.linalg.cross(a, b).norm(dim=-1), (a * b).sum(-1))


class Exact:
    """TRiSK/HTC tendency and RK4 (plain, k2, apvm, pxt16) of one mesh."""

    def __init__(self, m, scheme, dt):
        A = m.arrays
        opt = SCHEMES[scheme]
        self.dt, self.pvs, self.k2 = dt, opt.get("pvspar", 0.0), opt.get("k2", 0.0)
        self.px = opt.get("wrap") == "pxt16"

        def ids(k, w):
            return tensor(A[k].reshape(-1, w), torch.int64) - 1

        self.ev, self.esh, self.tv, self.te = ids("ed_v", 2), ids("ed_sh", 2), ids("tr_v", 3), ids("tr_ed", 3)
        ved = ids("v_ed", 6)
        self.ok = (ved >= 0).double()
        self.ved = ved.clamp(min=0)
        self.nnb = tensor(A["v_nnb"], torch.int64)
        self.ttg, tnr = tensor(A["hx_ttgout"].reshape(-1, 6)), tensor(A["hx_tnrccw"].reshape(-1, 6))
        self.tnr = tnr
        self.l, self.dl = tensor(A["ed_leng"]), tensor(A["edhx_leng"])
        self.Av, At = tensor(A["hx_areag"]), tensor(A["tr_areag"])
        self.f = 2.0 * OMEGA * torch.sin(tensor(A["tr_clat"]))
        self.curl = self.l[self.te] * tensor(A["tr_tg"].reshape(-1, 3)) / (At * ERAD_REF)[:, None]
        self.div = self.ok * self.ttg * self.dl[self.ved] / (self.Av * ERAD_REF)[:, None]
        kw = self.ok * 0.25 * (self.l * self.dl)[self.ved]
        self.kw = kw / kw.sum(1, keepdim=True)
        self.ht = tensor(A["tr_trhx_area"].reshape(-1, 3)) / At[:, None]
        P, C = tensor(A["v_p"].reshape(-1, 3)), tensor(A["tr_c"].reshape(-1, 3))
        E = tensor(A["ed_c"].reshape(-1, 3))
        a, b = P[self.ev[:, 0]], P[self.ev[:, 1]]
        self.nr = unit(torch.linalg.cross(a, b))
        self.tt = torch.sign((self.nr * (C[self.esh[:, 1]] - C[self.esh[:, 0]])).sum(-1))
        # where each edge sits in the rings of its two cells
        slot = torch.arange(ved.numel(), device=_DEV)
        self.at = torch.zeros((len(self.l), 2), dtype=torch.int64, device=_DEV)
        for q in range(2):
            mine = (self.ev[:, q][self.ved] == torch.arange(len(P), device=_DEV)[:, None]) & (ved >= 0)
            self.at[self.ved[mine], q] = slot.reshape(-1, 6)[mine]
        if not self.px:
            # TRiSK weight times sign(ttgout_j tnrccw_i) times the dual length of j
            w = tensor(A["hx_trskw"].reshape(-1, 6, 6))
            self.w = w * self.ttg[:, None, :] * tnr[:, :, None] * (self.ok * self.dl[self.ved])[:, None, :]
        if self.px or self.pvs:
            self.perot = self.tangent((self.ttg * self.ok * self.dl[self.ved])[..., None]
                                      * (E[self.ved] - P[:, None]) / self.Av[:, None, None], P)
        if self.pvs:
            te = self.te
            self.perot_t = self.tangent((-tensor(A["tr_tg"].reshape(-1, 3)) * self.l[te])[..., None]
                                        * (E[te] - C[:, None]) / At[:, None, None], C)
        if self.px:
            p = P[self.tv]
            ht = torch.stack([torch.linalg.cross(C, p[:, (i + 1) % 3]).mul(p[:, (i + 2) % 3]).sum(-1).abs()
                              for i in range(3)], 1)
            self.ht = ht / ht.sum(1, keepdim=True)
            d = arc(E[:, None], C[self.esh])
            self.eq = d.flip(1) / d.sum(1, keepdim=True)
            self.E = E

    @staticmethod
    def tangent(v, p):
        return v - (v * p[:, None]).sum(-1, keepdim=True) * p[:, None]

    def grad(self, x):
        return (x[self.ev[:, 1]] - x[self.ev[:, 0]]) / (self.l * ERAD_REF)

    def tendency(self, h, u):
        uh = u * h[self.ev].mean(1)
        zeta = (u[self.te] * self.curl).sum(1)
        q = (zeta + self.f) / (self.ht * h[self.tv]).sum(1)
        qe = (q[self.esh] * self.eq).sum(1) if self.px else q[self.esh].mean(1)
        if self.px or self.pvs:
            v = (self.perot * u[self.ved][..., None]).sum(1)
        if self.pvs:
            gq = self.tt * (q[self.esh[:, 1]] - q[self.esh[:, 0]]) / (self.dl * ERAD_REF)
            g = (self.perot_t * gq[self.te][..., None]).sum(1)
            qe = qe - self.pvs * self.dt * (g[self.esh].sum(1) * v[self.ev].sum(1)).sum(-1)
        K = 0.5 * (v * v).sum(-1) if self.px else (self.kw * u[self.ved] ** 2).sum(1)
        if self.px:
            a, b = ((self.perot * x[self.ved][..., None]).sum(1) for x in (uh, uh * qe))
            w = 0.25 * (qe[:, None] * a[self.ev].sum(1) + b[self.ev].sum(1))
            w = w - (w * self.E).sum(-1, keepdim=True) * self.E
            perp = -(w * self.nr).sum(-1)
        else:
            G, r = uh[self.ved], qe[self.ved]
            part = 0.5 * (r * (self.w * G[:, None, :]).sum(-1) + (self.w * (G * r)[:, None, :]).sum(-1))
            perp = part.reshape(-1)[self.at].sum(1) / self.l
        du = -self.grad(GRAV * h + K) - perp
        if self.k2:
            cz = self.k2 * zeta
            du = du + self.grad(self.k2 * (self.div * u[self.ved]).sum(1)) \
                - self.tt * (cz[self.esh[:, 1]] - cz[self.esh[:, 0]]) / (self.dl * ERAD_REF)
        return -(self.div * uh[self.ved]).sum(1), du

    def step(self, h, u):
        ah, au, x, y = 0.0, 0.0, h, u
        for c, w in ((0.5, 1.0), (0.5, 2.0), (1.0, 2.0), (0.0, 1.0)):
            dh, du = self.tendency(x, y)
            ah, au = ah + w / 6.0 * self.dt * dh, au + w / 6.0 * self.dt * du
            x, y = h + c * self.dt * dh, u + c * self.dt * du
        return h + ah, u + au

    # the correction's 48 features per edge (header of csrc/imx_learn.hip)
    def stencil(self, m):
        A, n = m.arrays, self.nnb
        nb = tensor(A["v_nb"].reshape(-1, 6), torch.int64) - 1
        edges, signs = [torch.arange(len(self.l), device=_DEV)], [torch.ones_like(self.l)]
        ring = {}
        for q in range(2):
            c, i = self.at[:, q] // 6, self.at[:, q] % 6
            for t in range(1, 6):
                j, good = (i + t) % n[c], t < n[c]
                edges.append(torch.where(good, self.ved[c, j], -1))
                signs.append(torch.where(good, torch.sign(self.ttg[c, j] * self.tnr[c, i]), 0.0))
                ring[q, t] = torch.where(t <= n[c] - 2, nb[c, j], -1)
        P = tensor(A["v_p"].reshape(-1, 3))
        c1, c2 = self.ev[:, 0], self.ev[:, 1]
        tri = self.tv[self.esh]  # the third vertex of each of the two triangles
        apex = tri.sum(-1) - c1[:, None] - c2[:, None]
        left = (self.nr * P[apex[:, 0]]).sum(-1) > 0
        cell = [c1, c2, torch.where(left, apex[:, 0], apex[:, 1]), torch.where(left, apex[:, 1], apex[:, 0])]
        cell += [ring[q, t] for q in range(2) for t in (2, 3, 4)]
        z = tensor(A["ed_c"].reshape(-1, 3))[:, 2]
        geo = [z, (1 - z * z).clamp(min=0).sqrt(), self.l / self.l.mean(), self.dl / self.dl.mean(),
               self.Av[c1] / self.Av.mean(), self.Av[c2] / self.Av.mean()]
        self.fe, self.fs, self.fc = torch.stack(edges, 1), torch.stack(signs, 1), torch.stack(cell, 1)
        self.geo = torch.stack(geo, 1)

    def features(self, h0, u0, h1, u1):
        e, c = self.fe.clamp(min=0), self.fc.clamp(min=0)
        good = (self.fc >= 0).double()
        return torch.cat([self.fs * u0[e], self.fs * (u1 - u0)[e], good * (h0 - H0_GEO)[c], good * (h1 - h0)[c],
                          self.geo], 1)

    def flux_div(self, F):
        return -self.Av.mean() / self.dl.mean() * ERAD_REF * (self.div * F[self.ved]).sum(1)


SHAPES = [(48, 128), (128,), (128, 128), (128,), (128, 128), (128,), (128, 2), (2,)]


def network(p, X):
    for k in range(0, 8, 2):
        X = X @ p[k] + p[k + 1]
        if k < 6:
            X = torch.nn.functional.gelu(X, approximate="tanh")
    return X


def unpack(p):
    at, parts = 0, []
    for s in SHAPES:
        n = int(np.prod(s))
        parts.append(tensor(p[at:at + n]).reshape(s))
        at += n
    return parts


def exact(case, seed):
    kind = case["kind"]
    if case.get("scheme", "plain") in ("hc", "gass18"):
        return None  # the plain case's arithmetic on other signs, and a scheme without a short closed form
    if kind == "ensemble":
        got = []
        for (h, u), g in zip(prepare(case, seed)["x"], levels(case)):
            X = Exact(mesh(g), "plain", ensemble_dt(mesh(g)))
            h, u = tensor(h), tensor(u)
            for _ in range(case["steps"]):
                h, u = X.step(h, u)
            got.append((h.cpu(), u.cpu()))
        return got
    m = mesh(case["glevel"])
    X = Exact(m, case.get("scheme", "plain"), time_step(case["glevel"]))
    if kind == "learned":
        state = prepare(case, seed)
        mu, sig, tsu, tsh = (tensor(x) for x in state["scaling"])
        p = unpack(state["L"].mlp.params())
        X.stencil(m)
    if kind == "fit":
        return exact_fit(case, prepare(case, seed), X)
    h, u = (tensor(x) for x in m.spectral(seed))
    if kind == "tendency":
        return tuple(x.cpu() for x in X.tendency(h, u))
    for _ in range(case["steps"]):
        h1, u1 = X.step(h, u)
        if kind == "learned":
            Y = network(p, (X.features(h, u, h1, u1) - mu) / sig)
            h1, u1 = h1 + X.flux_div(Y[:, 1]) / tsh, u1 + Y[:, 0] / tsu
        h, u = h1, u1
    return h.cpu(), u.cpu()


def exact_fit(case, state, X):
    """AdamW (0.9, 0.999, 1e-8; decay on the matrices) on samples drawn by
    SplitMix64, loss mean (Y0 - tu)^2 + mean (D Y1 - th)^2."""
    mu, sig, tsu, tsh = (tensor(x) for x in state["scaling"])
    data = [((tensor(raw) - mu) / sig, tensor(du) * tsu, tensor(dh) * tsh) for raw, du, dh in state["stored"]]
    state["L"].mlp.init(1)
    p = unpack(state["L"].mlp.params())
    M, V = [torch.zeros_like(x) for x in p], [torch.zeros_like(x) for x in p]
    lr0, lr1, wd, shuffle = FIT
    n, mask = case["steps"], (1 << 64) - 1
    for k in range(n):
        shuffle = (shuffle + 0x9E3779B97F4A7C15) & mask
        z = shuffle
        z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & mask
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
        F, tu, th = data[(z ^ (z >> 31)) % len(data)]
        p = [x.requires_grad_() for x in p]
        Y = network(p, F)
        loss = ((Y[:, 0] - tu) ** 2).mean() + ((X.flux_div(Y[:, 1]) - th) ** 2).mean()
        lr = lr0 + (lr1 - lr0) * k / max(1, n - 1)
        for i, g in enumerate(torch.autograd.grad(loss, p)):
            M[i], V[i] = 0.9 * M[i] + 0.1 * g, 0.999 * V[i] + 0.001 * g * g
            x = p[i].detach() * (1 - lr * wd if i % 2 == 0 else 1.0)
            p[i] = x - lr * (M[i] / (1 - 0.9 ** (k + 1))) / ((V[i] / (1 - 0.999 ** (k + 1))).sqrt() + 1e-8)
    return torch.cat([x.detach().reshape(-1) for x in p]).cpu()
