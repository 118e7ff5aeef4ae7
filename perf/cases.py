"""The workloads whose speed matters to a user of this library, as plain cases.

Every case is one complete call of the public package on the GPU, from the host data a
program holds (model, initial distribution, sample rows) to the host results it reads:

* ``krylov``    fixed-space transient solve of a time-invariant network (``solve`` with
                ``KrylovExpv``), telegraph or toggle switch, FP64 and FP32 storage;
* ``rk``        fixed-space solve of a time-varying network (``solve`` with ``RK45``): the
                four-state gene (separable law) or an induced toggle switch whose law is a
                sum that does not factor (joint law);
* ``sens``      forward sensitivities of the four-state gene, 13 blocks on a fixed space;
* ``batch``     many small instances of uneven size solved together (a parameter sweep);
* ``adaptive``  adaptive FSP: the telegraph model of the reference's documentation with
                state dropping, and the three-species cascade from an empty state;
* ``build``     expansion of a state space from one state, generator, one mat-vec, the
                marginals and the dense array of its result;
* ``adapter``   the adapter network on training records: logits, loss and gradient.

``exact`` gives the same outputs in FP64 from first principles: uniformization for
time-invariant networks, Taylor series in time for the others, on dense boxes of molecule
counts.
"""
from __future__ import annotations

import ctypes as C
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "numcme.jl_amd"))

import numcme_hip as nh  # noqa: E402
from numcme_hip import _lib as L  # noqa: E402


# ---- the cases ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest complete solve: gene expression with a few hundred mRNA, 21 outputs;
        # what a parameter fit calls thousands of times
        {"name": "telegraph_800_fp64", "kind": "krylov", "net": "telegraph", "n1": 400, "n2": 0, "prec": "fp64",
         "tol": 1e-9, "t": 200.0, "outs": 21},
        # the adaptive solve the reference's documentation times: R-step adapter with
        # dropping, default tolerances, a few hundred states
        {"name": "telegraph_adaptive", "kind": "adaptive", "net": "telegraph", "prec": "fp64", "R": 10, "t": 300.0,
         "outs": 11, "fsptol": 1e-6},
        # an ordinary two-species solve at the library's default tolerance, ragged box
        {"name": "toggle_301x259_fp64", "kind": "krylov", "net": "toggle", "n1": 301, "n2": 259, "prec": "fp64",
         "tol": 1e-12, "t": 10.0, "outs": 11},
        # the largest fixed solve, the benchmark's headline: 1024 x 1024 box, FP32 storage
        {"name": "toggle_1024_fp32", "kind": "krylov", "net": "toggle", "n1": 1024, "n2": 1024, "prec": "fp32",
         "tol": 1e-9, "t": 10.0, "outs": 11},
        # time-varying generator, separable law, a model fitted to mRNA counts
        {"name": "gene4_97_rk_fp32", "kind": "rk", "net": "gene4", "n1": 97, "n2": 97, "prec": "fp32", "rtol": 1e-8,
         "t": 120.0, "outs": 5},
        # time-varying generator, joint law evaluated for every state at every stage
        {"name": "toggle_induced_rk_fp64", "kind": "rk", "net": "induced", "n1": 101, "n2": 87, "prec": "fp64",
         "rtol": 1e-8, "t": 5.0, "outs": 6},
        # forward sensitivities to 12 parameters, an ordinary fit's space and precision
        {"name": "gene4_48_sens_fp64", "kind": "sens", "net": "gene4", "n1": 48, "n2": 48, "prec": "fp64",
         "rtol": 1e-8, "t": 120.0, "outs": 3},
        # the same on the largest space (262,144 states, 3.4 million unknowns), FP32 storage
        {"name": "gene4_256_sens_fp32", "kind": "sens", "net": "gene4", "n1": 256, "n2": 256, "prec": "fp32",
         "rtol": 1e-8, "t": 30.0, "outs": 2},
        # a parameter sweep: 48 telegraph and toggle instances of uneven size together
        {"name": "batch_48_fp32", "kind": "batch", "net": "mixed", "n": 48, "prec": "fp32", "t": 4.0, "outs": 3},
        # adaptive solve of a growing three-species space, selective expansion, no dropping
        {"name": "cascade_adaptive_fp32", "kind": "adaptive", "net": "cascade", "prec": "fp32", "R": 8, "t": 2.0,
         "outs": 3, "fsptol": 1e-4},
        # state-space expansion level by level, generator build, mat-vec, marginals, Array
        {"name": "toggle_build_400", "kind": "build", "net": "toggle", "levels": 400, "prec": "fp64"},
        # the adapter network over a training set: prediction, then loss and gradient
        {"name": "adapter_300k", "kind": "adapter", "net": "mlp", "n": 300_001, "prec": "bf16"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["krylov", "krylov", "krylov", "rk", "rk", "sens", "batch", "adaptive", "adaptive", "build",
                       "adapter"])
    prec = rng.choice(["fp32", "fp64"])
    if kind == "krylov":
        tol = rng.choice([1e-9, 1e-12])
        if rng.random() < 0.4:
            return {"kind": kind, "net": "telegraph", "n1": _log(rng, 40, 6000), "n2": 0, "prec": prec, "tol": tol,
                    "t": round(rng.uniform(10.0, 40.0), 2), "outs": rng.randint(2, 12)}
        n1 = _log(rng, 24, 800)
        return {"kind": kind, "net": "toggle", "n1": n1, "n2": max(16, min(800, int(n1 * rng.uniform(0.6, 1.4)))),
                "prec": prec, "tol": tol, "t": round(rng.uniform(2.0, 8.0), 2), "outs": rng.randint(2, 11)}
    if kind == "rk":
        n1 = _log(rng, 16, 150)
        net = rng.choice(["gene4", "induced"])
        return {"kind": kind, "net": net, "n1": n1, "n2": max(12, int(n1 * rng.uniform(0.7, 1.0))), "prec": prec,
                "rtol": 1e-8, "t": round(rng.uniform(20.0, 90.0) if net == "gene4" else rng.uniform(1.0, 5.0), 2),
                "outs": rng.randint(2, 6)}
    if kind == "sens":
        n1 = _log(rng, 16, 130)
        return {"kind": kind, "net": "gene4", "n1": n1, "n2": max(12, int(n1 * rng.uniform(0.7, 1.0))), "prec": prec,
                "rtol": 1e-8, "t": round(rng.uniform(10.0, 40.0), 2), "outs": rng.randint(2, 3)}
    if kind == "batch":
        return {"kind": kind, "net": "mixed", "n": rng.randint(5, 47), "prec": prec,
                "t": round(rng.uniform(1.0, 4.0), 2), "outs": rng.randint(2, 4)}
    if kind == "adaptive":
        if rng.random() < 0.5:
            return {"kind": kind, "net": "telegraph", "prec": prec, "R": rng.randint(5, 20),
                    "t": round(rng.uniform(60.0, 300.0), 1), "outs": rng.randint(2, 11), "fsptol": 1e-6}
        return {"kind": kind, "net": "cascade", "prec": prec, "R": rng.randint(5, 12),
                "t": round(rng.uniform(0.6, 1.8), 2), "outs": rng.randint(2, 4), "fsptol": 1e-4}
    if kind == "build":
        return {"kind": kind, "net": "toggle", "levels": _log(rng, 20, 390), "prec": prec}
    return {"kind": kind, "net": "mlp", "n": _log(rng, 500, 290_000), "prec": "bf16"}


# ---- networks ----------------------------------------------------------------------------
TELEGRAPH_S = np.array([[-1, 1, 0, 0], [1, -1, 0, 0], [0, 0, 1, -1]])
TOGGLE_S = np.array([[1, -1, 0, 0], [0, 0, 1, -1]])
CASCADE_S = np.array([[1, 0, 0, -1, 0, 0], [0, 1, 0, 0, -1, 0], [0, 0, 1, 0, 0, -1]])
GENE4_MOVES = [(0, 1), (1, 0), (1, 2), (2, 1), (2, 3), (3, 2)]
TELEGRAPH_THETA = (0.05, 0.1, 5.0, 0.05)
TELEGRAPH_ADAPTIVE_THETA = (0.05, 0.1, 5.0, 0.5)
TOGGLE_THETA = (50.0, 20.0, 2.5, 1.0, 1.0)
INDUCED_THETA = (20.0, 10.0, 2.5, 1.0, 1.0, 0.6)
GENE4_THETA = (1.3e-3, 3.2e-3, 5.9e-3, 2e-2, 1.5e-3, 4.6e-3, 0.01, 1e-2, 0.2, 1.5, 0.05, 1e-3)
CASCADE_THETA = (10.0, 2.0, 1.0, 0.5, 0.2, 0.1)
CASCADE_BOX = (72, 160, 160)  # holds all but 1e-9 of the cascade's mass over its time span
COUNTS = 512  # no species of the adaptive cases reaches this count
TELEGRAPH_BOX = (2, 256)
W = 1.0  # angular frequency of the induced toggle's signal


def _theta(base, seed, spread=0.05):
    """The network's rates, each scaled by its own factor: another seed is another model."""
    r = np.random.default_rng(seed)
    return [float(v) for v in np.asarray(base) * np.exp(r.uniform(-spread, spread, size=len(base)))]


def _telegraph(theta):
    return nh.CmeModel(TELEGRAPH_S, [nh.propensity(lambda x, p: p[0] * x[0]), nh.propensity(lambda x, p: p[1] * x[1]),
                                     nh.propensity(lambda x, p: p[2] * x[1]), nh.propensity(lambda x, p: p[3] * x[2])],
                       theta)


def _toggle(theta):
    return nh.CmeModel(TOGGLE_S, [nh.propensity(lambda x, p: p[3] + p[0] / (1.0 + (x[1] / p[1]) ** p[2])),
                                  nh.propensity(lambda x, p: p[4] * x[0]),
                                  nh.propensity(lambda x, p: p[3] + p[0] / (1.0 + (x[0] / p[1]) ** p[2])),
                                  nh.propensity(lambda x, p: p[4] * x[1])], theta)


def _induced(theta):
    """Toggle switch whose first promoter is driven by a periodic signal: basal plus
    (1 + p5 sin t) times the Hill law, a sum that stays a joint function of time and state."""
    nm = nh.nmath
    return nh.CmeModel(TOGGLE_S, [
        nh.JointTimeVaryingPropensity(
            lambda t, x, p: p[3] + p[0] * (1.0 + p[5] * nm.sin(t)) / (1.0 + (x[1] / p[1]) ** p[2])),
        nh.propensity(lambda x, p: p[4] * x[0]),
        nh.propensity(lambda x, p: p[3] + p[0] / (1.0 + (x[0] / p[1]) ** p[2])),
        nh.propensity(lambda x, p: p[4] * x[1])], theta)


def _gene4_stoich():
    S = np.zeros((6, 12), dtype=np.int64)
    for r, (a, b) in enumerate(GENE4_MOVES):
        S[a, r], S[b, r] = -1, 1
    S[4, 6:10] = 1
    S[4, 10], S[5, 10] = -1, 1
    S[5, 11] = -1
    return S


def _gene4(theta):
    nm = nh.nmath
    sig = lambda t: (1.0 - nm.exp(-6e-3 * t)) * nm.exp(-9e-3 * t)
    species = [0, 1, 1, 2, 2, 3, 0, 1, 2, 3, 4, 5]
    props = [nh.propensity((lambda r, s: lambda x, p: p[r] * x[s])(r, s)) for r, s in enumerate(species)]
    props[3] = nh.propensity(lambda x, p: x[2], tfactor=lambda t, p: nm.max(0.0, p[3] - 0.12 * sig(t)))
    return nh.CmeModel(_gene4_stoich(), props, theta)


def _cascade(theta):
    return nh.CmeModel(CASCADE_S, [
        nh.propensity(lambda x, p: p[0] + 0.0 * x[0]), nh.propensity(lambda x, p: p[1] * x[0]),
        nh.propensity(lambda x, p: p[2] * x[1]), nh.propensity(lambda x, p: p[3] * x[0]),
        nh.propensity(lambda x, p: p[4] * x[1]), nh.propensity(lambda x, p: p[5] * x[2])], theta)


def _telegraph_states(n):
    m = np.arange(n)
    one, zero = np.ones_like(m), np.zeros_like(m)
    return np.concatenate([np.stack([one, zero, m], axis=1), np.stack([zero, one, m], axis=1)])


def _box_states(n1, n2):
    out = np.empty((n1 * n2, 2), dtype=np.int64)
    out[:, 0] = np.tile(np.arange(n1), n2)
    out[:, 1] = np.repeat(np.arange(n2), n1)
    return out


def _gene4_states(n1, n2):
    g = np.repeat(np.eye(4, dtype=np.int64), n1 * n2, axis=0)
    return np.concatenate([g, np.tile(_box_states(n1, n2), (4, 1))], axis=1)


def _batch_specs(case, seed):
    """(net, theta, n) of each instance: telegraph spaces of 200 to about 2,000 states and
    toggle boxes of about 400 to 40,000, the sizes following the rates as in a sweep."""
    r = np.random.default_rng([seed, 1])
    sizes = np.random.default_rng(case["n"])  # the sizes belong to the case, the rates to the seed
    specs = []
    for i in range(case["n"]):
        if i % 2 == 0:
            th = np.asarray(TELEGRAPH_THETA) * np.exp(r.uniform(-0.7, 0.7, size=4))
            n = int(round(math.exp(sizes.uniform(math.log(100), math.log(1000)))))
            specs.append(("telegraph", [float(v) for v in th], n))
        else:
            th = np.asarray(TOGGLE_THETA) * np.exp(r.uniform(-0.3, 0.3, size=5))
            n = int(round(math.exp(sizes.uniform(math.log(20), math.log(200)))))
            specs.append(("toggle", [float(v) for v in th], n))
    return specs


def _times(case):
    return np.linspace(0.0, case["t"], case["outs"])


def _adapter_rows(case, seed):
    """Feature rows as an adaptive run records them (scaled counts, log probabilities and
    propensities, time, sink share) and their 0/1 labels."""
    r = np.random.default_rng(seed)
    n = case["n"]
    X = np.empty((n, 8), dtype=np.float32)
    X[:, 0:3] = r.random((n, 3), dtype=np.float32)
    X[:, 3] = -r.random(n, dtype=np.float32)
    X[:, 4] = r.random(n, dtype=np.float32)
    X[:, 5] = -r.random(n, dtype=np.float32)
    X[:, 6] = r.random(n, dtype=np.float32)
    X[:, 7] = np.round(r.random(n, dtype=np.float32) * 6) / 6
    Y = (X[:, 3] + 0.4 * X[:, 0] + 0.2 * X[:, 4] + 0.1 * r.standard_normal(n, dtype=np.float32) > -0.3)
    return X, Y.astype(np.float32)


def _adapter_params(seed):
    """Weights of a network in use: scaled normal, as its initialisation and training leave them."""
    r = np.random.default_rng([seed, 2])
    p = np.empty(4801, dtype=np.float32)
    p[:512] = r.standard_normal(512) / math.sqrt(8)
    p[512:576] = 0.05 * r.standard_normal(64)
    p[576:4672] = r.standard_normal(4096) / math.sqrt(64)
    p[4672:4736] = 0.05 * r.standard_normal(64)
    p[4736:4800] = r.standard_normal(64) / math.sqrt(64)
    p[4800] = 0.1
    return p


# ---- one pass ----------------------------------------------------------------------------
def prepare(case, seed):
    kind, net = case["kind"], case["net"]
    st = {"case": case}
    if kind == "batch":
        models, states, u0s = [], [], []
        base = {"telegraph": _telegraph(list(TELEGRAPH_THETA)), "toggle": _toggle(list(TOGGLE_THETA))}
        for name, th, n in _batch_specs(case, seed):
            models.append(base[name].with_parameters(th))
            states.append(_telegraph_states(n) if name == "telegraph" else _box_states(n, n))
            u0 = np.zeros(len(states[-1]) + 4)
            u0[0] = 1.0
            u0s.append(u0)
        st.update(models=models, states=states, u0s=u0s, ts=_times(case))
    elif kind == "adapter":
        X, Y = _adapter_rows(case, seed)
        mlp = nh.AdapterMlp(seed % (1 << 31))
        mlp.params = _adapter_params(seed)
        st.update(X=X, Y=Y, mlp=mlp)
    elif kind == "build":
        st.update(model=_toggle(_theta(TOGGLE_THETA, seed)))
    elif kind == "adaptive":
        if net == "telegraph":
            st.update(model=_telegraph(_theta(TELEGRAPH_ADAPTIVE_THETA, seed)),
                      p0=nh.FspVectorSparse([[1, 0, 0]], [1.0]), adapter=nh.RStepAdapter(5, case["R"], True),
                      ode=nh.KrylovExpv(precision=case["prec"], tol=1e-9))
        else:
            st.update(model=_cascade(_theta(CASCADE_THETA, seed)), p0=nh.FspVectorSparse([[0, 0, 0]], [1.0]),
                      adapter=nh.SelectiveRStepAdapter(2, case["R"], False),
                      ode=nh.RK45(rtol=1e-6, atol=1e-10, precision=case["prec"]))
    else:
        if net == "telegraph":
            model, states = _telegraph(_theta(TELEGRAPH_THETA, seed)), _telegraph_states(case["n1"])
        elif net == "toggle":
            model, states = _toggle(_theta(TOGGLE_THETA, seed)), _box_states(case["n1"], case["n2"])
        elif net == "induced":
            model, states = _induced(_theta(INDUCED_THETA, seed)), _box_states(case["n1"], case["n2"])
        else:
            model, states = _gene4(_theta(GENE4_THETA, seed)), _gene4_states(case["n1"], case["n2"])
        if kind == "sens":
            # the space and its sensitivity matrix are built once; a fit solves on them
            model = nh.CmeModelWithSensitivity(model)
            space = nh.StateSpaceSparse(model.get_stoich_matrix(), states)
            SA = nh.ForwardSensFspMatrixSparse(model, space, precision=case["prec"])
            u0 = np.zeros(SA.rowcount * (SA.parameter_count + 1))
            u0[0] = 1.0
            st.update(model=model, space=space, SA=SA, u0=u0, ts=_times(case))
        else:
            p = np.zeros(len(states))
            p[0] = 1.0
            ode = nh.KrylovExpv(precision=case["prec"], tol=case["tol"]) if kind == "krylov" else \
                nh.RK45(rtol=case["rtol"], atol=1e-14, precision=case["prec"])
            st.update(model=model, p0=nh.FspVectorSparse(states, p, copy=False), ode=ode)
    return st


def _dense(p):
    """The telegraph vector on the fixed box (G_on, mRNA)."""
    states = p.states
    out = np.zeros(TELEGRAPH_BOX)
    out[states[:, 1], states[:, 2]] = p.values
    return out


def _marginal(p, species):
    """Marginal distribution of one species (1-based), summed on the device."""
    out = np.zeros(COUNTS)
    m = p.sum([s for s in (1, 2, 3) if s != species]).to_array()
    out[:len(m)] = m
    return out


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind in ("krylov", "rk"):
        out = nh.solve(st["model"], st["p0"], (0.0, case["t"]), st["ode"], saveat=_times(case))
        return {"p": [q.values for q in out.p], "kept": 1.0 - np.stack(out.sinks)}
    if kind == "sens":
        o = L.nc_solve_opts()
        L.call("nc_solve_opts_default", C.byref(o))
        o.method, o.rtol, o.atol = L.NC_METHOD_RK45, case["rtol"], 1e-14
        u0, ts = st["u0"], st["ts"]
        res = np.empty((len(ts), u0.size))
        L.call("nc_solve_sens_fixed", st["SA"].handle, C.byref(o), L.ptr(u0, C.c_double), len(ts),
               L.ptr(ts, C.c_double), L.ptr(res, C.c_double), None)
        blocks = res.reshape(len(ts), 13, -1)
        # one output per block: the parameters' sensitivities differ by orders of magnitude
        return {"blocks": [blocks[-1, b] for b in range(13)], "p": [blocks[k, 0] for k in range(len(ts) - 1)]}
    if kind == "batch":
        B = nh.BatchFsp.from_models(st["models"], st["states"], case["prec"])
        B.solve(st["u0s"], st["ts"], fetch=False)
        return {"p": [np.concatenate(B.snapshots(k)) for k in range(len(st["ts"]))]}
    if kind == "adaptive":
        out = nh.solve(st["model"], st["p0"], (0.0, case["t"]),
                       nh.AdaptiveFspSparse(ode_method=st["ode"], space_adapter=st["adapter"]), saveat=_times(case),
                       fsptol=case["fsptol"])
        if case["net"] == "telegraph":
            # which states of probability near the rounding error are dropped is chance, so
            # the vectors are compared on a fixed box
            return {"t": np.asarray(out.t), "p": [_dense(q) for q in out.p]}
        return {"t": np.asarray(out.t), "states": [q.states for q in out.p], "p": [q.values for q in out.p],
                "kept": 1.0 - np.stack(out.sinks),
                "marginals": [[_marginal(q, s) for s in (1, 2, 3)] for q in out.p[:-1]]}
    if kind == "build":
        space = nh.StateSpaceSparse(TOGGLE_S, [[0, 0]])
        space.expand(case["levels"])
        A = nh.FspMatrixSparse(space, None, precision=case["prec"], model=st["model"])
        states = space.get_states()
        n = len(states)
        v = np.zeros(n + 4)
        v[:n] = _bump(states[:, 0], states[:, 1], case["levels"], np)
        y = A.matvec_(np.empty(n + 4), 0.0, v)
        p = nh.FspVectorSparse(states, y[:n], copy=False)
        return {"states": states, "y": y, "array": p.to_array(), "m1": p.sum([2]).to_array(),
                "m2": p.sum([1]).to_array()}
    logits = st["mlp"].forward(st["X"])
    grad, loss = st["mlp"].grad(st["X"], st["Y"])
    return {"logits": logits, "grad": grad, "loss": float(loss)}


def _bump(a, b, levels, xp):
    """A smooth two-peaked distribution over the expanded triangle."""
    s = 0.2 * levels + 2.0
    return xp.exp(-((a - 0.3 * levels) ** 2 + (b - 0.1 * levels) ** 2) / s) + \
        0.5 * xp.exp(-((a - 0.05 * levels) ** 2 + (b - 0.5 * levels) ** 2) / s)


# ---- what a pass cannot do without -------------------------------------------------------
def _matvecs(rate, t, tol):
    """Mat-vecs that any polynomial method needs over a span t: the degree at which a
    polynomial resolves exp on the generator's spectrum [-2 rate, 0] to the tolerance."""
    return math.ceil(math.sqrt(2.0 * rate * t * math.log(1.0 / tol)))


def work(case):
    """Bytes and FP64 operations of a pass: the host inputs once, the results once (eight
    bytes a value), and the integration's mat-vecs (``_matvecs``), each reading the stored
    nonzeros (value and column) and one vector and writing one."""
    kind, net = case["kind"], case["net"]
    vs = 4 if case["prec"] == "fp32" else 8
    if kind == "adapter":
        return {"bytes": 2.0 * 36 * case["n"], "flops": 4.0 * 9344 * case["n"]}
    if kind == "build":
        n = (case["levels"] + 1) * (case["levels"] + 2) / 2
        return {"bytes": n * (4 * 8 + 5 * (vs + 4) + 8 * 4), "flops": 2.0 * 5 * n}
    if kind == "batch":
        rows = row_mv = 0.0
        for name, th, n in _batch_specs(case, 0):
            r = 2 * n if name == "telegraph" else n * n
            rate = th[3] * n + 5.0 if name == "telegraph" else 2.0 * (th[4] * n + th[0])
            rows += r
            row_mv += _matvecs(rate, case["t"], 1e-8) * r
        return {"bytes": row_mv * (4 * (vs + 4) + 2 * vs) + rows * 8.0 * (1 + case["outs"]), "flops": 10.0 * row_mv}
    if kind == "adaptive":
        n, rate, tol = (200.0, 40.0, 1e-9) if net == "telegraph" else (30000.0 * case["t"] ** 3, 150.0, 1e-6)
        mv = _matvecs(rate, case["t"], tol)
        return {"bytes": n * (mv * (4 * (vs + 4) + 2 * vs) + 8.0 * case["outs"]), "flops": 10.0 * n * mv}
    if net == "telegraph":
        n, nnz, rate = 2 * case["n1"], 4, 0.05 * case["n1"] + 5.0
    elif net in ("toggle", "induced"):
        n, nnz, rate = case["n1"] * case["n2"], 5, case["n1"] + case["n2"] + 60.0
    else:
        n, nnz, rate = 4 * case["n1"] * case["n2"], 8, 0.05 * case["n1"] + 1e-3 * case["n2"] + 1.6
    blocks = 13 if kind == "sens" else 1
    mv = _matvecs(rate, case["t"], case["tol"] if kind == "krylov" else case["rtol"])
    return {"bytes": float(n * mv * (nnz * (vs + 4) + 2 * vs * blocks) + 8.0 * n * blocks * case["outs"]),
            "flops": float(2 * nnz * n * blocks * mv)}


def tolerance(case):
    """Relative 2-norm errors, about four times what another correct implementation of the
    same precision and solver tolerance shows against ``exact``."""
    kind, fp64 = case["kind"], case["prec"] == "fp64"
    if kind == "adapter":
        return {"rel": 2e-2, "max": 0.5}  # BF16 operands in the three layers
    if kind == "build":
        return {"rel": 1e-14 if fp64 else 1e-6, "max": 1e-5}
    if kind == "adaptive":  # the truncation that fsptol allows, and happy breakdown at 1e-7
        return {"rel": 4e-4, "max": 1e-2}
    if kind == "krylov":
        if case["net"] == "telegraph":  # happy breakdown at 1e-7 near the stationary state
            return {"rel": 2e-7 if fp64 else 1e-6, "max": 1e-3}
        return {"rel": (1e-9 if case["tol"] < 1e-10 else 1e-7) if fp64 else 1e-6, "max": 1e-3}
    if kind == "sens":  # the kinks of the pulse, met by error control alone
        return {"rel": 3e-5, "max": 1e-2}
    return {"rel": 4e-8 if fp64 else 1e-6, "max": 1e-3}


# ---- 64-bit results from first principles ------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


class _Reaction:
    """One reaction on a dense box: its rate over the box, the jump along the axes, and the
    cells it leaves the box from (its sink)."""

    def __init__(self, shape, rate, jump, only=None):
        rate = torch.broadcast_to(rate, shape).contiguous()
        src, dst, edge = [], [], []
        for ax, (n, s) in enumerate(zip(shape, jump)):
            if ax == 0 and only is not None:  # the one cell of the first axis with a nonzero rate
                src.append(slice(only, only + 1))
                dst.append(slice(only + s, only + s + 1))
                edge.append(slice(only, only + 1))
                continue
            src.append(slice(max(0, -s), n - max(0, s)))
            dst.append(slice(max(0, s), n + min(0, s)))
            edge.append(slice(max(0, -s), n) if s <= 0 else slice(n - s, n))
        leaves_box = any(s > 0 for ax, s in enumerate(jump) if not (ax == 0 and only is not None))
        self.src, self.dst, self.edge = (Ellipsis, *src), (Ellipsis, *dst), (Ellipsis, *edge)
        self.a, self.a_edge = rate[self.src].contiguous(), rate[self.edge].contiguous() if leaves_box else None
        self.rate, self.dims = rate, tuple(range(-len(shape), 0))
        # outflow counts only cells whose target has no negative count
        self.out = torch.zeros(shape, dtype=rate.dtype, device=rate.device)
        self.out[self.src] += rate[self.src]
        if self.a_edge is not None:
            self.out[self.edge] += rate[self.edge]

    def add(self, u, v):
        v[self.dst] += self.a * u[self.src]

    def sink(self, u):
        if self.a_edge is None:
            return torch.zeros(u.shape[:u.dim() - len(self.dims)], dtype=u.dtype, device=u.device)
        return (self.a_edge * u[self.edge]).sum(self.dims)


def _uniformize(reactions, u, times):
    """Snapshots (u, sinks) of a time-invariant network by uniformization: u(t) is the
    Poisson-weighted sum of P^k u, P = I + A / rate, every term non-negative."""
    out = sum(r.out for r in reactions)
    rate = float(out.max()) * 1.0000001
    stay = 1.0 - out / rate
    for r in reactions:
        r.a.div_(rate)
        if r.a_edge is not None:
            r.a_edge.div_(rate)
    sinks = torch.zeros(len(reactions), dtype=u.dtype, device=u.device)
    got, t = [], float(times[0])
    for target in times:
        span = float(target) - t
        steps = max(1, math.ceil(rate * span / 400.0)) if span > 0 else 0
        for _ in range(steps):
            lam = rate * span / steps
            terms = int(lam + 9.5 * math.sqrt(lam) + 30)
            w = np.exp(-lam + np.arange(terms + 1) * math.log(lam) - np.array([math.lgamma(k + 1.0)
                                                                            for k in range(terms + 1)]))
            tail = np.cumsum(w[::-1])[::-1] - w  # sum of the weights after k: a sink keeps what it got
            acc, acc_s = torch.zeros_like(u), sinks.clone()
            for k in range(terms + 1):
                acc.add_(u, alpha=float(w[k]))
                for i, r in enumerate(reactions):
                    if r.a_edge is not None:
                        acc_s[i] += float(tail[k]) * r.sink(u)
                v = stay * u
                for r in reactions:
                    r.add(u, v)
                u = v
            u, sinks = acc, acc_s
        t = float(target)
        got.append((u.clone(), sinks.clone()))
    return got


def _taylor(reactions, factors, blocks, u, times, breaks=(), terms=32, order=9):
    """Snapshots of u' = sum_r f_r(t) C_r u by Taylor series in time. ``factors[r]`` is a
    number or a function of t giving ``order`` Taylor coefficients; ``blocks`` maps extra
    leading blocks to the reaction whose derivative they are (with its factor's derivative
    as a function of t): S_i' = A S_i + g_i(t) C_i p. u: (blocks + 1, box) cells, sinks
    alongside as (blocks + 1, reactions)."""
    nb, R = u.shape[0], len(reactions)
    rate = 2.0 * float(sum(r.out * (abs(f) if not callable(f) else max(abs(f(0.0)[0]), abs(f(60.0)[0]), 1.0))
                           for r, f in zip(reactions, factors)).max())
    sinks = torch.zeros((nb, R), dtype=u.dtype, device=u.device)
    const = [(i, r, f) for i, (r, f) in enumerate(zip(reactions, factors)) if not callable(f)]
    varying = [(i, r, f) for i, (r, f) in enumerate(zip(reactions, factors)) if callable(f)]
    out_const = sum(r.out * f for _, r, f in const)
    got, t = [], float(times[0])
    for target in times:
        stops = [b for b in breaks if t < b < target] + [float(target)]
        for stop in stops:
            n = math.ceil(rate * (stop - t) / 4.0) if stop > t else 0
            h = (stop - t) / n if n else 0.0
            for k in range(n):
                t_k = t + k * h
                ser = [np.asarray(f(t_k + 1e-12 if k == 0 else t_k)) * h ** np.arange(order) for _, _, f in varying]
                gser = {b: g(t_k + 1e-12 if k == 0 else t_k) for b, (_, g) in blocks.items()}
                c, hist, tot, stot = u, [], u.clone(), sinks.clone()
                for q in range(terms):
                    d = c * (-out_const)
                    ds = torch.zeros_like(sinks)
                    for i, r, f in const:
                        d[r.dst] += f * (r.a * c[r.src])
                        if r.a_edge is not None:
                            ds[:, i] = f * r.sink(c)
                    d *= h
                    ds *= h
                    if varying:
                        hq = []
                        for i, r, f in varying:
                            m = -(r.out * c)
                            r.add(c, m)
                            hq.append((m, r.sink(c)))
                        hist.append(hq)
                        for e, (i, r, f) in enumerate(varying):
                            for o in range(min(order, q + 1)):
                                m, ms = hist[q - o][e]
                                d.add_(m, alpha=float(ser[e][o] * h))
                                if r.a_edge is not None:
                                    ds[:, i] += float(ser[e][o] * h) * ms
                    for b, (i, g) in blocks.items():
                        gc = gser[b]  # constant derivative factor between the breaks
                        if gc:
                            r = reactions[i]
                            m = -(r.out * c[0])
                            r.add(c[0], m)
                            d[b].add_(m, alpha=gc * h)
                            if r.a_edge is not None:
                                ds[b, i] += gc * h * r.sink(c[0])
                    c = d / (q + 1.0)
                    tot += c
                    stot += ds / (q + 1.0)
                u, sinks = tot, stot
            t = stop
        got.append((u.clone(), sinks.clone()))
    return got


def _telegraph_reactions(theta, n, dev):
    g = torch.tensor([[1.0], [0.0]], dtype=torch.float64, device=dev)  # axis 0: off, on
    m = torch.arange(n, dtype=torch.float64, device=dev)[None, :]
    shape = (2, n)
    return [_Reaction(shape, theta[0] * g, (1, 0), only=0), _Reaction(shape, theta[1] * (1 - g), (-1, 0), only=1),
            _Reaction(shape, theta[2] * (1 - g), (0, 1)), _Reaction(shape, theta[3] * m, (0, -1))]


def _hill(theta, x):
    return theta[0] / (1.0 + (x / theta[1]) ** theta[2])


def _toggle_reactions(theta, n1, n2, dev):
    x1 = torch.arange(n1, dtype=torch.float64, device=dev)[None, :]  # axes: species 2, species 1
    x2 = torch.arange(n2, dtype=torch.float64, device=dev)[:, None]
    shape = (n2, n1)
    return [_Reaction(shape, theta[3] + _hill(theta, x2), (0, 1)), _Reaction(shape, theta[4] * x1, (0, -1)),
            _Reaction(shape, theta[3] + _hill(theta, x1), (1, 0)), _Reaction(shape, theta[4] * x2, (-1, 0))]


def _gene4_reactions(n1, n2, dev):
    """The state factors of the twelve reactions on (gene, cytoplasmic, nuclear)."""
    shape = (4, n2, n1)
    g = torch.arange(4, device=dev)[:, None, None]
    nuc = torch.arange(n1, dtype=torch.float64, device=dev)[None, None, :]
    cyt = torch.arange(n2, dtype=torch.float64, device=dev)[None, :, None]
    at = lambda k: (g == k).to(torch.float64)
    rs = [_Reaction(shape, at(a), (b - a, 0, 0), only=a) for a, b in GENE4_MOVES]
    for k in range(4):
        r = _Reaction(shape, at(k), (0, 0, 1), only=k)
        rs.append(r)
    rs.append(_Reaction(shape, nuc.expand(shape), (0, 1, -1)))
    rs.append(_Reaction(shape, cyt.expand(shape), (0, -1, 0)))
    return rs


def _pulse(p3):
    """Taylor coefficients of max(0, p3 - 0.12 s(t)) and the times at which it changes branch."""
    s = lambda t: math.exp(-9e-3 * t) - math.exp(-15e-3 * t)

    def coeffs(t):
        if p3 - 0.12 * s(t) < 0.0:
            return np.zeros(9)
        c = np.array([-0.12 * (math.exp(-9e-3 * t) * (-9e-3) ** k - math.exp(-15e-3 * t) * (-15e-3) ** k)
                      / math.factorial(k) for k in range(9)])
        c[0] += p3
        return c

    grid = np.linspace(0.0, 1000.0, 20001)
    f = np.array([p3 - 0.12 * s(x) for x in grid])
    breaks = []
    for k in np.nonzero(f[1:] * f[:-1] < 0)[0]:
        lo, hi = grid[k], grid[k + 1]
        for _ in range(80):
            mid = 0.5 * (lo + hi)
            if (p3 - 0.12 * s(mid)) * (p3 - 0.12 * s(lo)) > 0:
                lo = mid
            else:
                hi = mid
        breaks.append(hi)
    return coeffs, breaks, lambda t: 1.0 if p3 - 0.12 * s(t) >= 0.0 else 0.0


def _numpy(x):
    return x.detach().cpu().numpy()


def exact(case, seed):
    kind, net, dev = case["kind"], case["net"], _device()
    f64 = dict(dtype=torch.float64, device=dev)
    if kind == "adapter":
        X, Y = _adapter_rows(case, seed)
        w = torch.tensor(_adapter_params(seed), **f64).requires_grad_()
        x, y = torch.tensor(X, **f64), torch.tensor(Y, **f64)
        h = torch.nn.functional.gelu(x @ w[:512].reshape(8, 64) + w[512:576], approximate="tanh")
        h = torch.nn.functional.gelu(h @ w[576:4672].reshape(64, 64) + w[4672:4736], approximate="tanh")
        z = h @ w[4736:4800] + w[4800]
        loss = torch.nn.functional.binary_cross_entropy_with_logits(z, y)
        loss.backward()
        return {"logits": _numpy(z), "grad": _numpy(w.grad), "loss": float(loss)}
    if kind == "build":
        n = case["levels"] + 1
        theta = _theta(TOGGLE_THETA, seed)
        x1 = np.arange(n, dtype=np.float64)[:, None]
        x2 = np.arange(n, dtype=np.float64)[None, :]
        inside = (x1 + x2 < n).astype(np.float64)
        v = _bump(x1, x2, case["levels"], np) * inside
        y = np.zeros((n, n))
        flows = [(theta[3] + _hill(theta, x2) + 0 * x1, (1, 0)), (theta[4] * x1 + 0 * x2, (-1, 0)),
                 (theta[3] + _hill(theta, x1) + 0 * x2, (0, 1)), (theta[4] * x2 + 0 * x1, (0, -1))]
        for a, (s1, s2) in flows:
            f = a * v
            y -= f
            y[max(0, s1):n + min(0, s1), max(0, s2):n + min(0, s2)] += f[max(0, -s1):n - max(0, s1),
                                                                         max(0, -s2):n - max(0, s2)]
        y *= inside
        return {"states": None, "y": None, "array": y, "m1": y.sum(1), "m2": y.sum(0)}
    if kind == "batch":
        if case["n"] > 60:
            return None
        ts, per_k = _times(case), [[] for _ in range(case["outs"])]
        for name, th, n in _batch_specs(case, seed):
            rs = _telegraph_reactions(th, n, dev) if name == "telegraph" else _toggle_reactions(th, n, n, dev)
            u = torch.zeros((2, n) if name == "telegraph" else (n, n), **f64)
            u[0, 0] = 1.0
            for k, (p, s) in enumerate(_uniformize(rs, u, ts)):
                per_k[k].append(torch.cat([p.reshape(-1), s]))
        return {"p": [_numpy(torch.cat(v)) for v in per_k]}
    if kind == "adaptive":
        ts = _times(case)
        if net == "telegraph":
            rs = _telegraph_reactions(_theta(TELEGRAPH_ADAPTIVE_THETA, seed), TELEGRAPH_BOX[1], dev)
            u = torch.zeros(TELEGRAPH_BOX, **f64)
        else:
            th = _theta(CASCADE_THETA, seed)
            a, b, c = (torch.arange(n, **f64).reshape([-1 if i == k else 1 for i in range(3)])
                       for k, n in enumerate(CASCADE_BOX))
            J = [(1, 0, 0), (0, 1, 0), (0, 0, 1), (-1, 0, 0), (0, -1, 0), (0, 0, -1)]
            rates = [th[0] + 0 * a, th[1] * a, th[2] * b, th[3] * a, th[4] * b, th[5] * c]
            rs = [_Reaction(CASCADE_BOX, r, j) for r, j in zip(rates, J)]
            u = torch.zeros(CASCADE_BOX, **f64)
        u.reshape(-1)[0] = 1.0
        got = [_numpy(p) for p, _ in _uniformize(rs, u, ts)]
        if net == "telegraph":  # the final snapshot appears twice
            return {"t": np.append(ts, ts[-1]), "p": got + got[-1:]}
        marg = [[np.pad(p.sum(tuple(a for a in range(3) if a != s)), (0, COUNTS - CASCADE_BOX[s])) for s in range(3)]
                for p in got]
        return {"t": np.append(ts, ts[-1]), "states": None, "p": None, "kept": None, "marginals": marg}
    ts = _times(case)
    if kind == "krylov":
        n1, n2 = case["n1"], case["n2"]
        if net == "telegraph":
            rs, shape = _telegraph_reactions(_theta(TELEGRAPH_THETA, seed), n1, dev), (2, n1)
        else:
            rs, shape = _toggle_reactions(_theta(TOGGLE_THETA, seed), n1, n2, dev), (n2, n1)
        u = torch.zeros(shape, **f64)
        u.reshape(-1)[0] = 1.0
        got = _uniformize(rs, u, ts)
        return {"p": [_numpy(p.reshape(-1)) for p, _ in got], "kept": 1.0 - np.stack([_numpy(s) for _, s in got])}
    if net == "induced":
        th = _theta(INDUCED_THETA, seed)
        n1, n2 = case["n1"], case["n2"]
        rs = _toggle_reactions(th, n1, n2, dev)
        x2 = torch.arange(n2, **f64)[:, None]
        # the driven part, (1 + p5 sin t) times the Hill law, split into constant and sine
        rs.append(_Reaction((n2, n1), th[5] * _hill(th, x2), (0, 1)))
        sine = lambda t: [math.sin(W * t + 0.5 * math.pi * k) * W ** k / math.factorial(k) for k in range(9)]
        u = torch.zeros((1, n2, n1), **f64)
        u.reshape(-1)[0] = 1.0
        got = _taylor(rs, [1.0] * 4 + [sine], {}, u, ts)
        sinks = []
        for _, s in got:
            s = s[0].clone()
            s[0] += s[4]
            sinks.append(_numpy(s[:4]))
        return {"p": [_numpy(p.reshape(-1)) for p, _ in got], "kept": 1.0 - np.stack(sinks)}
    th = _theta(GENE4_THETA, seed)
    n1, n2 = case["n1"], case["n2"]
    rs = _gene4_reactions(n1, n2, dev)
    pulse, breaks, dpulse = _pulse(th[3])
    factors = [pulse if r == 3 else th[r] for r in range(12)]
    blocks = {} if kind == "rk" else {r + 1: (r, dpulse if r == 3 else (lambda t: 1.0)) for r in range(12)}
    u = torch.zeros((1 + len(blocks), 4, n2, n1), **f64)
    u.reshape(-1)[0] = 1.0
    got = _taylor(rs, factors, blocks, u, ts, breaks)
    if kind == "rk":
        return {"p": [_numpy(p.reshape(-1)) for p, _ in got], "kept": 1.0 - np.stack([_numpy(s[0]) for _, s in got])}
    full = [torch.cat([p.reshape(13, -1), s], dim=1) for p, s in got]
    return {"blocks": [_numpy(full[-1][b]) for b in range(13)], "p": [_numpy(f[0]) for f in full[:-1]]}
