"""GPU tests of the Krylov process's three forms.

A Krylov basis vector of the device expv (the integrator that replaces the reference's ODE
call around matvec!, fspsolve.jl:10-41) is formed, multiplied and summed by one launch of
the stored generator's column kernel, by separate launches (timing mode 2 forces them on any
generator), or, on a small space, with all the others in one workgroup. The forms share the
arithmetic and the order of the sums: a solve must give the same snapshots bit for bit.
Sizes lie at the edges of the one-workgroup form's row counts, of the 512-row blocks and of
the workgroup groups; the generators have 4, 6 and 12 slots, computed, loaded and mixed
columns, and sink rows of 1 to 700 entries. The errors of FP64 and FP32 solves are held
against the exact exponential.
"""
import numpy as np
import pytest
import scipy.linalg

import models
import numcme_hip as nh
from numcme_hip.solve import _integrate

pytestmark = pytest.mark.gpu


def _solve(S, states, model, precision, time_kernels, ts, tol=1e-9, m=30):
    space = nh.StateSpaceSparse(S, states)
    A = nh.FspMatrixSparse(space, None, precision=precision, model=model)
    u0 = np.zeros(len(states) + space.get_sink_count())
    u0[len(states) // 3] = 0.75
    u0[0] += 0.25
    opts = nh.KrylovExpv(m=m, tol=tol, precision=precision, time_kernels=time_kernels).opts(1e-6, 1e-4)
    out = _integrate(A, opts, u0, 0.0, np.array(ts), space)
    return out, A


def _check(S, states, props, th, precision, ts):
    model = nh.CmeModel(S, models.to_product(props), th)
    one, A = _solve(S, states, model, precision, 0, ts)
    sep, _ = _solve(S, states, model, precision, 2, ts)
    assert one.stats["steps"] == sep.stats["steps"] >= 2
    for k in range(len(ts)):
        assert np.array_equal(one.p[k].values, sep.p[k].values), k
        assert np.array_equal(one.sinks[k], sep.sinks[k]), k
        # mass: the tolerance 1e-9 per unit time, and per basis vector the storage rounding
        tot = one.p[k].values.sum() + one.sinks[k].sum()
        assert abs(tot - 1.0) < (1e-8 if precision == "fp64" else 1e-5)
    return A


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("n", [1, 3, 32, 127, 256, 257, 511, 512, 513, 1024, 1025, 2047, 2048, 2049])
def test_telegraph_sizes(gpu, precision, n):
    S, props, th = models.telegraph()
    _check(S, np.asarray(models.telegraph_states(n - 1)), props, th, precision, (0.0, 0.5, 4.0))


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("box", [(6, 699), (60, 70), (21, 389), (150, 301)])
@pytest.mark.parametrize("order", ["lattice", "shuffled"])
def test_toggle_boxes(gpu, precision, box, order):
    # sink rows of 6 to 700 entries; (60, 70) is past the one-workgroup form, (150, 301) has
    # 89 blocks
    S, props, th = models.toggle()
    states = models.box_states(box)
    if order == "shuffled":
        states = states[np.random.default_rng(5).permutation(len(states))]
    A = _check(S, states, props, th, precision, (0.0, 0.2, 0.7))
    assert A.info()["computed_col_slots"] == (4 if order == "lattice" else 0)


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("levels", [11, 12, 13, 40])
def test_cascade_expanded(gpu, precision, levels):
    # six slots: the one-workgroup form holds 2,048 states, larger spaces spread their blocks
    # over workgroups; expansion order, mixed columns
    S, props, th = models.cascade()
    space = nh.StateSpaceSparse(S, [0, 0, 0])
    space.expand(levels + 6)
    _check(S, space.get_states(), props, th, precision, (0.0, 0.3, 1.0))


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("bounds", [(8, 8, 8), (16, 17, 18)])
def test_twelve_slots(gpu, precision, bounds):
    # more slots than the fixed-count kernels and the one-workgroup form: 2 and 12 blocks
    S, props, th = models.twelve_slot()
    _check(S, models.box_states(bounds), props, th, precision, (0.0, 0.2, 0.5))


def test_max_steps_leaves_the_state_reached(gpu):
    # the combination that a small space's next process would have taken is applied before
    # the error
    import ctypes as C

    from numcme_hip import _lib as L

    S, props, th = models.telegraph()
    states = np.asarray(models.telegraph_states(99))
    model = nh.CmeModel(S, models.to_product(props), th)
    A = nh.FspMatrixSparse(nh.StateSpaceSparse(S, states), None, model=model)
    u0 = np.zeros(len(states) + 4)
    u0[0] = 1.0
    got = []
    for time_kernels in (0, 2):
        o = nh.KrylovExpv(tol=1e-9, time_kernels=time_kernels).opts(1e-6, 1e-4)
        o.max_steps = 2
        h, t, u = C.c_void_p(), C.c_double(), np.empty_like(u0)
        L.call("nc_solver_create", A.handle, C.byref(o), C.byref(h))
        L.call("nc_solver_set_state", h, 0.0, L.ptr(u0, C.c_double))
        with pytest.raises(nh.NumCmeHipError):
            L.call("nc_solver_run", h, 1, L.ptr(np.array([200.0]), C.c_double))
        L.call("nc_solver_get_state", h, C.byref(t), L.ptr(u, C.c_double))
        L.call("nc_solver_destroy", h)
        got.append((t.value, u))
    assert got[0][0] == got[1][0] > 0.0
    assert np.array_equal(got[0][1], got[1][1])
    assert abs(got[0][1].sum() - 1.0) < 1e-9


def _telegraph_exact(n, theta, dt, K):
    """Exact states at K + 1 times of the box of n counts, from a distribution on two states,
    and how much the exponential amplifies an error in the 2-norm over that time: at most, and
    in the mean square over errors of independent entries."""
    states = np.asarray(models.telegraph_states(n - 1))
    N = 2 * n
    G = np.zeros((N + 4, N + 4))
    for j, (off, on, m) in enumerate(states.tolist()):
        gene = (n + m, theta[0]) if off else (m, theta[1])
        for i, rate in (gene, (j + 1 if m + 1 < n else N + 2, theta[2] * on), (j - 1, theta[3] * m)):
            if rate:
                G[i, j] += rate
                G[j, j] -= rate
    E, s, amp, rms = scipy.linalg.expm(G * (dt / 16)), dt / 16, 1.0, 1.0
    while True:
        amp, rms = max(amp, np.linalg.norm(E, 2)), max(rms, np.linalg.norm(E) / np.sqrt(N))
        if s == dt:
            P = E
        if s >= dt * K:
            break
        E, s = E @ E, 2 * s
    u = np.zeros(N + 4)
    u[n // 3 * 2], u[0] = 0.75, 0.25
    ref = [u]
    for _ in range(K):
        ref.append(P @ ref[-1])
    return states, ref, amp, rms


def _telegraph_solve(n, theta, dt, K, tol, precision):
    states, ref, amp, rms = _telegraph_exact(n, theta, dt, K)
    S, props, th = models.telegraph(theta)
    model = nh.CmeModel(S, models.to_product(props), th)
    space = nh.StateSpaceSparse(S, states)
    A = nh.FspMatrixSparse(space, None, precision=precision, model=model)
    ts = dt * np.arange(K + 1)
    out = _integrate(A, nh.KrylovExpv(m=30, tol=tol, precision=precision).opts(1e-6, 1e-4), ref[0], 0.0, ts, space)
    err = [np.linalg.norm(np.concatenate([p.values, s]) - r) for p, s, r in zip(out.p, out.sinks, ref)]
    return out.stats["steps"], ts, np.array(err), amp, rms * max(np.linalg.norm(r) for r in ref[1:])


@pytest.mark.parametrize("n", [120, 300])
def test_fp32_near_stationary_steps(gpu, n):
    # Rates that FP32 holds exactly, ten relaxation times past the transient: what is left for
    # a step to follow is the rounding of its first vector, 2^-24 of each entry at most, and
    # asking for less than a quarter of that takes no more steps (1e-12 took 1.4 times the
    # steps of 1e-9). The errors of the steps add up as a random walk: four deviations
    theta = (0.0625, 0.5, 15.0, 1.0)
    steps = {}
    for tol in (1e-9, 1e-12):
        steps[tol], ts, err, _, size = _telegraph_solve(n, theta, 10.0, 20, tol, "fp32")
        k = steps[tol]
        assert err.max() <= 4 * np.sqrt(k) * 2.0 ** -24 * size
    assert steps[1e-12] <= 1.1 * steps[1e-9]


@pytest.mark.parametrize("n,theta,tol", [(120, (0.05, 0.1, 5.0, 0.05), 1e-6), (120, (0.05, 0.1, 5.0, 0.05), 1e-9),
                                         (400, (0.05, 0.1, 5.0, 0.05), 1e-9), (300, (0.01, 0.01, 3.0, 0.02), 1e-9),
                                         (400, (0.01, 0.01, 3.0, 0.02), 1e-6)])
def test_fp64_errors(gpu, n, theta, tol):
    # boxes whose Krylov space is never exhausted: at 30 vectors a step's error estimate is
    # held to 1.2e-3 of the tolerance per unit time; 2e-13 for the roundings of the steps
    _, ts, err, amp, _ = _telegraph_solve(n, theta, 10.0, 20, tol, "fp64")
    assert (err <= amp * 1.2e-3 * tol * ts + 2e-13).all()


@pytest.mark.parametrize("n,theta,tol", [(300, (0.05, 0.5, 15.0, 1.0), 1e-9), (700, (0.05, 0.5, 15.0, 1.0), 1e-6),
                                         (700, (0.02, 0.2, 30.0, 0.5), 1e-6), (300, (0.5, 5.0, 100.0, 1.0), 1e-6)])
def test_near_stationary_states(gpu, n, theta, tol):
    # stiff boxes far above the law's support, run to ten relaxation times: the step's error
    # estimate falls slowly with the step there, and the step control has to get by with its
    # ten rejections
    S, props, th = models.telegraph(theta)
    states = np.asarray(models.telegraph_states(n - 1))
    dt, K = 10.0, 20
    N = 2 * n
    G = np.zeros((N + 4, N + 4))
    for j, (off, on, m) in enumerate(states.tolist()):
        gene = (n + m, theta[0]) if off else (m, theta[1])
        for i, rate in (gene, (j + 1 if m + 1 < n else N + 2, theta[2] * on), (j - 1, theta[3] * m)):
            if rate:
                G[i, j] += rate
                G[j, j] -= rate
    P = scipy.linalg.expm(G * dt)
    ref = np.zeros(N + 4)
    ref[n // 3 * 2], ref[0] = 0.75, 0.25
    ts = dt * np.arange(K + 1)
    model = nh.CmeModel(S, models.to_product(props), th)
    space = nh.StateSpaceSparse(S, states)
    A = nh.FspMatrixSparse(space, None, precision="fp64", model=model)
    out = _integrate(A, nh.KrylovExpv(m=30, tol=tol, precision="fp64").opts(1e-6, 1e-4), ref, 0.0, ts, space)
    for k in range(K + 1):
        got = np.concatenate([out.p[k].values, out.sinks[k]])
        # per unit time a step accepts 1.2e-3 tol and an exhausted space leaves at most tol, or
        # 1e-8; the semigroup does not amplify it in the 1-norm, which 2-norm errors bound
        # within sqrt(N)
        assert np.linalg.norm(got - ref) <= (1.2e-3 * tol + min(tol, 1e-8)) * ts[k] * np.sqrt(N) + 1e-12
        ref = P @ ref
