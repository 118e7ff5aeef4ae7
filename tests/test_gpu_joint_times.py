"""Joint values prepared for several stage times at once (_update_sparsematrix!,
fspsparsematrix.jl:154-166, run ahead of the mat-vecs of an integrator step).

A generator whose integrator has prepared value sets must multiply at any time, among them
times no set holds and times that sets of an earlier step held, exactly as a generator that
never integrated. Programs within and beyond the register evaluator's stack, several
workgroups with a partial last one, two joint reactions next to a separable one.
"""
import numpy as np
import pytest

import models
import numcme_hip as nh
from numcme_hip.solve import _integrate

pytestmark = pytest.mark.gpu


def _model(deep):
    def prod(t, x, p):
        v = p[3] + p[0] * (1.0 + 0.5 * nh.nmath.sin(t)) / (1.0 + (x[1] / p[1]) ** p[2])
        if deep:  # right-nested sums: a stack of 11 entries, beyond the register evaluator's 8
            v = v + (x[0] + (x[1] + (t + (p[0] + (p[1] + (p[2] + (p[3] + (p[4] + (x[0] + t))))))))) * 1e-6
        return v

    props = [
        nh.JointTimeVaryingPropensity(prod),
        nh.JointTimeVaryingPropensity(lambda t, x, p: p[4] * x[0] / (1.0 + 0.1 * t * x[0])),
        nh.propensity(lambda x, p: p[3] + p[0] / (1.0 + (x[0] / p[1]) ** p[2])),
        nh.propensity(lambda x, p: x[1], tfactor=lambda t, p: p[4] * (1.0 + 0.2 * nh.nmath.cos(t))),
    ]
    return nh.CmeModel(models.TOGGLE_S, props, [5.0, 4.0, 2.0, 1.0, 1.0])


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("deep", [False, True])
@pytest.mark.parametrize("bounds", [(2, 3), (15, 15), (40, 31)])
def test_prepared_times_leave_matvec_unchanged(gpu, precision, deep, bounds):
    model = _model(deep)
    states = models.box_states(bounds)
    space = nh.StateSpaceSparse(models.TOGGLE_S, states)
    used = nh.FspMatrixSparse(space, None, precision=precision, model=model)
    fresh = nh.FspMatrixSparse(space, None, precision=precision, model=model)
    n = len(states)
    u0 = np.zeros(n + 4)
    u0[0] = 1.0
    v = np.random.default_rng(1).random(n + 4)
    opts = nh.RK45(rtol=1e-6, atol=1e-10, precision=precision).opts(1e-6, 1e-4)
    h = 0.0
    for ts in ((0.0, 0.3), (0.1, 0.2, 0.7)):
        out = _integrate(used, opts, u0, ts[0], np.array(ts), space)
        total = out.p[-1].values.sum() + out.sinks[-1].sum()
        # mass: 1e-6 relative per step of error control, FP32 columns sum to zero exactly
        assert abs(total - 1.0) < 1e-5
        for t in (ts[-1], 0.0, 0.25, ts[0], ts[-1] - 0.01, h, 1.7):
            a, b = np.empty(n + 4), np.empty(n + 4)
            used.matvec_(a, t, v)
            fresh.matvec_(b, t, v)
            assert np.array_equal(a, b), t
        h = 0.5 * (ts[0] + ts[-1])
