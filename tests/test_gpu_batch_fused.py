"""Batched DP5(4): the fused stage and error forms (four rows per thread) against the separate
passes (one and two rows per thread).

The forms share the stage arithmetic; the error norm is summed in another order, so a step
may differ in its last bits: the solutions agree to the integrator's tolerance. Instances
lie at the edges of a 256-row granule, single and many, with slot counts 3, 4, 6 and 12,
computed and loaded columns and empty sink rows. The controller folds the error sums of up to
64 instances itself; 65 take the separate fold.
"""
import numpy as np
import pytest

import models
import numcme_hip as nh

pytestmark = pytest.mark.gpu


def _instances(kind, precision):
    out = []

    def add(S, props, th, states):
        sp = nh.StateSpaceSparse(S, states)
        out.append((nh.FspMatrixSparse(sp, models.to_product(props), th, precision=precision), len(states) + S.shape[1]))

    S, props, th = models.telegraph((0.5, 0.7, 2.0, 0.3))
    if kind == "edges":
        for n in (1, 2, 125, 126, 127, 128, 129, 254, 256):
            add(S, props, th, np.asarray(models.telegraph_states(n - 1)))
    elif kind in ("n64", "n65"):
        for i in range(int(kind[1:])):
            add(S, props, np.asarray(th) * (1.0 + 0.01 * i), np.asarray(models.telegraph_states(3 + 5 * i)))
    elif kind == "one":
        add(S, props, th, np.asarray(models.telegraph_states(200)))
    else:
        rng = np.random.default_rng(4)
        T, tp, tt = models.toggle((5.0, 4.0, 2.0, 1.0, 1.0))
        add(T, tp, tt, models.box_states([30, 17]))
        st = models.box_states([17, 30])
        add(T, tp, tt, st[rng.permutation(len(st))])
        C, cp, ct = models.cascade((2.0, 1.0, 0.5, 0.5, 0.2, 0.1))
        add(C, cp, ct, models.box_states([9, 9, 9]))
        if kind == "twelve":
            W, wp, wt = models.twelve_slot()
            add(W, wp, wt, models.box_states([6, 6, 6]))
        for n in (3, 700):
            add(S, props, th, np.asarray(models.telegraph_states(n)))
    return out


@pytest.mark.parametrize("precision,bar", [("fp64", 1e-9), ("fp32", 1e-6)])
@pytest.mark.parametrize("kind", ["one", "edges", "mixed", "twelve", "n64", "n65"])
def test_fused_against_separate(gpu, precision, bar, kind):
    inst = _instances(kind, precision)
    u0s = []
    for _, n in inst:
        u = np.zeros(n)
        u[0] = 1.0
        u0s.append(u)
    ts = np.array([0.0, 0.4, 1.5])
    B = nh.BatchFsp([m for m, _ in inst])
    got = {}
    for rows in (4, 2, 1):
        B.set_rows_per_thread(rows)
        # rtol 1e-11: local errors of the two step sequences stay below the bar
        got[rows] = B.solve(u0s, ts, rtol=1e-11, atol=1e-16)
    for i in range(len(inst)):
        for k in range(len(ts)):
            assert np.abs(got[4][i][k] - got[2][i][k]).sum() <= bar
            assert np.abs(got[4][i][k] - got[1][i][k]).sum() <= bar
            assert abs(got[4][i][k].sum() - 1.0) <= bar
