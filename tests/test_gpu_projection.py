"""GPU tests of the Krylov columns on spaces past the one-workgroup form.

Each column of the device expv (the Krylov integrator that replaces the reference's ODE
call around matvec!, fspsolve.jl:10-41 with fspsparsematrix.jl:196-247) forms a basis vector,
multiplies it and sums five products over the rows. On a stored generator one launch does
all three (timing mode 0); launches of their own form, multiply and sum on every other
generator and, in timing mode 2, on any. Both sum in the same order, so a solve must give the
same snapshots bit for bit. Spaces here have more than 4,096 states, which the one-workgroup
form does not take, and from one block of 512 rows per workgroup to four.
The solves' accuracy against the oracle is tested elsewhere (the C1/C2 parity tests).
"""
import numpy as np
import pytest

import models
import numcme_hip as nh
from numcme_hip.solve import _integrate

pytestmark = pytest.mark.gpu


def _solve(S, states, model, precision, time_kernels, m=30, ts=(0.0, 0.5, 2.0), rows=2):
    space = nh.StateSpaceSparse(S, states)
    A = nh.FspMatrixSparse(space, model.propensities, model.parameters, precision=precision, model=model)
    A.set_rows_per_thread(rows)
    p0 = np.zeros(len(states))
    p0[int(np.flatnonzero((states == 0).all(axis=1))[0])] = 1.0
    u0 = np.concatenate([p0, np.zeros(space.get_sink_count())])
    opts = nh.KrylovExpv(m=m, tol=1e-9, precision=precision, time_kernels=time_kernels).opts(1e-6, 1e-4)
    out = _integrate(A, opts, u0, 0.0, np.array(ts), space)
    return [(p.values, np.asarray(s)) for p, s in zip(out.p, out.sinks)], A


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("order", ["lattice", "shuffled"])
def test_column_equals_separate_launches(gpu, precision, order):
    # lattice order: every slot's columns computed; shuffled: every slot's loaded. 200 x 300
    # states is not a multiple of 512 rows: the last of 118 blocks, each a workgroup's only
    # one, is partly past the states, and the 4 sink rows are added by the fold.
    S, props, th = models.toggle()
    states = models.box_states([199, 299])
    if order == "shuffled":
        states = states[np.random.default_rng(3).permutation(len(states))]
    model = nh.CmeModel(S, models.to_product(props), th)
    fused, A = _solve(S, states, model, precision, 0)
    inf = A.info()
    assert inf["rows_per_thread"] == 2 and inf["matrix_free"] == 0
    assert inf["computed_col_slots"] == (4 if order == "lattice" else 0)
    plain, _ = _solve(S, states, model, precision, 2)
    for (pa, sa), (pb, sb) in zip(fused, plain):
        assert np.array_equal(pa, pb) and np.array_equal(sa, sb)
    tot = fused[-1][0].sum() + fused[-1][1].sum()
    assert abs(tot - 1.0) < (1e-6 if precision == "fp32" else 1e-9)


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("order", ["lattice", "shuffled"])
@pytest.mark.parametrize("box", [(599, 521), (1400, 740)])
def test_several_blocks_per_workgroup(gpu, precision, order, box):
    # 313,200 states in 612 blocks and 1,038,141 in 2,028: 512 workgroups of one or two, and
    # of three or four blocks
    S, props, th = models.toggle()
    states = models.box_states(box)
    assert len(states) > 512 * 512 and len(states) % 512
    if order == "shuffled":
        states = states[np.random.default_rng(7).permutation(len(states))]
    model = nh.CmeModel(S, models.to_product(props), th)
    ts = (0.0, 0.01, 0.03)
    one, A = _solve(S, states, model, precision, 0, ts=ts)
    assert A.info()["computed_col_slots"] == (4 if order == "lattice" else 0)
    sep, _ = _solve(S, states, model, precision, 2, ts=ts)
    for (pa, sa), (pb, sb) in zip(one, sep):
        assert np.array_equal(pa, pb) and np.array_equal(sa, sb)
    tot = one[-1][0].sum() + one[-1][1].sum()
    assert abs(tot - 1.0) < (1e-6 if precision == "fp32" else 1e-9)


@pytest.mark.parametrize("m", [3, 5, 17, 31])
def test_every_basis_count(gpu, m):
    # 66 x 66 states, 9 workgroups: Krylov dimensions up to the largest, of
    # which the last column alone has no successor to fold its sums. Timing mode 1 runs the
    # column kernel one launch at a time, mode 0 as a graph.
    S, props, th = models.toggle()
    states = models.box_states([65, 65])
    model = nh.CmeModel(S, models.to_product(props), th)
    ts = (0.0, 0.02, 0.05) if m < 5 else (0.0, 0.5, 2.0)
    plain, _ = _solve(S, states, model, "fp32", 2, m=m, ts=ts)
    for time_kernels in (0, 1):
        fused, _ = _solve(S, states, model, "fp32", time_kernels, m=m, ts=ts)
        for (pa, sa), (pb, sb) in zip(fused, plain):
            assert np.array_equal(pa, pb) and np.array_equal(sa, sb)


@pytest.mark.parametrize("m", [3, 5, 17, 31])
def test_every_basis_count_one_workgroup(gpu, m):
    # 64 x 64 states: mode 0 is the one-workgroup form, mode 1 the column kernel with one
    # workgroup over the eight blocks, mode 2 the separate launches
    S, props, th = models.toggle()
    states = models.box_states([63, 63])
    model = nh.CmeModel(S, models.to_product(props), th)
    ts = (0.0, 0.02, 0.05) if m < 5 else (0.0, 0.5, 2.0)
    plain, _ = _solve(S, states, model, "fp32", 2, m=m, ts=ts)
    for time_kernels in (0, 1):
        got, _ = _solve(S, states, model, "fp32", time_kernels, m=m, ts=ts)
        for (pa, sa), (pb, sb) in zip(got, plain):
            assert np.array_equal(pa, pb) and np.array_equal(sa, sb)


@pytest.mark.parametrize("rows", [1, 4])
def test_every_mat_vec_shape(gpu, rows):
    # the column kernel has its own split of the rows: a generator whose mat-vec was tuned to
    # another one has the form as well, and the solve gives the same bits
    S, props, th = models.toggle()
    states = models.box_states([99, 70])
    model = nh.CmeModel(S, models.to_product(props), th)
    ref, _ = _solve(S, states, model, "fp32", 0)
    got, A = _solve(S, states, model, "fp32", 0, rows=rows)
    assert A.info()["rows_per_thread"] == rows and A.bench_projection(4, reps=1) > 0.0
    for (pa, sa), (pb, sb) in zip(ref, got):
        assert np.array_equal(pa, pb) and np.array_equal(sa, sb)


def test_bench_projection(gpu):
    S, props, th = models.toggle()
    states = models.box_states([127, 127])
    space = nh.StateSpaceSparse(S, states)
    A = nh.FspMatrixSparse(space, models.to_product(props), th, precision="fp32")
    for nv in (1, 4, 5, 30):
        assert A.bench_projection(nv, reps=3) > 0.0
    with pytest.raises(nh.NumCmeHipError):
        A.bench_projection(33, reps=1)
    # the computed-values mode has no column form
    A.set_matrix_free(1)
    with pytest.raises(nh.NumCmeHipError):
        A.bench_projection(4, reps=1)
    A.set_matrix_free(0)
    assert A.bench_projection(2, reps=1) > 0.0
    # sink rows of 9,001 entries, which the mat-vec reduces in chunks
    space = nh.StateSpaceSparse(S, models.box_states([9000, 1]))
    A = nh.FspMatrixSparse(space, models.to_product(props), th, precision="fp32")
    for nv in (1, 2, 32):
        assert A.bench_projection(nv, reps=3) > 0.0


def test_large_space_against_rk(gpu):
    # 1500 x 1450 = 2,175,000 states, 4,249 blocks: eight or nine per workgroup; checked
    # against the device DP5(4) solve
    S, props, th = models.toggle()
    states = models.box_states([1499, 1449])
    assert len(states) > 8 * 512 * 512
    model = nh.CmeModel(S, models.to_product(props), th)
    space = nh.StateSpaceSparse(S, states)
    A = nh.FspMatrixSparse(space, model.propensities, model.parameters, precision="fp64", model=model)
    p0 = np.zeros(len(states))
    p0[int(np.flatnonzero((states[:, 0] == 20) & (states[:, 1] == 5))[0])] = 1.0
    u0 = np.concatenate([p0, np.zeros(space.get_sink_count())])
    ts = np.array([0.0, 0.05, 0.1])
    kr = _integrate(A, nh.KrylovExpv(m=30, tol=1e-12).opts(1e-6, 1e-4), u0, 0.0, ts, space)
    rk = _integrate(A, nh.RK45(rtol=1e-10, atol=1e-16).opts(1e-6, 1e-4), u0, 0.0, ts, space)
    for pk, pr, sk, sr in zip(kr.p, rk.p, kr.sinks, rk.sinks):
        assert np.abs(pk.values - pr.values).sum() + np.abs(np.asarray(sk) - np.asarray(sr)).sum() < 1e-8
    assert abs(kr.p[-1].values.sum() + np.sum(kr.sinks[-1]) - 1.0) < 1e-10
