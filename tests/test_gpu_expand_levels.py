"""State-space expansion across the one-workgroup and the launched levels.

expand! (sparsestatespace.jl:153-194) must give the reference's states in the reference's
order, with its connectivity and sinks, whichever form ran a level: levels of at most 4,096
candidates of a space run in one workgroup, several to a launch; larger ones by launches of
their own. The cases start small, cross the limit and come back below it, stop for room,
restrict the reactions, and cover the species counts the kernels are built for.
"""
import numpy as np
import pytest

import models
import numcme_hip as nh
from oracle.statespace import StateSpace

pytestmark = pytest.mark.gpu


def _same(d, o):
    assert np.array_equal(d.get_states(), o.states)
    assert np.array_equal(d.get_state_connectivity(), o.state_conn)
    assert np.array_equal(d.get_sink_connectivity(), o.sink_conn)
    assert np.array_equal(d.lookup(o.states[:: max(1, len(o.states) // 50)]),
                          np.arange(len(o.states))[:: max(1, len(o.states) // 50)] + 1)


def _chain(ns):
    """A conversion chain with birth at the first and death at the last of ns species."""
    S = np.zeros((ns, ns + 1), dtype=np.int64)
    S[0, 0] = 1
    for s in range(ns - 1):
        S[s, s + 1], S[s + 1, s + 1] = -1, 1
    S[ns - 1, ns] = -1
    return S


@pytest.mark.parametrize("ns,levels", [(1, 700), (2, 60), (3, 30), (4, 16), (5, 11), (6, 9), (7, 8), (8, 7), (9, 7), (16, 4)])
def test_species_counts(gpu, ns, levels):
    S = _chain(ns)
    d, o = nh.StateSpaceSparse(S, [0] * ns if ns > 1 else [[0]]), StateSpace(S, [[0] * ns])
    for step in (levels, 1, 2):
        d.expand(step)
        o.expand(step)
        _same(d, o)


@pytest.mark.parametrize("only", [(), (1,), (3, 1), (2, 4)])
@pytest.mark.parametrize("init", [1, 4095, 4096, 4097, 9000])
def test_toggle_from_lists(gpu, only, init):
    # first levels of a line of states: candidates below, at and above the limit, and spaces
    # whose explorables are listed by the launches (more than 4,096 states)
    S = models.TOGGLE_S
    x = [[k, 0] for k in range(init)]
    d, o = nh.StateSpaceSparse(S, x), StateSpace(S, x)
    for step in (1, 3):
        d.expand(step, only)
        o.expand(step, only)
        _same(d, o)


def test_wide_then_narrow(gpu):
    # 50 x 50 x 50 births of three species: levels pass 4,096 candidates and fall below again
    # once the species' counts are capped by the reactions listed
    S = models.CASCADE_S
    d, o = nh.StateSpaceSparse(S, [0, 0, 0]), StateSpace(S, [[0, 0, 0]])
    for step, only in ((45, ()), (40, (1,)), (3, ())):
        d.expand(step, only)
        o.expand(step, only)
        _same(d, o)


def test_after_deletion(gpu):
    # holes: the table is rebuilt and the sinks recomputed before the next levels
    S = models.TOGGLE_S
    d, o = nh.StateSpaceSparse(S, [0, 0]), StateSpace(S, [[0, 0]])
    d.expand(30)
    o.expand(30)
    ids = np.random.default_rng(2).choice(len(o.states), 200, replace=False)
    ids.sort()
    d.deleteat(ids + 1)
    o.deleteat(ids + 1)
    _same(d, o)
    d.expand(4, (1, 2))
    o.expand(4, (1, 2))
    _same(d, o)
