"""Fixed-order folds at the edges of their work split.

The marginal sum(p, dims) (fspvector.jl:66-99) is the reference's left fold in state order,
bit for bit: a thread per group for short groups, a wave per group from a mean length of 32
on. The adapter gradient's partials are folded by eight waves, sixteen loads at a time; the
sample counts give 1, 7, 8, 9, 127, 129 and 512 partials.
"""
import numpy as np
import pytest

import numcme_hip as nh
from oracle import mlp as om

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lengths", [(1,), (31, 31), (32, 32), (33, 33, 33), (64,), (63, 65, 64), (1, 2000, 5),
                                     (1, 1, 1, 700, 128), tuple(range(20, 60))])
def test_marginal_group_lengths(gpu, lengths):
    rng = np.random.default_rng(len(lengths))
    group = np.repeat(np.arange(len(lengths)), lengths)
    states = np.stack([group, np.concatenate([np.arange(n) for n in lengths])], axis=1)
    order = rng.permutation(len(states))
    states = states[order]
    vals = rng.standard_normal(len(states)) * 10.0 ** rng.integers(-18, 3, len(states))
    vals[rng.random(len(states)) < 0.1] = -0.0
    vals[states[:, 0] == 0] = -0.0  # a group of negative zeros keeps its sign
    m = nh.FspVectorSparse(states, vals).sum([2])
    want = {}
    for g, v in zip(states[:, 0], vals):  # in state order
        want[g] = v if g not in want else want[g] + v
    assert m.states[:, 0].tolist() == list(want)  # first appearance
    got, ref = m.values, np.array(list(want.values()))
    assert np.array_equal(got, ref) and np.array_equal(np.signbit(got), np.signbit(ref))


@pytest.mark.parametrize("blocks", [1, 7, 8, 9, 127, 129, 512])
def test_gradient_partial_counts(gpu, blocks):
    n = 64 * blocks
    rng = np.random.default_rng(blocks)
    X = rng.normal(size=(n, om.F)).astype(np.float32)
    Y = (rng.random(n) < 0.3).astype(np.float32)
    net = nh.AdapterMlp(seed=5)
    g, loss = net.grad(X, Y)
    go, lo = om.grad(net.params.astype(np.float64), X, Y, bf16_ops=True)
    # the bounds of the gradient test: FP32 accumulation of BF16 products, activations that
    # cross a BF16 rounding boundary
    assert abs(loss - lo) <= 1e-5 * max(1.0, abs(lo))
    assert np.linalg.norm(g - go) <= 2e-3 * np.linalg.norm(go)
