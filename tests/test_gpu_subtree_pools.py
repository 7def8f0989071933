"""Subtrees staged in LDS by the build and the summary: those that fit the pool,
those just past it, and those that fit none (chains of one-child cells above
pairs of bodies, about 18 cells a pair), with the bodies in the pairs' slots, in
level-21 buckets and hanging beside cells; by both builds; and enough bodies
that the subtrees go to two pools.  The tree is compared cell for cell and bit
for bit with the oracle's (no tolerance)."""
import numpy as np
import pytest

import nns_amd

from test_gpu_parity import check_tree, run_to_forces

pytestmark = pytest.mark.gpu


def deep_pairs(pairs, plain, seed):
    """`pairs` pairs 2^-17 of the box apart, a triple at one place, `plain` bodies; all in one unit box."""
    r = np.random.default_rng(seed)
    p = r.uniform(-1, 1, (pairs, 3))
    three = np.repeat(r.uniform(-1, 1, (1, 3)), 3, axis=0)
    p = np.concatenate([p, p + 2.0 ** -16 * r.choice([-1.0, 1.0], (pairs, 3)), three, r.uniform(-1, 1, (plain, 3))])
    p = r.permutation(p).astype(np.float32)
    v = np.zeros((len(p), 3), np.float32)
    m = (r.uniform(0.5, 1.5, len(p)) / len(p)).astype(np.float32)
    return (*p.T.copy(), *v.T.copy(), m)


@pytest.mark.parametrize("locked", [0, 1])
@pytest.mark.parametrize("pairs,plain", [(0, 2), (16, 990), (24, 970), (30, 960), (60, 900), (512, 0), (300, 3000)])
def test_subtrees_in_and_past_the_pool(oracle, pairs, plain, locked):
    import torch
    assert torch.cuda.is_available()
    print(f"case subtree pools pairs={pairs} plain={plain} locked={locked}", flush=True)
    arrs = deep_pairs(pairs, plain, 10 * pairs + locked)
    n = len(arrs[0])
    bh = run_to_forces(*arrs, nns_amd.default_params(build_locked=locked), m_nodes=24 * n + 12000)
    t = oracle.KeyTree(arrs[0], arrs[1], arrs[2], arrs[6])
    assert t.err == 0
    check_tree(bh, t)


def test_subtrees_in_two_pools(oracle):
    import torch
    assert torch.cuda.is_available()
    n = (1 << 22) + 77
    print(f"case subtree pools n={n}", flush=True)
    arrs = [a.copy() for a in nns_amd.initial_conditions("plummer", n, seed=3)]
    deep = deep_pairs(2000, 0, 9)
    for a, d in zip(arrs[:3], deep[:3]):
        a[:len(d)] = d
    bh = run_to_forces(*arrs)
    t = oracle.KeyTree(arrs[0], arrs[1], arrs[2], arrs[6])
    assert t.err == 0
    check_tree(bh, t)
