"""The merge sort of (key, index) pairs and the group order read off the tree.

Sort: against a stable numpy argsort, at the edges of a chunk (4,096 pairs), of
a merge (two, three, five chunks) and of a thread (8 pairs), with repeated keys
and with the largest key, which is also what the sort pads chunks with.  Exact.

Ensemble: systems at both sides of a chunk's end, sorted each by itself: keys in
order and stable within every system.  Exact.

Group order: the walk's child steps and frames depend on which bodies share a
group, so they equal the oracle's count over its own order (a stable sort by
the coarse Hilbert key) only if the orders agree; on trees of deep one-child
chains (subtrees of more than 1,024 cells), tight clusters and a few bodies that
hang from the root."""
import numpy as np
import pytest

import nns_amd

from test_gpu_parity import make_case

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 7, 8, 9, 65, 511, 513, 4095, 4096, 4097, 8192, 8193, 12289, 20481, 300001]


@pytest.mark.parametrize("n", SIZES)
def test_merge_sort_is_stable(n):
    import torch
    assert torch.cuda.is_available()
    print(f"case merge sort n={n}", flush=True)
    r = np.random.default_rng(n)
    k = r.integers(0, 2 ** 63, n, dtype=np.int64).view(np.uint64) * np.uint64(2)
    k[r.integers(0, n, n // 3)] = k[r.integers(0, n, n // 3)]
    k[r.integers(0, n, n // 5 + 1)] = np.uint64(2 ** 64 - 1)
    kw = nns_amd.KernelsWrapper(nns_amd.Context(n))
    keys = torch.as_tensor(k.view(np.int64), device="cuda")
    sk, p = torch.zeros_like(keys), torch.full((n,), -1, dtype=torch.int32, device="cuda")
    kw.sortKeys(keys, n, sk, p)
    ref = np.argsort(k, kind="stable")
    assert np.array_equal(p.cpu().numpy(), ref)
    assert np.array_equal(sk.cpu().numpy().view(np.uint64), k[ref])
    assert np.array_equal(keys.cpu().numpy().view(np.uint64), k)


def test_ensemble_sorts_every_system_by_itself():
    import torch
    assert torch.cuda.is_available()
    sizes = [4096, 1, 4097, 4095, 9000, 2, 12289]
    print(f"case ensemble sort sizes={sizes}", flush=True)
    parts = [make_case("coincident", n, seed=s) for s, n in enumerate(sizes)]
    b = nns_amd.Batch(*[np.concatenate([q[k] for q in parts]) for k in range(7)], sizes, [0.5] * len(sizes))
    b.step()
    torch.cuda.synchronize()
    keys = b.copy_buffer(nns_amd.BUF_KEYS, b.N, np.uint64)
    skeys = b.copy_buffer(nns_amd.BUF_SORTED_KEYS, b.N, np.uint64)
    perm = b.copy_buffer(nns_amd.BUF_PERM, b.N, np.int32)
    for lo, hi in zip(b.off[:-1], b.off[1:]):
        ref = lo + np.argsort(keys[lo:hi], kind="stable")
        assert np.array_equal(perm[lo:hi], ref)
        assert np.array_equal(skeys[lo:hi], keys[ref])


def lone(n):
    """A tight cluster and three bodies far off, each alone in an octant of the root."""
    x, y, z, vx, vy, vz, m = make_case("plummer", n)
    x, y, z = x * 1e-3, y * 1e-3, z * 1e-3
    x[:3], y[:3], z[:3] = [1, -1, 1], [1, 1, -1], [1, -1, 1]
    return x, y, z, vx, vy, vz, m


@pytest.mark.parametrize("kind,n", [("coincident", 6000), ("cluster", 30000), ("line", 5000), ("lone", 5003),
                                    ("plummer", 2), ("far_clumps", 3000)])
def test_group_order_gives_the_oracles_walk(oracle, kind, n):
    import torch
    assert torch.cuda.is_available()
    print(f"case group order {kind} n={n}", flush=True)
    arrs = lone(n) if kind == "lone" else make_case(kind, n)
    deep = kind in ("coincident", "line", "cluster")
    bh = nns_amd.BarnesHut(*arrs, m=24 * n + 12000 if deep else None)
    bh.rebuild()
    w = bh.walk_stats()
    bh.ctx.check()
    t = oracle.KeyTree(*arrs[:3], arrs[6], cap=23 * n + 12000 if deep else 0)
    assert np.array_equal(bh.host("sorted"), t.perm)
    steps, frames = t.group_walk(0.5, float(np.float32(np.float32(bh.ctx.params.softening) ** 2)))
    assert (w["child_steps"], w["frames"]) == (int(steps.sum()), int(frames.sum()))
