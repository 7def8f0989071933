"""Prefix sums that a launch's workgroups form themselves for few bodies, at both
sides of their limits: the top table (2,048 entries: 97 and 98 samples of 1,024
bodies), the subtrees' cells (65,536 bodies), the frame blocks' runs (96 runs of
1,024 nodes), and the bounding box of one workgroup (8,192 bodies).  The tree is
compared bit for bit with the oracle's, the bounding box exactly, and the walk's
steps and frames, which depend on every block's place, as counts."""
import numpy as np
import pytest

import nns_amd

from test_gpu_parity import check_tree, make_case, run_to_forces

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,n,extra", [("plummer", 1, 0), ("plummer", 1024, 0), ("cluster", 8192, 0),
                                          ("cluster", 8193, 0), ("binary_disk", 65536, 0), ("binary_disk", 65537, 0),
                                          ("plummer", 99328, 0), ("plummer", 99329, 0),
                                          ("plummer", 20000, 96 * 1024 - 1), ("plummer", 20000, 96 * 1024)])
def test_trees_at_the_limits(oracle, kind, n, extra):
    import torch
    assert torch.cuda.is_available()
    print(f"case small scans {kind} n={n} extra nodes={extra}", flush=True)
    arrs = make_case(kind, n)
    m = n + extra if extra else 24 * n + 12000 if kind == "cluster" else None
    bh = run_to_forces(*arrs, m_nodes=m)
    for k, (lo, hi) in enumerate([("minX", "maxX"), ("minY", "maxY"), ("minZ", "maxZ")]):
        assert bh.host(lo)[0] == arrs[k].min() and bh.host(hi)[0] == arrs[k].max()
    if n == 1:  # the oracle makes no tree of one body: no cell, no force
        assert int(bh.host("index")[0]) == 1 and bh.host("ax")[0] == 0.0
        return
    t = oracle.KeyTree(arrs[0], arrs[1], arrs[2], arrs[6])
    assert t.err == 0
    check_tree(bh, t)
    eps2 = float(np.float32(np.float32(bh.ctx.params.softening) ** 2))
    _, cnt = t.accel(bh.ctx.params.theta, eps2, mac_mode=1)
    assert np.array_equal(bh.count_interactions().cpu().numpy(), cnt)
