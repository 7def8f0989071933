"""Top cells summed in one workgroup's LDS, in levels by several workgroups first,
and with more roots than fit beside them: around the limit of top cells (some 230,
330 and 500 of them), by both builds, and ensembles of few and many systems with and
without top cells.  Sums against the oracle's, bit for bit (no tolerance)."""
import numpy as np
import pytest

import nns_amd

from test_gpu_parity import check_tree, run_to_forces

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,n,locked", [("plummer", 240000, 0), ("plummer", 340000, 0), ("plummer", 340000, 1),
                                           ("binary_disk", 420000, 0), ("plummer", 500000, 0),
                                           ("plummer", 620000, 1)])
def test_top_cells_around_the_limit(oracle, kind, n, locked):
    import torch
    assert torch.cuda.is_available()
    print(f"case top cells {kind} n={n} locked={locked}", flush=True)
    arrs = nns_amd.initial_conditions(kind, n, 6)
    bh = run_to_forces(*arrs, nns_amd.default_params(build_locked=locked))
    t = oracle.KeyTree(arrs[0], arrs[1], arrs[2], arrs[6])
    assert t.err == 0
    check_tree(bh, t)


@pytest.mark.parametrize("sizes", [[2, 3000, 40000], [1100] * 100, [1100] * 300, [30] * 449, [1500] * 460])
def test_roots_of_ensembles(oracle, sizes):
    import torch
    assert torch.cuda.is_available()
    print(f"case roots of {len(sizes)} systems, {sum(sizes)} bodies", flush=True)
    parts = [nns_amd.initial_conditions("plummer", n, s + 1) for s, n in enumerate(sizes)]
    b = nns_amd.Batch(*[np.concatenate([q[k] for q in parts]) for k in range(7)], sizes, [0.5] * len(sizes))
    b.step()
    torch.cuda.synchronize()
    N, S = b.N, len(sizes)
    mass = b.copy_buffer(nns_amd.BUF_CELL_MASS64, N + S, np.float64)[N:]
    com = b.copy_buffer(nns_amd.BUF_CELL_COM64, 3 * (N + S), np.float64).reshape(-1, 3)[N:]
    for s, q in enumerate(parts):
        t = oracle.KeyTree(q[0], q[1], q[2], q[6])
        assert mass[s] == t.mass[0] and np.array_equal(com[s], t.com[0]), s
