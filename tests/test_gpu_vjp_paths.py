"""The paths of nbx_force_vjp against the oracle's FP64 product of the same
interaction lists (orc_tree_vjp, mac_mode 1):
  walk  -- 16 waves per group up to 640 groups of 64 bodies, 8 up to 5,120, 4 up to
           10,240, then one: both sides of the first two lines;
  sums  -- the log's node sums: bins of 2^10, 2^11 or 2^12 node ids, or the sorted form, by
           the context's n_max + m_max: a small system in contexts of each size;
  log   -- theta = 0 at n = 8,192 logs more than the log holds: the rest goes by
           atomics.
Bar: the FP32 terms of a body's list and of a node's bodies carry about 1e-6 of the
gradient norm; 2e-5 as for the other sizes."""
import numpy as np
import pytest

import nns_amd

pytestmark = pytest.mark.gpu

CASES = [("plummer", 640 * 64, 0.7, None), ("plummer", 640 * 64 + 1, 0.7, None),
         ("binary_disk", 5120 * 64, 0.8, None), ("binary_disk", 5120 * 64 + 1, 0.8, None),
         ("plummer", 3001, 0.5, 400000), ("plummer", 3001, 0.5, 700000), ("plummer", 3001, 0.5, 1500000),
         ("plummer", 8192, 0.0, None), ("plummer", 2, 0.5, None)]


def rel_err(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-300))


@pytest.mark.parametrize("kind,n,theta,n_max", CASES)
def test_vjp_path_matches_oracle(oracle, kind, n, theta, n_max):
    import torch
    assert torch.cuda.is_available()
    print(f"case vjp path {kind} n={n} theta={theta} n_max={n_max}", flush=True)
    arrs = nns_amd.initial_conditions(kind, n, 2)
    p = nns_amd.default_params(theta=theta)
    ctx = nns_amd.Context(n_max, params=p) if n_max else None
    bh = nns_amd.BarnesHut(*arrs, params=p, ctx=ctx)
    bh.rebuild()
    u = np.random.default_rng(9).normal(size=(n, 3)).astype(np.float32)
    ut = [torch.as_tensor(u[:, k].copy(), device=bh.dev) for k in range(3)]
    t = oracle.KeyTree(*arrs[:3], arrs[6])
    ogx, ogm = t.vjp(float(np.float32(theta)), float(np.float32(p.softening)) ** 2, u.astype(np.float64), mac_mode=1)
    for _ in range(2):
        gx, gy, gz, gm = [g.cpu().numpy() for g in bh.vjp(*ut)]
        bh.ctx.check()
        assert rel_err(np.stack([gx, gy, gz], 1), ogx) <= 2e-5, rel_err(np.stack([gx, gy, gz], 1), ogx)
        assert rel_err(gm, ogm) <= 2e-5, rel_err(gm, ogm)
