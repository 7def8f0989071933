"""nbx_force_vjp of systems with few nodes, taken three times on one context: the counters
of its log (65 lines of 32 words) are more words than four per body and node, and every
call must find them at zero.  n + m on both sides of 504, where the two are as many; and a
small system in a context of 65,536 bodies, whose log has the most parts.
Reference: the oracle's FP64 product of the same interaction lists (orc_tree_vjp, mac_mode 1).
Bar: the FP32 terms carry about 1e-6 of the gradient norm; 2e-5 as for the other sizes."""
import numpy as np
import pytest

import nns_amd

pytestmark = pytest.mark.gpu

# bodies, nodes, bodies of the context (None: as many as the system's)
CASES = [(2, 8, None), (64, 200, None), (100, 300, None), (100, 404, None), (100, 405, None), (150, 450, None),
         (64, 200, 65536)]


def rel_err(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-300))


@pytest.mark.parametrize("n,m,n_max", CASES)
def test_vjp_of_few_nodes(oracle, n, m, n_max):
    import torch
    assert torch.cuda.is_available()
    print(f"case vjp few nodes n={n} m={m} n_max={n_max}", flush=True)
    arrs = nns_amd.initial_conditions("plummer", n, 6)
    p = nns_amd.default_params(theta=0.5)
    ctx = nns_amd.Context(n_max, params=p) if n_max else None
    bh = nns_amd.BarnesHut(*arrs, params=p, m=m, ctx=ctx)
    bh.rebuild()
    u = np.random.default_rng(5).normal(size=(n, 3)).astype(np.float32)
    ut = [torch.as_tensor(u[:, k].copy(), device=bh.dev) for k in range(3)]
    t = oracle.KeyTree(*arrs[:3], arrs[6])
    ogx, ogm = t.vjp(0.5, float(np.float32(p.softening)) ** 2, u.astype(np.float64), mac_mode=1)
    for call in range(3):
        gx, gy, gz, gm = [g.cpu().numpy() for g in bh.vjp(*ut)]
        bh.ctx.check()
        err = rel_err(np.stack([gx, gy, gz], 1), ogx), rel_err(gm, ogm)
        assert max(err) <= 2e-5, (call, err)
