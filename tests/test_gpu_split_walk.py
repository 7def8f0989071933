"""Force launches of few groups share each group's walk among the waves of a
workgroup: 16 up to 640 groups of 64 bodies, 8 up to 2,560, 4 up to 5,120.  At
both sides of each line, at the smallest sizes and on a tree whose every node is
opened (theta = 0, equal keys: the deepest stacks), the accelerations are those
of the oracle's FP64 walk of the same lists, and the same on every run.

Bars: per body, an FP32 sum of a few hundred to some thousand monopoles, each
with a few roundings of 6e-8 and differences of coordinates of up to ~1e-4
relative to their distance: RMS 1e-5, maximum 2e-3 (as for the one-wave walk)."""
import numpy as np
import pytest

import nns_amd

from test_gpu_parity import make_case

pytestmark = pytest.mark.gpu

CASES = [("plummer", 2, 0.5, {}), ("plummer", 64, 0.5, {}), ("plummer", 65, 0.5, {"kahan": 0}),
         ("coincident", 2000, 0.0, {}), ("plummer", 640 * 64, 0.6, {}), ("plummer", 640 * 64 + 1, 0.6, {}),
         ("binary_disk", 2560 * 64, 0.5, {"softening": 0.0}), ("binary_disk", 2560 * 64 + 1, 0.5, {}),
         ("plummer", 5120 * 64, 0.8, {"kahan": 0}), ("plummer", 5120 * 64 + 1, 0.8, {})]


@pytest.mark.parametrize("kind,n,theta,extra", CASES)
def test_shared_walk_matches_oracle(oracle, kind, n, theta, extra):
    import torch
    assert torch.cuda.is_available()
    print(f"case shared walk {kind} n={n} theta={theta} {extra}", flush=True)
    x, y, z, vx, vy, vz, m = make_case(kind, n)
    p = nns_amd.default_params(theta=theta, **extra)
    bh = nns_amd.BarnesHut(x, y, z, vx, vy, vz, m, params=p, m=24 * n + 12000 if kind == "coincident" else None)
    bh.rebuild()
    bh.forces()
    bh.ctx.check()
    a = np.stack([bh.host(k) for k in ("ax", "ay", "az")], 1)
    bh.forces()
    bh.ctx.check()
    assert np.array_equal(np.stack([bh.host(k) for k in ("ax", "ay", "az")], 1), a)
    t = oracle.KeyTree(x, y, z, m, cap=23 * n + 12000 if kind == "coincident" else 0)
    tgt = np.sort(np.random.default_rng(3).choice(n, size=min(n, 2000), replace=False)).astype(np.int32)
    eps2 = float(np.float32(np.float32(p.softening) ** 2))
    acc, _ = t.accel(float(np.float32(theta)), eps2, mac_mode=1, targets=tgt)
    rel = np.linalg.norm(a[tgt].astype(np.float64) - acc, axis=1) / np.linalg.norm(acc, axis=1)
    assert np.sqrt((rel ** 2).mean()) < 1e-5 and rel.max() < 2e-3, (np.sqrt((rel ** 2).mean()), rel.max())
