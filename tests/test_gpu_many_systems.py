"""Ensembles of many small systems: the build adds up the subtrees' cells in its own
workgroups up to 192 systems, in a launch of its own above.  Both sides of the line, mixed sizes
from one body on, and thousands of systems of a few bodies.  With theta = 0 every body of a
system is met exactly once, so a step's accelerations are the direct sums of each system.
Bar: FP32 sums of at most 400 terms against FP64, each term to a few roundings of 6e-8 of itself:
1e-5 of the sum of the terms' norms (the sum itself may cancel)."""
import numpy as np
import pytest

import nns_amd

pytestmark = pytest.mark.gpu

CASES = [(191, 1, 40), (192, 1, 300), (193, 1, 300), (193, 1, 3), (193, 300, 400), (1000, 30, 60), (8192, 8, 8),
         (47662, 1, 2)]


@pytest.mark.parametrize("systems,lo,hi", CASES)
def test_ensemble_of_many_systems(systems, lo, hi):
    import torch
    assert torch.cuda.is_available()
    print(f"case many systems {systems} of {lo}..{hi}", flush=True)
    rng = np.random.default_rng(systems + hi)
    sizes = rng.integers(lo, hi + 1, systems).astype(np.int32)
    n = int(sizes.sum())
    p = rng.normal(size=(3, n)).astype(np.float32)
    m = rng.uniform(0.5, 1.5, n).astype(np.float32)
    z = np.zeros(n, np.float32)
    b = nns_amd.Batch(*p, z, z, z, m, sizes, params=nns_amd.default_params(theta=0.0, softening=0.1, timestep=0.0))
    for _ in range(2):
        b.step()
        b.check()
    a = np.stack([b.host(k) for k in ("ax", "ay", "az")], 1)
    off = np.concatenate([[0], np.cumsum(sizes)])
    eps2 = float(np.float32(np.float32(0.1) ** 2))
    for s in range(0, systems, max(1, systems // 2000)):
        x = p[:, off[s]:off[s + 1]].astype(np.float64)
        d = x[:, None, :] - x[:, :, None]
        w = m[off[s]:off[s + 1]].astype(np.float64) * ((d ** 2).sum(0) + eps2) ** -1.5
        want = (w * d).sum(2).T
        scale = (w * np.sqrt((d ** 2).sum(0))).sum(1) + 1e-30
        err = np.linalg.norm(a[off[s]:off[s + 1]] - want, axis=1) / scale
        assert err.max() <= 1e-5, (s, int(sizes[s]), err.max())
