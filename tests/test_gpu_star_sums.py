"""Star sums met by a whole workgroup per star, at the ends of its range: one
star and the most allowed; no body, one, fewer than a workgroup, one more than
a workgroup, more partials than a star's workgroup has threads can take at once.

Tolerance: sums run in FP64 and are stored once in FP32, so every component is
within 2^-24 of itself plus FP64 rounding; the largest partial sums here are
below 1e4 times the result (random signs over at most 70,000 terms), 1e4 * 2^-53
is far below that, and 1e-6 leaves a factor of 16."""
import numpy as np
import pytest

import nns_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns", [1, 2, nns_amd.MAX_STARS])
@pytest.mark.parametrize("n", [1, 255, 257, 70001])
def test_star_sums_match_oracle(oracle, n, ns):
    import torch
    assert torch.cuda.is_available()
    print(f"case star sums n={n} stars={ns}", flush=True)
    r = np.random.default_rng(100 * n + ns)
    b = [r.normal(0, 1, n).astype(np.float32) for _ in range(3)] + [r.uniform(0.5, 1.5, n).astype(np.float32) / n]
    s = [r.normal(0, 1, ns).astype(np.float32) for _ in range(3)] + [r.uniform(0.2, 0.5, ns).astype(np.float32)]
    p = nns_amd.default_params()
    ctx = nns_amd.Context(n, params=p)
    T = lambda a: torch.as_tensor(a, device="cuda")
    acc, sacc = [torch.zeros(n, device="cuda") for _ in range(3)], [torch.zeros(ns, device="cuda") for _ in range(3)]
    nns_amd.KernelsWrapper(ctx).starForces(*(T(a) for a in s), *sacc, ns, *(T(a) for a in b), *acc, n, 1.0)
    ctx.check()
    eps2 = float(np.float32(np.float32(p.softening) ** 2))
    sa, _ = oracle.star_forces((s[3], *s[:3]), (b[3], *b[:3]), kernel=1, eps2=eps2)
    got = np.stack([t.cpu().numpy() for t in sacc], 1).astype(np.float64)
    rel = np.linalg.norm(got - sa, axis=1) / np.linalg.norm(sa, axis=1)
    assert rel.max() <= 1e-6, rel.max()
