"""The split search of the merge passes, whose probes lie at multiples of 64, 2,048,
2^17 and 2^23 pairs from 1,310,720 pairs on and are spread evenly below, against a
stable numpy argsort: at both sides of that line and with runs of every round's
length (the longest past 8,388,608 pairs), with ends that are no multiple of a step,
and for keys whose splits lie at the ends of the range.  Exact."""
import numpy as np
import pytest

import nns_amd

from test_gpu_rank_merge import make_keys

pytestmark = pytest.mark.gpu

CASES = [(kind, n) for kind in ("random", "ordered", "reversed", "equal", "nested")
         for n in (131073, 526401, 1310719, 1310720, 2099265)] + [("random", 16777217 + 70001), ("few", 33554432 + 63)]


@pytest.mark.parametrize("kind,n", CASES)
def test_merge_passes_are_stable(kind, n):
    import torch
    assert torch.cuda.is_available()
    print(f"case merge split {kind} n={n}", flush=True)
    k = make_keys(kind, n, np.random.default_rng(n))
    kw = nns_amd.KernelsWrapper(nns_amd.Context(n))
    keys = torch.as_tensor(k.view(np.int64), device="cuda")
    sk, p = torch.zeros_like(keys), torch.full((n,), -1, dtype=torch.int32, device="cuda")
    kw.sortKeys(keys, n, sk, p)
    ref = np.argsort(k, kind="stable")
    assert np.array_equal(p.cpu().numpy(), ref)
    assert np.array_equal(sk.cpu().numpy().view(np.uint64), k[ref])
