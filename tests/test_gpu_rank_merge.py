"""The one-launch merge of up to 17 sorted chunks of 4,096 pairs, against a stable
numpy argsort, at both sides of its ranges and for keys that bracket badly: in
order, in reverse, all equal, a few values (with the largest), one chunk inside a
gap of another, and a narrow cluster below a wide spread.  Exact."""
import numpy as np
import pytest

import nns_amd

pytestmark = pytest.mark.gpu

KINDS = ["random", "ordered", "reversed", "equal", "few", "nested"]


def make_keys(kind, n, r):
    wide = r.integers(0, 2 ** 63, n, dtype=np.uint64) * np.uint64(2) + r.integers(0, 2, n, dtype=np.uint64)
    if kind == "ordered":
        return np.sort(wide)
    if kind == "reversed":
        return np.sort(wide)[::-1].copy()
    if kind == "equal":
        return np.full(n, 2 ** 64 - 1, np.uint64)
    if kind == "few":
        return np.array([0, 5, 2 ** 40, 2 ** 64 - 1], np.uint64)[r.integers(0, 4, n)]
    if kind == "nested":  # every second chunk within a narrow band
        band = (np.arange(n) // 4096) % 2 == 1
        wide[band] = np.uint64(2 ** 62) + r.integers(0, 1000, int(band.sum()), dtype=np.uint64)
    return wide


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n", [4097, 4160, 8192, 16447, 36865, 69631, 69632, 69633])
def test_rank_merge_is_stable(kind, n):
    import torch
    assert torch.cuda.is_available()
    print(f"case rank merge {kind} n={n}", flush=True)
    k = make_keys(kind, n, np.random.default_rng(n))
    kw = nns_amd.KernelsWrapper(nns_amd.Context(n))
    keys = torch.as_tensor(k.view(np.int64), device="cuda")
    sk, p = torch.zeros_like(keys), torch.full((n,), -1, dtype=torch.int32, device="cuda")
    kw.sortKeys(keys, n, sk, p)
    ref = np.argsort(k, kind="stable")
    assert np.array_equal(p.cpu().numpy(), ref)
    assert np.array_equal(sk.cpu().numpy().view(np.uint64), k[ref])


@pytest.mark.parametrize("sizes", [[8200, 1, 4096, 12300, 2], [4097] * 31, [4097] * 33, [70000, 30]])
def test_rank_merge_of_ensembles(sizes):
    import torch
    assert torch.cuda.is_available()
    print(f"case rank merge ensemble of {len(sizes)}, {sum(sizes)} bodies", flush=True)
    parts = [nns_amd.initial_conditions("plummer", n, s + 1) for s, n in enumerate(sizes)]
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
