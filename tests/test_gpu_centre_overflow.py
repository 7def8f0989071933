"""A cell whose centre of mass is past FP32 (masses 1, -1 and 2^-140 in three octants: moments
of 1e-3 over a mass of 7e-43) below a parent whose centre is not (a fourth body of mass 1).
The bodies that took the parent must not feel what happens below it, whichever of their wave's
lanes went on: their accelerations are finite and those of the oracle's FP64 walk.
Through the shared walk (one system) and the one-wave walk (an ensemble of more groups than
the shared walk takes).
Bar: an FP32 sum of some twenty monopoles, 1e-5 of the acceleration."""
import numpy as np
import pytest

import nns_amd

pytestmark = pytest.mark.gpu

FAR = np.arange(21, dtype=np.int32)


def bodies():
    far = np.random.default_rng(3).uniform(0.0, 0.35, (20, 3))
    small = 0.9 + np.array([[0.0, 0.0, 0.0], [2e-3, 0.0, 0.0], [0.0, 2e-3, 0.0], [9e-3, 9e-3, 9e-3]])
    corners = np.array([[0.0, 0.0, 0.0], [1.0, 1.0, 1.0]])
    p = np.concatenate([far, corners[:1], small, corners[1:]]).astype(np.float32)
    m = np.concatenate([np.ones(21), [1.0, -1.0, 2.0 ** -140, 1.0], [1.0]]).astype(np.float32)
    z = np.zeros(len(m), np.float32)
    return [p[:, 0].copy(), p[:, 1].copy(), p[:, 2].copy(), z, z, z, m]


def expected(oracle, theta, eps):
    a = bodies()
    t = oracle.KeyTree(*a[:3], a[6])
    return t.accel(theta, float(np.float32(np.float32(eps) ** 2)), mac_mode=1, targets=FAR)[0]


def compare(got, want):
    assert np.isfinite(got).all()
    err = np.linalg.norm(got.astype(np.float64) - want, axis=1) / np.linalg.norm(want, axis=1)
    assert err.max() <= 1e-5, err.max()


@pytest.mark.parametrize("soft,kahan", [(0.0, 1), (0.0, 0), (1e-3, 1), (1e-3, 0)])
def test_bodies_that_took_the_parent_stay_finite(oracle, soft, kahan):
    import torch
    assert torch.cuda.is_available()
    print(f"case centre overflow soft={soft} kahan={kahan}", flush=True)
    kw = dict(theta=0.5, softening=soft, kahan=kahan)
    want = expected(oracle, 0.5, soft)
    assert np.isfinite(want).all()
    bh = nns_amd.BarnesHut(*bodies(), params=nns_amd.default_params(**kw))
    bh.rebuild()
    bh.forces()
    bh.ctx.check()
    centres = bh.host("x", int(bh.arr["index"].item()))[bh.n:]
    assert np.isinf(centres).any()  # the cell is there
    compare(np.stack([bh.host(k) for k in ("ax", "ay", "az")], 1)[FAR], want)
    systems, n = 5121, len(bodies()[6])
    b = nns_amd.Batch(*[np.tile(v, systems) for v in bodies()], np.full(systems, n, np.int32),
                      params=nns_amd.default_params(timestep=0.0, **kw))
    b.step()
    b.check()
    a = np.stack([b.host(k) for k in ("ax", "ay", "az")], 1).reshape(systems, n, 3)
    assert np.array_equal(a[0, FAR], a[-1, FAR])
    compare(a[0, FAR], want)
