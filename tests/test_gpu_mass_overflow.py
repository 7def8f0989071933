"""A cell whose mass is past FP32 (2 x 2e38) below a parent that is not (a third body of
-2.5e38): the bodies that took the parent must not feel what happens below it, whichever of
their wave's lanes went on.  The acceleration of the far bodies is finite and that of the
oracle's FP64 walk.  Through the shared walk (one system) and the one-wave walk (an ensemble of
more groups than the shared walk takes).
Bar: an FP32 sum of some twenty monopoles, 1e-5 of the acceleration."""
import numpy as np
import pytest

import nns_amd

pytestmark = pytest.mark.gpu


def bodies():
    far = np.random.default_rng(2).uniform(0.0, 0.35, (20, 3))
    heavy = 0.9 + np.array([[0.0, 0.0, 0.0], [1e-4, 0.0, 0.0], [8e-3, 8e-3, 8e-3]])
    corners = np.array([[0.0, 0.0, 0.0], [1.0, 1.0, 1.0]])
    p = np.concatenate([far, corners[:1], heavy, corners[1:]]).astype(np.float32)
    m = np.concatenate([np.ones(21), [2e38, 2e38, -2.5e38], [1.0]]).astype(np.float32)
    z = np.zeros(len(m), np.float32)
    return [p[:, 0].copy(), p[:, 1].copy(), p[:, 2].copy(), z, z, z, m]


FAR = np.arange(21, dtype=np.int32)


def expected(oracle, theta, eps):
    a = bodies()
    t = oracle.KeyTree(*a[:3], a[6])
    acc, _ = t.accel(theta, float(np.float32(np.float32(eps) ** 2)), mac_mode=1, targets=FAR)
    return acc


def compare(got, want):
    assert np.isfinite(got).all()
    err = np.linalg.norm(got.astype(np.float64) - want, axis=1) / np.linalg.norm(want, axis=1)
    assert err.max() <= 1e-5, err.max()


@pytest.mark.parametrize("soft,kahan", [(1e-3, 1), (1e-3, 0), (0.0, 1), (0.0, 0)])
def test_bodies_that_took_the_parent_stay_finite(oracle, soft, kahan):
    import torch
    assert torch.cuda.is_available()
    print(f"case mass overflow soft={soft} kahan={kahan}", flush=True)
    p = nns_amd.default_params(theta=0.5, softening=soft, kahan=kahan)
    want = expected(oracle, 0.5, soft)
    bh = nns_amd.BarnesHut(*bodies(), params=p)
    bh.rebuild()
    bh.forces()
    bh.ctx.check()
    compare(np.stack([bh.host(k) for k in ("ax", "ay", "az")], 1)[FAR], want)
    systems, n = 5121, len(bodies()[6])
    b = nns_amd.Batch(*[np.tile(v, systems) for v in bodies()], np.full(systems, n, np.int32),
                      params=nns_amd.default_params(theta=0.5, softening=soft, kahan=kahan, timestep=0.0))
    b.step()
    b.check()
    a = np.stack([b.host(k) for k in ("ax", "ay", "az")], 1).reshape(systems, n, 3)
    assert np.array_equal(a[0, FAR], a[-1, FAR])
    compare(a[0, FAR], want)
