"""Where the waves of a block share a group (up to 5,120 groups of 64 bodies) the waves per
block follow from the groups: the tuner has nothing to choose there and leaves the setting,
which the counting walk and a later, larger system on the same context use.  Above, it takes one
of the three that it times.  The line is met from both sides."""
import numpy as np
import pytest

import nns_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [64, 3000, 5120 * 64])
@pytest.mark.parametrize("waves", [2, 4, 8])
def test_setting_stays_where_groups_are_shared(n, waves):
    import torch
    assert torch.cuda.is_available()
    print(f"case autotune n={n} waves={waves}", flush=True)
    bh = nns_amd.BarnesHut(*nns_amd.initial_conditions("plummer", n, 5),
                           params=nns_amd.default_params(force_waves=waves))
    bh.rebuild()
    assert nns_amd.autotune(bh.ctx) == waves
    assert bh.ctx.get_params().force_waves == waves
    bh.forces()
    bh.ctx.check()


@pytest.mark.parametrize("waves", [2, 4, 8])
def test_ensemble_keeps_its_setting(waves):
    sizes = [700, 65, 300]
    parts = [nns_amd.initial_conditions("plummer", k, k) for k in sizes]
    b = nns_amd.Batch(*[np.concatenate([p[k] for p in parts]) for k in range(7)], sizes,
                      params=nns_amd.default_params(force_waves=waves))
    b.step()
    assert b.autotune() == waves
    b.check()


def test_one_wave_per_group_is_tuned():
    n = 5120 * 64 + 1
    bh = nns_amd.BarnesHut(*nns_amd.initial_conditions("plummer", n, 5))
    bh.rebuild()
    w = nns_amd.autotune(bh.ctx)
    assert w in (2, 4, 8) and bh.ctx.get_params().force_waves == w
