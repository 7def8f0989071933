"""A rollout of no steps is the identity: its states are its inputs, the gradients of positions and
velocities are the cotangents themselves, and that of the masses is exactly zero, also after
inputs and results were changed in place.  Equality, since nothing is computed."""
import pytest

import nns_amd

pytestmark = pytest.mark.gpu


def test_no_steps_is_the_identity():
    import torch
    from nns_amd.adjoint import Slots, rollout
    assert torch.cuda.is_available()
    n = 777
    ins = [torch.tensor(a, device="cuda", requires_grad=True) for a in nns_amd.initial_conditions("plummer", n, 4)]
    was = [t.detach().clone() for t in ins]
    u = [torch.randn(n, device="cuda") for _ in range(6)]
    slots = Slots(n, 2)
    out = rollout(slots, *ins, steps=0, dt=1e-3, every=2)
    assert all(torch.equal(o, w) for o, w in zip(out, was))
    with torch.no_grad():
        for t in ins[:6]:
            t.mul_(-3.0)
        for t in out:
            t.detach().add_(5.0)
    torch.autograd.backward(out, u)
    slots.check()
    assert all(torch.equal(t.grad, v) for t, v in zip(ins[:6], u))
    assert torch.equal(ins[6].grad, torch.zeros_like(ins[6]))
