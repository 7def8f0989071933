"""A rollout's states are its own: inputs and results changed in place between the
forward and the backward leave the gradients alone, with the last checkpoint at
the first step, in the middle and one step before the end.

Tolerance: the two gradients are the same sums of the same terms, added in FP64 in an
order that may differ and rounded to FP32 once a step: 5 steps of 2^-24, relative to the
largest gradient, carried along a map close to the identity; 1e-5 leaves a factor of 30."""
import pytest

import nns_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps,every", [(1, 8), (5, 8), (5, 2), (4, 3), (0, 2)])
def test_states_changed_after_the_forward(steps, every):
    import torch
    from nns_amd.adjoint import Slots, rollout
    assert torch.cuda.is_available()
    print(f"case rollout states steps={steps} every={every}", flush=True)
    n = 3001
    arrs = nns_amd.initial_conditions("plummer", n, 4)
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    u = [torch.randn(n, device="cuda", generator=g) for _ in range(6)]
    grads = []
    for change in (False, True):
        ins = [torch.tensor(a, device="cuda", requires_grad=True) for a in arrs]
        slots = Slots(n, every)
        out = rollout(slots, *ins, steps=steps, dt=1e-3, every=every)
        if change:
            with torch.no_grad():
                for t in ins[:6]:
                    t.mul_(-3.0)
                for t in out:
                    t.detach().add_(5.0)
        torch.autograd.backward(out, u)
        slots.check()
        grads.append([t.grad for t in ins])
    for a, b in zip(*grads):
        assert float((a - b).abs().max()) <= 1e-5 * float(a.abs().max()) or not bool(a.any())
