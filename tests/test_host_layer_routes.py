"""Which calls the torch host layer takes: ordinary eager ones.  Anything that has to see the operators, or that they refuse,
goes to the Python operators as before."""
import pytest
import torch
from torch.autograd import forward_ad
from torch.utils._python_dispatch import TorchDispatchMode

from stickbreaking_attention import _native, sb_attn


class Watch(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def takes(q):
    return _native.use_ext() and _native.ext().ordinary(q, torch.zeros(1, 2, 8), torch.zeros(1, 2, 8))


def test_only_ordinary_calls_go_through_the_host_layer():
    x = torch.zeros(1, 2, 8)
    seen = []

    def note(q):
        seen.append(takes(q))
        return q * 1

    assert takes(x) and takes(torch.nn.Parameter(x)) and takes(x.clone().requires_grad_())
    with torch.no_grad():
        assert takes(x)
    torch.func.vmap(note)(torch.zeros(3, 1, 2, 8))
    torch.func.grad(lambda q: note(q).sum())(x)
    torch.jit.trace(note, (x,), check_trace=False)
    with Watch():
        note(x)
    with torch._subclasses.FakeTensorMode() as fake:
        fake_x = fake.from_tensor(x)
    note(fake_x)
    with forward_ad.dual_level():
        note(forward_ad.make_dual(x, torch.ones_like(x)))
    assert seen == [False] * 6
    assert takes(x)      # and nothing lingers


@pytest.mark.gpu
def test_forward_mode_derivatives_stay_refused(gpu_device):
    q, k, v = (torch.randn(1, 2, 40, 64, device=gpu_device, dtype=torch.bfloat16) for _ in range(3))
    with torch.no_grad(), forward_ad.dual_level():
        with pytest.raises(RuntimeError):
            sb_attn(forward_ad.make_dual(q, torch.ones_like(q)), k, v)
