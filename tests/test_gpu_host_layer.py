"""The torch host layer of eager calls: gradients arriving through only one of the two outputs, and graphs kept for a second
backward, against the same call with both gradients given."""
import pytest
import torch

from stickbreaking_attention import sb_attn, sb_attn_varlen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("through", ["o", "rem", "both"])
def test_gradient_through_either_output_and_a_second_backward(gpu_device, through, packed, dtype):
    H, L, D = 8, 200, 128
    g = torch.Generator(device=gpu_device).manual_seed(3)
    shape = (H, L, D) if packed else (1, H, L, D)
    q, k, v = (torch.randn(shape, generator=g, device=gpu_device, dtype=torch.float32).to(dtype).requires_grad_() for _ in range(3))
    do, drem = torch.randn_like(q), torch.randn_like(q[..., 0])
    if packed:
        o, rem = sb_attn_varlen(q, k, v, torch.tensor([70, L], dtype=torch.int32), 130, zero_start=False)
    else:
        o, rem = sb_attn(q, k, v)
    do, drem = (do if through != "rem" else torch.zeros_like(do)), (drem if through != "o" else torch.zeros_like(drem))
    both = torch.autograd.grad([o, rem], [q, k, v], [do, drem], retain_graph=True)
    outs, grads = {"o": ([o], [do]), "rem": ([rem], [drem]), "both": ([o, rem], [do, drem])}[through]
    for got, want in zip(torch.autograd.grad(outs, [q, k, v], grads), both):
        assert torch.equal(got, want)
    assert all(t.abs().max() > 0 for t in both[:2])
