"""A backward whose workspace does not fit the memory that is left runs with a smaller one: on the two kernels, or some heads at a time."""
import pytest
import torch

pytestmark = pytest.mark.gpu

MB = 1 << 20


@pytest.mark.parametrize("host_layer", [True, False])
@pytest.mark.parametrize("D,H,left", [(128, 16, 200), (128, 16, 60), (64, 12, 130)])      # MB left: the backward asks for 360 and 162, the two
def test_backward_with_little_memory_left(gpu_device, monkeypatch, D, H, left, host_layer):      # kernels for 141 and 106
    from stickbreaking_attention import _native, sb_attn_varlen

    lengths, device = [4096, 2048, 4096, 4096, 2048], torch.cuda.current_device()
    g = torch.Generator().manual_seed(D)
    q, k, v, do = (torch.randn(H, sum(lengths), D, generator=g).bfloat16().to(gpu_device) for _ in range(4))
    drem = torch.randn(H, sum(lengths), generator=g).bfloat16().to(gpu_device)
    for t in (q, k, v):
        t.requires_grad_()
    cu = torch.tensor(lengths).cumsum(0).int().to(gpu_device)
    if not host_layer:
        monkeypatch.setattr(_native, "use_ext", lambda: False)
    o, rem = sb_attn_varlen(q, k, v, cu, max(lengths), zero_start=False, save_carry=False)

    def backward():
        return torch.autograd.grad([o, rem], [q, k, v], [do, drem], retain_graph=True)

    whole = backward()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    outputs = 3 * q.numel() * 2
    total = torch.cuda.get_device_properties(device).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + outputs + left * MB) / total)
    try:
        with_less = backward()
        torch.cuda.synchronize()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    for n, a, b in zip(("dq", "dk", "dv"), with_less, whole):
        assert torch.isfinite(a.float()).all()
        excess = (a.float() - b.float()).abs() - 2 * torch.maximum(torch.full_like(b.float(), 2e-2), b.float().abs() * 2.0 ** -7)      # two orders of summation
        assert excess.max().item() <= 0, f"{n}: {excess.max().item():.2e} beyond twice the bound"
