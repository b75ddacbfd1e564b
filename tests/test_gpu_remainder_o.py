"""The forward's share of the remainder at head_dims that no kernel is made for: o + rem * v in one rounding, against the two outputs of the plain
call.  With u = 2^-8 (f16, of 11 bits: 2^-11) the largest relative error of a rounding to 8 bits, what they differ by is at most the rounding of o, of rem and of the sum."""
import pytest
import torch

from test_gpu_parity import run_varlen, small_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,u", [(torch.bfloat16, 2.0 ** -8), (torch.float16, 2.0 ** -11)])
@pytest.mark.parametrize("H", [1, 24])      # rows split over the waves of a workgroup, and tiles of 128 rows
@pytest.mark.parametrize("D", [8, 9, 33, 50, 63, 65, 72, 96, 97, 127])
def test_sum_in_one_rounding(gpu_device, D, H, dtype, u):
    lengths = [1, 2, 31, 32, 33, 64, 65, 127, 128, 129, 161, 300, 515]
    _, dev, cu = small_case(H, D, lengths, dtype, seed=D)
    q, k, v = (t * 0.25 for t in dev[:3])
    plain, fused = (run_varlen(q, k, v, cu.to(gpu_device), lengths, False, False, None, None, add_remainder=a) for a in (False, True))
    o, rem, both = plain[0].detach().double(), plain[1].detach().double(), fused[0].detach().double()
    share = rem.unsqueeze(-1) * v.double()
    # (2^-24: the smallest step of f16; 1e-6: fp32 arithmetic)
    bound = (u + 1e-6) * (o.abs() + share.abs() + both.abs()) * (1 + 2 * u) + 2 * 2.0 ** -24 * (1 + v.double().abs())
    assert torch.equal(plain[1], fused[1])
    assert ((both - (o + share)).abs() <= bound).all()
