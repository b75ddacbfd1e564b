"""The kernel that rebuilds the forward's products at head_dim 128 sweeps 64 keys at a time: lengths around its tiles, with an odd and an even number
of 32-key sub-tiles, against the gradients that the kept products give, bit for bit."""
import pytest
import torch

from test_gpu_parity import NAMES, run_varlen, small_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("attend_current", [False, True])
@pytest.mark.parametrize("lengths", [[1, 2, 31, 32, 33, 34, 63, 64, 65, 66] * 20, [96, 97, 127, 128, 129, 160, 161, 192, 193, 255, 256, 257, 258] * 4,
                                     [2017, 1, 2080, 2081, 33]])
def test_rebuilt_as_recorded(gpu_device, lengths, attend_current, dtype):
    H = 32      # (tiles of 128 rows, not split over the waves)
    _, dev, cu = small_case(H, 128, lengths, dtype, seed=len(lengths), qk_std=2.0)
    kept, rebuilt = (run_varlen(dev[0], dev[1], dev[2], cu.to(gpu_device), lengths, False, attend_current, dev[3], dev[4], save_carry=s)
                     for s in (True, False))
    for n, a, b in zip(NAMES, kept, rebuilt):
        assert torch.equal(a, b), n
