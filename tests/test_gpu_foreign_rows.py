"""Rows behind a sequence's last one (the next sequence's, the next head's, rows of no sequence) are loaded with its last tiles and enter their
contractions as zeros.  Every second sequence, and the rows of no sequence, hold NaN or infinities here: the other sequences must come out
bit for bit as beside ordinary numbers.  Lengths end anywhere in the kernels' tiles of 32, 64, 128 and 256 rows."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

LENGTHS = [70, 1, 33, 255, 129, 31, 320, 257, 64, 95, 300, 289, 97, 513]      # odd places are kept
CASES = {
    # heads, head_dim, lengths, dtype, options
    "row-tiles": (40, 128, LENGTHS, torch.bfloat16, {}),
    "row-tiles-64": (16, 64, [70, 1300, 31, 1153, 600, 1029], torch.bfloat16, {}),
    "row-tiles-remainder": (40, 128, LENGTHS, torch.float16, dict(add_remainder=True, attend_current=True)),
    "row-tiles-64-remainder-rebuilt": (16, 64, [70, 1300, 31, 1153, 600, 1029], torch.float16, dict(add_remainder=True, save_carry=False)),
    "two-kernels": (40, 128, LENGTHS, torch.bfloat16, dict(kernels=1)),
    "two-kernels-64": (40, 64, LENGTHS, torch.bfloat16, dict(kernels=1)),
    "key-tiles": (8, 128, LENGTHS, torch.bfloat16, dict(kernels=2)),
    "split": (2, 64, LENGTHS, torch.bfloat16, dict(add_remainder=True)),
    "padded": (40, 50, LENGTHS, torch.bfloat16, dict(add_remainder=True)),
    "fp32": (8, 64, LENGTHS, torch.float32, dict(add_remainder=True)),
    "fp32-padded": (8, 127, LENGTHS, torch.float32, {}),
    "fp32-few": (1, 128, LENGTHS, torch.float32, {}),
}


@pytest.mark.parametrize("token_major", [False, True])
@pytest.mark.parametrize("label", CASES)
def test_foreign_rows_are_zeros(gpu_device, label, token_major):
    from stickbreaking_attention import _native, sb_attn_varlen

    H, D, lengths, dtype, opts = CASES[label]
    opts, pad, T = dict(opts), 67, sum(lengths)
    kernels = opts.pop("kernels", 0)
    if label.startswith("row-tiles"):
        assert T * H >= 64 << 10      # (fewer do not reach the kernel)
    ends = np.cumsum(lengths)
    keep = torch.zeros(T + pad, dtype=torch.bool, device=gpu_device)
    for i in range(1, len(lengths), 2):
        keep[ends[i - 1]:ends[i]] = True
    g = torch.Generator().manual_seed(D)
    clean = [torch.randn(H, T + pad, D, generator=g) for _ in range(4)] + [torch.randn(H, T + pad, generator=g)]
    clean = [t.to(dtype).to(gpu_device) for t in clean]
    cu = torch.tensor(ends, dtype=torch.int32, device=gpu_device)

    def run(fill):
        x = [t.clone() for t in clean]
        if fill is not None:
            for t in x:
                t[:, ~keep] = fill
        if token_major:
            x = [t.transpose(0, 1).contiguous().transpose(0, 1) for t in x]
        q, k, v = (t.requires_grad_() for t in x[:3])
        o, rem = sb_attn_varlen(q, k, v, cu, max(lengths), zero_start=False, **opts)
        return o, rem, *torch.autograd.grad([o, rem], [q, k, v], [x[3], x[4]])

    saved = _native.BACKWARD_KERNELS
    try:
        _native.BACKWARD_KERNELS = kernels
        ref = run(None)
        for fill in (float("nan"), float("inf"), torch.finfo(dtype).min):
            for n, a, b in zip(("o", "rem", "dq", "dk", "dv"), run(fill), ref):
                assert torch.isfinite(b[:, keep].float()).all()
                assert torch.equal(a[:, keep], b[:, keep]), f"{label}: {n} beside rows of {fill}"
                assert (a[:, T:] == 0).all(), f"{label}: {n}, rows of no sequence"
    finally:
        _native.BACKWARD_KERNELS = saved
