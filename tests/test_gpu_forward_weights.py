"""The forward's two ways through a tile's weights: groups of keys whose odds multiply up to any size (the lane then takes them
one by one), next to tame ones in the same wave, against the float64 oracle; and that neither way shows in another row's bits."""
import pytest
import torch

from oracle import sb_oracle as orc
from stickbreaking_attention import sb_attn, sb_attn_varlen
from test_gpu_parity import NAMES, run_varlen, tol_check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 80, 128])
@pytest.mark.parametrize("low,high", [(-20.0, 20.0), (15.0, 30.0), (-200.0, 200.0), (50.0, 400.0)])
def test_logits_of_any_size(gpu_device, D, low, high):
    lengths = [33, 200]
    T, H = sum(lengths), 2
    g = torch.Generator().manual_seed(int(high) + D)
    # one column carries the logits: z_ij = k_j for every row, so that every size of odds meets every other
    q, k, v, do = (torch.zeros(H, T, D), 0.01 * torch.randn(H, T, D, generator=g), *(torch.randn(H, T, D, generator=g) for _ in range(2)))
    q[..., 0] = 1
    k[..., 0] = low + (high - low) * torch.rand(H, T, generator=g)
    drem = torch.randn(H, T, generator=g)
    host = [t.bfloat16() for t in (q, k, v, do, drem)]
    cu = torch.tensor([33, 233], dtype=torch.int32)
    ref = orc.varlen_stream(*host[:3], cu, do=host[3], drem=host[4], dtype=torch.float64, scale=1.0)
    dev = [t.to(gpu_device) for t in host]
    got = run_varlen(dev[0], dev[1], dev[2], cu.to(gpu_device), lengths, False, False, dev[3], dev[4], scale=1.0)
    for n, a, b in list(zip(NAMES, got, ref))[:2]:
        tol_check(n, a, b, torch.bfloat16, f"logits {low}..{high}")
    assert all(torch.isfinite(t).all() for t in got)


@pytest.mark.parametrize("H,D", [(2, 64), (2, 80), (2, 128), (100, 64), (100, 50), (100, 96), (100, 128)])
def test_a_rows_bits_depend_on_no_other_row(gpu_device, H, D):
    """Few and many heads: the kernels that split the keys over the waves, and those that do not."""
    T, odd = 700, [3, 40, 131, 699]
    g = torch.Generator(device=gpu_device).manual_seed(D)
    q, k, v, do = (torch.randn(H, T, D, generator=g, device=gpu_device).bfloat16() for _ in range(4))
    cu = torch.tensor([T], dtype=torch.int32, device=gpu_device)
    saturated = q.clone()
    saturated[:, odd] *= 100

    def run(q):
        q = q.requires_grad_()
        o, rem = sb_attn_varlen(q, k, v, cu, T, zero_start=False)
        return o, rem, torch.autograd.grad(o, q, do)[0]

    others = [i for i in range(T) if i not in odd]
    for n, a, b in zip(("o", "rem", "dq"), run(q), run(saturated)):
        assert torch.equal(a[:, others], b[:, others]), n
        assert not torch.equal(a[:, odd], b[:, odd]), n


@pytest.mark.parametrize("attend_current", [False, True])
@pytest.mark.parametrize("D", [50, 64, 128])
@pytest.mark.parametrize("H", [2, 1000])
def test_a_rows_bits_do_not_depend_on_the_rows_behind_it(gpu_device, H, D, attend_current):
    """Sequences that end just behind, just before and well behind a multiple of 32 and 128 rows: the rows they have in common, in the kernels
    that split the keys over the waves (few heads) and those that do not."""
    most, outs = 700, {}
    g = torch.Generator(device=gpu_device).manual_seed(D)
    q, k, v, do = (torch.randn(H, most, D, generator=g, device=gpu_device).bfloat16() for _ in range(4))
    q, k = 0.25 * q + 0.8, 0.25 * k - 0.8      # (sticks that last for hundreds of keys)
    for T in (33, 129, 130, 160, 161, 257, 289, 290, 385, 386, 513, 514, 641, 642, most):
        x = [t[:, :T].contiguous().requires_grad_() for t in (q, k, v)]
        cu = torch.tensor([T], dtype=torch.int32, device=gpu_device)
        o, rem = sb_attn_varlen(*x, cu, T, zero_start=False, attend_current=attend_current)
        outs[T] = dict(o=o.detach(), rem=rem.detach())
        if H == 2:
            outs[T]["dq"] = torch.autograd.grad(o, x[0], do[:, :T])[0]
    for T, got in outs.items():
        for n, a in got.items():
            assert torch.equal(a, outs[most][n][:, :T]), f"{n}, {T} rows"


@pytest.mark.parametrize("attend_current", [False, True])
@pytest.mark.parametrize("D", [50, 64, 128])
@pytest.mark.parametrize("H,count", [(1, 1), (12, 1), (100, 1), (1000, 1), (4, 3)])
def test_a_short_prompts_bits_stay_when_it_grows(gpu_device, H, count, D, attend_current):
    """Prompts that grow from one and two sub-tiles of keys to three, at head counts on both sides of the line between the kernels."""
    g = torch.Generator(device=gpu_device).manual_seed(D)
    q, k, v = (torch.randn(count, H, 70, D, generator=g, device=gpu_device).bfloat16() for _ in range(3))
    outs = {T: sb_attn(*(t[:, :, :T] for t in (q, k, v)), attend_current=attend_current) for T in (1, 31, 32, 33, 63, 64, 65, 70)}
    for T, got in outs.items():
        for n, a, b in zip(("o", "rem"), got, outs[70]):
            assert torch.equal(a, b[:, :, :T]), f"{n}, {T} rows"
