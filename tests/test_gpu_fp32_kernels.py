"""The fp32 kernels at the edges of their tiles: head_dims around the multiples of 32 (exact and padded variants), lengths
around the 32-key sub-tiles, the 128-key steps of the four waves and the 128-row query tiles, and odds around the smallest normal number, against the float64
oracle; and rows further apart than 32-bit offsets reach."""
import pytest
import torch

from oracle import sb_oracle as orc
from stickbreaking_attention import sb_attn_varlen
from test_gpu_parity import NAMES, run_varlen, small_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qk_std,attend_current,add_remainder", [(1.0, False, True), (6.0, True, False)])
@pytest.mark.parametrize("H", [3, 6])      # 4743 and 9486 rows x heads: products of fp32 numbers, and of triples
@pytest.mark.parametrize("D", [1, 31, 32, 33, 64, 66, 96, 97, 127, 128])
def test_fp32_tile_edges_against_oracle(gpu_device, D, H, qk_std, attend_current, add_remainder):
    lengths = [1, 31, 32, 33, 127, 128, 129, 161, 255, 257, 2, 385]
    (q, k, v, do, drem), dev, cu = small_case(H, D, lengths, torch.float32, seed=D, qk_std=qk_std)
    outs = run_varlen(dev[0], dev[1], dev[2], cu.to(gpu_device), lengths, False, attend_current, dev[3], dev[4],
                      add_remainder=add_remainder)
    again = run_varlen(dev[0], dev[1], dev[2], cu.to(gpu_device), lengths, False, attend_current, dev[3], dev[4],
                       add_remainder=add_remainder)
    d = [t.double() for t in (q, k, v, do, drem)]
    if add_remainder:
        d[4] = orc.remainder_drem(d[3], d[4], d[2])
    ref = orc.varlen_stream(d[0], d[1], d[2], cu, attend_current=attend_current, do=d[3], drem=d[4], dtype=torch.float64)
    if add_remainder:
        ref = orc.with_remainder(ref, d[2], d[3])
    for n, a, b, r in zip(NAMES, outs, again, ref):
        rel = (a.detach().double().cpu() - r).norm() / r.norm()
        print(f"D={D} {n}: relative error {rel.item():.2e}", flush=True)
        assert rel < 1e-5, f"{n}: {rel.item():.2e}"
        assert torch.equal(a, b), f"{n}: two runs differ"


@pytest.mark.parametrize("D", [20, 64, 96, 128])
def test_single_products_are_rounded_once(gpu_device, D):
    """Sequences of two tokens: every contraction over keys or rows has one term.  Column 0 of q, k, v and d_o is 1, so column 0 of an
    output is the other factor, and the rest are its products rounded to fp32: within 2^-24 of them."""
    H, n = 32, 200      # (12800 rows x heads: products of triples elsewhere)
    (q, k, v, do, drem), _, cu = small_case(H, D, [2] * n, torch.float32, seed=D)
    for t in (q, k, v, do):
        t[..., 0] = 1
    dev = [t.to(gpu_device) for t in (q, k, v, do, drem)]
    got = dict(zip(NAMES, run_varlen(dev[0], dev[1], dev[2], cu.to(gpu_device), [2] * n, False, False, dev[3], dev[4], scale=1.0)))
    for name, vec, row, other in (("o", v, 1, 0), ("dq", k, 1, 0), ("dk", q, 0, 1), ("dv", do, 0, 1)):
        out = got[name].detach().double().cpu()[:, row::2]
        exact = out[..., :1] * vec.double()[:, other::2]
        worst = ((out - exact).abs() * 2.0 ** 24 - exact.abs()).max().item()
        print(f"D={D} {name}: {worst:.2e}", flush=True)
        assert worst <= 0, name


@pytest.mark.parametrize("values", ["normal", "slow"])
@pytest.mark.parametrize("D", [3, 16, 64, 128])
def test_triples_are_no_less_accurate_than_fp32_products(gpu_device, D, values):
    """Eight heads together (9600 rows x heads) form their products of triples, one at a time of fp32 numbers: the error against float64, in
    norm, may not be larger than 1.02 times theirs (a rms over 8 x 1200 rows x D numbers is known to about 1 %; measured: 0.80 to 1.00)."""
    lengths, H = [40, 97, 33, 65, 129, 50, 71, 200, 300, 215], 8
    (q, k, v, do, drem), _, cu = small_case(H, D, lengths, torch.float32, seed=D)
    if values == "slow":
        q, k, v = 0.25 * (q + 1), 0.25 * (k - 1), 0.25 * v
    dev = [t.to(gpu_device) for t in (q, k, v, do, drem)]
    run = lambda h: run_varlen(*(t[h] for t in dev[:3]), cu.to(gpu_device), lengths, False, False, dev[3][h], dev[4][h])
    triples = run(slice(0, H))
    parts = [run(slice(h, h + 1)) for h in range(H)]
    ref = orc.varlen_stream(*(t.double() for t in (q, k, v)), cu, do=do.double(), drem=drem.double(), dtype=torch.float64)
    for i, n in enumerate(NAMES):
        a, b = ((t.detach().double().cpu() - ref[i]).norm().item() for t in (triples[i], torch.cat([p[i] for p in parts])))
        print(f"D={D} {values} {n}: error of triples / of fp32 products {a / b:.3f}", flush=True)
        assert a <= 1.02 * b, n


@pytest.mark.parametrize("D", [32, 64, 128])
def test_head_groups_give_the_bits_of_one_pass(gpu_device, D):
    """A call large enough for products of triples, under workspace limits that leave groups of heads that are not."""
    from stickbreaking_attention import _native

    lengths, H = [200, 33, 1, 385], 16      # (9904 rows x heads; a line at 8192)
    host, dev, cu = small_case(H, D, lengths, torch.float32, seed=D)
    run = lambda: run_varlen(*dev[:3], cu.to(gpu_device), lengths, False, False, dev[3], dev[4])
    whole = run()
    try:
        for limit in (1, 100000, 300000):
            _native.set_backward_workspace_limit(limit)
            for n, a, b in zip(NAMES, run(), whole):
                assert torch.equal(a, b), f"{n}, limit {limit}"
    finally:
        _native.set_backward_workspace_limit(None)


@pytest.mark.parametrize("D", [64, 128])
def test_odds_below_the_smallest_normal_number(gpu_device, D):
    """Logits of -92 to -86, odds of 2^-133 to 2^-124.  A logit in octaves has an error of up to 2^-17.9 (133 octaves, two
    roundings), which is 3e-6 of the odds at most and the same again where they are multiplied; the odds' own last place lies
    at 2^-149, 4e-6 of the mean of 2^-128."""
    H, T = 2, 300
    g = torch.Generator().manual_seed(D)
    q, k = torch.zeros(H, T, D), torch.zeros(H, T, D)
    q[..., 0] = 1
    k[..., 0] = -92 + 6 * torch.rand(H, T, generator=g)
    v, do = (2.0 ** 20 * torch.randn(H, T, D, generator=g) for _ in range(2))
    drem = torch.randn(H, T, generator=g)
    cu = torch.tensor([T], dtype=torch.int32)
    ref = orc.varlen_stream(*(t.double() for t in (q, k, v)), cu, do=do.double(), drem=drem.double(), dtype=torch.float64, scale=1.0)
    dev = [t.to(gpu_device) for t in (q, k, v, do, drem)]
    got = run_varlen(dev[0], dev[1], dev[2], cu.to(gpu_device), [T], False, False, dev[3], dev[4], scale=1.0)
    for n, a, b in zip(NAMES, got, ref):
        rel = (a.detach().double().cpu() - b).norm() / b.norm()
        print(f"D={D} {n}: relative error {rel.item():.2e}", flush=True)
        assert rel < 1e-5, f"{n}: {rel.item():.2e}"


@pytest.mark.parametrize("D", [128, 50, 9])
@pytest.mark.parametrize("far", ["all", "do"])
def test_rows_further_apart_than_32_bit_offsets_reach(gpu_device, far, D):
    H, T, stride = 2, 40, (1 << 24) + 8
    buf = torch.empty(T * stride, device=gpu_device)
    near = [torch.randn(H, T, D, device=gpu_device) for _ in range(4)]
    drem = torch.randn(H, T, device=gpu_device)
    cu = torch.tensor([7, T], dtype=torch.int32)
    views = [buf.as_strided((H, T, D), (D, stride, 1), 2 * i * D) for i in range(4)]
    for view, t in zip(views, near):
        view.copy_(t)
    if far == "do":
        views[:3] = near[:3]

    def run(q, k, v, do):      # (without the copies run_varlen makes)
        for t in (q, k, v):
            t.requires_grad_()
        o, rem = sb_attn_varlen(q, k, v, cu, T - 7, zero_start=False, attend_current=True, add_remainder=True)
        return o, rem, *torch.autograd.grad([o, rem], [q, k, v], [do, drem])

    for n, a, b in zip(NAMES, run(*views), run(*near)):
        assert (a - b).norm() < 1e-6 * b.norm(), n
