"""From 8192 rows x heads on the fp32 kernels form their products of bf16 triples.  Workgroups that meet numbers which triples do not hold form
them of fp32 numbers instead.  Tensors at both ends of fp32's range, alone and with partners that bring the products back to the middle,
against the float64 oracle, 1e-5 in norm: a gradient is a difference of prefix sums of up to 161 terms, 161 x 2^-24 = 0.96e-5 at worst
where nothing cancels (measured: up to 1.3e-6).  An operand of 2^-122 whose last bits were lost (those below 2^-133) would be 2^-12 = 2.4e-4
off.  An infinite key against a large one: the logit saturates for both."""
import pytest
import torch

from oracle import sb_oracle as orc
from test_gpu_parity import NAMES, run_varlen, small_case

pytestmark = pytest.mark.gpu

LENGTHS, HEADS = [1, 33, 64, 161], 32      # (8288 rows x heads, more than which triples are used from)
ZERO = -1000      # (2.0 ** ZERO is 0 in fp32)
CASES = {      # exponents added to q, k, v, do, drem
    "middle": (0, 0, 0, 0, 0),
    "tiny-values": (0, 0, -122, 0, 0),
    "tiny-gradients": (0, 0, 0, -122, -122),
    "tiny-values-and-drem": (0, 0, -122, 0, -122),
    "tiny-keys-huge-queries": (122, -122, 0, 0, 0),
    "huge-keys-tiny-queries": (-122, 122, 0, 0, 0),
    "huge-values-tiny-gradients": (0, 0, 122, -122, 0),
    # tiny numbers that are streamed past, and another operand that brings the results back: dP of V and of dO, then K and Q
    "tiny-values-large-keys": (-60, 60, -122, 0, ZERO),
    "tiny-gradients-large-queries": (60, -60, 0, -122, ZERO),
    "tiny-keys-large-gradients": (45, -122, 0, 60, 60),
    "tiny-queries-large-gradients": (-122, 45, 0, 60, 60),
}


@pytest.mark.parametrize("label", CASES)
@pytest.mark.parametrize("D", [36, 64, 127, 128])
def test_ends_of_the_range(gpu_device, D, label):
    host, _, cu = small_case(HEADS, D, LENGTHS, torch.float32, seed=D)
    host = [t * 2.0 ** e for t, e in zip(host, CASES[label])]
    dev = [t.to(gpu_device) for t in host]
    outs = run_varlen(dev[0], dev[1], dev[2], cu.to(gpu_device), LENGTHS, False, False, dev[3], dev[4])
    d = [t.double() for t in host]
    ref = orc.varlen_stream(d[0], d[1], d[2], cu, do=d[3], drem=d[4], dtype=torch.float64)
    for n, a, r in zip(NAMES, outs, ref):
        if not 2.0 ** -126 < r.abs().max().item() < 2.0 ** 127:      # beyond fp32
            continue
        rel = ((a.detach().double().cpu() - r).norm() / r.norm()).item()
        print(f"{label} D={D} {n}: relative error {rel:.2e}", flush=True)
        assert rel < 1e-5, f"{n}: {rel:.2e}"


@pytest.mark.parametrize("D", [36, 128])
def test_infinite_key(gpu_device, D):
    host, _, cu = small_case(HEADS, D, LENGTHS, torch.float32, seed=D)
    host[0][..., 0] = 1
    got = []
    for value in (float("inf"), 1e30):
        host[1][:, 50, 0] = value
        dev = [t.to(gpu_device) for t in host]
        got.append(run_varlen(dev[0], dev[1], dev[2], cu.to(gpu_device), LENGTHS, False, False, dev[3], dev[4]))
    for n, a, b in zip(NAMES[:2], *got):
        assert torch.isfinite(a).all() and ((a - b).norm() / b.norm()).item() < 1e-5, n
