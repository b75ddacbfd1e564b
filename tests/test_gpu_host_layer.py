"""The torch host layer of eager calls: gradients arriving through only one of the two outputs, and graphs kept for a second
backward, against the same call with both gradients given; other Python threads while a call waits for the GPU;
what saved-tensor hooks and checkpointing hand back to the backward; what is held between the passes."""
import threading
import time

import pytest
import torch
from torch.utils.checkpoint import checkpoint

from stickbreaking_attention import _native, sb_attn, sb_attn_varlen

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


@pytest.mark.parametrize("where", ["device", "host"])
def test_other_threads_run_while_a_call_waits_for_the_gpu(gpu_device, where):
    """Reading the lengths back (or sending them) waits for everything the stream holds; the interpreter is not held meanwhile."""
    q, k, v = (torch.randn(2, 200, 64, device=gpu_device, dtype=torch.bfloat16) for _ in range(3))
    cu = torch.tensor([0, 70, 200], dtype=torch.int32, device=gpu_device if where == "device" else "cpu")
    sb_attn_varlen(q, k, v, cu, 130)
    start, end = torch.cuda.Event(True), torch.cuda.Event(True)
    torch.cuda._sleep(1 << 20)
    start.record()
    torch.cuda._sleep(1 << 20)
    end.record()
    torch.cuda.synchronize()
    cycles = int((1 << 20) * 150 / start.elapsed_time(end))      # of a kernel of 150 ms
    ticks, stop = [], threading.Event()

    def tick():
        while not stop.wait(0.0005):
            ticks.append(time.perf_counter())

    thread = threading.Thread(target=tick)
    thread.start()
    try:
        time.sleep(0.01)
        torch.cuda._sleep(cycles)
        t0 = time.perf_counter()
        sb_attn_varlen(q, k, v, cu, 130)
        t1 = time.perf_counter()
    finally:
        stop.set()
        thread.join()
    print(f"{where}: the call took {1e3 * (t1 - t0):.1f} ms", flush=True)
    assert where == "host" or t1 - t0 > 0.04
    assert t1 - t0 < 0.04 or sum(t0 < t < t1 for t in ticks) > (t1 - t0) / 0.02


def moved_by_a_byte(t):
    if t.dtype != torch.uint8:
        return t
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    buf[1:] = t
    return buf[1:]


def other_strides(t):
    return t.transpose(-1, -2).contiguous().transpose(-1, -2) if t.dim() >= 3 else t


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("how", ["host and back", "by a byte", "other strides", "left on the host", "checkpoint", "reentrant checkpoint"])
def test_saved_tensors_that_come_back_different(gpu_device, how, packed, dtype):
    H, L, D = 8, 200, 128
    shape = (H, L, D) if packed else (1, H, L, D)
    q, k, v, do = (torch.randn(shape, device=gpu_device).to(dtype) for _ in range(4))
    drem = torch.randn(shape[:-1], device=gpu_device).to(dtype)
    for t in (q, k, v):
        t.requires_grad_()
    cu = torch.tensor([70, L], dtype=torch.int32, device=gpu_device)

    def call(q, k, v):
        return sb_attn_varlen(q, k, v, cu, 130, zero_start=False) if packed else sb_attn(q, k, v)

    def grads(out):
        return torch.autograd.grad(out, [q, k, v], [do, drem])

    want = grads(call(q, k, v))
    if "checkpoint" in how:
        leaves = [t.detach().requires_grad_() for t in (q, k, v)]      # (a reentrant one needs .backward())
        torch.autograd.backward(checkpoint(call, *leaves, use_reentrant=how.startswith("re")), [do, drem])
        got = [t.grad for t in leaves]
    else:
        pack, unpack = {"host and back": (lambda t: t.cpu(), lambda t: t.to(gpu_device)), "by a byte": (lambda t: t, moved_by_a_byte),
                        "other strides": (lambda t: t, other_strides), "left on the host": (lambda t: t.cpu(), lambda t: t)}[how]
        with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
            out = call(q, k, v)
        if how == "left on the host":
            with pytest.raises(RuntimeError, match="GPU only"):
                grads(out)
            return
        got = grads(out)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("limit", [False, True])
@pytest.mark.parametrize("add_remainder", [False, True])
@pytest.mark.parametrize("save_carry", [False, True])
@pytest.mark.parametrize("H,L", [(32, 2048), (12, 2048)])
def test_what_is_held_between_the_passes(gpu_device, H, L, save_carry, add_remainder, limit):
    """save_carry=False holds no more than tile lists (32 bytes per 128 rows and per 64 keys), and with the remainder term a
    number per row; save_carry=True the products and, where a schedule is prepared, up to 13 bytes per row and head.  Either backward
    is the same with a workspace limit, under which nothing is prepared."""
    D, rows = 128, H * L
    q, k, v, do = (torch.randn(H, L, D, device=gpu_device).bfloat16() for _ in range(4))
    for t in (q, k, v):
        t.requires_grad_()
    cu = torch.tensor([L], dtype=torch.int32)
    options = dict(zero_start=False, add_remainder=add_remainder, save_carry=save_carry)
    want = torch.autograd.grad(sb_attn_varlen(q, k, v, cu, L, **options)[0], [q, k, v], do)
    saved = []

    def note(t):
        saved.append(t.nbytes)
        return t

    try:
        if limit:
            _native.set_backward_workspace_limit(1 << 40)
        with torch.autograd.graph.saved_tensors_hooks(note, lambda t: t):
            o, rem = sb_attn_varlen(q, k, v, cu, L, **options)
        held = sum(saved) - 3 * q.nbytes
        got = torch.autograd.grad(o, [q, k, v], do)
    finally:
        _native.set_backward_workspace_limit(None)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    lists = 4096 + 32 * (L // 128 + L // 64 + 2)
    products = 4 * H * _native.plan_host(cu, False, L).carry_slots
    allowed = lists + (products + (4 if limit else 13) * rows if save_carry else 4 * rows * add_remainder)
    print(f"held {held} bytes, allowed {allowed}", flush=True)
    assert held <= allowed + 2048


def test_anomaly_detection(gpu_device):
    """The node's forward runs without the interpreter's lock; anomaly detection records a Python traceback there."""
    q, k, v = (torch.randn(2, 100, 64, device=gpu_device).bfloat16().requires_grad_() for _ in range(3))
    cu = torch.tensor([100], dtype=torch.int32)
    want = torch.autograd.grad(sb_attn_varlen(q, k, v, cu, 100, zero_start=False)[0].sum(), [q, k, v])
    with torch.autograd.set_detect_anomaly(True):
        got = torch.autograd.grad(sb_attn_varlen(q, k, v, cu, 100, zero_start=False)[0].sum(), [q, k, v])
    assert all(torch.equal(a, b) for a, b in zip(got, want))
