"""The schedule a forward prepares for its backward, where the two do not simply follow one another: both captured in a graph and
replayed, a captured forward with eager backwards, and several threads with streams of their own.  Against the same calls
made eagerly, bit for bit."""
import threading

import pytest
import torch

from stickbreaking_attention import _native, sb_attn_varlen

pytestmark = pytest.mark.gpu

# (heads, head_dim, ends, dtype): the kernels that split the keys, the wide ones, the one-kernel backward, fp32
CASES = {"split": (3, 64, [200, 201, 700], torch.bfloat16), "wide": (100, 64, [513, 700], torch.bfloat16),
         "wide128": (100, 128, [513, 700], torch.float16), "chained": (8, 128, [2600, 2730], torch.bfloat16), "fp32": (3, 64, [100, 300], torch.float32)}


class Calls:
    """One call and its gradients on tensors that stay where they are."""

    def __init__(self, case, device, seed, save_carry=True):
        self.H, D, ends, dtype = CASES[case]
        self.ends, self.save_carry = ends, save_carry
        self.cu = torch.tensor(ends, dtype=torch.int32, device=device)
        shape = (self.H, ends[-1], D)
        self.q, self.k, self.v, self.do = (torch.empty(shape, device=device, dtype=dtype) for _ in range(4))
        self.drem = torch.empty(shape[:2], device=device, dtype=dtype)
        self.fill(seed)
        for t in (self.q, self.k, self.v):
            t.requires_grad_()

    def fill(self, seed):
        g = torch.Generator(device=self.q.device).manual_seed(seed)
        for t in (self.q, self.k, self.v, self.do, self.drem):      # (.data: a captured forward's backwards follow new values)
            t.data.copy_(torch.randn(t.shape, generator=g, device=t.device))

    def forward(self):
        return sb_attn_varlen(self.q, self.k, self.v, self.cu, max(self.ends), zero_start=False, save_carry=self.save_carry)

    def backward(self, out, **kw):
        return torch.autograd.grad(out, [self.q, self.k, self.v], [self.do, self.drem], **kw)

    def both(self):
        out = self.forward()
        return [t.detach() for t in out] + list(self.backward(out))


def captured(run):
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        run()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = run()
    return graph, out


@pytest.mark.parametrize("save_carry", [True, False])
@pytest.mark.parametrize("case", CASES)
def test_both_passes_in_a_graph(gpu_device, monkeypatch, case, save_carry):
    monkeypatch.setattr(_native, "DEBUG_CHECK", False)      # (its synchronisation cannot be captured)
    calls = Calls(case, gpu_device, 0, save_carry)
    graph, out = captured(calls.both)
    for seed in (1, 2, 3):
        calls.fill(seed)
        want = calls.both()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, want)), seed


@pytest.mark.parametrize("case", CASES)
def test_captured_forward_with_eager_backwards(gpu_device, monkeypatch, case):
    monkeypatch.setattr(_native, "DEBUG_CHECK", False)
    calls = Calls(case, gpu_device, 0)
    graph, out = captured(calls.forward)
    for seed in (1, 2, 3):      # the first backward may take the schedule as the replay left it, the others may not
        calls.fill(seed)
        want = calls.both()[2:]
        graph.replay()
        for _ in range(2):
            assert all(torch.equal(a, b) for a, b in zip(calls.backward(out, retain_graph=True), want)), seed


def test_threads_with_streams_of_their_own(gpu_device):
    work = [Calls(case, gpu_device, i) for i, case in enumerate(["split", "wide", "wide128", "fp32"])]
    want = [calls.both() for calls in work]
    torch.cuda.synchronize()
    wrong = []

    def run(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(10):
                got = work[i].both()
                torch.cuda.current_stream().synchronize()
                if not all(torch.equal(a, b) for a, b in zip(got, want[i])):
                    wrong.append(i)

    threads = [threading.Thread(target=run, args=(i,)) for i in range(len(work))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert wrong == []
