"""Persistent recurrent launches on several streams of one process.

The workgroups of a persistent launch wait for each other, one per CU, so two launches that
together exceed the chip's CUs must not run side by side.  The library orders them; launches
that fit side by side stay independent.
"""

import threading
import time

import pytest
import torch

import prlstm_amd
from prlstm_amd import _lib
from prlstm_amd.graph import GraphedTrainStep

pytestmark = pytest.mark.gpu


def _module(dev, D, H, seed=0):
    torch.manual_seed(seed)
    m = prlstm_amd.HeadStartLSTM(D, H).to(dev)
    with torch.no_grad():
        m.a.fill_(0.3)
    return m


def _sleep_cycles(seconds):
    t = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
    n = 1 << 20
    while True:
        t[0].record()
        torch.cuda._sleep(n)
        t[1].record()
        torch.cuda.synchronize()
        ms = t[0].elapsed_time(t[1])
        if ms > 5.0:
            return int(n * seconds * 1e3 / ms)
        n *= 4


@pytest.mark.parametrize("B,H,ordered", [(4, 1024, True),   # 256 workgroups
                                         (40, 512, True),   # 256, two launches
                                         (4, 64, False)])   # 32: 64 fit side by side
@pytest.mark.parametrize("graphed", [False, True])
def test_calls_that_do_not_fit_together_are_ordered(dev, B, H, ordered, graphed):
    """A call queued behind a sleeping stream keeps a later call of another stream waiting when
    the two would not fit, and only then."""
    T, D, lib = 20, 16, _lib.load()
    print(f"two streams B={B} H={H} graphed={graphed}", flush=True)
    m, x = _module(dev, D, H), torch.randn(T, B, D, device=dev)
    if graphed:
        step = GraphedTrainStep(m, x)
        run = step.step
    else:
        def run():
            with torch.no_grad():
                return m(x)[0]
    lib.hsl_launched_workgroups(1)
    want = run().clone()
    assert graphed or lib.hsl_launched_workgroups(0) == (256 if ordered else 32)
    cycles = _sleep_cycles(0.4)
    first = torch.cuda.Stream()
    others = [torch.cuda.Stream() for _ in range(6)]  # some share a hardware queue with the first
    torch.cuda.synchronize()
    slept, ends, free, outs = torch.cuda.Event(), [], [], []
    with torch.cuda.stream(first):
        torch.cuda._sleep(cycles)
        slept.record()
        outs.append(run())
    for s in others:
        with torch.cuda.stream(s):
            free.append(torch.cuda.Event())
            x.sum()
            free[-1].record()
            outs.append(run())
            ends.append(torch.cuda.Event())
            ends[-1].record()
    time.sleep(0.1)
    done, ran, asleep = [e.query() for e in ends], [e.query() for e in free], not slept.query()
    torch.cuda.synchronize()
    assert asleep and any(ran)  # other streams ran while the first slept
    assert not any(done) if ordered else any(done)
    for o in outs:
        assert torch.equal(o, want)
    prlstm_amd.check_errors()


def test_two_threads_on_two_streams(dev):
    """Training steps of two threads, each on its own stream and each of launches as wide as the
    chip, give what they give alone, with no wait timed out."""
    shapes = [(24, 8, 32, 700), (24, 48, 32, 512)]  # the wide kernels; two launches each way
    mods = [_module(dev, D, H, i) for i, (_, _, D, H) in enumerate(shapes)]
    xs = [torch.randn(T, B, D, device=dev) for T, B, D, _ in shapes]

    def step(i):
        m = mods[i]
        m.zero_grad(set_to_none=True)
        out = m(xs[i])[0]
        out.sum().backward()
        return [out.detach()] + [p.grad for p in m.parameters()]

    want = [step(i) for i in range(2)]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for k in range(25):
                got = step(i)
                torch.cuda.current_stream().synchronize()
                if not all(torch.equal(a, b) for a, b in zip(got, want[i])):
                    bad.append((i, k))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    prlstm_amd.check_errors()
    assert not bad, bad


def test_replay_order_is_one_at_a_time(dev):
    lib = _lib.load()
    s = _lib.stream_of(dev)
    assert lib.hsl_replay_end() == 1 and b"no hsl_replay_begin" in lib.hsl_last_error()
    assert lib.hsl_replay_begin(256, s) == 0
    assert lib.hsl_replay_begin(256, s) == 1 and b"not ended" in lib.hsl_last_error()
    m, x = _module(dev, 16, 64), torch.randn(5, 4, 16, device=dev)
    assert torch.isfinite(m(x)[0]).all()  # a call of the thread that holds the lock
    assert lib.hsl_replay_end() == 0
