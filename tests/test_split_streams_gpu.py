"""Split calls on several streams: a stream whose queue is held up does not hold
up the split calls of three others (each stream has a workspace of its own), and
with more streams than workspaces every call still gets the result that it gets
alone.
"""
from __future__ import annotations

import time

import pytest

pytestmark = pytest.mark.gpu

# heads, M, N, d: batched split, split decode, batched split at 64 features, split decode
SHAPES = [(4, 300, 3000, 128), (8, 4, 6000, 128), (6, 200, 2500, 64), (5, 16, 3000, 72)]


def _calls(tm, count):
    """(call(stream), O, O of the call alone) of `count` split calls, each with its own tensors."""
    import torch

    made = []
    for i in range(count):
        heads, M, N, d = SHAPES[i % len(SHAPES)]
        gen = torch.Generator(device="cuda")
        gen.manual_seed(i)
        Q, K, V = (torch.randn(heads, r, d, generator=gen, device="cuda").half() for r in (M, N, N))
        O = torch.empty(heads, M, d, device="cuda")
        args = tm.BatchedArgs(Q=Q, K=K, V=V, O=O, heads=heads, M=M, N=N, d=d, score_scale=d ** -0.5)
        tm.check(tm.attention_batched(args))
        torch.cuda.synchronize()
        alone = O.clone()
        O.fill_(float("nan"))
        made.append((lambda stream, args=args: tm.check(tm.attention_batched(args, stream)), O, alone))
    torch.cuda.synchronize()
    return made


def _hold_ticks(seconds):
    """Ticks of torch.cuda._sleep that take about `seconds`."""
    import torch

    ticks = 1_000_000
    begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    torch.cuda._sleep(ticks)
    begin.record()
    torch.cuda._sleep(ticks)
    end.record()
    torch.cuda.synchronize()
    return int(ticks * seconds * 1e3 / max(begin.elapsed_time(end), 1e-3))


def _finished(events, seconds):
    """Which of the events are done within `seconds`."""
    limit = time.monotonic() + seconds
    while time.monotonic() < limit and not all(e.query() for e in events):
        time.sleep(0.002)
    return [e.query() for e in events]


def test_a_held_stream_holds_up_no_other(tm, cuda):
    import torch

    calls = _calls(tm, 4)
    ticks = _hold_ticks(1.0)
    held, others = torch.cuda.Stream(), [torch.cuda.Stream() for _ in range(8)]
    done = [torch.cuda.Event() for _ in others]
    # Streams that share a hardware queue with the held one wait for it by themselves.
    print("streams beside a held one", flush=True)
    with torch.cuda.stream(held):
        torch.cuda._sleep(ticks)
    for stream, event in zip(others, done):
        with torch.cuda.stream(stream):
            torch.zeros(1, device="cuda")
        event.record(stream)
    beside = [s for s, free in zip(others, _finished(done, 0.5)) if free][:3]
    torch.cuda.synchronize()
    assert beside, "no stream runs beside the held one"
    print(f"split calls on {len(beside)} streams beside a held one", flush=True)
    done = [torch.cuda.Event() for _ in range(len(beside) + 1)]
    with torch.cuda.stream(held):
        torch.cuda._sleep(ticks)
    for stream, event, (call, _, _) in zip([held] + beside, done, calls):
        call(stream)
        event.record(stream)
    finished = _finished(done[1:], 0.8)
    still_held = not done[0].query()
    torch.cuda.synchronize()
    assert all(finished) and still_held, (finished, still_held)
    for _, O, alone in calls[:len(done)]:
        assert torch.equal(O.view(torch.int32), alone.view(torch.int32))


def test_more_streams_than_workspaces(tm, cuda):
    import torch

    calls = _calls(tm, 8)
    streams = [torch.cuda.Stream() for _ in range(6)]
    torch.cuda.synchronize()
    print("split calls on six streams", flush=True)
    for round_ in range(6):
        for i, (call, _, _) in enumerate(calls):
            call(streams[(i + round_) % len(streams)])
        for stream in streams:  # a call's O is its own; the next round may run on another stream
            torch.cuda.current_stream().wait_stream(stream)
        for stream in streams:
            stream.wait_stream(torch.cuda.current_stream())
    torch.cuda.synchronize()
    for _, O, alone in calls:
        assert torch.equal(O.view(torch.int32), alone.view(torch.int32))
