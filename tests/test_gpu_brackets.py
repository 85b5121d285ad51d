"""Folds between "the queue waits for torch's stream" and "torch's stream waits for the queue".  What comes
behind what, and what does not: each test closes several such brackets at once, opens the next one, then goes
on in every way there is, behind a producer that is still running."""
import time

import pytest
import torch

from mccl_amd import _lib as L
from mccl_amd import kernels as K

pytestmark = pytest.mark.gpu

N = 3_000_001


def scale(q, x, out, factor=0.5):
    plan = K.make_plan(L.F32, 2, scale_mode=L.SCALE_VIEW, scale=factor)
    q.fold(plan, [K.make_seg(out.data_ptr(), 0, [x.data_ptr(), x.data_ptr()], x.numel())])


def joined_queue(n=N, brackets=12):
    """A queue whose brackets have been closed at once, and its next one opened behind a running producer."""
    q = K.ReduceQueue(0)
    x, out = torch.zeros(n, device="cuda"), torch.zeros(n, device="cuda")
    torch.cuda.synchronize()
    scale(q, x, out)
    q.drain()
    for i in range(brackets):
        x.fill_(i + 1)
        q.wait_torch_stream()
        scale(q, x, out)
        q.torch_stream_wait()
        out.add_(1)
        if i in (2, brackets - 1):
            assert bool((out == i + 2).all())
    away = q.away_launch_count()
    torch.cuda._sleep(1_000_000)
    x.fill_(64)
    q.wait_torch_stream()
    return q, x, out, away


@pytest.mark.parametrize("n", [5, 32 * 256 * 4, N])
@pytest.mark.parametrize("end", ["closed", "drain", "wait", "ticket", "other_stream", "copy", "exposed", "graph", "ordered", "left_open",
                                 "two_folds", "another_producer", "table"])
def test_every_way_to_go_on(n, end):
    q, x, out, away = joined_queue(n)
    other = torch.cuda.Stream()
    got = torch.zeros_like(out)
    want = 64.0
    if end == "table":  # more segments than travel by value: through the queue
        plan = K.make_plan(L.F32, 2, scale_mode=L.SCALE_VIEW, scale=0.5)
        step = -(-n // 40)
        q.fold(plan, [K.make_seg(out.data_ptr() + 4 * i, 0, [x.data_ptr() + 4 * i] * 2, min(step, n - i)) for i in range(0, n, step)])
    elif end != "left_open":
        scale(q, x, out)
        assert q.away_launch_count() == away
    if end in ("closed", "table"):
        q.torch_stream_wait()
        got.copy_(out)
    elif end == "two_folds":
        scale(q, out, out, 1.0)
        q.torch_stream_wait()
        got.copy_(out)
        want = 128.0
    elif end == "drain":
        q.drain()
        with torch.cuda.stream(other):
            got.copy_(out)
    elif end == "wait":
        q.wait_results()
        with torch.cuda.stream(other):
            got.copy_(out)
    elif end == "ticket":
        q.wait(q.record())
        with torch.cuda.stream(other):
            got.copy_(out)
    elif end == "other_stream":
        q.torch_stream_wait(other)
        with torch.cuda.stream(other):
            got.copy_(out)
    elif end == "copy":
        q.copy(got.data_ptr(), out.data_ptr(), 4 * n)
        q.drain()
    elif end == "exposed":
        with torch.cuda.stream(torch.cuda.ExternalStream(q.stream)):
            got.copy_(out)
        scale(q, x, out)
    elif end == "graph":
        q.graph_begin()
        q.copy(got.data_ptr(), out.data_ptr(), 4 * n)
        g = q.graph_end()
        for _ in range(3):
            q.graph_launch(g)
            q.drain()
        q.graph_destroy(g)
    elif end == "ordered":
        K.hip_scale_inplace(out, 2.0, queue=q)
        q.torch_stream_wait(other)
        with torch.cuda.stream(other):
            got.copy_(out)
        want = 128.0
    elif end == "left_open":        # the queue's next operation is behind the producer all the same
        q.copy(got.data_ptr(), x.data_ptr(), 4 * n)
        q.torch_stream_wait(other)
        with torch.cuda.stream(other):
            got.add_(0)
    elif end == "another_producer":
        with torch.cuda.stream(other):
            torch.cuda._sleep(1_000_000)
            got.fill_(3)
        q.wait_torch_stream(other)
        plan = K.make_plan(L.F32, 2)
        q.fold(plan, [K.make_seg(got.data_ptr(), 0, [out.data_ptr(), got.data_ptr()], n)])
        q.drain()
        want = 67.0
    torch.cuda.synchronize()
    assert bool((got == want).all())
    q.close()


def test_the_queues_later_work_is_behind_a_closed_bracket():
    for consumer in range(3):
        got = torch.zeros(N, device="cuda")
        q, x, out, _ = joined_queue()
        scale(q, x, out)
        q.torch_stream_wait()
        if consumer == 0:
            q.copy(got.data_ptr(), out.data_ptr(), 4 * N)
        elif consumer == 1:
            plan = K.make_plan(L.F32, 1)
            q.fold(plan, [K.make_seg(got.data_ptr(), 0, [out.data_ptr()], N)])
        else:
            side = torch.cuda.Stream()
            q.torch_stream_wait(side)
            with torch.cuda.stream(side):
                got.copy_(out)
        q.drain()
        torch.cuda.synchronize()
        assert bool((got == 64.0).all()), consumer
        q.close()


def test_work_put_between_a_fold_and_the_second_ordering_runs_beside_it():
    """A caller whose brackets stay open while they go on has their folds on the queue: the host, waiting
    for the queue, does not wait for what the default stream has been given since."""
    q = K.ReduceQueue(0)
    x, out = torch.ones(N, device="cuda"), torch.zeros(N, device="cuda")
    torch.cuda.synchronize()
    for i in range(16):
        q.wait_torch_stream()
        scale(q, x, out)
        time.sleep(100e-6)
        q.torch_stream_wait()
    torch.cuda.synchronize()
    assert q.away_launch_count() == 0
    q.wait_torch_stream()
    scale(q, x, out)
    ticket = q.record()  # (a drain's own marker may share a hardware queue with what follows)
    torch.cuda._sleep(100_000_000)
    t = time.perf_counter()
    q.wait(ticket)
    waited = time.perf_counter() - t
    torch.cuda.synchronize()
    assert waited < (time.perf_counter() - t) / 2
    q.close()


def test_brackets_of_several_threads_on_one_queue():
    import threading
    q = K.ReduceQueue(0)
    wrong = []

    def work(i):
        torch.cuda.set_device(0)
        n = 40_001 + i
        x, out = torch.zeros(n, device="cuda"), torch.zeros(n, device="cuda")
        for rep in range(150):
            torch.cuda._sleep(20_000 * (rep % 3))
            x.fill_(rep + i)
            q.wait_torch_stream()
            scale(q, x, out)
            q.torch_stream_wait()
            if rep % 10 == 9 and not bool((out == rep + i).all()):
                wrong.append((i, rep))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    q.drain()
    q.close()
    assert not wrong


def test_a_wait_said_by_another_caller_survives_the_end_of_the_first_ones_bracket():
    """wait, fold, [another caller's work and wait], end of the first bracket, the other's fold: it has to
    be behind the other's work."""
    for end_first in (True, False):
        q, x, out, away = joined_queue()
        y, res = torch.zeros(N, device="cuda"), torch.zeros(N, device="cuda")
        scale(q, x, out)
        torch.cuda._sleep(2_000_000)
        y.fill_(7)
        q.wait_torch_stream()
        if end_first:
            q.torch_stream_wait()
        scale(q, y, res)
        q.torch_stream_wait()
        torch.cuda.synchronize()
        assert bool((out == 64.0).all()) and bool((res == 7.0).all()), end_first
        q.close()


LONG = 100_000_000  # cycles of a kernel that runs for some 50 ms


def early(attempt, tries=8):
    """Does `attempt` come back well before the long kernel that it has put on the default stream ends?  Two streams
    may share a hardware queue, where one waits for the other whatever the library does: one try of several."""
    for _ in range(tries):
        t = time.perf_counter()
        attempt()
        waited = time.perf_counter() - t
        torch.cuda.synchronize()
        if waited < (time.perf_counter() - t) / 2:
            return True
    return False


@pytest.mark.parametrize("what", ["fold", "copy", "nothing"])
def test_the_first_ordering_covers_what_was_enqueued_before_it_and_no_more(what):
    """However quickly the brackets before it were closed: work that the default stream is given behind the first
    ordering, in front of the fold or another operation of the queue, runs beside it."""
    def attempt():
        q, x, out, _ = joined_queue()
        torch.cuda._sleep(LONG)
        if what == "fold":
            scale(q, x, out)
        elif what == "copy":
            q.copy(out.data_ptr(), x.data_ptr(), 4 * N)
        if what == "nothing":
            q.drain()
        else:
            q.wait(q.record())
        made.append((q, x, out))

    made = []
    assert early(attempt)
    for q, x, out in made:
        assert bool((out == {"fold": 64.0, "copy": 64.0, "nothing": 13.0}[what]).all())
        q.close()


def test_folds_between_orderings_stay_on_the_queue():
    """Whatever follows the fold, and however soon the bracket is closed: a quickly issued kernel in between, two
    queues with their brackets interleaved, a collective that waits for its own launches."""
    from mccl_amd import harness as H
    a, b = K.ReduceQueue(0), K.ReduceQueue(0)
    x, y = torch.ones(N, device="cuda"), torch.ones(N, device="cuda")
    out, res, other = torch.zeros_like(x), torch.zeros_like(x), torch.zeros(4_097, device="cuda")
    ts = [torch.full((100_003,), float(i), device="cuda") for i in range(3)]
    torch.cuda.synchronize()
    for i in range(16):
        a.wait_torch_stream()
        b.wait_torch_stream()
        scale(a, x, out)
        scale(b, y, res)
        if i % 2:
            other.add_(1)
        a.torch_stream_wait()
        b.torch_stream_wait()
    a.wait_torch_stream()
    H.allreduce_replay(ts, "sum", L.ALGO_BUTTERFLY, wire_bf16=True, mode=L.REPLAY_FUSED, queue=a)
    torch.cuda.synchronize()
    assert a.away_launch_count() == 0 and b.away_launch_count() == 0
    assert bool((out == 1).all()) and bool((res == 1).all()) and bool((other == 8).all())
    assert all(bool((t == 3).all()) for t in ts)
    a.close()
    b.close()
