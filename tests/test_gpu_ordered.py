"""The tensor variants' ordering: one launch behind everything on torch's stream and on the reduce
queue, in front of what either gets next -- wherever the launch itself runs (on torch's stream where
the queue is idle, on the queue otherwise).  Every consumer reads a result without further waits of
its own, behind a producer that is still running when the call is made."""
import pytest
import torch

from mccl_amd import kernels as K

pytestmark = pytest.mark.gpu

N = 8_000_003  # some 10 us of device time a launch, several times what a call takes the host


def _produce(n=N):
    """(dst, src) of small whole numbers, the last of a chain of passes still under way."""
    base = torch.arange(n, device="cuda", dtype=torch.float32).remainder_(64)
    dst, src = base.clone(), torch.zeros_like(base)
    for _ in range(40):
        src.add_(1)
    return base, dst, src


def _streams():
    return [("default", torch.cuda.default_stream()), ("side", torch.cuda.Stream())]


@pytest.mark.parametrize("which", [0, 1])
@pytest.mark.parametrize("consumer", ["torch", "queue", "other_stream", "ticket", "drain", "other_caller"])
@pytest.mark.parametrize("queue_state", ["idle", "busy", "exposed"])
def test_result_is_seen_by_every_consumer(which, consumer, queue_state):
    q = K.ReduceQueue(0)
    if queue_state == "exposed":
        assert q.stream
    st = _streams()[which][1]
    torch.cuda.synchronize()
    with torch.cuda.stream(st):
        base, dst, src = _produce()
        got = torch.zeros_like(dst)
        filler = torch.zeros(64_000_000, device="cuda", dtype=torch.float32)
        if queue_state == "busy":
            for _ in range(4):
                q.copy(filler.data_ptr(), filler.data_ptr() + 128_000_000, 128_000_000)
        for _ in range(3):
            K.hip_reduce_op(dst, src, "sum", queue=q)
        want = base + 3 * 40
        if consumer == "torch":
            got.copy_(dst)
        elif consumer == "queue":          # a raw launch on the queue, then the host waits for the queue
            q.copy(got.data_ptr(), dst.data_ptr(), 4 * N)
            q.drain()
        elif consumer == "other_stream":
            other = torch.cuda.Stream()
            q.torch_stream_wait(other)
            with torch.cuda.stream(other):
                got.copy_(dst)
            other.synchronize()
        elif consumer == "ticket":
            q.wait(q.record())
            other = torch.cuda.Stream()
            with torch.cuda.stream(other):
                got.copy_(dst)
            other.synchronize()
        elif consumer == "drain":
            q.drain()
            other = torch.cuda.Stream()
            with torch.cuda.stream(other):
                got.copy_(dst)
            other.synchronize()
        else:                              # the same queue called from another stream: behind the first caller's launches
            other = torch.cuda.Stream()
            with torch.cuda.stream(other):
                K.hip_reduce_op(got, dst, "sum", queue=q)
            other.synchronize()
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    q.close()


@pytest.mark.parametrize("n", [1, 63, 4_097, 2_000_003])
def test_codec_round_trips_on_an_idle_and_a_busy_queue(n):
    q = K.ReduceQueue(0)
    x = torch.randn(n, device="cuda")
    want = x.to(torch.bfloat16)
    big = torch.zeros(32_000_000, device="cuda")
    torch.cuda.synchronize()
    for busy in (False, True, False):
        if busy:
            q.copy(big.data_ptr(), big.data_ptr() + 64_000_000, 64_000_000)
        w = K.encode_bf16(x, queue=q)
        back = K.decode_bf16(w, queue=q)
        assert torch.equal(w.view(torch.int16), want.view(torch.int16))
        assert torch.equal(back, want.float())
        q.drain()
    K.hip_scale_inplace(back, 0.5, queue=q)
    assert torch.equal(back, want.float() * 0.5)
    q.close()


def test_errors_are_the_same_on_either_route():
    q = K.ReduceQueue(0)
    a = torch.zeros(8, device="cuda")
    for _ in range(2):
        with pytest.raises(K.MCCLError, match="Unsupported ReduceOp"):
            K.hip_reduce_op(a, a, 9, queue=q)
        assert q.stream  # from here on through the queue
    q.graph_begin()
    with pytest.raises(K.MCCLError, match="not allowed between graph_begin and graph_end"):
        K.hip_reduce_op(a, a, "sum", queue=q)
    q.copy(a.data_ptr(), a.data_ptr() + 16, 16)
    q.graph_destroy(q.graph_end())
    q.close()


def test_a_borrowed_streams_own_later_work_is_behind_the_launch():
    """A queue on a stream of the caller's: what they enqueue there themselves comes after the call."""
    mine, other = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(mine):
        q = K.ReduceQueue(0, on_torch_stream=True)
        got = torch.zeros(N, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.stream(other):
        base, dst, src = _produce()
        K.hip_reduce_op(dst, src, "sum", queue=q)
    with torch.cuda.stream(mine):
        got.copy_(dst)
    torch.cuda.synchronize()
    assert torch.equal(got, base + 40)
    q.close()


def test_callers_on_alternating_streams_come_one_after_the_other():
    """Launches of one queue keep their order whichever streams they are called from."""
    q = K.ReduceQueue(0)
    streams = [torch.cuda.default_stream(), torch.cuda.Stream(), torch.cuda.Stream()]
    dst = torch.zeros(N, device="cuda")
    one = torch.ones(N, device="cuda")
    torch.cuda.synchronize()
    for i in range(24):
        with torch.cuda.stream(streams[i % 3]):
            K.hip_reduce_op(dst, one, "sum", queue=q)
            K.hip_scale_inplace(dst, 2.0, queue=q)
            if i % 4 == 3:
                K.hip_scale_inplace(dst, 2.0 ** -4, queue=q)
    q.drain()
    want = 0.0
    for i in range(24):
        want = (want + 1) * 2 * (2.0 ** -4 if i % 4 == 3 else 1)
    assert torch.equal(dst, torch.full_like(dst, want))
    q.close()


@pytest.mark.parametrize("which", [0, 1])
def test_a_recording_stream_may_wait_for_an_idle_queue(which):
    """The wait has nothing to record where the queue's work is done -- also when the newest launch
    ran in the queue's place, on a stream of which, or beside which, the caller now records."""
    q = K.ReduceQueue(0)
    side = torch.cuda.Stream()
    dst, src = torch.zeros(4_097, device="cuda"), torch.ones(4_097, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.default_stream() if which == 0 else side):
        K.hip_reduce_op(dst, src, "sum", queue=q)
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=side, capture_error_mode="relaxed"):
            q.torch_stream_wait()
            dst.add_(src)
            q.drain()
        for rep in range(3):
            g.replay()
            side.synchronize()
            assert torch.equal(dst, torch.full_like(dst, 2.0 + rep)), rep
        K.hip_reduce_op(dst, src, "sum", queue=q)
        assert torch.equal(dst, torch.full_like(dst, 5.0))
    q.close()


# Small launches in a row, up to one packet a lane in 32 blocks of 256 lanes and beyond.
@pytest.mark.parametrize("dtype,most", [(torch.float32, 32 * 256 * 4), (torch.bfloat16, 32 * 256 * 8), (torch.float16, 32 * 256 * 8)])
@pytest.mark.parametrize("consumer", ["torch", "queue", "other_stream", "ticket", "drain", "wait", "exposed"])
@pytest.mark.parametrize("behind", ["nothing", "a_running_kernel"])
def test_small_launches_in_a_row(dtype, most, consumer, behind):
    q = K.ReduceQueue(0)
    other = torch.cuda.Stream()
    for n in (1, 4_097, most - 1, most, most + 1, 4 * most + 3):
        dst = torch.full((n,), 3.0, device="cuda", dtype=dtype)
        src = torch.full((n,), 2.0, device="cuda", dtype=dtype)
        got = torch.zeros_like(dst)
        torch.cuda.synchronize()
        if behind == "a_running_kernel":
            torch.cuda._sleep(300_000)
        src.add_(1)
        K.hip_reduce_op(dst, src, "sum", queue=q)
        K.hip_scale_inplace(dst, 0.5, queue=q)
        if consumer == "torch":
            got.copy_(dst)
        elif consumer == "queue":
            q.copy(got.data_ptr(), dst.data_ptr(), n * dst.element_size())
            q.drain()
        elif consumer == "other_stream":
            q.torch_stream_wait(other)
            with torch.cuda.stream(other):
                got.copy_(dst)
            other.synchronize()
        else:
            if consumer == "ticket":
                q.wait(q.record())
            elif consumer == "drain":
                q.drain()
            elif consumer == "wait":
                q.wait_results()
            else:
                torch.cuda.ExternalStream(q.stream).synchronize()
            with torch.cuda.stream(other):
                got.copy_(dst)
            other.synchronize()
        torch.cuda.synchronize()
        assert bool((got == 3.0).all()), n
    assert q.away_launch_count() > 0  # (the queue was idle, and its stream not handed out, at the first of the sizes)
    q.close()


def test_codec_and_scaling_at_the_edges_of_blocks():
    q = K.ReduceQueue(0)
    for blocks in (1, 2, 31, 32, 33):
        for extra in (-1, 0, 1):
            n = blocks * 256 * 4 + extra
            x = torch.randn(n, device="cuda")
            y = x.clone()
            w = K.encode_bf16(x, queue=q)
            back = K.decode_bf16(w, queue=q)
            K.hip_accumulate_and_scale(y, x, 0.25, queue=q)
            assert torch.equal(w.view(torch.int16), x.to(torch.bfloat16).view(torch.int16))
            assert torch.equal(back, w.float()) and torch.equal(y, (x + x) * 0.25)
    q.close()


def test_a_host_that_waits_for_a_small_launch_does_not_wait_for_what_came_behind_it():
    import time
    q = K.ReduceQueue(0)
    dst, src = torch.zeros(4_097, device="cuda"), torch.ones(4_097, device="cuda")
    K.hip_reduce_op(dst, src, "sum", queue=q)
    torch.cuda.synchronize()
    for _ in range(3):
        K.hip_reduce_op(dst, src, "sum", queue=q)
    torch.cuda._sleep(100_000_000)  # some 50 ms
    t = time.perf_counter()
    q.drain()
    waited = time.perf_counter() - t
    t = time.perf_counter()
    torch.cuda.synchronize()
    slept = time.perf_counter() - t
    assert waited < slept / 2, (waited, slept)
    assert bool((dst == 4.0).all())
    q.close()


@pytest.mark.parametrize("who", ["drain", "wait", "ticket", "queue", "other_stream"])
def test_who_asks_for_a_launch_that_is_still_running_waits_for_it_and_no_more(who):
    """Behind small calls in a row, the newest of which are still to run, the caller puts a long kernel on their stream:
    the host, the queue and other streams get the results long before that kernel ends.  (Two streams may share a
    hardware queue, where one waits for the other whatever the library does: one try of several.)"""
    import time
    on_time = False
    for _ in range(8):
        q, side = K.ReduceQueue(0), torch.cuda.Stream()
        dst, src, got = torch.zeros(4_097, device="cuda"), torch.ones(4_097, device="cuda"), torch.zeros(4_097, device="cuda")
        host = torch.zeros(4_097, pin_memory=True)
        K.hip_reduce_op(dst, src, "sum", queue=q)
        torch.cuda.synchronize()
        torch.cuda._sleep(8_000_000)  # some 4 ms
        for _ in range(8):
            K.hip_reduce_op(dst, src, "sum", queue=q)
        torch.cuda._sleep(100_000_000)  # some 50 ms
        t = time.perf_counter()
        if who == "drain":
            q.drain()
        elif who == "wait":
            q.wait_results()
        elif who == "ticket":
            q.wait(q.record())
        elif who == "queue":
            q.copy(got.data_ptr(), dst.data_ptr(), 4 * 4_097)
            q.wait(q.record())
        else:
            q.torch_stream_wait(side)
            with torch.cuda.stream(side):
                got.copy_(dst)
                host.copy_(dst, non_blocking=True)
            side.synchronize()
            assert bool((host == 9.0).all())
        waited = time.perf_counter() - t
        torch.cuda.synchronize()
        whole = time.perf_counter() - t
        assert bool((dst == 9.0).all()) and (who not in ("queue", "other_stream") or bool((got == 9.0).all()))
        q.close()
        on_time = on_time or waited < whole / 2
        if on_time:
            break
    assert on_time


def test_a_queue_that_the_default_stream_waits_for_counts_as_idle():
    """The launch is behind the queue's work on that stream already; what the queue is given next is behind the launch."""
    from mccl_amd import _lib as L
    q = K.ReduceQueue(0)
    x, out, got = torch.zeros(N, device="cuda"), torch.zeros(N, device="cuda"), torch.zeros(N, device="cuda")
    torch.cuda.synchronize()
    plan = K.make_plan(L.F32, 2, scale_mode=L.SCALE_VIEW, scale=0.5)
    for i in range(1, 9):
        torch.cuda._sleep(300_000)
        x.fill_(i)
        q.wait_torch_stream()
        q.fold(plan, [K.make_seg(out.data_ptr(), 0, [x.data_ptr(), x.data_ptr()], N)])
        q.torch_stream_wait()
        K.hip_scale_inplace(out, 2.0, queue=q)
        assert q.away_launch_count() == i
        q.copy(got.data_ptr(), out.data_ptr(), 4 * N)
        if i % 2:
            K.hip_scale_inplace(out, 4.0, queue=q)   # the queue's copy is still to run: through the queue
            assert q.away_launch_count() == i
        q.drain()
        torch.cuda.synchronize()
        assert bool((got == 2 * i).all()) and bool((out == (8 * i if i % 2 else 2 * i)).all()), i
    q.close()
