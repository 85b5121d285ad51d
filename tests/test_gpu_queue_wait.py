"""mcclx_queue_wait: the host leaves on a word that the queue's end writes.  Results in device memory
have to be there for whatever comes next, and the queue has to count as idle for the calls that ask."""
import ctypes as C
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    from mccl_amd import _lib as L, kernels as K
    return L, K


@pytest.mark.parametrize("spin_us", [0, 1, 1000])
@pytest.mark.parametrize("numel", [1, 4097, 6_553_601])
def test_results_are_there_for_a_kernel_and_a_copy_on_other_streams(env, spin_us, numel):
    L, K = env
    q = K.ReduceQueue(0)
    try:
        side = torch.cuda.Stream()
        for rep in range(8):
            x = torch.full((numel,), float(rep + 1), device="cuda")
            y = torch.full((numel,), 0.5, device="cuda")
            torch.cuda.synchronize()
            L.check(L.lib().mcclx_reduce(q.handle, x.data_ptr(), y.data_ptr(), L.F32, numel, L.SUM))
            L.check(L.lib().mcclx_queue_wait(q.handle, spin_us))
            with torch.cuda.stream(side):
                doubled = x * 2
            assert x.cpu().eq(rep + 1.5).all()
            side.synchronize()
            assert doubled.cpu().eq(2 * rep + 3.0).all()
    finally:
        q.close()


def test_the_queue_counts_as_idle_afterwards_and_as_busy_behind_a_wait(env):
    """An ordered launch goes to the default stream where the queue is idle.  A queue that waits for
    another stream is not: what it is given runs behind that stream's work."""
    L, K = env
    q = K.ReduceQueue(0)
    side = torch.cuda.Stream()
    try:
        a = torch.ones(1_000_000, device="cuda")
        b = torch.ones(1_000_000, device="cuda")
        torch.cuda.synchronize()
        for _ in range(4):  # launches on the queue and on the default stream in turn
            L.check(L.lib().mcclx_reduce(q.handle, a.data_ptr(), b.data_ptr(), L.F32, a.numel(), L.SUM))
            q.wait_results()
            K.hip_accumulate_chunk(a, b, queue=q)
        torch.cuda.synchronize()
        q.drain()
        assert a.cpu().eq(9).all()
        x = torch.zeros(1_000_000, device="cuda")
        torch.cuda.synchronize()
        q.wait_results()
        with torch.cuda.stream(side):
            torch.cuda._sleep(20_000_000)
            x.fill_(3)
        q.wait_torch_stream(side)
        K.hip_accumulate_chunk(x, b, queue=q)  # 3 + 1, not 0 + 1
        torch.cuda.synchronize()
        assert x.cpu().eq(4).all()
    finally:
        q.close()


def test_waits_of_several_threads_on_one_queue(env):
    L, K = env
    q = K.ReduceQueue(0)
    ones = torch.ones(50_000, device="cuda")
    wrong = []

    def work(i):
        torch.cuda.set_device(0)
        x = torch.zeros(50_000, device="cuda")
        torch.cuda.current_stream().synchronize()
        for rep in range(200):
            L.check(L.lib().mcclx_reduce(q.handle, x.data_ptr(), ones.data_ptr(), L.F32, x.numel(), L.SUM))
            L.check(L.lib().mcclx_queue_wait(q.handle, 1000))
            if rep % 50 == 49 and not x.cpu().eq(rep + 1).all():
                wrong.append((i, rep))

    torch.cuda.synchronize()
    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    q.close()
    assert not wrong


def test_refused_while_recording_and_usable_after(env):
    L, K = env
    q = K.ReduceQueue(0)
    try:
        x = torch.ones(1000, device="cuda")
        torch.cuda.synchronize()
        q.graph_begin()
        L.check(L.lib().mcclx_scale(q.handle, x.data_ptr(), L.F32, 1000, 2.0, L.SCALE_VIEW))
        assert L.lib().mcclx_queue_wait(q.handle, 1000) == L.ERR_STATE
        g = q.graph_end()
        q.wait_results()
        assert x.cpu().eq(1).all()
        for rep in range(3):
            q.graph_launch(g)
            q.wait_results()
            assert x.cpu().eq(2.0 ** (rep + 1)).all()
        q.graph_destroy(g)
    finally:
        q.close()


def test_without_a_context(env):
    L, _ = env
    assert L.lib().mcclx_queue_wait(C.c_void_p(None), 1000) == L.ERR_STATE


@pytest.mark.parametrize("streams", [1, 2])
@pytest.mark.parametrize("drain_every", [0, 5])
def test_every_wait_holds_whether_or_not_the_stream_was_asked(env, streams, drain_every):
    """Waits for a stream that was busy are not preceded by a query for a while: in a run of them, with
    the host catching up in between or not, each orders the queue behind what the stream was given last."""
    _, K = env
    q = K.ReduceQueue(0)
    sides = [torch.cuda.Stream() for _ in range(streams)]
    n = 200_003
    xs = [torch.zeros(n, device="cuda") for _ in range(24)]
    seen = [torch.zeros(n, device="cuda") for _ in range(24)]
    torch.cuda.synchronize()
    try:
        for i, (x, y) in enumerate(zip(xs, seen)):
            side = sides[i % streams]
            with torch.cuda.stream(side):
                torch.cuda._sleep(200_000)
                x.fill_(i + 1)
            q.wait_torch_stream(side)
            q.copy(y.data_ptr(), x.data_ptr(), 4 * n)
            q.torch_stream_wait(side)   # the queue's newest operation is a kernel: not asked either
            with torch.cuda.stream(side):
                y.mul_(2)
            if drain_every and i % drain_every == drain_every - 1:
                q.wait_results()
        torch.cuda.synchronize()
        for i, y in enumerate(seen):
            assert y.cpu().eq(2 * (i + 1)).all(), i
    finally:
        q.close()
