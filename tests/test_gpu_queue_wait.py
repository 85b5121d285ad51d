"""mcclx_queue_wait: the host leaves on a word that the queue's end writes.  Results in device memory
have to be there for whatever comes next, and the queue has to count as idle for the calls that ask."""
import ctypes as C
import statistics
import threading
import time

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


def test_a_wait_for_an_idle_stream_does_not_stand_behind_a_staging_copy(env):
    """mcclx_stage_for_send holds the context's lock while 512 MB come off the device (10 ms): a wait for an
    idle stream on another thread needs nothing of what it guards."""
    L, K = env
    q = K.ReduceQueue(0)
    try:
        big = torch.ones(128 << 20, device="cuda")
        side = torch.cuda.Stream()
        torch.cuda.synchronize()
        host = C.c_void_p()
        stage = lambda: L.check(L.lib().mcclx_stage_for_send(q.handle, big.data_ptr(), 4 * big.numel(), C.byref(host)))
        stage()  # the pinned buffer is there from now on
        longest = []
        for _ in range(3):
            copying = threading.Thread(target=stage)
            started = time.perf_counter()
            copying.start()
            waits = [0.0]
            while copying.is_alive():
                t = time.perf_counter()
                q.wait_torch_stream(side)
                waits.append(time.perf_counter() - t)
                time.sleep(1e-4)
            longest.append(max(waits) / (time.perf_counter() - started))
            copying.join()
        assert min(longest) < 0.3, longest
    finally:
        q.close()


@pytest.mark.parametrize("what", ["allreduce", "reduce_scatter", "allgather"])
def test_a_synchronisation_behind_each_call_finds_a_signal_to_wait_for(env, what):
    """A device synchronisation behind a call takes as long in a run of such calls as behind one that
    stands alone: some 5.5 us, where one that has to put a marker on the queue first takes 11."""
    L, K = env
    from mccl_amd import harness as H
    K.hip_kernels_init(0)
    a, b = torch.ones(2, 4_000, device="cuda"), torch.ones(2, 8_000, device="cuda")
    short, long = list(a), list(b)
    call = {"allreduce": lambda: H.allreduce(short, "max"),
            "reduce_scatter": lambda: H.reduce_scatter_replay(short, long, "max"),
            "allgather": lambda: H.allgather_replay(long, short)}[what]

    def median_sync(pause):
        took = []
        for _ in range(100):
            if pause:
                time.sleep(pause)
            call()
            t = time.perf_counter()
            torch.cuda.synchronize()
            took.append(time.perf_counter() - t)
        return statistics.median(took[20:])

    alone = min(median_sync(1e-3) for _ in range(2))
    assert min(median_sync(0) for _ in range(3)) < 1.5 * alone


@pytest.mark.parametrize("gap_us", [0, 6, 10_000_000])
def test_results_hold_with_any_gap(env, gap_us):
    """An event behind every call, behind some and behind none."""
    L, K = env
    from mccl_amd import harness as H
    q = K.ReduceQueue(0)
    try:
        L.check(L.lib().mcclx_set_wait_gap(q.handle, gap_us))
        for n in (1_000, 100_001):
            a, b = torch.zeros(n, device="cuda"), torch.ones(n, device="cuda")
            for rep in range(20):
                b.fill_(1)
                H.allreduce_replay([a, b], "sum", L.ALGO_TREE, queue=q)
                if rep % 3 == 0:
                    torch.cuda.synchronize()
                K.hip_accumulate_chunk(a, b, queue=q)
                a.sub_(b)
            assert a.cpu().eq(20).all()
        assert L.lib().mcclx_set_wait_gap(C.c_void_p(None), 1) == L.ERR_STATE
    finally:
        q.close()


def test_making_a_queue_does_not_wait_for_the_default_stream(env):
    _, K = env
    K.ReduceQueue(0).close()  # what a process does once is done
    torch.cuda.synchronize()
    torch.cuda._sleep(400_000_000)
    busy = torch.cuda.Event()
    busy.record()
    q = K.ReduceQueue(0)
    still = not busy.query()
    torch.cuda.synchronize()
    q.close()
    assert still


@pytest.mark.parametrize("borrowed", [False, True])
@pytest.mark.parametrize("thread", ["the recording one", "another"])
def test_a_queue_made_and_one_closed_while_a_stream_records(env, thread, borrowed):
    """The memory that a queue sets up for its waits is allocated and given back in a way that a recording in
    the strictest mode survives, on the thread that records and on others."""
    L, K = env
    K.ReduceQueue(0).close()  # what a process does once is done
    x = torch.zeros(1000, device="cuda")
    side, other = torch.cuda.Stream(), torch.cuda.Stream()
    made, old = [], K.ReduceQueue(0)

    def make():
        torch.cuda.set_device(0)
        with torch.cuda.stream(other):
            made.append(K.ReduceQueue(0, on_torch_stream=borrowed))
            old.close()

    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=side):  # capture_error_mode="global"
        x.add_(1)
        if thread == "another":
            t = threading.Thread(target=make)
            t.start()
            t.join()
        else:
            make()
        x.mul_(2)
    want = 0.0
    q = made[0]
    try:
        for rep in range(3):
            g.replay()
            torch.cuda.synchronize()
            want = 2 * (want + 1)
            assert x.cpu().eq(want).all()
            y = torch.full((5_000,), float(rep), device="cuda")
            torch.cuda.synchronize()
            L.check(L.lib().mcclx_reduce(q.handle, y.data_ptr(), y.data_ptr(), L.F32, y.numel(), L.SUM))
            q.wait_results()
            assert y.cpu().eq(2.0 * rep).all()
    finally:
        q.close()


@pytest.mark.parametrize("world,dtype", [(2, "fp32"), (3, "bf16"), (4, "wire"), (5, "fp16"), (8, "fp32"), (8, "wire")])
def test_small_allreduces_that_tell_of_their_own_end(env, world, dtype):
    """Launches of few blocks write the word themselves, others have a wave behind them for it: in turn,
    on tensors that change, each call returns with its result in place for a copy to the host, a kernel on
    another stream and the next call."""
    L, K = env
    from mccl_amd import harness as H
    K.hip_kernels_init(0)
    dt = {"fp32": torch.float32, "wire": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}[dtype]
    side = torch.cuda.Stream()
    q = K._q(None)
    sizes = [1, world, 63, 255, 1_000, 4_097, 8_192 * world, 300_000, 16_385, 2_047, 70_001, 500, 32_768, 33_000]
    for op in ("sum", "max"):
        for rep in range(3):
            for n in sizes:
                ts = [((torch.arange(n, device="cuda") * (r + 2) + rep) % 9 - 4).to(dt) for r in range(world)]
                stack = torch.stack([t.float() for t in ts])
                want = stack.sum(0) if op == "sum" else stack.amax(0)
                told = q.marked_launch_count()
                H.allreduce_replay(ts, op, L.ALGO_BUTTERFLY if n >= world else L.ALGO_TREE, wire_bf16=dtype == "wire", mode=L.REPLAY_DIRECT)
                told = q.marked_launch_count() - told
                assert told == 1 if n <= 4_097 else told == 0 if n >= 70_001 else told <= 1, n
                with torch.cuda.stream(side):
                    doubled = [t.float() * 2 for t in ts]
                host = [t.cpu().float() for t in ts]
                side.synchronize()
                want = want.cpu()
                for r in range(world):
                    assert torch.equal(host[r], want), (op, n, r)
                    assert torch.equal(doubled[r].cpu(), 2 * want), (op, n, r)
    assert L.lib().mcclx_allreduce_replay_wait(C.c_void_p(None), None, 0, 1000) == L.ERR_STATE


def test_marked_calls_from_threads_on_queues_of_their_own_and_on_one(env):
    L, K = env
    from mccl_amd import harness as H
    shared = K.ReduceQueue(0)
    wrong = []

    def work(i):
        torch.cuda.set_device(0)
        q = shared if i % 2 else K.ReduceQueue(0)
        a = torch.zeros(3_000, device="cuda")
        b = torch.ones(3_000, device="cuda")
        torch.cuda.current_stream().synchronize()
        for rep in range(150):
            b.fill_(1)
            torch.cuda.current_stream().synchronize()
            H.allreduce_replay([a, b], "sum", L.ALGO_TREE, mode=L.REPLAY_DIRECT, queue=q)
            if rep % 30 == 29 and not (a.cpu().eq(rep + 1).all() and b.cpu().eq(rep + 1).all()):
                wrong.append((i, rep))
        if q is not shared:
            q.close()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    shared.close()
    assert not wrong
