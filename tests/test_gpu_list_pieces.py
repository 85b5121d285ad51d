"""Lists of many large enough messages go out in pieces of 2048, one run of launches each: results
and the order of entries that share tensors are those of the whole list."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    from mccl_amd import _lib as L, harness as H, kernels as K
    K.hip_kernels_init(0)
    return L, H, K


def _average(ts):
    """The tree of two or three ranks on the host: ranks 0 and 1, then rank 2, then the factor, each rounded."""
    acc = ts[0] + ts[1]
    if len(ts) == 3:
        acc = acc + ts[2]
    return acc * torch.tensor(1.0 / len(ts), dtype=torch.float32)


@pytest.mark.parametrize("messages,numel,world,launches", [
    (2_047, 4_001, 2, 1),     # just below a piece
    (2_048, 4_001, 2, 1),     # one piece, whole
    (2_049, 4_001, 2, 2),     # and one entry left over
    (5_000, 2_731, 3, 3),
    (5_000, 64, 3, 1),        # too little to keep the device busy: one launch
])
def test_pieces_of_a_list(env, messages, numel, world, launches):
    L, H, K = env
    g = torch.Generator(device="cuda").manual_seed(5)
    flat = [torch.randn(messages * numel, generator=g, device="cuda") for _ in range(world)]
    groups = [list(ts) for ts in zip(*[f.split(numel) for f in flat])]
    host = [f.cpu().split(numel) for f in flat]
    want = [_average(ts) for ts in zip(*host)]
    q = K._q(None)
    before = q.launch_count()
    H.allreduce_replay_many(groups, "avg", L.ALGO_TREE)
    assert q.launch_count() - before == launches
    want = torch.cat(want)
    for f in flat:
        assert torch.equal(f.cpu().view(torch.int32), want.view(torch.int32))


def test_an_entry_named_in_two_pieces_and_twice_in_one(env):
    L, H, K = env
    n, messages, world = 5_000, 4_200, 2
    g = torch.Generator(device="cuda").manual_seed(6)
    ts = [[torch.randn(n, generator=g, device="cuda") for _ in range(world)] for _ in range(messages)]
    order = list(range(messages)) + [3, 2_700, 2_700]
    order.insert(2_500, 5)
    state = [[t.cpu() for t in pair] for pair in ts]
    for i in order:
        mean = _average(state[i])
        state[i] = [mean] * world
    H.allreduce_replay_many([ts[i] for i in order], "avg", L.ALGO_TREE)
    for pair, want in zip(ts, state):
        for t, w in zip(pair, want):
            assert torch.equal(t.cpu().view(torch.int32), w.view(torch.int32))


def test_more_table_launches_than_staging_slots_without_a_drain(env):
    """The staging ring's slots are taken again while earlier launches are still queued."""
    L, H, K = env
    q = K.ReduceQueue(0)
    try:
        n, m = 4_099, 300
        x = torch.zeros(m * n, device="cuda")
        y = torch.ones(m * n, device="cuda")
        torch.cuda.synchronize()
        plan = K.make_plan(L.F32, 2)
        for rep in range(12):
            lo = rep % 5  # another table each time
            segs = [K.make_seg(a, 0, [a, b], n) for a, b in
                    ((x.data_ptr() + 4 * n * i, y.data_ptr() + 4 * n * i) for i in range(lo, m))]
            q.fold(plan, segs)
        q.drain()
        counts = torch.tensor([sum(1 for rep in range(12) if i >= rep % 5) for i in range(m)], dtype=torch.float32)
        assert torch.equal(x.cpu().view(m, n), counts[:, None].expand(m, n))
        assert torch.equal(y, torch.ones_like(y))
    finally:
        q.close()


@pytest.mark.parametrize("layout", ["in_order", "reversed", "interleaved", "scattered"])
def test_entries_of_any_layout_and_one_that_overlaps(env, layout):
    """What a run has touched is kept as intervals that usually just grow: lists whose tensors lie the other
    way round, rank by rank in one buffer, or anywhere, and an entry that shares half of an earlier one's tensor."""
    L, H, _ = env
    n, messages, world = 1_000, 700, 3
    g = torch.Generator(device="cuda").manual_seed(7)
    buf = torch.randint(-50, 50, (messages * world * n,), generator=g, device="cuda").float()
    at = {"in_order": lambda i, r: r * messages + i, "reversed": lambda i, r: r * messages + messages - 1 - i,
          "interleaved": lambda i, r: i * world + r, "scattered": lambda i, r: (i * 389 + 7) % messages * world + r}[layout]
    starts = [[at(i, r) * n for r in range(world)] for i in range(messages)]
    starts.append([starts[400][0], starts[10][1] + n // 2, starts[20][2]])  # half of an earlier tensor, half of its neighbour
    host = buf.cpu()
    for s in starts:
        total = sum(host[a:a + n].clone() for a in s)
        for a in s:
            host[a:a + n] = total
    H.allreduce_replay_many([[buf[a:a + n] for a in s] for s in starts], "sum", L.ALGO_TREE)
    assert torch.equal(buf.cpu(), host)
