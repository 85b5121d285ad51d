"""Allreduce with the wire copies in pinned host memory: from some megabytes on the schedule is cut
into pieces whose folds and encodes share launches.  Same bits as the launches one by one in HBM."""
import ctypes as C

import pytest
import torch

from mccl_amd import _lib as L
from mccl_amd import harness as H
from mccl_amd import kernels as K

pytestmark = pytest.mark.gpu

ALGOS = {"ring": L.ALGO_RING, "butterfly": L.ALGO_BUTTERFLY}


def _pieces(world, numel, algo):
    """Pieces P with P^2 * 1.5 MB of what every rank sends: all chunks but its own, two bytes an element."""
    own = sum(c[1] for c in H.chunkize(numel, 4, world))
    nbytes = 2 * (world - 1) * own
    p = 1
    while (p + 1) ** 2 * 1_500_000 <= nbytes:
        p += 1
    return p


def _tensors(world, numel, seed=1):
    g = torch.Generator(device="cuda").manual_seed(seed)
    out = [torch.randn(numel, device="cuda", generator=g) for _ in range(world)]
    special = torch.tensor([float("inf"), float("-inf"), float("nan"), -0.0, 1e-40, 3.3e38], device="cuda")
    for r, t in enumerate(out):
        at = torch.arange(r, numel, 100_003, device="cuda")
        t[at] = special[at % 6]
    return out


def _pinned(q, world, numel, algo):
    r = L.Replay()
    r.world, r.algo, r.op, r.dtype, r.wire_bf16, r.mode, r.numel = world, algo, K.op_code("avg"), L.F32, 1, L.REPLAY_STEPWISE, numel
    return H.Workspace(q, L.lib().mcclx_replay_workspace_bytes(C.byref(r)), pinned_host=True)


@pytest.mark.parametrize("world,numel", [
    (2, 1_499_999),            # two launches, as ever
    (2, 3_000_000),            # two pieces exactly
    (2, 2 * (1_500_000 + 65)),  # the last piece shorter by what rounding to 64 leaves
    (3, 2_000_003), (3, 7_000_001),
    (4, 1_000_001), (4, 4_000_002), (4, 9_999_997),
])
@pytest.mark.parametrize("algo", list(ALGOS))
@pytest.mark.parametrize("op", ["avg", "sum"])
def test_same_bits_as_the_stepwise_schedule(world, numel, algo, op):
    q = K.hip_kernels_init(0)
    base = _tensors(world, numel)
    want = [t.clone() for t in base]
    H.allreduce_replay(want, op, ALGOS[algo], wire_bf16=True, mode=L.REPLAY_STEPWISE)
    ws = _pinned(q, world, numel, ALGOS[algo])
    try:
        got = [t.clone() for t in base]
        before = q.launch_count()
        H.allreduce_replay(got, op, ALGOS[algo], wire_bf16=True, workspace=ws)
        pieces = _pieces(world, numel, algo)
        assert q.launch_count() - before == pieces + 1
        for r in range(world):
            assert torch.equal(got[r].view(torch.int32), want[r].view(torch.int32)), f"rank {r}"
    finally:
        ws.free()


def test_odd_addresses_and_replays_of_a_recording():
    """Tensors that start off a 16-byte boundary, recorded once and replayed on fresh values."""
    q = K.hip_kernels_init(0)
    world, numel = 3, 2_500_001
    room = [torch.empty(numel + 3, device="cuda") for _ in range(world)]
    got = [t[1 + r:1 + r + numel] for r, t in enumerate(room)]
    ws = _pinned(q, world, numel, L.ALGO_RING)
    r = L.Replay()
    r.world, r.algo, r.op, r.dtype, r.wire_bf16, r.mode, r.numel = world, L.ALGO_RING, K.op_code("avg"), L.F32, 1, L.REPLAY_FUSED, numel
    ptrs = (C.c_void_p * world)(*[t.data_ptr() for t in got])
    r.tensors, r.workspace, r.workspace_bytes = ptrs, ws.ptr, ws.nbytes
    torch.cuda.synchronize()
    q.graph_begin()
    L.check(L.lib().mcclx_allreduce_replay(q.handle, C.byref(r)))
    graph = q.graph_end()
    try:
        for seed in (1, 2, 3):
            base = _tensors(world, numel, seed)
            for t, b in zip(got, base):
                t.copy_(b)
            want = [b.clone() for b in base]
            H.allreduce_replay(want, "avg", L.ALGO_RING, wire_bf16=True, mode=L.REPLAY_STEPWISE)
            torch.cuda.synchronize()
            q.graph_launch(graph)
            q.drain()
            for k in range(world):
                assert torch.equal(got[k].view(torch.int32), want[k].view(torch.int32)), (seed, k)
    finally:
        q.graph_destroy(graph)
        ws.free()
