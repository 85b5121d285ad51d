"""By-value launches in blocks of one and of four wavefronts (launch_few in fold_kernels.hip): every
element over a range of sizes and on both sides of each boundary, where the shape that was taken is
asserted too, with sums of small whole numbers, which are exact in every dtype and order."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DT = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16, "wire": torch.float32}


@pytest.fixture(scope="module")
def env():
    from mccl_amd import _lib as L, harness as H, kernels as K
    K.hip_kernels_init(0)
    return L, H, K


def _whole(rank, numel, dtype):
    x = (torch.arange(numel, device="cuda") * (rank + 3) + rank) % 17 - 8
    return x.to(DT[dtype])


E = {"fp32": 4, "wire": 4, "fp16": 8, "bf16": 8}  # elements of a lane's packet


def _numel(dtype, waves, segs, off):
    """Elements of a tensor whose launch of `segs` equal segments has about that many one-wavefront tiles."""
    return 64 * (4 if dtype in ("fp32", "wire") else 8) * waves + segs * off


@pytest.mark.parametrize("waves", [40, 479, 481, 959, 961, 2047, 2049, 4607, 4609, 6143, 6145, 7679, 7681, 12_300])
@pytest.mark.parametrize("world,dtype", [(2, "fp32"), (2, "wire"), (3, "bf16"), (4, "fp16"), (4, "wire"), (5, "fp32"),
                                         (5, "bf16"), (8, "bf16"), (8, "wire"), (8, "fp16")])
def test_allreduce_in_place(env, world, dtype, waves):
    L, H, _ = env
    for op, off in (("sum", 0), ("sum", 3), ("max", -5)):
        numel = _numel(dtype, waves, world, off)
        ts = [_whole(r, numel, dtype) for r in range(world)]
        want = torch.stack([t.float() for t in ts]).sum(0) if op == "sum" else torch.stack([t.float() for t in ts]).amax(0)
        H.allreduce_replay(ts, op, L.ALGO_BUTTERFLY, wire_bf16=dtype == "wire", mode=L.REPLAY_DIRECT)
        for r, t in enumerate(ts):
            assert torch.equal(t.float(), want), (op, off, r)


@pytest.mark.parametrize("waves", [40, 479, 481, 961, 2049, 4609, 6145, 7681])
@pytest.mark.parametrize("world,dtype", [(2, "fp32"), (4, "bf16"), (8, "bf16"), (8, "fp16")])
def test_reduce_scatter(env, world, dtype, waves):
    L, H, _ = env
    for off in (0, 1):
        chunk = _numel(dtype, max(1, waves // world), 1, off)
        ins = [_whole(r, world * chunk, dtype) for r in range(world)]
        outs = [torch.full((chunk,), 77, dtype=DT[dtype], device="cuda") for _ in range(world)]
        H.reduce_scatter_replay(outs, ins, "sum")
        want = torch.stack([t.float() for t in ins]).sum(0)
        assert torch.equal(torch.cat(outs).float(), want)


@pytest.mark.parametrize("dtype", ["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("waves", [1, 40, 959, 961, 2049, 4609, 7679, 7681])
def test_received_chunk_off_the_lines(env, dtype, waves):
    _, _, K = env
    numel = _numel(dtype, waves, 1, 1)
    for shift in (0, 1, 31):  # elements in front of the operands, as of a chunk inside a tensor
        a, b = _whole(0, numel + shift, dtype), _whole(1, numel + shift, dtype)
        want = a.clone()
        want[shift:] += b[shift:]
        K.hip_reduce_op(a[shift:], b[shift:], "sum")
        assert torch.equal(a, want)


def _shape(q, call):
    """(launches in blocks of four wavefronts, launches that told of their end) of a call of one launch."""
    before = q.launch_count(), q.four_wave_launch_count(), q.marked_launch_count()
    call()
    after = q.launch_count(), q.four_wave_launch_count(), q.marked_launch_count()
    assert after[0] - before[0] == 1
    return after[1] - before[1], after[2] - before[2]


@pytest.mark.parametrize("off", [0, 1, 5])
@pytest.mark.parametrize("side", [-1, 0])
@pytest.mark.parametrize("waves", [1_280, 4_096, 6_144])
@pytest.mark.parametrize("world,dtype", [(4, "fp32"), (5, "fp32"), (5, "fp16"), (7, "bf16"), (8, "fp32"), (8, "bf16")])
def test_shape_of_folds_into_one(env, world, dtype, waves, side, off):
    """Five operands or more take blocks of four from four of them a CU on; the tiles of a segment are a whole
    number, so the launch has the last count below `waves` or the first one that reaches it."""
    L, H, K = env
    q = K._q(None)
    tiles = -(-waves // world) + side
    chunk = 64 * E[dtype] * tiles - off
    ins = [_whole(r, world * chunk, dtype) for r in range(world)]
    outs = [torch.full((chunk,), 77, dtype=DT[dtype], device="cuda") for _ in range(world)]
    four, _ = _shape(q, lambda: H.reduce_scatter_replay(outs, ins, "sum"))
    assert four == (world >= 5 and tiles * world >= 16 * q.compute_units)
    want = torch.stack([t.float() for t in ins]).sum(0)
    assert torch.equal(torch.cat(outs).float(), want)


@pytest.mark.parametrize("tiles", [1, 4, 5, 6, 8, 12, 13, 16, 17, 32, 33, 43, 64, 65, 256])
@pytest.mark.parametrize("world,dtype", [(2, "fp32"), (3, "bf16"), (4, "wire"), (5, "fp16"), (8, "fp32"), (8, "bf16")])
def test_shape_of_small_allreduces(env, world, dtype, tiles):
    """Up to 32 blocks tell of their own end: blocks of one wavefront, or of four where those are too many."""
    L, H, K = env
    q = K._q(None)
    for off in (0, 1, world + 1):
        numel = world * 64 * E[dtype] * tiles - off
        if off > world and tiles == 1:
            continue
        ts = [_whole(r, numel, dtype) for r in range(world)]
        want = torch.stack([t.float() for t in ts]).sum(0)
        chunk = -(-numel // world)
        t = -(-chunk // (64 * E[dtype]))
        four, marked = _shape(q, lambda: H.allreduce_replay(ts, "sum", L.ALGO_BUTTERFLY, wire_bf16=dtype == "wire", mode=L.REPLAY_DIRECT))
        assert four == (32 < t * world <= 128)
        assert marked == (t * world <= 32 or (four and -(-t // 4) * world <= 32))
        for x in ts:
            assert torch.equal(x.float(), want), off
