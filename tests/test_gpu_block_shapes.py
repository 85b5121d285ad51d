"""By-value launches in blocks of one and of four wavefronts (four_waves in fold_kernels.hip): every
element on both sides of each boundary, with sums of small whole numbers, which are exact in every
dtype and order."""
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
