"""The to-all form of a fold (the result goes back into every operand's buffer: a whole allreduce
of five to eight ranks, or of any op, in one launch) against the oracle's replay of the
reference, bit for bit: every dtype, op, algorithm and number of ranks, sizes at the edges of
packets and tiles, tensors off the 16-byte grid, and the sizes from which large replays take it."""
import re

import numpy as np
import pytest
import torch

from oracle import oracle as orc
from oracle.oracle import AVG, BF16, BUTTERFLY, F16, F32, MAX, MIN, PRODUCT, RING, SUM, TREE

pytestmark = pytest.mark.gpu
NAMES = {RING: "ring", TREE: "tree", BUTTERFLY: "butterfly"}


def replay(world, n, dtype, op, algo, wire, launches, offset=0, specials=True):
    import gpu_util as U
    from mccl_amd import _lib as L, harness as H, kernels as K
    q = K.hip_kernels_init(0)
    rng = np.random.default_rng(world * 1000 + n + 7 * op + algo)
    xs = [U.rand_values(rng, n, dtype, specials=specials) for _ in range(world)]
    full = [U.to_dev(np.concatenate([x[:1].repeat(offset), x, x[:1].repeat(5)]), dtype) for x in xs]
    ts = [f[offset:offset + n] for f in full]
    torch.cuda.synchronize()
    before = q.launch_count()
    H.allreduce_replay(ts, op, algo, wire_bf16=wire, mode=L.REPLAY_DIRECT if wire else L.REPLAY_FUSED)
    assert q.launch_count() - before == launches
    want = [x.copy() for x in xs]
    rc, used = orc.pg_allreduce(want, dtype, op, wire_bf16=wire, env_algo=NAMES[algo], threads=orc.max_threads())
    assert rc == 0 and used == algo
    for r in range(world):
        U.assert_same_bits(ts[r], want[r], dtype, f"w{world} n={n} dtype {dtype} op {op} algo {algo} wire {wire} rank {r}")
        assert torch.equal(full[r][offset + n:].view(torch.int16), U.to_dev(xs[r][:1].repeat(5), dtype).view(torch.int16)), "past the end"


@pytest.mark.parametrize("dtype,wire", [(F32, False), (F16, False), (BF16, False), (F32, True)])
@pytest.mark.parametrize("algo", [RING, TREE, BUTTERFLY])
@pytest.mark.parametrize("op", [SUM, AVG, MIN, MAX, PRODUCT])
def test_small_replays_against_the_oracle(dtype, wire, algo, op):
    for world in ([2, 3, 4] if op in (MIN, MAX, PRODUCT) else []) + [5, 6, 7, 8]:
        for n, offset in ((world, 0), (63, 1), (511, 0), (1024, 3), (2049, 0), (4099, 7), (15_013, 2)):
            replay(world, n, dtype, op, algo, wire, 1, offset, specials=dtype != F16)  # fp16 NaN payloads are the hardware's


@pytest.mark.parametrize("world,n,dtype,op,algo,wire", [
    (8, 524_288, BF16, AVG, RING, False), (8, 262_147, F32, SUM, BUTTERFLY, True), (5, 419_431, F32, AVG, TREE, False),
    (3, 699_053, F32, MAX, RING, True), (2, 2_097_153, F16, MIN, BUTTERFLY, False),
    (8, 5_000_011, BF16, AVG, RING, False), (6, 3_500_003, F32, AVG, RING, True)])  # the last two: fewer waves resident
def test_large_replays_against_the_oracle(world, n, dtype, op, algo, wire):
    replay(world, n, dtype, op, algo, wire, 1, offset=1, specials=False)


def test_to_all_validation():
    from mccl_amd import _lib as L, kernels as K
    q = K.hip_kernels_init(0)
    a, b = torch.zeros(64, device="cuda"), torch.zeros(64, device="cuda")
    seg = lambda out, ins, wire=0: [K.make_seg(out, wire, ins, 32)]
    pa, pb = a.data_ptr(), b.data_ptr()
    for plan, segs, frag in (
            (K.make_plan(L.F32, 1, flags=L.PLAN_TO_ALL), seg(pa, [pa]), "two operands"),
            (K.make_plan(L.BF16, 2, acc=L.ACC_F32, flags=L.PLAN_TO_ALL), seg(pa, [pa, pb]), "per-step rounding"),
            (K.make_plan(L.BF16, 2, io=L.IO_OWN_FIRST_F32, flags=L.PLAN_TO_ALL), seg(pa, [pa, pb]), "form of the result"),
            (K.make_plan(L.F32, 2, flags=L.PLAN_TO_ALL, fanout=1), seg(pa, [pa, pb, pb]), "excludes fan-out"),
            (K.make_plan(L.F32, 2, flags=L.PLAN_TO_ALL), seg(pb, [pa, pb]), "to be in[0]"),
            (K.make_plan(L.BF16, 2, flags=L.PLAN_TO_ALL), seg(pa, [pa, pb], pb), "no wire_out"),
            (K.make_plan(L.F32, 2, flags=L.PLAN_TO_ALL), seg(pa, [pa, pa + 16]), "overlap")):
        with pytest.raises(Exception, match=re.escape(frag)):
            q.fold(plan, segs)
