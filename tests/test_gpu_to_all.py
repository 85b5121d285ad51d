"""The to-all form of a fold (the result goes back into every operand's buffer: a whole allreduce
of five to eight ranks, or of any op, in one launch) against the oracle's replay of the
reference, bit for bit: every dtype, op, algorithm and number of ranks, sizes at the edges of
packets and tiles, tensors off the 16-byte grid, and large replays."""
import ctypes as C
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
    (5, 60_001, F32, SUM, RING, False), (8, 100_003, F32, AVG, RING, True), (3, 300_007, F32, MAX, BUTTERFLY, True),
    (6, 200_001, BF16, AVG, TREE, False), (7, 150_001, F16, MIN, RING, False), (4, 400_003, F32, PRODUCT, TREE, False),
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


KINDS = ["f32", "bf16", "f16", "all_f32"]


def to_all_against_one_output(L, K, U, q, kind, k, op, counts, seed, noalloc=False, topo=0, scale=None):
    """The to-all launch over `counts` against the same operands folded into buffers of their own
    (the one-output form, which the oracle's tests hold): every operand becomes the result, and
    what lies between the segments stays."""
    W = {"f32": F32, "bf16": BF16, "f16": F16, "all_f32": BF16}[kind]
    io = L.IO_ALL_F32 if kind == "all_f32" else L.IO_PURE
    stored = F32 if kind == "all_f32" else W
    es = 4 if stored == F32 else 2
    gap = 5  # elements behind every segment: odd starts, and a guard
    starts = np.concatenate([[0], np.cumsum([c + gap for c in counts])])
    rng = np.random.default_rng(seed)
    tdt = U.TORCH_DT[stored]
    full = [torch.from_numpy(rng.standard_normal(int(starts[-1])).astype(np.float32)).cuda().to(tdt) for _ in range(k)]
    out = torch.zeros_like(full[0])
    kw = dict(io=io, op=op, topo=topo)
    if scale is not None:
        kw.update(scale_mode=L.SCALE_VIEW, scale=scale)
    at = lambda t, i: t.data_ptr() + es * int(starts[i])  # noqa: E731
    fn = L.lib().mcclx_fold_batched_noalloc if noalloc else L.lib().mcclx_fold_batched

    def launch(flags, out_of):
        arr = (L.Seg * len(counts))(*[K.make_seg(out_of(i), 0, [at(t, i) for t in full], c) for i, c in enumerate(counts)])
        plan = K.make_plan(W, k, flags=flags, **kw)
        L.check(fn(q.handle, C.byref(plan), arr, len(counts)))

    torch.cuda.synchronize()
    want = [f.clone() for f in full]
    torch.cuda.synchronize()
    launch(0, lambda i: at(out, i))
    held = q.hold_launch_count()
    launch(L.PLAN_TO_ALL, lambda i: at(full[0], i))
    assert q.hold_launch_count() == held, "to-all has no hold form"
    q.drain()
    bits = torch.int32 if es == 4 else torch.int16
    inside = torch.zeros(int(starts[-1]), dtype=torch.bool, device="cuda")
    for i, c in enumerate(counts):
        inside[int(starts[i]):int(starts[i]) + c] = True
    for j in range(k):
        expect = torch.where(inside, out.view(bits), want[j].view(bits))
        assert torch.equal(full[j].view(bits), expect), f"{kind} k={k} op={op} operand {j} segs {len(counts)} noalloc {noalloc}"


@pytest.fixture(scope="module")
def env():
    import gpu_util as U
    from mccl_amd import _lib as L, kernels as K
    return L, K, U, K.hip_kernels_init(0)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("k", [2, 3, 4, 8])
def test_to_all_launches_by_value(env, kind, k):
    """One to 32 segments in the kernel arguments, through both entry points: a size of a few
    elements, tiles and their edges, and sums from where other plans take the hold form to where
    fewer waves stay resident (160 MB moved)."""
    L, K, U, q = env
    es = 2 if kind in ("bf16", "f16") else 4
    for noalloc in (False, True):
        for counts in ([1], [7, 63, 64, 65], [4097, 5000, 4099], [1023] * 32):
            to_all_against_one_output(L, K, U, q, kind, k, SUM, counts, 11 + k, noalloc, scale=1 / 3)
    for bytes_read in (20 << 20, 34 << 20, 110_000_000):
        n = bytes_read // (es * k) // 3
        to_all_against_one_output(L, K, U, q, kind, k, SUM, [n, n, n + 1], 12 + k)
    if kind != "all_f32":
        to_all_against_one_output(L, K, U, q, kind, k, MAX, [4097, 5000, 4099], 13 + k)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("k", [2, 5, 8])
def test_to_all_launches_over_a_table(env, kind, k):
    """More segments than fit the kernel arguments, ragged ones and equal ones, from a table the
    library uploads and from the one it writes with kernels."""
    L, K, U, q = env
    rng = np.random.default_rng(k)
    ragged = [int(c) for c in rng.integers(1, 9000, size=90)] + [40_001, 1]
    for noalloc in (False, True):
        for counts in (ragged, [2048] * 100, [513] * 33):
            to_all_against_one_output(L, K, U, q, kind, k, SUM, counts, 21 + k, noalloc, scale=0.25)
        if kind != "all_f32":
            to_all_against_one_output(L, K, U, q, kind, k, PRODUCT, ragged, 22 + k, noalloc)
    n = 260_000_000 // (2 * k * (2 if kind in ("bf16", "f16") else 4)) // 200  # enough bytes for the residency limit
    to_all_against_one_output(L, K, U, q, kind, k, SUM, [n] * 200, 23 + k)
    if k >= 4:
        to_all_against_one_output(L, K, U, q, kind, k, SUM, ragged, 24 + k, topo=L.TOPO_BINOMIAL)


@pytest.mark.parametrize("world,dtype", [(7, "fp32"), (8, "fp32"), (7, "fp16")])
def test_large_max_takes_about_as_long_as_the_average(world, dtype):
    """Both move the same bytes.  The kernels of MAX compute longer between loads and stores and need more waves
    under way for that: with as few as a sum, 16-25 % more time, with those they get 2-6 %."""
    import time
    from mccl_amd import _lib as L, harness as H, kernels as K
    K.hip_kernels_init(0)
    dt = {"fp32": torch.float32, "fp16": torch.float16}[dtype]
    n = 400_000_000 // (world * dt.itemsize)
    ts = [torch.full((n,), 1.0 + r, dtype=dt, device="cuda") for r in range(world)]
    best = {}
    for _ in range(6):
        for op in ("avg", "max"):
            H.allreduce_replay(ts, op, L.ALGO_RING, mode=L.REPLAY_DIRECT)
            torch.cuda.synchronize()
            t = time.perf_counter()
            for _ in range(10):
                H.allreduce_replay(ts, op, L.ALGO_RING, mode=L.REPLAY_DIRECT)
            best[op] = min(best.get(op, 1.0), time.perf_counter() - t)
    assert best["max"] < 1.11 * best["avg"], best
