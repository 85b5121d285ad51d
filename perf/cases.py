"""The work that users of this framework have it do, as a fixed set of cases to time.

`listed()` names them, `draw(rng)` gives further ones of the same ranges, `prepare` builds what a
program holds before the call, `run` makes one pass through the public entry points, `work` and
`tolerance` say what a pass cannot do without and how close two correct results are.

The kinds of work, and who does it:

  reduce_op     one received chunk reduced into a local one (the reference's metal_reduce_op)
  scale         the same with the averaging step fused in (metal_accumulate_and_scale)
  codec         a tensor to its bf16 wire form and back
  fold          an integrator's launch: one plan over the chunks of a bucket on the reduce queue
  allreduce     a collective over tensors that share the GPU, algorithm and wire form from the
                MCCL_* environment as in production
  pinned        the same where the wire delivers into pinned host memory (zero-copy peers)
  list          one allreduce over a list of tensors (a model's many small gradients)
  reduce_scatter, allgather   the two halves of a sharded (ZeRO) step
  c10d          ranks that call the torch.distributed backend, each on its own thread

In-place collectives average, as DDP does, or take a maximum: a repeated pass keeps its values in
range, where a sum would run away from the distribution the path meets.
"""
from __future__ import annotations

import atexit
import datetime
import os
import queue
import threading

import torch
import torch.distributed as dist

import mccl_amd
from mccl_amd import _lib as L
from mccl_amd import harness as H
from mccl_amd import kernels as K

DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
MIB_25 = 6_553_600  # fp32 elements of torch DDP's default bucket


def listed():
    return [
        # A received chunk of a small bf16 layer reduced in place: launch latency and nothing else.
        {"name": "reduce_op_small", "kind": "reduce_op", "dtype": "bf16", "numel": 4_097, "op": "sum"},
        # Metrics, overflow flags and gradient norms of eight ranks: a few kilobytes, maximum, tree.
        {"name": "metrics_max_w8", "kind": "allreduce", "world": 8, "numel": 1_000, "dtype": "fp32", "op": "max",
         "algo": "auto", "wire": False},
        # The wire codec on one odd-sized bucket: encode for sending, decode on arrival.
        {"name": "codec_bucket", "kind": "codec", "numel": MIB_25 + 1},
        # The launch an integrator of the C ABI issues per DDP bucket: own fp32 chunk + two bf16 peers -> average.
        {"name": "fold_bucket_w3", "kind": "fold", "world": 3, "numel": MIB_25, "dtype": "fp32", "wire": True},
        # The whole allreduce of that bucket: butterfly, bf16 wire, average over three ranks.
        {"name": "ddp_bucket_w3", "kind": "allreduce", "world": 3, "numel": MIB_25, "dtype": "fp32", "op": "avg",
         "algo": "butterfly", "wire": True},
        # Mixed-precision training on a full node: bf16 gradients of eight ranks, ring, ragged tail.
        {"name": "bf16_grads_w8", "kind": "allreduce", "world": 8, "numel": 12_500_003, "dtype": "bf16", "op": "avg",
         "algo": "auto", "wire": False},
        # A 110M-parameter model's flattened gradient over four ranks: ring, bf16 wire, ragged tail.
        {"name": "flat_grad_w4", "kind": "allreduce", "world": 4, "numel": 110_000_002, "dtype": "fp32", "op": "avg",
         "algo": "ring", "wire": True},
        # The same gradient with the wire copies in pinned host memory, read over PCIe.
        {"name": "flat_grad_pinned_w4", "kind": "pinned", "world": 4, "numel": 110_000_002, "algo": "ring"},
        # 4096 messages of 64 KiB, below the tree threshold, in one list call.
        {"name": "tree_messages_w3", "kind": "list", "world": 3, "messages": 4_096, "numel": 16_384, "wire": False},
        # ZeRO, eight ranks of 512 MiB bf16: the gradients' reduce_scatter ...
        {"name": "reduce_scatter_w8", "kind": "reduce_scatter", "world": 8, "chunk": 33_554_432, "dtype": "bf16"},
        # ... and the parameters' allgather.
        {"name": "allgather_w8", "kind": "allgather", "world": 8, "chunk": 33_554_432, "dtype": "bf16"},
        # A DDP step through torch.distributed's backend: two ranks, eight 25 MiB buckets back to back.
        {"name": "c10d_step_w2", "kind": "c10d", "world": 2, "buckets": 8, "numel": MIB_25, "wire": True},
    ]


def _log_int(rng, lo, hi):
    """A whole number spread over the logarithm of its range, odd ones as likely as even ones."""
    return max(lo, min(hi, int(lo * (hi / lo) ** rng.random()) + rng.randrange(2)))


def draw(rng):
    kind = rng.choice(["reduce_op", "scale", "codec", "fold", "allreduce", "allreduce", "allreduce", "pinned", "list",
                       "reduce_scatter", "allgather", "c10d"])
    if kind == "reduce_op":
        return {"kind": kind, "dtype": rng.choice(list(DTYPES)), "numel": _log_int(rng, 1_000, 100_000_000),
                "op": rng.choice(["sum", "sum", "max", "min"])}
    if kind == "scale":
        return {"kind": kind, "dtype": rng.choice(list(DTYPES)), "numel": _log_int(rng, 1_000, 100_000_000)}
    if kind == "codec":
        return {"kind": kind, "numel": _log_int(rng, 1_000, 100_000_000)}
    if kind == "fold":
        dtype = rng.choice(list(DTYPES))
        return {"kind": kind, "world": rng.randint(2, 8), "numel": _log_int(rng, 10_000, 50_000_000), "dtype": dtype,
                "wire": dtype == "fp32" and rng.random() < 0.7}
    if kind == "allreduce":
        dtype = rng.choice(["fp32", "fp32", "bf16", "fp16"])
        world = rng.randint(2, 8)
        return {"kind": kind, "world": world, "numel": _log_int(rng, 500, 400_000_000 // world), "dtype": dtype,
                "op": rng.choice(["avg", "avg", "avg", "max"]),
                "algo": rng.choice(["auto", "auto", "ring", "butterfly"]),
                "wire": dtype == "fp32" and rng.random() < 0.7}
    if kind == "pinned":
        world = rng.randint(2, 4)
        return {"kind": kind, "world": world, "numel": _log_int(rng, 1_000_000, 400_000_000 // world),
                "algo": rng.choice(["ring", "butterfly"])}
    if kind == "list":
        messages = _log_int(rng, 32, 4_096)
        return {"kind": kind, "world": rng.choice([2, 3]), "messages": messages,
                "numel": _log_int(rng, 256, 16_384), "wire": rng.random() < 0.3}
    if kind in ("reduce_scatter", "allgather"):
        world = rng.choice([2, 4, 8])
        return {"kind": kind, "world": world, "chunk": _log_int(rng, 10_000, 33_000_000),
                "dtype": rng.choice(["bf16", "fp32"] if world < 8 else ["bf16"])}
    return {"kind": kind, "world": rng.choice([2, 3, 4]), "buckets": rng.randint(1, 8),
            "numel": _log_int(rng, 100_000, MIB_25), "wire": rng.random() < 0.7}


# ---- inputs ------------------------------------------------------------------------------


def _values(seed, index, numel, dtype, spread):
    """Gradients as they come: N(0, spread), one in a thousand an outlier a hundred thousand times that size."""
    g = torch.Generator(device="cuda").manual_seed(seed * 1_009 + index)
    x = torch.randn(numel, generator=g, device="cuda").mul_(spread)
    at = torch.randint(0, numel, (max(1, numel // 1000),), generator=g, device="cuda")
    x[at] = torch.where(at % 2 == 0, 1.0, -1.0) * min(1e5 * spread, 1e2)
    return x.to(DTYPES[dtype])


def _bf16_specials(x):
    """NaN, infinities, zeros of both signs and the extreme finite values at fixed places of a bf16 tensor."""
    bits = torch.tensor([0x7FC0, 0x7F80, 0xFF80, 0x0000, 0x8000, 0x0001, 0x007F, 0x7F7F, 0xFF7F], dtype=torch.int32)
    at = torch.arange(0, x.numel(), 1_000_003)
    x.view(torch.int16)[at.cuda()] = bits.to(torch.int16)[at % bits.numel()].cuda()
    return x


def _environment(algo, wire):
    """What a program exports before it starts: the reference's own two switches."""
    os.environ["MCCL_ALLREDUCE_ALGO"] = algo
    if wire:
        os.environ["MCCL_WIRE_DTYPE"] = "bf16"
    else:
        os.environ.pop("MCCL_WIRE_DTYPE", None)


def _workspace_bytes(case):
    """One bf16 copy of the tensor per rank, and each rank's receive slots."""
    world, per = case["world"], -(-case["numel"] // case["world"])
    slots = world - 1 if case["algo"] == "butterfly" else 1
    return world * sum((2 * n + 255) // 256 * 256 for n in (case["numel"], slots * per))


class _Pinned:
    """Pinned, device-mapped memory for the wire copies; given back with the state that holds it."""

    def __init__(self, q, nbytes):
        self.workspace = H.Workspace(q, nbytes, pinned_host=True)

    def __del__(self):
        self.workspace.free()


class _Ranks:
    """The ranks of a job: threads that each own a process group of backend "mccl" and take their
    turn of work from a queue."""

    def __init__(self, world):
        store = dist.HashStore()
        self.todo = [queue.SimpleQueue() for _ in range(world)]
        self.done = queue.SimpleQueue()
        self.threads = [threading.Thread(target=self._rank, args=(store, r, world), daemon=True) for r in range(world)]
        for t in self.threads:
            t.start()
        atexit.register(self.close)

    def _rank(self, store, rank, world):
        torch.cuda.set_device(0)
        group = mccl_amd._C._create_process_group_mccl(store, rank, world, datetime.timedelta(seconds=60))
        options = dist.AllreduceOptions()
        options.reduceOp = dist.ReduceOp.AVG
        while True:
            buckets = self.todo[rank].get()
            if buckets is None:
                break
            failure = None
            try:
                works = [group.allreduce([b], options) for b in buckets]
                for w in works:
                    w.wait()
            except Exception as e:  # noqa: BLE001  (handed to the thread that asked)
                failure = e
            self.done.put(failure)
        del group

    def step(self, tensors):
        for q, buckets in zip(self.todo, tensors):
            q.put(buckets)
        for failure in [self.done.get() for _ in self.todo]:
            if failure is not None:
                raise failure

    def close(self):
        for q in self.todo:
            q.put(None)
        for t in self.threads:
            t.join(30)


_ranks = {}


def _ranks_for(world):
    if world not in _ranks:
        _ranks[world] = _Ranks(world)
    return _ranks[world]


def prepare(case, seed):
    q = K.hip_kernels_init(0)
    kind, s = case["kind"], {"case": case, "q": q}
    if kind in ("reduce_op", "scale"):
        s["dst"] = _values(seed, 0, case["numel"], case["dtype"], 1e-3)
        s["src"] = _values(seed, 1, case["numel"], case["dtype"], 1e-3)
    elif kind == "codec":
        s["x"] = _values(seed, 0, case["numel"], "fp32", 1e-3)
    elif kind == "fold":
        _prepare_fold(case, seed, s)
    elif kind in ("allreduce", "pinned", "c10d"):
        _environment(case.get("algo", "auto"), case.get("wire", True))
        world, numel, dtype = case["world"], case["numel"], case.get("dtype", "fp32")
        if kind == "c10d":
            s["ranks"] = _ranks_for(world)
            s["tensors"] = [[_values(seed, r * 64 + b, numel, dtype, 1e-3) for b in range(case["buckets"])]
                            for r in range(world)]
        else:
            s["tensors"] = [_values(seed, r, numel, dtype, 1e-3 if numel <= 50_000_000 else 1e-4) for r in range(world)]
        if kind == "pinned":
            s["pinned"] = _Pinned(q, _workspace_bytes(case))
    elif kind == "list":
        _environment("auto", case["wire"])
        m, n = case["messages"], case["numel"]
        g = torch.Generator(device="cuda").manual_seed(seed)
        s["flat"] = [torch.rand(m * n, generator=g, device="cuda").mul_(2).sub_(1) for _ in range(case["world"])]
        split = [f.split(n) for f in s["flat"]]
        s["groups"] = [list(ranks) for ranks in zip(*split)]
    elif kind in ("reduce_scatter", "allgather"):
        world, chunk = case["world"], case["chunk"]
        whole = world * chunk
        long, short = (whole, chunk) if kind == "reduce_scatter" else (chunk, whole)
        s["ins"] = [_values(seed, r, long, case["dtype"], 1e-2) for r in range(world)]
        if case["dtype"] == "bf16":
            for x in s["ins"]:
                _bf16_specials(x)
        s["outs"] = [torch.empty(short, dtype=DTYPES[case["dtype"]], device="cuda") for _ in range(world)]
    return s


def _prepare_fold(case, seed, s):
    """Butterfly's launch for every rank of a bucket: chunk r = rank r's own elements + the peers', in ascending order."""
    world, numel, wire = case["world"], case["numel"], case["wire"]
    own = [_values(seed, r, numel, case["dtype"], 1e-3) for r in range(world)]
    peers = [K.encode_bf16(t) for t in own] if wire else own
    outs = [torch.empty(numel, dtype=own[0].dtype, device="cuda") for _ in range(world)]
    s["plan"] = K.make_plan(L.BF16 if wire else K.dtype_code(own[0]), world,
                            io=L.IO_OWN_FIRST_F32 if wire else L.IO_PURE, scale_mode=L.SCALE_VIEW, scale=1.0 / world)
    eo, ep = own[0].element_size(), peers[0].element_size()
    chunks = H.chunkize(numel, eo, world)
    s["segs"] = [K.make_seg(outs[r].data_ptr() + eo * at, 0,
                            [own[r].data_ptr() + eo * at] +
                            [peers[p].data_ptr() + ep * at for p in range(world) if p != r], n)
                 for r, (at, n, _, _) in enumerate(chunks) if n]
    s["keep"] = own, peers
    s["out"] = [outs[r][at:at + n] for r, (at, n, _, _) in enumerate(chunks) if n]


# ---- one pass ----------------------------------------------------------------------------


def run(state):
    case, q = state["case"], state["q"]
    kind = case["kind"]
    if kind == "reduce_op":
        return K.hip_reduce_op(state["dst"], state["src"], case["op"])
    if kind == "scale":
        return K.hip_accumulate_and_scale(state["dst"], state["src"], 0.5)
    if kind == "codec":
        wire = K.encode_bf16(state["x"])
        return wire, K.decode_bf16(wire)
    if kind == "fold":
        q.wait_torch_stream()
        q.fold(state["plan"], state["segs"])
        q.torch_stream_wait()
        return state["out"]
    if kind == "allreduce":
        H.allreduce(state["tensors"], case["op"])
        return state["tensors"]
    if kind == "pinned":
        H.allreduce_replay(state["tensors"], "avg", H.ALGO_NAMES[case["algo"]], wire_bf16=True,
                           workspace=state["pinned"].workspace)
        return state["tensors"]
    if kind == "list":
        H.allreduce_replay_many(state["groups"], "avg", L.ALGO_TREE, wire_bf16=case["wire"])
        return state["flat"]
    if kind == "reduce_scatter":
        H.reduce_scatter_replay(state["outs"], state["ins"], "avg")
        return state["outs"]
    if kind == "allgather":
        H.allgather_replay(state["outs"], state["ins"])
        return state["outs"]
    state["ranks"].step(state["tensors"])
    return state["tensors"]


def work(case):
    """Bytes: every input read once, every output written once.  Flops: one per operand after the
    first and one for the factor, per result element."""
    kind, n, world = case["kind"], case.get("numel", 0), case.get("world", 1)
    size = 4 if case.get("dtype", "fp32") == "fp32" else 2
    if kind in ("reduce_op", "scale"):
        return {"bytes": 3 * n * size, "flops": n if kind == "reduce_op" else 2 * n}
    if kind == "codec":
        return {"bytes": 12 * n, "flops": n}
    if kind == "fold":
        peer = 2 if case["wire"] else size
        return {"bytes": n * (size + (world - 1) * peer + size), "flops": n * world}
    if kind in ("reduce_scatter", "allgather"):
        chunk = case["chunk"]
        if kind == "reduce_scatter":
            return {"bytes": (world + 1) * world * chunk * size, "flops": world * world * chunk}
        return {"bytes": (world + 1) * world * chunk * size, "flops": 0}
    n *= case.get("messages", 1) * case.get("buckets", 1)
    return {"bytes": 2 * world * n * size, "flops": n * world}


def tolerance(case):
    """Every path rounds after every operation in the reference's order (or moves bytes): results are
    the same bits whatever the launches look like.  Measured: two runs, and runs of the stepwise, the
    fused and the direct schedule, do not differ in a single bit."""
    return "exact"
