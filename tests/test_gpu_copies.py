"""Batched copies of one source to several destinations: consecutive descriptors of one source
travel as one, the source is read once.  Bytes must arrive unchanged and nothing around a
destination may be touched, at every edge of the packet grid (16-byte packets that start on a
128-byte boundary of the first destination), in both block shapes and with the resident waves
limited (launches that move 160 MB and more)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def deliver(q, nbytes, fan, src_off, dst_offs, repeat=1):
    rng = np.random.default_rng(nbytes * 31 + fan * 7 + src_off)
    host = rng.integers(0, 256, repeat * nbytes + 64, dtype=np.uint8)
    src = torch.from_numpy(host).cuda()
    outs = [torch.full((repeat * nbytes + 512,), 0xA5, dtype=torch.uint8, device="cuda") for _ in range(fan)]
    descs = [(outs[f].data_ptr() + 128 + dst_offs[f % len(dst_offs)] + s * nbytes, src.data_ptr() + src_off + s * nbytes, nbytes)
             for s in range(repeat) for f in range(fan)]
    torch.cuda.synchronize()
    before = q.launch_count()
    q.copy_batched(descs)
    q.drain()
    for f in range(fan):
        lo = 128 + dst_offs[f % len(dst_offs)]
        want = np.full(repeat * nbytes + 512, 0xA5, dtype=np.uint8)
        want[lo:lo + repeat * nbytes] = host[src_off:src_off + repeat * nbytes]
        assert np.array_equal(outs[f].cpu().numpy(), want), (nbytes, fan, src_off, f)
    return q.launch_count() - before


@pytest.mark.parametrize("fan", [1, 2, 7, 8, 9])
@pytest.mark.parametrize("src_off,dst_offs", [(0, [0]), (4, [8, 100]), (2, [2]), (1, [3, 0, 77])])
def test_one_source_to_several_destinations(fan, src_off, dst_offs):
    from mccl_amd import kernels as K
    q = K.hip_kernels_init(0)
    for nbytes in (1, 15, 16, 17, 127, 128, 129, 255, 1023, 1024, 1025, 4096, 4097, 65_537):
        assert deliver(q, nbytes, fan, src_off, dst_offs) == 1
    assert deliver(q, 1021, fan, src_off, dst_offs, repeat=40) == 1      # 40 sources or more: the table launch
    # several destinations one after another, one and the ninth alone in blocks of four wavefronts up to 12,288 of them, then of one
    deliver(q, 9_000_001, fan, src_off, dst_offs)
    deliver(q, 13_000_003, fan, src_off, dst_offs)


@pytest.mark.parametrize("fan,nbytes", [(8, 18_000_005), (4, 33_000_001), (2, 54_000_001), (1, 81_000_003)])
def test_large_launches_with_fewer_waves_resident(fan, nbytes):
    from mccl_amd import kernels as K
    assert deliver(K.hip_kernels_init(0), nbytes, fan, 2, [6]) == 1


@pytest.mark.parametrize("world", [2, 3, 8])
@pytest.mark.parametrize("in_place", [False, True])
def test_allgather_of_odd_chunks(world, in_place):
    """Chunks of an odd number of elements leave every destination but the first off the packet
    grid; in place, a rank's own chunk is already where it belongs and is not copied."""
    from mccl_amd import harness as H
    for chunk in (1, 63, 4099, 300_001):
        outs = [torch.zeros(world * chunk, dtype=torch.bfloat16, device="cuda") for _ in range(world)]
        parts = [torch.randn(chunk, device="cuda").to(torch.bfloat16) for _ in range(world)]
        ins = [outs[r][r * chunk:(r + 1) * chunk].copy_(parts[r]) for r in range(world)] if in_place else parts
        H.allgather_replay(outs, ins)
        want = torch.cat(parts)
        assert all(torch.equal(o.view(torch.int16), want.view(torch.int16)) for o in outs), chunk


# A block moves 8 KiB, an XCD takes up to 64 of them in a row, a piece of the source is at most 8 MiB.
PIECE = 8 << 20


@pytest.mark.parametrize("fan", [2, 3, 4, 8])
@pytest.mark.parametrize("nbytes", [8191, 8192 * 8 + 1, 8192 * 512, 8192 * 512 + 15, PIECE - 1, PIECE + 34, 2 * PIECE + 8192, 3 * PIECE + 1])
def test_destination_after_destination_at_the_edges_of_tiles_and_pieces(fan, nbytes):
    """The short ones beside a source of 8 MB, which takes the launch to that form."""
    from mccl_amd import kernels as K
    q = K.hip_kernels_init(0)
    for src_off, offs in ((0, [0]), (2, [6, 100, 129])):
        assert deliver(q, nbytes, fan, src_off, offs) == 1
        long = torch.randint(0, 256, (8_000_000,), dtype=torch.uint8, device="cuda")
        src = torch.randint(0, 256, (nbytes + 4,), dtype=torch.uint8, device="cuda")
        copies = [torch.zeros_like(long) for _ in range(fan)]
        outs = [torch.full((nbytes + 512,), 0xA5, dtype=torch.uint8, device="cuda") for _ in range(fan)]
        at = [128 + offs[f % len(offs)] for f in range(fan)]
        sources = [(src.data_ptr() + src_off, [o.data_ptr() + a for o, a in zip(outs, at)], nbytes),
                   (long.data_ptr(), [c.data_ptr() for c in copies], long.numel())]
        torch.cuda.synchronize()
        before = q.spread_copy_count()
        q.copy_batched([(d, s, n) for s, ds, n in sources for d in ds])
        q.drain()
        assert q.spread_copy_count() == before + 1
        for o, a in zip(outs, at):
            assert torch.equal(o[a:a + nbytes], src[src_off:src_off + nbytes])
            assert bool((o[:a] == 0xA5).all()) and bool((o[a + nbytes:] == 0xA5).all())
        assert all(torch.equal(c, long) for c in copies)


def test_sources_of_many_lengths_share_a_launch_of_several_destinations():
    from mccl_amd import kernels as K
    q = K.hip_kernels_init(0)
    lengths = [9_000_001, 8_999_987, 6_000_000, 1, 4_000_003, 16, 8192 * 700]
    srcs = [torch.randint(0, 256, (n,), dtype=torch.uint8, device="cuda") for n in lengths]
    outs = [[torch.full((n + 64,), 0xA5, dtype=torch.uint8, device="cuda") for _ in range(5)] for n in lengths]
    torch.cuda.synchronize()
    q.copy_batched([(o.data_ptr() + 3 * f, s.data_ptr(), n) for s, group, n in zip(srcs, outs, lengths)
                    for f, o in enumerate(group)])
    q.drain()
    for s, group, n in zip(srcs, outs, lengths):
        for f, o in enumerate(group):
            assert torch.equal(o[3 * f:3 * f + n], s), (n, f)
            assert bool((o[:3 * f] == 0xA5).all()) and bool((o[3 * f + n:] == 0xA5).all()), (n, f)


# Destination after destination is for memory of this device alone; what lies elsewhere is written side by side, in blocks
# of four wavefronts up to 12,288 of them and of one beyond.
@pytest.mark.parametrize("fan", range(2, 9))
@pytest.mark.parametrize("n", [4_099, 5_000_003, 12_288 * 1024 - 17, 12_288 * 1024 + 1029, 20_000_003])
def test_a_source_in_pinned_host_memory_goes_to_several_destinations(fan, n):
    import ctypes
    from mccl_amd import kernels as K
    q = K.hip_kernels_init(0)
    host, dev = q.host_alloc(n + 1)
    data = np.random.default_rng(7).integers(0, 256, n + 1, dtype=np.uint8)
    ctypes.memmove(host, data.ctypes.data, n + 1)
    want = torch.from_numpy(data[1:]).cuda()
    outs = [torch.zeros(n + 32, dtype=torch.uint8, device="cuda") for _ in range(fan)]
    torch.cuda.synchronize()
    before = q.spread_copy_count(), q.launch_count()
    q.copy_batched([(o.data_ptr() + f, dev + 1, n) for f, o in enumerate(outs)])
    q.drain()
    assert (q.spread_copy_count(), q.launch_count()) == (before[0], before[1] + 1)
    q.host_free(host)
    for f, o in enumerate(outs):
        assert torch.equal(o[f:f + n], want) and not bool(o[:f].any()) and not bool(o[f + n:].any())


@pytest.mark.parametrize("fan", [2, 4, 8])
def test_destinations_in_pinned_host_memory_are_written_side_by_side(fan):
    import ctypes
    from mccl_amd import kernels as K
    q = K.hip_kernels_init(0)
    n = 12_000_001
    src = torch.randint(0, 256, (n,), dtype=torch.uint8, device="cuda")
    mem = [q.host_alloc(n) for _ in range(fan)]
    torch.cuda.synchronize()
    before = q.spread_copy_count()
    q.copy_batched([(dev, src.data_ptr(), n) for _, dev in mem])
    q.drain()
    assert q.spread_copy_count() == before
    want = src.cpu().numpy()
    for host, _ in mem:
        assert np.array_equal(np.ctypeslib.as_array((ctypes.c_uint8 * n).from_address(host)), want)
        q.host_free(host)


@pytest.mark.parametrize("fan,lo,hi", [(2, 20_000_000, 150_000_000), (3, 20_000_000, 150_000_000), (4, 20_000_000, None), (8, 20_000_000, None)])
def test_either_form_at_the_sizes_where_it_changes(fan, lo, hi):
    """By the bytes moved, the source once and each destination; from the upper line on, two and three destinations are
    written side by side again."""
    from mccl_amd import kernels as K
    q = K.hip_kernels_init(0)
    for line, below in ((lo, 0), (hi, 1)):
        if line is None:
            continue
        n = -(-line // (fan + 1))
        for nbytes, spread in ((n - 1, below), (n, 1 - below)):
            before = q.spread_copy_count()
            assert deliver(q, nbytes, fan, 1, [3, 0, 77]) == 1
            assert q.spread_copy_count() - before == spread, nbytes
