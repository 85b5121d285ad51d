"""The wire codec on one tensor, at the sizes where the number of packets a lane takes changes (in waves of one
packet a lane: three fifths, three quarters, one, one and a half, two, three and seven generations of the device), at
the edges of a tile and off the lines of memory, bit for bit: encode against torch's cast, decode against
the bits moved up by sixteen."""
import pytest
import torch

from mccl_amd import _lib as L
from mccl_amd import kernels as K

pytestmark = pytest.mark.gpu

GEN = 8192 * 256  # elements of one generation of waves on 256 compute units


def special(n, offset):
    """Random values with the ones a cast can get wrong spread through them, at the ends too."""
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn(n + offset, generator=g, device="cuda")[offset:]
    bits = torch.tensor([0x7FC00000, 0x7F800001, -0x3FFFFF, 0x7F800000, -0x800000, 0, -0x80000000, 1, 0x007FFFFF, 0x7F7FFFFF, 0x3F808000,
                         0x3F818000, 0x3F807FFF, 0x7F7F8000], dtype=torch.int32, device="cuda")
    at = torch.cat([torch.arange(0, n, 9973, device="cuda"), torch.arange(max(0, n - 70), n, device="cuda"),
                    torch.arange(0, min(n, 70), device="cuda")])
    x.view(torch.int32)[at] = bits[at % bits.numel()]
    return x


SIZES = [1, 3, 4, 63, 64, 65, 1023, 1025, 33_000, 40_001]
SIZES += [GEN * a // b + d for a, b in ((3, 5), (3, 4), (1, 1), (3, 2), (2, 1), (3, 1), (7, 1)) for d in (-1, 0, 1, 259)]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("src_off,dst_off", [(0, 0), (1, 0), (0, 3), (5, 7)])
def test_casts_at_every_change_of_shape(n, src_off, dst_off):
    q = K.hip_kernels_init(0)
    x = special(n, src_off)
    wire = torch.full((n + dst_off + 8,), -5.0, device="cuda", dtype=torch.bfloat16)
    torch.cuda.synchronize()
    L.check(L.lib().mcclx_encode_bf16(q.handle, wire.data_ptr() + 2 * dst_off, x.data_ptr(), n))
    q.drain()
    got = wire[dst_off:dst_off + n].view(torch.int16)
    want = x.to(torch.bfloat16).view(torch.int16)
    want[x != x] = 0x7FC0
    assert torch.equal(got, want)
    assert bool((wire[:dst_off] == -5).all()) and bool((wire[dst_off + n:] == -5).all())
    src = wire[dst_off:dst_off + n]
    src.view(torch.int16)[::1013] = 0x7F81   # NaN payloads go through a decode as they are
    back = torch.full((n + src_off + 8,), -5.0, device="cuda")
    torch.cuda.synchronize()
    L.check(L.lib().mcclx_decode_bf16(q.handle, back.data_ptr() + 4 * src_off, src.data_ptr(), n))
    q.drain()
    assert torch.equal(back[src_off:src_off + n].view(torch.int32), src.view(torch.int16).to(torch.int32) << 16)
    assert bool((back[:src_off] == -5).all()) and bool((back[src_off + n:] == -5).all())


@pytest.mark.parametrize("n", [GEN * 2 - 1, GEN * 2 + 1029, GEN * 3 + 1, GEN * 7 + 5])
def test_decode_into_pinned_host_memory(n):
    import ctypes
    import numpy as np
    q = K.hip_kernels_init(0)
    wire = special(n, 0).to(torch.bfloat16)
    host, dev = q.host_alloc(4 * n + 64)
    ctypes.memset(host, 0x5A, 4 * n + 64)
    torch.cuda.synchronize()
    L.check(L.lib().mcclx_decode_bf16(q.handle, dev, wire.data_ptr(), n))
    q.drain()
    got = np.ctypeslib.as_array((ctypes.c_uint32 * (n + 16)).from_address(host))
    want = wire.view(torch.int16).cpu().numpy().view(np.uint16).astype(np.uint32) << 16
    same = np.array_equal(got[:n], want) and bool((got[n:] == 0x5A5A5A5A).all())
    q.host_free(host)
    assert same


def test_the_same_plan_with_a_scale_or_two_outputs_is_not_taken_for_a_cast():
    q = K.hip_kernels_init(0)
    n = 50_003
    x = torch.randn(n, device="cuda")
    out, wire = torch.zeros(n, device="cuda"), torch.zeros(n, device="cuda", dtype=torch.bfloat16)
    torch.cuda.synchronize()
    plan = K.make_plan(L.BF16, 1, io=L.IO_OWN_FIRST_F32, scale_mode=L.SCALE_VIEW, scale=0.25)
    q.fold(plan, [K.make_seg(0, wire.data_ptr(), [x.data_ptr()], n)])
    q.drain()
    assert torch.equal(wire, x.to(torch.bfloat16) * 0.25)
    plan = K.make_plan(L.BF16, 1, io=L.IO_OWN_FIRST_F32)
    q.fold(plan, [K.make_seg(out.data_ptr(), wire.data_ptr(), [x.data_ptr()], n)])
    q.drain()
    assert torch.equal(wire, x.to(torch.bfloat16)) and torch.equal(out, wire.float())
    q.fold(plan, [K.make_seg(0, wire.data_ptr() + 2 * a, [x.data_ptr() + 4 * a], b) for a, b in ((0, 20_000), (20_000, 30_003))])
    q.drain()
    assert torch.equal(wire, x.to(torch.bfloat16))
