"""By-value fold launches at the sizes where their block shape changes (blocks of four wavefronts
below 12,288 of them, an encode below 20,480; one-wavefront blocks above) and from where a large
launch of several streams keeps fewer waves on a CU (160 MB moved), bit for bit against the same
arithmetic in torch: one rounding to the operands' type after every operation, in order."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    from mccl_amd import kernels
    kernels.hip_kernels_init(0)
    return kernels


def operands(k, n, dtype, offset=0):
    g = torch.Generator(device="cuda").manual_seed(n + 17 * k)
    return [torch.randn(n + offset, generator=g, device="cuda").to(dtype)[offset:] for _ in range(k)]


def same(a, b):
    return torch.equal(a.contiguous().view(torch.int16), b.contiguous().view(torch.int16))


@pytest.mark.parametrize("elems", [12_288 * 256 - 257, 12_288 * 256, 12_288 * 256 + 129, 20_480 * 256 - 1, 20_480 * 256 + 1])
@pytest.mark.parametrize("offset", [0, 1])
def test_one_and_two_operand_launches_around_the_change_of_block(K, elems, offset):
    x, = operands(1, elems, torch.float32, offset)
    wire = K.encode_bf16(x)
    assert same(wire, x.to(torch.bfloat16))
    for part in (wire, wire[:elems // 2 + 1]):       # a cast's wavefront covers twice as many elements
        assert same(K.decode_bf16(part), part.float())
    for dtype in (torch.float32, torch.bfloat16, torch.float16):
        a, b = operands(2, elems * (1 if dtype == torch.float32 else 2) + 3, dtype, offset)
        want = a * 0.25
        assert same(K.hip_scale_inplace(a.clone(), 0.25), want), dtype
        assert same(K.hip_reduce_op(a.clone(), b, "sum"), a + b), dtype


@pytest.mark.parametrize("k,dtype,n", [(3, torch.float32, 10_000_003), (4, torch.float32, 8_000_001), (6, torch.bfloat16, 11_500_007),
                                       (8, torch.bfloat16, 8_900_001), (8, torch.float16, 8_900_001), (5, torch.float32, 6_700_001)])
def test_many_operands_with_fewer_waves_resident(K, k, dtype, n):
    from mccl_amd import _lib as L
    q = K._q(None)
    ins = operands(k, n, dtype, 1)
    out = torch.full((n + 8,), 7.0, dtype=dtype, device="cuda")
    plan = K.make_plan(K.dtype_code(ins[0]), k)
    torch.cuda.synchronize()
    q.fold(plan, [K.make_seg(out.data_ptr(), 0, [t.data_ptr() for t in ins], n)])
    q.drain()
    want = ins[0]
    for t in ins[1:]:
        want = want + t
    assert same(out[:n], want) and bool((out[n:] == 7.0).all())


@pytest.mark.parametrize("world,fan", [(4, 3), (2, 6), (3, 0), (8, 0)])
def test_wire_folds_with_fewer_waves_resident(K, world, fan):
    """Own fp32 operand + bf16 peers, averaged, into one tensor or several."""
    from mccl_amd import _lib as L
    q = K._q(None)
    n = 9_500_003
    own, = operands(1, n, torch.float32)
    peers = operands(world - 1, n, torch.bfloat16)
    outs = [torch.full((n + 8,), 7.0, device="cuda") for _ in range(fan + 1)]
    plan = K.make_plan(L.BF16, world, io=L.IO_OWN_FIRST_F32, scale_mode=L.SCALE_VIEW, scale=0.25, fanout=fan)
    ins = [own.data_ptr()] + [p.data_ptr() for p in peers] + [o.data_ptr() for o in outs[1:]]
    torch.cuda.synchronize()
    q.fold(plan, [K.make_seg(outs[0].data_ptr(), 0, ins, n)])
    q.drain()
    want = own.to(torch.bfloat16)
    for p in peers:
        want = want + p
    want = (want * 0.25).float()
    for o in outs:
        assert same(o[:n], want) and bool((o[n:] == 7.0).all())
