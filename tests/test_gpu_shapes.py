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


@pytest.mark.parametrize("n", [1, 40, 300, 70_003, 3_200_017])
@pytest.mark.parametrize("own_off,wire_off", [(0, 32), (32, 0), (1, 1), (33, 1), (0, 7), (31, 63), (5, 4)])
def test_wire_operands_on_and_off_the_lines_of_the_output(K, n, own_off, wire_off):
    """The packet grid starts where the fp32 output and the first 16-bit operand both start a line
    of memory, if they ever do (elements off it are done one by one), and a large launch takes
    larger blocks if they do not."""
    from mccl_amd import _lib as L
    q = K._q(None)
    for k, last in ((2, False), (3, True), (4, False)):
        own, = operands(1, n, torch.float32, own_off)
        peers = operands(k - 1, n, torch.bfloat16, wire_off)
        outs = [torch.full((n + own_off + wire_off + 8,), 7.0, device="cuda") for _ in range(2)]
        wire = torch.full((n + wire_off + 8,), 7.0, dtype=torch.bfloat16, device="cuda")
        ops = peers + [own] if last else [own] + peers
        want = ops[0].to(torch.bfloat16)
        for t in ops[1:]:
            want = want + t.to(torch.bfloat16)
        want = want * 0.25
        kw = dict(io=L.IO_OWN_LAST_F32 if last else L.IO_OWN_FIRST_F32, scale_mode=L.SCALE_VIEW, scale=0.25)
        ins = [t.data_ptr() for t in ops]
        at = [o.data_ptr() + 4 * own_off for o in outs]
        torch.cuda.synchronize()
        q.fold(K.make_plan(L.BF16, k, **kw), [K.make_seg(at[0], wire.data_ptr() + 2 * wire_off, ins, n)])
        q.drain()
        assert same(outs[0][own_off:own_off + n], want.float()) and same(wire[wire_off:wire_off + n], want)
        for o in outs:
            o.fill_(7.0)
        torch.cuda.synchronize()
        q.fold(K.make_plan(L.BF16, k, fanout=1, **kw), [K.make_seg(at[0], 0, ins + [outs[1].data_ptr() + 4 * wire_off], n)])
        q.drain()
        for o, off in ((outs[0], own_off), (outs[1], wire_off)):
            assert same(o[off:off + n], want.float()) and bool((o[:off] == 7.0).all()) and bool((o[off + n:] == 7.0).all())
        assert bool((wire[:wire_off] == 7.0).all()) and bool((wire[wire_off + n:] == 7.0).all())


@pytest.mark.parametrize("n", [70_003, 5_300_021])
@pytest.mark.parametrize("f_off,h_off", [(0, 1), (1, 0), (32, 33), (3, 64)])
def test_codec_passes_on_and_off_the_lines(K, n, f_off, h_off):
    x, = operands(1, n, torch.float32, f_off)
    full = torch.full((n + h_off + 8,), 7.0, dtype=torch.bfloat16, device="cuda")
    K.encode_bf16(x, out=full[h_off:h_off + n])
    want = x.to(torch.bfloat16)
    assert same(full[h_off:h_off + n], want) and bool((full[:h_off] == 7.0).all()) and bool((full[h_off + n:] == 7.0).all())
    back = torch.full((n + f_off + 8,), 7.0, device="cuda")
    K.decode_bf16(full[h_off:h_off + n], out=back[f_off:f_off + n])
    assert same(back[f_off:f_off + n], want.float()) and bool((back[:f_off] == 7.0).all()) and bool((back[f_off + n:] == 7.0).all())


def test_an_encode_of_more_elements_than_a_grid_has_threads_for(K):
    """A grid has at most 2^32 threads: one packet of four elements per lane ends at 2^34 elements."""
    n = 2**34 + 4099
    if torch.cuda.mem_get_info()[0] < 120 * 2**30:
        pytest.skip("needs 100 GB of device memory")
    x = torch.full((n,), 1.25, device="cuda")
    marks = [0, 1, 2**33 + 5, 2**34 - 1, 2**34, 2**34 + 4097, n - 1]
    for i, at in enumerate(marks):
        x[at] = float(i + 3)
    out = torch.zeros(n, dtype=torch.bfloat16, device="cuda")
    K.encode_bf16(x, out=out)
    del x
    assert [float(out[at]) for at in marks] == [float(i + 3) for i in range(len(marks))]
    for at in marks:
        out[at] = 1.25
    for lo in range(0, n, 2**31):
        assert bool((out[lo:lo + 2**31] == 1.25).all()), lo
    del out
    torch.cuda.empty_cache()


def test_a_fold_and_a_copy_longer_than_a_grid(K):
    from mccl_amd import _lib as L
    if torch.cuda.mem_get_info()[0] < 160 * 2**30:
        pytest.skip("needs 140 GB of device memory")
    q = K._q(None)
    n = 2**34 + 4099  # 64 GiB of fp32
    marks = [0, 1, 2**33 + 5, 2**34 - 1, 2**34, n - 1]
    a, b = torch.full((n,), 1.25, device="cuda"), torch.full((n,), 0.5, device="cuda")
    for i, at in enumerate(marks):
        a[at] = float(i + 3)

    def check(t, base, plus):
        assert [float(t[at]) for at in marks] == [i + 3 + plus for i in range(len(marks))]
        keep = [float(t[at]) for at in marks]
        for at in marks:
            t[at] = base
        for lo in range(0, n, 2**31):
            assert bool((t[lo:lo + 2**31] == base).all()), lo
        for at, v in zip(marks, keep):
            t[at] = v

    K.hip_reduce_op(a, b, "sum")
    check(a, 1.75, 0.5)
    torch.cuda.synchronize()
    q.copy(b.data_ptr(), a.data_ptr(), 4 * n)
    q.drain()
    check(b, 1.75, 0.5)
    b.zero_()
    torch.cuda.synchronize()
    q.copy_batched([(b.data_ptr(), a.data_ptr(), 4 * n)])
    q.drain()
    check(b, 1.75, 0.5)
    del a, b
    torch.cuda.empty_cache()
