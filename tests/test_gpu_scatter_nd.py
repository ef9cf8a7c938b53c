"""scatter_nd through the torch op and the C ABI against the CPU oracle.  Shapes follow
tests/python/test_scatter_nd.py (data [7,8,9,10], 5 index rows of depth 2, three dtypes); unlike
that test the tensors keep their shapes and the expectation is accumulation, which is what the
reference kernel computes."""

import pytest
import torch

from oracle import numerics as N

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=lambda d: str(d).split(".")[-1])
@pytest.mark.parametrize("depth", [1, 2, 4])
def test_scatter_nd_accumulates(dtype, depth):
    from tilefusion_amd.ops import scatter_nd
    g = torch.Generator().manual_seed(1234 + depth)
    shape = [7, 8, 9, 10]
    data = torch.full(shape, 5.0, dtype=dtype)
    rows = 5 if depth < 4 else 300
    idx = torch.stack([torch.randint(0, shape[j], (rows,), generator=g) for j in range(depth)], dim=1)
    idx[1] = idx[0]                                               # a duplicate row must accumulate
    upd = torch.randint(-4, 5, (rows, *shape[depth:]), generator=g).to(dtype)   # small integers: exact in bf16
    want = N.scatter_nd_ref(data, idx, upd)
    dev = data.to(DEV)
    scatter_nd(dev, idx.to(DEV), upd.to(DEV))
    assert torch.equal(dev.float().cpu(), want)


def test_out_of_range_rows_are_skipped_and_shapes_checked():
    from tilefusion_amd.ops import scatter_nd
    data = torch.zeros(4, 6, device=DEV)
    idx = torch.tensor([[1], [9], [-1], [3]], device=DEV)
    upd = torch.ones(4, 6, device=DEV)
    scatter_nd(data, idx, upd)
    assert data.sum().item() == 12 and data[1].sum().item() == 6 and data[3].sum().item() == 6
    with pytest.raises(RuntimeError, match="updates must hold"):
        scatter_nd(data, idx, torch.ones(3, 6, device=DEV))
    with pytest.raises(RuntimeError, match="int64"):
        scatter_nd(data, idx.int(), upd)


# Up to 1024 updates go straight to memory; beyond, workgroups sort 16 at a time (a few 16-bit updates, up to 2048) or own a
# share of the targets of a chunk; lanes take words of 32
# bits, so odd slices and an odd start of a 16-bit array split pairs.  Values of
# -1, 0, 1 keep every partial sum well below 256 (the hottest row takes 1367 of them: a standard
# deviation of 30): exact in all types, whatever the order.
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=lambda d: str(d).split(".")[-1])
@pytest.mark.parametrize("rows,slice_,n,start", [(5, 1, 1, 0), (7, 3, 17, 1), (300, 130, 1024, 0), (300, 131, 1025, 1),
                                                 (300, 64, 2048, 0), (3000, 66, 2049, 0), (2000, 257, 4100, 1),
                                                 (3000, 1290, 4096, 0), (64, 33, 2500, 0), (40, 128, 2500, 0)])
def test_scatter_nd_sorted_workgroups(dtype, rows, slice_, n, start):
    from tilefusion_amd.ops import scatter_nd
    g = torch.Generator().manual_seed(rows + n)
    data = torch.randint(-2, 3, (rows, slice_), generator=g).to(dtype)
    idx = torch.randint(0, rows, (n, 1), generator=g)
    idx[::3] = rows // 2                                          # a row hit in every workgroup
    upd = torch.randint(-1, 2, (n, slice_), generator=g).to(dtype)
    want = N.scatter_nd_ref(data, idx, upd)
    bad = torch.cat([idx, torch.tensor([[rows], [-1]])])          # skipped
    upd = torch.cat([upd, torch.ones(2, slice_, dtype=dtype)])
    buf = torch.full((start + data.numel() + 1,), 3.0, dtype=dtype, device=DEV)
    dev = buf[start:start + data.numel()].view(rows, slice_)
    dev.copy_(data)
    scatter_nd(dev, bad.to(DEV), upd.to(DEV))
    assert torch.equal(dev.float().cpu(), want)
    assert buf[-1].item() == 3.0 and (start == 0 or buf[0].item() == 3.0)


# Owners of targets: one and several chunks of 1024 and 2048 updates, the last as long as the others or shorter, chunks of 4096
# from 20000 on, slices of a few lanes, of one word a lane and two, of more column ranges than one, indices of one and of three numbers, all updates to one target, and to none.
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=lambda d: str(d).split(".")[-1])
@pytest.mark.parametrize("dims,depth,n,start", [
    ((500, 40), 1, 2048, 0), ((500, 3), 1, 2049, 1), ((6, 5, 7, 260), 3, 4097, 0), ((3000, 517), 1, 4096, 1), ((300, 1026), 1, 2500, 0),
    ((1200, 34), 1, 9001, 1), ((5000, 66), 1, 19999, 0), ((5000, 65), 1, 20001, 0), ((70, 60, 130), 2, 20000, 0), ((2000, 8), 1, 33000, 0),
    ((900, 6), 1, 16385, 0)])
def test_scatter_nd_owners_of_targets(dtype, dims, depth, n, start):
    from tilefusion_amd.ops import scatter_nd
    g = torch.Generator().manual_seed(n + dims[0])
    data = torch.randint(-2, 3, dims, generator=g).to(dtype)
    idx = torch.stack([torch.randint(0, dims[j], (n,), generator=g) for j in range(depth)], dim=1)
    idx[::97] = torch.tensor([d // 2 for d in dims[:depth]])      # a target of every chunk
    idx[5], idx[n - 1] = -1, dims[0]                              # skipped
    upd = torch.randint(-1, 2, (n, *dims[depth:]), generator=g).to(dtype)
    keep = (idx >= 0).all(1) & (idx[:, 0] < dims[0])
    want = N.scatter_nd_ref(data, idx[keep], upd[keep])
    buf = torch.full((start + data.numel() + 1,), 3.0, dtype=dtype, device=DEV)
    dev = buf[start:start + data.numel()].view(dims)
    dev.copy_(data)
    scatter_nd(dev, idx.to(DEV), upd.to(DEV))
    assert torch.equal(dev.float().cpu(), want)
    assert buf[-1].item() == 3.0 and (start == 0 or buf[0].item() == 3.0)
    one = torch.zeros(3, *dims[depth:], dtype=dtype, device=DEV)   # every update to one target: alternating signs
    at = torch.ones(n, 1, dtype=torch.int64, device=DEV)
    sign = (1 - 2 * (torch.arange(n, device=DEV) % 2)).to(dtype).view(-1, *[1] * (len(dims) - depth))
    scatter_nd(one, at, (sign * torch.ones(n, *dims[depth:], dtype=dtype, device=DEV)).contiguous())
    assert torch.equal(one[1].float().cpu(), torch.full(dims[depth:], float(n % 2))) and not one[[0, 2]].any()
    scatter_nd(one, at * 3, sign.expand(n, *dims[depth:]).contiguous())
    assert not one[[0, 2]].any()


# Wide slices: each update for itself, sorted by 16, by 1024 and 2048 a chunk with a word or two a lane, around the numbers of updates, words
# and workgroups where one takes over.
# Sums of integers: at most ~1450 updates a target, none or one each way, keep every partial sum below 256 (8 deviations), which all types hold.
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=lambda d: str(d).split(".")[-1])
@pytest.mark.parametrize("rows,slice_,n", [(900, 1026, 4097), (900, 1024, 8193), (900, 514, 4097), (300, 4226, 4500), (200, 1154, 19999),
                                           (5000, 1030, 4096), (900, 4226, 400), (900, 6148, 1023), (300, 3090, 1025), (300, 1030, 1281), (900, 514, 2048)])
def test_scatter_nd_chunks_of_wide_slices(dtype, rows, slice_, n):
    from tilefusion_amd.ops import scatter_nd
    g = torch.Generator().manual_seed(rows + n)
    data = torch.randint(-2, 3, (rows, slice_), generator=g).to(dtype)
    idx = (rows * torch.rand(n, generator=g) ** 2).long()
    idx[5], idx[n - 1] = -1, rows                                 # skipped
    keep = (idx >= 0) & (idx < rows)
    upd = torch.randint(-1, 2, (n, slice_), generator=g).to(dtype)
    want = data.float().index_add(0, idx[keep], upd[keep].float())
    assert want.abs().max() <= 256
    dev = data.to(DEV)
    scatter_nd(dev, idx.unsqueeze(1).to(DEV), upd.to(DEV))
    assert torch.equal(dev.cpu().float(), want)


# Few but wide updates in one chunk, from the fewest on: rows x 32-bit words of a slice x updates, and what test_capi_cpu.py's plan says of
# them (1: a chunk of all, two of up to 1280; 0: one of the forms for fewer updates).
FEW_WIDE = [(60, 12290, 128, 1), (60, 12290, 127, 0), (64, 12288, 128, 1), (65, 12290, 128, 0), (3, 7500, 300, 1), (300, 65536, 256, 1),
            (300, 65535, 256, 0), (2000, 16384, 1024, 1), (512, 3070, 1025, 1), (640, 2458, 1280, 1), (640, 2457, 1280, 0),
            (641, 2458, 1280, 0), (20, 24580, 131, 1)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=lambda d: str(d).split(".")[-1])
@pytest.mark.parametrize("rows,words,n,chunk", FEW_WIDE)
def test_scatter_nd_few_but_wide_updates(dtype, rows, words, n, chunk):
    g = torch.Generator(device=DEV).manual_seed(rows + n)
    slice_ = words * (4 // dtype.itemsize)
    data = torch.randint(-2, 3, (rows, slice_), device=DEV, generator=g).to(dtype)
    idx = (rows * torch.rand(n, device=DEV, generator=g) ** 2).long()
    idx[5], idx[n - 1], idx[n // 2] = -1, rows, rows - 1          # two of them skipped
    upd = torch.randint(-1, 2, (n, slice_), device=DEV, generator=g).to(dtype)
    keep = (idx >= 0) & (idx < rows)
    want = data.cpu().float().index_add_(0, idx[keep].cpu(), upd[keep].cpu().float())
    assert want.abs().max() <= 256                                # exact in every type, whatever the order
    from tilefusion_amd.ops import scatter_nd
    scatter_nd(data, idx.unsqueeze(1), upd)
    assert torch.equal(data.cpu().float(), want)


# Targets with a large part of a chunk's updates: half of them to one row, an eighth to a second and a thirtieth to a third, in
# chunks of 1024, 2048 and 4096 updates, one and two words a lane, unpaired halves, slices of one element.  All workgroups of a
# chunk have to agree on who adds what: every update once.
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=lambda d: str(d).split(".")[-1])
@pytest.mark.parametrize("rows,slice_,n,start", [
    (900, 20, 1281, 0), (900, 520, 2049, 0), (300, 1, 2500, 0), (300, 1, 9000, 1), (5000, 64, 4096, 0), (70, 33, 5000, 1), (2000, 1026, 3000, 0),
    (4000, 640, 9001, 0), (4000, 8, 8193, 0), (4000, 40, 20011, 0), (3000, 530, 20000, 0), (500, 7, 33001, 0), (8, 16, 24000, 0)])
def test_scatter_nd_hot_targets(dtype, rows, slice_, n, start):
    from tilefusion_amd.ops import scatter_nd
    g = torch.Generator().manual_seed(rows + n)
    data = torch.randint(-2, 3, (rows, slice_), generator=g).to(dtype)
    idx = torch.randint(0, rows, (n,), generator=g)
    u = torch.rand(n, generator=g)
    idx[u < 0.5], idx[(u >= 0.5) & (u < 0.625)], idx[(u >= 0.625) & (u < 0.658)] = rows // 3, rows - 1, 0
    idx[7], idx[n - 1] = -1, rows
    keep = (idx >= 0) & (idx < rows)
    upd = torch.randint(-1, 2, (n, slice_), generator=g).to(dtype)
    upd[(idx == rows // 3).nonzero()[100:, 0]] = 0.0               # sums stay exact in bf16 in any order
    upd[(idx == rows - 1).nonzero()[100:, 0]] = 0.0
    want = N.scatter_nd_ref(data, idx[keep].unsqueeze(1), upd[keep])
    assert float(want.abs().max()) <= 128
    for shift in (0, n // 3):                                      # the updates that count at the front, and elsewhere
        buf = torch.full((start + data.numel() + 1,), 3.0, dtype=dtype, device=DEV)
        dev = buf[start:start + data.numel()].view(rows, slice_)
        dev.copy_(data)
        scatter_nd(dev, idx.roll(shift).unsqueeze(1).to(DEV), upd.roll(shift, 0).to(DEV))
        assert torch.equal(dev.float().cpu(), want)
        assert buf[-1].item() == 3.0 and (start == 0 or buf[0].item() == 3.0)


# Updates of one target are added up, 128 at least, before they are rounded to the target's type: whole numbers up to
# 256 times 128 come out exactly in bf16, which added eight at a time stop at 2048.
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=lambda d: str(d).split(".")[-1])
@pytest.mark.parametrize("n", [4096, 8192, 16384, 24576])
@pytest.mark.parametrize("slice_", [1, 33, 40, 520])
def test_scatter_nd_sums_one_target_before_rounding(dtype, n, slice_):
    from tilefusion_amd.ops import scatter_nd
    data = torch.zeros(300, slice_, dtype=dtype, device=DEV)
    scatter_nd(data, torch.full((n, 1), 150, device=DEV), torch.ones(n, slice_, dtype=dtype, device=DEV))
    assert torch.equal(data[150].float(), torch.full((slice_,), float(n), device=DEV))
    assert not data[:150].any() and not data[151:].any()


# Few targets, each with many updates: they are rounded no more often than by workgroups that add up 128 updates as they come, one
# rounding a target and workgroup.  (Errors against 64 bits of four draws together: 0.97 to 1.06 of that; 1.20 to 1.36 with the ends of a
# target's run rounded by themselves.)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=lambda d: str(d).split(".")[-1])
@pytest.mark.parametrize("rows,slice_,n", [(2, 702, 3224), (3, 694, 5493), (3, 329, 2494), (3, 276, 3496), (7, 218, 14576)])
def test_scatter_nd_rounds_a_run_of_one_target_once(dtype, rows, slice_, n):
    from tilefusion_amd.ops import scatter_nd
    square, allowed = 0.0, 0.0
    for seed in range(4):
        g = torch.Generator().manual_seed(rows + n + seed)
        idx = torch.randint(0, rows, (n,), generator=g)
        data = torch.randn(rows, slice_, generator=g).to(dtype)
        upd = (torch.randn(n, slice_, generator=g) / 64).to(dtype)
        exact = data.double().index_add_(0, idx, upd.double())
        dev = data.to(DEV)
        scatter_nd(dev, idx.unsqueeze(1).to(DEV), upd.to(DEV))
        model = data.clone()
        for i in range(0, n, 128):
            part = torch.zeros(rows, slice_).index_add_(0, idx[i:i + 128], upd[i:i + 128].float())
            model = (model.float() + part.to(dtype).float()).to(dtype)
        square += float((dev.double().cpu() - exact).square().sum())
        allowed += float((model.double() - exact).square().sum())
    assert square <= 1.15 ** 2 * allowed


def test_scatter_nd_fp16_sum_of_duplicates_beyond_its_range():
    from tilefusion_amd.ops import scatter_nd
    data = torch.full((2, 2), -60000.0, dtype=torch.float16, device=DEV)
    upd = torch.full((2, 2), 60000.0, dtype=torch.float16, device=DEV)
    scatter_nd(data, torch.tensor([[1], [1]], device=DEV), upd)
    assert data[1].tolist() == [60000.0, 60000.0] and data[0].tolist() == [-60000.0, -60000.0]


@pytest.mark.parametrize("dtype,big", [(torch.float32, 3e38), (torch.float16, 60000.0), (torch.bfloat16, 3e38)],
                         ids=["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("slice_", [4, 5])
@pytest.mark.parametrize("n", [1500, 2500])
def test_scatter_nd_sums_beyond_the_range_of_the_type(dtype, big, slice_, n):
    # the sum of the two updates is beyond the type's range, the result is not; sums with infinities stay theirs
    from tilefusion_amd.ops import scatter_nd
    data = torch.zeros(1000, slice_, dtype=dtype, device=DEV)
    data[7] = -big
    upd = torch.zeros(n, slice_, dtype=dtype, device=DEV)
    idx = 8 + torch.arange(n, device=DEV) % 900
    idx[[3, 9, 5, 6]] = torch.tensor([7, 7, 950, 950], device=DEV)
    upd[[3, 9]], upd[5], upd[6] = big, float("inf"), 1.0
    want = data.clone()
    want[7], want[950] = upd[3], float("inf")
    scatter_nd(data, idx.unsqueeze(1), upd)
    assert torch.equal(data, want)


# Of a word of two 16-bit elements a slice may hold one: the other one, of a neighbouring row, keeps its value
# (the smallest subnormal number here), and memory outside the tensor its bits, also those of a signalling NaN.
@pytest.mark.parametrize("dtype,bits", [(torch.float16, 0x7D01), (torch.bfloat16, 0x7F81), (torch.float32, 0x7F800001)],
                         ids=["float16", "bfloat16", "float32"])
@pytest.mark.parametrize("start", [0, 1, 2, 3])
@pytest.mark.parametrize("slice_", [1, 3, 66, 131])
@pytest.mark.parametrize("n", [2, 1500])
@pytest.mark.parametrize("rows_,first,second", [(5, 0, 4), (5, 1, 3), (6, 0, 5), (6, 2, 3)])   # odd and even totals
def test_scatter_nd_leaves_what_lies_next_to_a_slice_alone(dtype, bits, start, slice_, n, rows_, first, second):
    from tilefusion_amd.ops import scatter_nd
    ints = torch.int32 if dtype == torch.float32 else torch.int16
    buf = torch.full((start + rows_ * slice_ + 3,), bits, dtype=ints, device=DEV)
    inside = buf[start:start + rows_ * slice_]
    inside.fill_(1)
    data = inside.view(dtype).view(rows_, slice_)
    data[first], data[second] = 1.0, 2.0
    want = buf.clone()
    rows = want.view(dtype)[start:start + rows_ * slice_].view(rows_, slice_)
    rows[first], rows[second] = 4.0, 6.0
    upd = torch.zeros(n, slice_, dtype=dtype, device=DEV)
    upd[0], upd[1] = 3.0, 4.0
    scatter_nd(data, (torch.arange(n, device=DEV) % 2 * (second - first) + first).unsqueeze(1), upd)
    assert torch.equal(buf, want)


@pytest.mark.parametrize("dtype,tiny", [(torch.float16, 2.0 ** -24), (torch.bfloat16, 2.0 ** -133), (torch.float32, 2.0 ** -149)],
                         ids=["float16", "bfloat16", "float32"])
@pytest.mark.parametrize("slice_", [8, 7])
@pytest.mark.parametrize("n", [3, 1500, 3000])
def test_scatter_nd_adds_subnormal_numbers_exactly(dtype, tiny, slice_, n):
    from tilefusion_amd.ops import scatter_nd
    data = ((torch.arange(64 * slice_) % 7).double() * tiny).to(dtype).view(64, slice_)
    idx = torch.arange(n) % 64
    upd = ((torch.arange(n * slice_) % 5 - 2).double() * tiny).to(dtype).view(n, slice_)
    want = data.double().index_add(0, idx, upd.double())
    dev = data.to(DEV)
    scatter_nd(dev, idx.unsqueeze(1).to(DEV), upd.to(DEV))
    assert torch.equal(dev.double().cpu(), want)


# Hardware floating-point atomics are defined for a device's ordinary memory only.  Elsewhere every element
# is added by compare-and-swap, which shows in the rows next to an odd slice: a signalling NaN keeps its bits.
@pytest.mark.parametrize("dtype,bits", [(torch.float16, 0x7D01), (torch.bfloat16, 0x7F81), (torch.float32, 0x7F800001)],
                         ids=["float16", "bfloat16", "float32"])
@pytest.mark.parametrize("slice_,n", [(5, 3), (64, 3000), (77, 5000)])
def test_scatter_nd_into_fine_grained_memory_adds_by_compare_and_swap(dtype, bits, slice_, n):
    import ctypes

    from tilefusion_amd import _capi
    hip = ctypes.CDLL("libamdhip64.so")
    rows, size = 9, torch.empty(0, dtype=dtype).element_size()
    ints = torch.int32 if size == 4 else torch.int16
    g = torch.Generator().manual_seed(n)
    host = torch.randint(-2, 3, (rows, slice_), generator=g).to(dtype)
    idx = torch.randint(0, rows, (n, 1), generator=g)
    idx[idx == 4] = 3                                             # row 4 is not hit
    host[4].view(ints).fill_(bits)
    upd = torch.randint(-1, 2, (n, slice_), generator=g).to(dtype)
    for i in range(rows):                                         # sums of hundreds of them stay exact: 0 for most
        upd[(idx[:, 0] == i).nonzero()[32:, 0]] = 0.0
    want = N.scatter_nd_ref(host, idx, upd)
    p, flags_fine_grained = ctypes.c_void_p(), 1
    assert hip.hipExtMallocWithFlags(ctypes.byref(p), ctypes.c_size_t(host.numel() * size), flags_fine_grained) == 0
    to_device, to_host = 1, 2
    assert hip.hipMemcpy(p, ctypes.c_void_p(host.data_ptr()), ctypes.c_size_t(host.numel() * size), to_device) == 0
    upd_d, idx_d = upd.to(DEV), idx.to(DEV)
    dims = (ctypes.c_int64 * 2)(rows, slice_)
    _capi.check(_capi.load().tf_scatter_nd(upd_d.data_ptr(), p, idx_d.data_ptr(), dims, 2, n, 1,
                                           {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}[dtype],
                                           torch.cuda.current_stream().cuda_stream), "tf_scatter_nd")
    torch.cuda.synchronize()
    got = torch.empty_like(host)
    assert hip.hipMemcpy(ctypes.c_void_p(got.data_ptr()), p, ctypes.c_size_t(host.numel() * size), to_host) == 0
    assert hip.hipFree(p) == 0
    assert (got[4].view(ints) == torch.tensor(bits, dtype=torch.int64).to(ints)).all()
    keep = [i for i in range(rows) if i != 4]
    assert torch.equal(got[keep].float(), want[keep])


def test_scatter_nd_in_a_graph():
    from tilefusion_amd.ops import scatter_nd
    g = torch.Generator().manual_seed(3)
    idx = torch.randint(0, 50, (1500, 1), generator=g).to(DEV)
    upd = torch.randint(-1, 2, (1500, 33), generator=g).to(torch.bfloat16).to(DEV)
    data, other = torch.zeros(50, 33, dtype=torch.bfloat16, device=DEV), torch.zeros(50, 33, dtype=torch.bfloat16, device=DEV)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        scatter_nd(data, idx, upd)
    for _ in range(3):
        data.zero_(), other.zero_()
        graph.replay()
        scatter_nd(other, idx, upd)
        torch.cuda.synchronize()
        assert torch.equal(data, other)
