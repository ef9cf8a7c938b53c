"""GPU parity of split-KV flash-decoding (split kernel + combine kernel) through the C ABI
against the fp32 CPU oracle.  Tolerance: rel-L2 <= 1e-3, max-abs <= 2e-2.
The reference has no decoding kernel: the oracle is the closed form, itself pinned by the
split/combine identity and an independent C loop (tests/test_oracle_numerics.py)."""

import ctypes
import math

import pytest
import torch

import oracle
from oracle import numerics as N
from tests.gpu_util import DEV, c_decode, stream
from tilefusion_amd import _capi, ops

pytestmark = pytest.mark.gpu


def _slices(bh, lkv):
    qs, ks, vs = zip(*[oracle.make_c5_decode_slice(i // 32, i % 32, kv_len=lkv) for i in range(bh)])
    return torch.stack(qs), torch.stack(ks), torch.stack(vs)


@pytest.mark.parametrize("bh,lkv,splits", [(4, 1000, 3), (2, 777, 64), (3, 1, 1), (3, 5, 8), (8, 4096, 1),
                                           (8, 4096, 64), (2, 32768, 64), (1, 20000, 7), (5, 128, 128),
                                           (2, 128, 1), (2, 256, 1), (2, 384, 1), (3, 129, 1), (3, 257, 2)])
def test_shapes_and_ragged_splits(bh, lkv, splits):
    q, k, v = _slices(bh, lkv)
    o = c_decode(q.to(DEV), k.to(DEV), v.to(DEV), splits)
    assert not torch.isnan(o).any()
    ok, r, m = N.check_close(o, N.flash_decode_ref(q, k, v))
    assert ok, f"rel_l2={r:.3e} max_abs={m:.3e}"


# The kernels are templates of the element type and the head dimension (the reference's 16-bit
# types, include/kernels/dispatch_macros.hpp:6-23).  bf16: the oracle consumes the bf16-rounded
# inputs in fp32, what is left is the rounding of the output to 8 mantissa bits (rel-L2 <= 4e-3,
# max-abs <= 4e-2); head dimension 64 puts two key rows in a 16-lane group (8-lane reductions).
@pytest.mark.parametrize("dtype,tol", [(torch.float16, (1e-3, 2e-2)), (torch.bfloat16, (4e-3, 4e-2))])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("bh,lkv,splits", [(4, 1000, 3), (3, 5, 8), (2, 32768, 64), (5, 128, 128), (3, 257, 2),
                                           (16, 4096, 16), (2, 2048, 1)])
def test_element_types_and_head_dimensions(dtype, tol, d, bh, lkv, splits):
    g = torch.Generator().manual_seed(bh * 100 + lkv + d)
    q = torch.randn(bh, d, generator=g).to(dtype)
    k = torch.randn(bh, lkv, d, generator=g).to(dtype)
    v = torch.randn(bh, lkv, d, generator=g).to(dtype)
    o = c_decode(q.to(DEV), k.to(DEV), v.to(DEV), splits)
    assert o.dtype == dtype and not torch.isnan(o).any()
    ref = N.flash_decode_ref(q, k, v, 1.0 / math.sqrt(d))
    assert N.rel_l2(o, ref) <= tol[0] and N.max_abs(o, ref) <= tol[1], (N.rel_l2(o, ref), N.max_abs(o, ref))


def test_one_hot_keys_pick_single_value_rows_exactly():
    # a key that dominates by a wide margin makes the output that key's value row, bit for bit,
    # in every type and head dimension (a wrong lane-group reduction or row mapping cannot hide)
    for dtype in (torch.float16, torch.bfloat16):
        for d in (64, 128):
            g = torch.Generator().manual_seed(d)
            bh, lkv = 6, 3000
            q = torch.zeros(bh, d); q[:, 0] = 8.0
            k = torch.zeros(bh, lkv, d)
            hot = torch.randint(0, lkv, (bh,), generator=g)
            k[torch.arange(bh), hot, 0] = 16.0          # logit 128 * scale against 0 everywhere else
            v = torch.randint(-8, 9, (bh, lkv, d), generator=g).float()
            o = c_decode(q.to(dtype).to(DEV), k.to(dtype).to(DEV), v.to(dtype).to(DEV), 7, 1.0)
            assert torch.equal(o.float().cpu(), v[torch.arange(bh), hot]), (dtype, d)


def test_scale_and_extreme_logits():
    q, k, v = _slices(4, 2048)
    for scale in (1.0, 1e-3, -0.2):
        o = c_decode(q.to(DEV), k.to(DEV), v.to(DEV), 16, scale)
        ok, r, m = N.check_close(o, N.flash_decode_ref(q, k, v, scale))
        assert ok, f"scale={scale}: rel_l2={r:.3e} max_abs={m:.3e}"


def test_split_count_invariance_and_invariants():
    q, k, v = _slices(4, 4096)
    qd, kd, vd = q.to(DEV), k.to(DEV), v.to(DEV)
    base = c_decode(qd, kd, vd, 1).float()
    for splits in (2, 16, 64, 257):
        assert (c_decode(qd, kd, vd, splits).float() - base).abs().max() < 2e-3
    assert (c_decode(qd, kd, torch.ones_like(vd), 64).float() - 1).abs().max() < 2e-3
    # one dominant key: the output is that key's value row
    k2 = k.clone(); k2[:, 1234] = q * 8
    o = c_decode(qd, k2.to(DEV), vd, 64)
    assert N.max_abs(o, v[:, 1234]) < 2e-3


def test_c5_full_size():
    # B16 H32 q1 KV32768 D128, 64 splits: 8 GiB of K,V are drawn on the device; a sample of
    # (batch, head) slices is copied back so the oracle consumes identical values, and other cuts
    # (3 ranges; none, finished in one kernel) give the same for every slice.
    bh, lkv, d = 512, 32768, 128
    g = torch.Generator(device=DEV).manual_seed(oracle.SEEDS["c5"])
    q = torch.randn(bh, d, device=DEV, dtype=torch.float16, generator=g)
    k = torch.randn(bh, lkv, d, device=DEV, dtype=torch.float16, generator=g)
    v = torch.randn(bh, lkv, d, device=DEV, dtype=torch.float16, generator=g)
    o = c_decode(q, k, v, 64)
    assert not torch.isnan(o).any()
    for i in (0, 100, 255, 511):
        ok, r, m = N.check_close(o[i], N.flash_decode_ref(q[i].cpu(), k[i].cpu(), v[i].cpu()))
        assert ok, f"slice {i}: rel_l2={r:.3e} max_abs={m:.3e}"
    for splits in (3, 1):
        assert (o.float() - c_decode(q, k, v, splits).float()).abs().max() < 1e-3


# Not cut: one kernel that leaves the workspace alone.
@pytest.mark.parametrize("bh,lkv,d,splits", [(127, 2111, 128, 64), (128, 1500, 128, 2), (200, 4099, 128, 3), (520, 63, 64, 3)])
def test_uncut_slices_take_no_workspace(bh, lkv, d, splits):
    lib, waves = _capi.load(), ctypes.c_int()
    assert lib.tf_flash_decode_plan(bh, lkv, d, splits, ctypes.byref(waves)) == 1
    g = torch.Generator(device=DEV).manual_seed(lkv)
    q, k, v = (torch.randn(*shape, device=DEV, generator=g).half() for shape in ((bh, d), (bh, lkv, d), (bh, lkv, d)))
    ws = torch.full((lib.tf_flash_decode_workspace_bytes(bh, d, splits) + 256 * bh,), 0xA5, device=DEV, dtype=torch.uint8)
    o = torch.empty_like(q)
    _capi.check(lib.tf_flash_decode(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), 1, ws.data_ptr(), ws.numel(), bh, lkv, d,
                                    splits, 1.0 / math.sqrt(d), stream()), "tf_flash_decode")
    assert (ws == 0xA5).all() and torch.equal(o, ops.flash_decode(q, k, v, splits))


# The cut is the library's: one workgroup of 8 or (from 512 slices on) 4 wavefronts per slice and no
# partials, or up to num_splits ranges reduced by workgroups of 8 (fewer than 1024 of them) or 4
# wavefronts; slices of more than 4 MiB, 2.75 GB together, come in ranges of 2 MiB in any case.  Lengths around the
# rows of a load step (32 or 64) and of the two batches in flight.
CUTS = [(3, 31, 128, 64), (3, 65, 64, 64), (513, 33, 128, 64), (520, 63, 64, 3),
        (600, 300, 64, 64), (4, 2047, 128, 64), (5, 4097, 64, 64),
        (2, 9000, 128, 2), (40, 6000, 64, 64), (270, 2100, 128, 9), (1, 1, 64, 2),
        (136, 4099, 64, 64), (256, 8192, 128, 64), (256, 8193, 128, 64), (768, 8200, 128, 64),
        (250, 17001, 64, 2), (130, 16500, 64, 64)]


@pytest.mark.parametrize("dtype,tol", [(torch.float16, (1e-3, 2e-2)), (torch.bfloat16, (4e-3, 4e-2))])
@pytest.mark.parametrize("bh,lkv,d,splits", CUTS)
def test_every_way_to_cut(bh, lkv, d, splits, dtype, tol):
    g = torch.Generator(device=DEV).manual_seed(bh + lkv)
    q = torch.randn(bh, d, device=DEV, generator=g).to(dtype)
    k = torch.randn(bh, lkv, d, device=DEV, generator=g).to(dtype)
    v = torch.randn(bh, lkv, d, device=DEV, generator=g).to(dtype)
    scores = (k.float() * q.float()[:, None]).sum(-1) / math.sqrt(d)
    ref = (torch.softmax(scores, -1)[..., None] * v.float()).sum(1)
    o = c_decode(q, k, v, splits)
    assert o.dtype == dtype and N.rel_l2(o, ref) <= tol[0] and N.max_abs(o, ref) <= tol[1]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bh,lkv,d,splits", [(8, 4096, 128, 64), (8, 4096, 64, 64), (4, 8192, 128, 5), (300, 8192, 64, 64),
                                             (3, 1001, 128, 1), (3, 4099, 64, 7), (520, 1003, 128, 64), (4, 9, 64, 3)])
def test_infinite_values_in_any_split_stay_infinite(bh, lkv, d, splits, dtype):
    # every weight is positive: an infinite value makes its column that infinity, whichever split holds it
    g = torch.Generator(device=DEV).manual_seed(lkv + d)
    q, k, v = (torch.randn(*shape, device=DEV, generator=g).to(dtype) for shape in ((bh, d), (bh, lkv, d), (bh, lkv, d)))
    v[:, 0, 1], v[:, lkv // 2, 2], v[:, lkv - 1, 3] = math.inf, -math.inf, math.inf
    o = c_decode(q, k, v, splits)
    want = torch.zeros(d, device=DEV)
    want[1], want[2], want[3] = math.inf, -math.inf, math.inf
    assert torch.equal(torch.where(o.isfinite(), torch.zeros_like(o), o).float(), want.expand(bh, d))


@pytest.mark.parametrize("dtype,tol", [(torch.float16, (1e-3, 2e-2)), (torch.bfloat16, (4e-3, 4e-2))])
@pytest.mark.parametrize("start", [1, 2, 5])
@pytest.mark.parametrize("bh,lkv,d,splits", [(5, 301, 128, 64), (5, 4097, 64, 64), (3, 2000, 128, 1)])
def test_operands_that_start_anywhere(bh, lkv, d, splits, start, dtype, tol):
    # operands at the alignment of their elements, between numbers that must not count
    g = torch.Generator(device=DEV).manual_seed(start + lkv)

    def inside(*shape):
        n = math.prod(shape)
        buf = torch.full((n + 16,), 100.0, device=DEV, dtype=dtype)
        x = buf[start:start + n].view(*shape)
        return x.copy_(torch.randn(*shape, device=DEV, generator=g))

    q, k, v = inside(bh, d), inside(bh, lkv, d), inside(bh, lkv, d)
    assert k.data_ptr() % 16 == start * 2
    scores = (k.float() * q.float()[:, None]).sum(-1) / math.sqrt(d)
    ref = (torch.softmax(scores, -1)[..., None] * v.float()).sum(1)
    o = c_decode(q, k, v, splits)
    assert N.rel_l2(o, ref) <= tol[0] and N.max_abs(o, ref) <= tol[1]


# Where the workspace has 256 bytes a slice beyond the partials of the ranges taken, the workgroup that is done last puts a slice together,
# instead of a second kernel: the same sums in the same order, so the same bits, whatever the workspace held before.  Two and many
# ranges, more than one turn of the loop that merges them (64 at D = 128, 128 at 64), up to 1023 workgroups.  The two kernels it is
# compared with are those that a workspace outside the device's memory gets.
MERGED = [(1, 30000, 128, 64), (3, 1001, 64, 2), (32, 1999, 64, 64), (1, 31360, 128, 70), (1, 38400, 64, 150), (100, 8192, 128, 2),
          (127, 8192, 64, 2), (341, 8192, 64, 3), (2, 40000, 64, 257)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bh,lkv,d,splits", MERGED)
def test_last_workgroup_merges(bh, lkv, d, splits, dtype):
    g = torch.Generator(device=DEV).manual_seed(lkv)
    q, k, v = (torch.randn(*shape, device=DEV, generator=g).to(dtype) for shape in ((bh, d), (bh, lkv, d), (bh, lkv, d)))
    lib, code = _capi.load(), 2 if dtype == torch.bfloat16 else 1
    partials = lib.tf_flash_decode_workspace_bytes(bh, d, splits)
    nbytes = partials + 256 * bh
    o = torch.empty_like(q)

    def run(ws):
        o.fill_(math.nan)
        _capi.check(lib.tf_flash_decode(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), code, ws.data_ptr(), ws.numel(),
                                        bh, lkv, d, splits, 1.0 / math.sqrt(d), stream()), "tf_flash_decode")

    host = torch.empty(partials, dtype=torch.uint8, pin_memory=True)
    run(host)
    torch.cuda.synchronize()
    want = o.clone()
    assert torch.equal(c_decode(q, k, v, splits), want) and not torch.isnan(want).any()
    # it does merge: the last to arrive leaves a zero behind
    ranges = lib.tf_flash_decode_plan(bh, lkv, d, splits, ctypes.byref(ctypes.c_int()))
    ws = torch.full((nbytes,), 0xA5, device=DEV, dtype=torch.uint8)
    run(ws)
    words = ws[lib.tf_flash_decode_workspace_bytes(bh, d, ranges):][:256 * bh].view(bh, 256)
    assert not words[:, :8].any() and (words[:, 8:] == 0xA5).all()

    for held in (0, 255, 1, None):
        ws = torch.randint(0, 256, (nbytes,), device=DEV, dtype=torch.uint8, generator=g)
        if held is not None:
            ws.fill_(held)
        for _ in range(3):
            run(ws)
            assert torch.equal(o, want)
    assert torch.equal(ops.flash_decode(q.unsqueeze(1), k, v, splits).squeeze(1), want)
    # replays, with other contents of the workspace and eager calls between them
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        run(ws)
    for i in range(4):
        ws.fill_(37 * i)
        graph.replay()
        graph.replay()
        assert torch.equal(o, want)
        assert torch.equal(ops.flash_decode(q, k, v, splits), want)


def test_output_has_the_strides_of_the_query():
    # also those of extents of 1, whichever way the wrapper takes
    k, v = (torch.randn(3, 65, 64, device=DEV, dtype=torch.float16) for _ in range(2))
    long = torch.randn(3, 10, 64, device=DEV, dtype=torch.float16)
    for q, key, value in ((long[:1, :1], k[:1], v[:1]), (long[:1, :1].squeeze(1), k[:1], v[:1]), (long[:, 2], k, v),
                          (long[:, :1].contiguous(), k, v), (long[:1, 3:4], k[:1], v[:1])):
        out = ops.flash_decode(q, key, value, 4)
        assert out.shape == q.shape and out.stride() == torch.empty_like(q).stride()


def test_workspace_outside_device_memory_holds_partials_only():
    # whose arrivals are counted by atomics in memory that is ordinary for the device: elsewhere two kernels run, however large it is
    bh, lkv, d, splits = 3, 1001, 64, 2
    lib = _capi.load()
    assert lib.tf_flash_decode_plan(bh, lkv, d, splits, ctypes.byref(ctypes.c_int())) == splits
    g = torch.Generator(device=DEV).manual_seed(lkv)
    q, k, v = (torch.randn(*shape, device=DEV, generator=g).half() for shape in ((bh, d), (bh, lkv, d), (bh, lkv, d)))
    partials = lib.tf_flash_decode_workspace_bytes(bh, d, splits)
    ws = torch.empty(partials + 4096, dtype=torch.uint8, pin_memory=True).fill_(0xA5)
    o = torch.empty_like(q)
    _capi.check(lib.tf_flash_decode(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), 1, ws.data_ptr(), ws.numel(), bh, lkv, d,
                                    splits, 1.0 / math.sqrt(d), stream()), "tf_flash_decode")
    torch.cuda.synchronize()
    assert torch.equal(o, c_decode(q, k, v, splits))
    assert (ws[partials:] == 0xA5).all() and not (ws[:partials] == 0xA5).all()
