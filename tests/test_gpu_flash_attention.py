"""GPU parity of flash-attention forward through the C ABI against the fp32 CPU oracle.
Tolerance: rel-L2 <= 1e-3, max-abs <= 2e-2 (fp16 in/out, fp32 scores and statistics)."""

import math

import pytest
import torch

import oracle
from oracle import numerics as N
from tests.gpu_util import DEV, c_attention
from tilefusion_amd import _capi, ops

pytestmark = pytest.mark.gpu


def _inputs(b, lq, lkv, d, seed):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(b, lq, d, generator=g).half(), torch.randn(b, lkv, d, generator=g).half(),
            torch.randn(b, lkv, d, generator=g).half())


# tests/python/test_flash_attn.py:202-233: (Lq, Lkv, D, Dv) = (64,128,128,128) non-causal and
# (128,128,128,128) causal, tiles (64,128,128,128), seed 1234; V handed over transposed as the
# reference op receives it
@pytest.mark.parametrize("lq,lkv,causal", [(64, 128, False), (128, 128, True)])
@pytest.mark.parametrize("v_transposed", [True, False])
def test_reference_cases(lq, lkv, causal, v_transposed):
    q, k, v = _inputs(1, lq, lkv, 128, 1234)
    vd = v.transpose(1, 2).contiguous() if v_transposed else v
    o = c_attention(q.to(DEV), k.to(DEV), vd.to(DEV), causal, 1.0 / math.sqrt(128), v_transposed, (64, 128, 128, 128))
    ok, r, m = N.check_close(o, N.attention_ref(q, k, v, causal=causal))
    assert ok, f"rel_l2={r:.3e} max_abs={m:.3e}"


@pytest.mark.parametrize("b,lq,lkv,d", [(3, 200, 136, 128), (2, 1, 16, 128), (2, 128, 1000, 128), (1, 513, 513, 128),
                                        (2, 256, 512, 64), (4, 96, 72, 64), (1, 1024, 2048, 128),
                                        (2, 256, 512, 96), (3, 200, 136, 96), (1, 1024, 1100, 96), (2, 100, 40, 96)])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("v_transposed", [False, True])
def test_shapes(b, lq, lkv, d, causal, v_transposed):
    q, k, v = _inputs(b, lq, lkv, d, b * 7 + lq + lkv)
    vd = v.transpose(1, 2).contiguous() if v_transposed else v
    if v_transposed and lkv % 8:
        # rows of a transposed V must stay 16-byte aligned: rejected, not mis-computed
        with pytest.raises(RuntimeError, match="Lkv % 8"):
            c_attention(q.to(DEV), k.to(DEV), vd.to(DEV), causal, None, v_transposed)
        return
    o = c_attention(q.to(DEV), k.to(DEV), vd.to(DEV), causal, None, v_transposed)
    assert not torch.isnan(o).any()
    ok, r, m = N.check_close(o, N.attention_ref(q, k, v, causal=causal))
    assert ok, f"rel_l2={r:.3e} max_abs={m:.3e}"


# The 256- and 128-query workgroups keep a five-tile ring with two tiles live and request three tiles
# ahead: key ranges of one to seven tiles, with and without a ragged last tile, exercise its fill,
# the clamped requests past the end and the hand-over between the two wavefront sets; the 64-query workgroup has
# a ring of four tiles and one set.  (The number of slices decides which of them runs.)
RING_CASES = [(64, 2), (128, 128), (256, 256)]   # query rows per workgroup, slices of 256 queries


@pytest.mark.parametrize("lkv", [8, 64, 72, 128, 192, 200, 256, 320, 384, 448])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("rows,b", RING_CASES)
def test_short_key_ranges_through_the_eight_wavefront_ring(rows, b, lkv, causal):
    assert _capi.load().tf_flash_attention_rows(b, 256, lkv, 128, int(causal)) == rows
    q, k, v = _inputs(b, 256, lkv, 128, 900 + lkv)
    o = c_attention(q.to(DEV), k.to(DEV), v.to(DEV), causal, None, False)
    assert not torch.isnan(o).any()
    pick = sorted({0, b // 2, b - 1})
    ok, r, m = N.check_close(o[pick], N.attention_ref(q[pick], k[pick], v[pick], causal=causal))
    assert ok, f"rel_l2={r:.3e} max_abs={m:.3e}"


# Single causal tiles of 64 queries: an odd and an even number of them, a ragged last one.
@pytest.mark.parametrize("lq,d", [(512, 128), (768, 128), (1024, 64), (300, 128), (512, 96), (768, 96)])
def test_causal_pass_orders(lq, d):
    q, k, v = _inputs(3, lq, lq, d, 77 + lq)
    o = c_attention(q.to(DEV), k.to(DEV), v.to(DEV), True, None, False)
    ok, r, m = N.check_close(o, N.attention_ref(q, k, v, causal=True))
    assert ok, f"rel_l2={r:.3e} max_abs={m:.3e}"


# Whole rounds of pairs (256 and 512 of them), a ragged last query tile, and a nearly empty last round that
# runs single tiles instead: every slice against the same slice alone, which is never paired (bit for bit).
@pytest.mark.parametrize("bh,lq", [(256, 512), (256, 500), (512, 300), (264, 512)])
@pytest.mark.parametrize("d", [64, 128])
def test_causal_pairs_and_single_tiles_agree(bh, lq, d):
    q, k, v = (x.to(DEV) for x in _inputs(bh, lq, lq, d, bh + lq + d))
    o = c_attention(q, k, v, True)
    for i in (0, 1, 7, 8, bh // 2, bh - 1):
        alone = c_attention(q[i:i + 1].contiguous(), k[i:i + 1].contiguous(), v[i:i + 1].contiguous(), True)
        assert torch.equal(o[i:i + 1], alone), i
    ok, r, m = N.check_close(o[-1:].cpu(), N.attention_ref(q[-1:].cpu(), k[-1:].cpu(), v[-1:].cpu(), causal=True))
    assert ok, f"rel_l2={r:.3e} max_abs={m:.3e}"


# Causal pairs and single tiles at every workgroup size and head dimension, with ragged last query and key tiles: the second
# pass of a pair fills the ring behind the clamped requests of the first.  Every order of K and V, and rows of
# fewer elements, against a slice alone, which runs single tiles (bit for bit), and the oracle.
PAIR_CASES = [(64, 512, 250, 256, 64), (128, 229, 385, 392, 64), (256, 512, 300, 304, 64),
              (64, 21, 1531, 1536, 96), (128, 52, 961, 968, 96), (256, 192, 300, 304, 96),
              (64, 26, 1100, 1104, 128), (128, 43, 1217, 1224, 128), (256, 192, 300, 304, 128)]
SINGLE_CASES = [(64, 5, 257, 264, 64), (128, 88, 129, 136, 64), (256, 88, 385, 392, 64),
                (64, 5, 257, 264, 96), (128, 88, 129, 136, 96), (256, 88, 257, 264, 96),
                (64, 5, 257, 264, 128), (128, 88, 129, 136, 128), (256, 88, 257, 264, 128)]


@pytest.mark.parametrize("rows,b,lq,lkv,d", PAIR_CASES + SINGLE_CASES)
@pytest.mark.parametrize("less", [0, 16])
def test_causal_forms(rows, b, lq, lkv, d, less):
    assert _capi.load().tf_flash_attention_rows(b, lq, lkv, d, 1) == rows
    e = d - less
    q, k, v = (x.to(DEV) for x in _inputs(b, lq, lkv, e, rows + b + lq + e))

    def natural(q, k, v):
        o = torch.full_like(q, float("nan"))
        torch.ops.tilefusion.flash_attention_fwd(q, k, v, o, e ** -0.5, True)
        return o
    o = natural(q, k, v)
    for i in (0, 7 % b, b // 2, b - 1):
        one = slice(i, i + 1)
        assert torch.equal(o[one], natural(q[one].contiguous(), k[one].contiguous(), v[one].contiguous())), i
    ok, r, m = N.check_close(o[-1:].cpu(), N.attention_ref(q[-1:].cpu(), k[-1:].cpu(), v[-1:].cpu(), causal=True))
    assert ok, f"rel_l2={r:.3e} max_abs={m:.3e}"
    assert not torch.isnan(o).any()
    if not less:
        assert torch.equal(ops.flash_attention(q, k.transpose(1, 2).contiguous(), v, 1, 1, d, d, d ** -0.5, True), o)
        assert torch.equal(c_attention(q, k, v.transpose(1, 2).contiguous(), True, None, True), o)


# A key stored [D, Lkv] is read as it is: the same products in the same order as on the transposed key, so the same
# bits; a length that is no multiple of 8, or a key that starts off a 16-byte boundary, takes the copy.
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("d", [64, 96, 128])
@pytest.mark.parametrize("lq,lkv", [(1, 8), (17, 72), (128, 64), (129, 128), (300, 200), (520, 520), (257, 333)])
@pytest.mark.parametrize("causal", [False, True])
def test_key_stored_transposed(lq, lkv, d, causal, dtype):
    q, k, v = (x.to(DEV, dtype) for x in _inputs(3, lq, lkv, d, lq + lkv + d))
    kt = k.transpose(-1, -2).contiguous()
    o = ops.flash_attention(q, kt, v, 1, 1, d, d, d ** -0.5, causal)
    want = ops.flash_attention(q, k.transpose(-1, -2), v, 1, 1, d, d, d ** -0.5, causal)
    assert torch.equal(o, want)
    odd = torch.empty(kt.numel() + 1, device=DEV, dtype=dtype)[1:].view_as(kt).copy_(kt)
    assert torch.equal(ops.flash_attention(q, odd, v, 1, 1, d, d, d ** -0.5, causal), want)
    rel = 1e-3 if dtype == torch.float16 else 4e-3
    ref = N.attention_ref(q.cpu(), k.cpu(), v.cpu(), causal=causal)
    assert (o.float().cpu() - ref.float()).norm() <= rel * ref.float().norm()


# The copy of a key [D, Lkv] that no kernel reads as it is: edges of the 64 x 64 tiles, rows off every boundary, the
# stores of 16 bytes (D a multiple of 8) and of 2.  Nothing beyond the copy may be written.
@pytest.mark.parametrize("b,rows,cols", [(1, 1, 1), (2, 7, 9), (3, 64, 64), (2, 72, 65), (1, 63, 127), (4, 160, 333),
                                         (2, 256, 96), (5, 130, 70), (70, 80, 3)])
def test_transposed_copy(b, rows, cols):
    x = torch.randint(-2 ** 15, 2 ** 15, (b * rows * cols + 1,), dtype=torch.int16, device=DEV)
    for start in (0, 1):
        src = x[start:start + b * rows * cols].view(b, rows, cols)
        out = torch.full((b * rows * cols + 64,), 77, dtype=torch.int16, device=DEV)
        _capi.check(_capi.load().tf_transpose_16bit(src.data_ptr(), out.data_ptr(), b, rows, cols,
                                                    torch.cuda.current_stream().cuda_stream), "transpose")
        assert torch.equal(out[:-64].view(b, cols, rows), src.transpose(1, 2))
        assert bool((out[-64:] == 77).all())


# Head dimensions between the tuned ones take the next tuned kernel on rows as they are: the bits of the operands padded
# with zeros, at every workgroup size and remainder, with K and V of other heads (and nothing of them) around; an
# infinity in the last chunk of K meets no zero of the padding, and no element beyond O is written.
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("b,lq,lkv,d", [(2, 1, 8, 40), (3, 17, 72, 80), (2, 64, 64, 88), (5, 129, 130, 72), (3, 300, 333, 104),
                                        (1, 513, 440, 48), (130, 128, 192, 80), (256, 250, 320, 112), (2, 70, 1, 56)])
@pytest.mark.parametrize("causal", [False, True])
def test_rows_between_head_dimensions(b, lq, lkv, d, causal, dtype):
    q, k, v = (x.to(DEV, dtype) for x in _inputs(b, lq, lkv, d, lq + lkv + d))
    k[0, lkv // 2, d - 1] = float("inf")
    store = torch.full((q.numel() + 64,), 77, device=DEV, dtype=dtype)
    _capi.check(_capi.load().tf_flash_attention_fwd_d8(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), store.data_ptr(),
        _capi.TF_DTYPE_F16 if dtype == torch.float16 else _capi.TF_DTYPE_BF16, b, lq, lkv, d,
        d ** -0.5, int(causal), torch.cuda.current_stream().cuda_stream), "between")
    pad = (64 if d < 64 else 96 if d < 96 else 128) - d
    want = c_attention(*(torch.nn.functional.pad(x, (0, pad)) for x in (q, k, v)), causal, d ** -0.5)[..., :d]
    o = store[:-64].view_as(q)
    assert torch.equal(o.isnan(), want.isnan()) and torch.equal(o.nan_to_num(), want.nan_to_num())
    assert bool((store[-64:] == 77).all())
    for key in (k.transpose(1, 2), k.transpose(1, 2).contiguous()):
        assert torch.equal(ops.flash_attention(q, key, v, 1, 1, d, d, d ** -0.5, causal).nan_to_num(), want.nan_to_num())
    if b > 1:
        ref = N.attention_ref(q[-1:].cpu(), k[-1:].cpu(), v[-1:].cpu(), causal=causal)
        assert (o[-1:].float().cpu() - ref.float()).norm() <= (1e-3 if dtype == torch.float16 else 4e-3) * ref.float().norm()


# Keys in parts (few queries, many keys), against 64 bits and the kernel on all keys, with the workspace full of NaN:
# remainders of queries, keys and parts, both orders of K, rows between the tuned sizes.  The error is that of 16-bit weights and
# results in either case: the same bound, and no more than 1.1 of the other's (samples of 16 x 40 elements and up).
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("b,lq,lkv,d", [(1, 16, 1500, 40), (1, 63, 5056, 128), (9, 65, 648, 128), (3, 129, 2001, 64),
                                        (12, 20, 1280, 96), (5, 300, 4104, 80), (70, 64, 4096, 128), (2, 1708, 1664, 96),
                                        (16, 63, 4096, 256), (3, 130, 1056, 192), (8, 250, 768, 160)])
def test_keys_in_parts(b, lq, lkv, d, dtype):
    lib, stream = _capi.load(), torch.cuda.current_stream().cuda_stream
    bytes_ = lib.tf_flash_attention_split_workspace(b, lq, lkv, d)
    assert bytes_ > 0
    q, k, v = (x.to(DEV, dtype) for x in _inputs(b, lq, lkv, d, lq + lkv + d))
    want = torch.softmax(q.double() @ k.double().transpose(1, 2).contiguous() * d ** -0.5, -1) @ v.double()
    code = _capi.TF_DTYPE_F16 if dtype == torch.float16 else _capi.TF_DTYPE_BF16
    if d in (64, 96, 128):
        whole = c_attention(q, k, v)
    elif d > 128:
        whole = torch.empty_like(q)
        _capi.check(lib.tf_flash_attention_fwd_wide(q.data_ptr(), k.data_ptr(), v.data_ptr(), whole.data_ptr(), code, b, lq, lkv,
                                                    d, d ** -0.5, 0, stream), "whole")
    else:
        whole = torch.empty_like(q)
        _capi.check(lib.tf_flash_attention_fwd_d8(q.data_ptr(), k.data_ptr(), v.data_ptr(), whole.data_ptr(), code, b, lq, lkv,
                                                  d, d ** -0.5, 0, stream), "whole")
    bound = 1.1 * (whole.double() - want).norm()
    for kt in (False, True):
        if kt and (lkv % 8 or d not in (64, 96, 128)):
            continue
        key = k.transpose(1, 2).contiguous() if kt else k
        room = torch.full((bytes_ // 4 + 64,), float("nan"), device=DEV)
        store = torch.full((q.numel() + 64,), 77, device=DEV, dtype=dtype)
        _capi.check(lib.tf_flash_attention_fwd_split(q.data_ptr(), key.data_ptr(), v.data_ptr(), store.data_ptr(), code, b, lq,
                                                     lkv, d, int(kt), d ** -0.5, room.data_ptr(), stream), "parts")
        o = store[:-64].view_as(q)
        assert (o.double() - want).norm() <= bound
        assert bool((store[-64:] == 77).all()) and bool(room[-64:].isnan().all())
        assert torch.equal(ops.flash_attention(q, k.transpose(1, 2) if not kt else key, v, 1, 1, d, d, d ** -0.5, False), o)


# ... a part whose scores are all -inf takes no weight, and a row without a score is NaN as it is in one piece
def test_keys_in_parts_without_scores():
    q, k, v = (x.to(DEV) for x in _inputs(2, 40, 4096, 64, 5))
    q[..., 0] = 1.0
    k[0, 512:3000, 0] = float("-inf")
    k[1, :, 0] = float("-inf")
    assert _capi.load().tf_flash_attention_split_workspace(2, 40, 4096, 64) > 0
    o = ops.flash_attention(q, k.transpose(1, 2), v, 1, 1, 64, 64, 0.125, False)
    whole = c_attention(q, k, v, False, 0.125)
    assert bool(o[1].isnan().all()) and bool(whole[1].isnan().all())
    assert (o[0].float() - whole[0].float()).norm() <= 1e-3 * whole[0].float().norm()


# The three workgroup sizes (256, 128, 64 query rows), at remainders of their tiles and of the key tiles, with all
# orders of K and V; the library's pick is checked with them.
@pytest.mark.parametrize("rows,b,lq,lkv,d", [
    (64, 2, 1, 8, 64), (64, 3, 63, 200, 96), (64, 2, 65, 64, 128), (64, 5, 257, 136, 64), (64, 3, 300, 328, 128),
    (128, 250, 128, 72, 64), (128, 130, 128, 192, 96), (128, 128, 129, 264, 128), (128, 64, 449, 448, 128),
    (128, 300, 70, 128, 64), (256, 256, 200, 200, 128), (256, 512, 513, 72, 64), (256, 256, 250, 320, 96)])
@pytest.mark.parametrize("causal", [False, True])
def test_every_workgroup_size(rows, b, lq, lkv, d, causal):
    if not causal:
        assert _capi.load().tf_flash_attention_rows(b, lq, lkv, d, 0) == rows
    q, k, v = _inputs(b, lq, lkv, d, rows + lq + lkv)
    o = c_attention(q.to(DEV), k.to(DEV), v.to(DEV), causal)
    pick = [0, b // 2, b - 1]
    ok, r, m = N.check_close(o[pick], N.attention_ref(q[pick], k[pick], v[pick], causal=causal))
    assert ok, f"rel_l2={r:.3e} max_abs={m:.3e}"
    vt = v.transpose(-1, -2).contiguous().to(DEV)
    assert torch.equal(c_attention(q.to(DEV), k.to(DEV), vt, causal, None, True), o)
    kt = k.transpose(-1, -2).contiguous().to(DEV)
    assert torch.equal(ops.flash_attention(q.to(DEV), kt, v.to(DEV), 1, 1, d, d, d ** -0.5, causal), o)


# Single causal tiles dealt by XCD (slice counts that 8 does not divide) and not, and pairs of 64-query tiles of wide
# heads: every tile of every slice is done once, with the bits of the slice alone.
@pytest.mark.parametrize("bh,lq", [(31, 320), (30, 160), (63, 192), (61, 544), (9, 96), (150, 384), (225, 256)])
@pytest.mark.parametrize("d", [64, 128, 192, 256])
def test_causal_orders_agree(bh, lq, d):
    q, k, v = (x.to(DEV) for x in _inputs(bh, lq, lq, d, bh + lq + d))
    o = torch.full_like(q, float("nan"))
    torch.ops.tilefusion.flash_attention_fwd(q, k, v, o, d ** -0.5, True)
    assert not torch.isnan(o).any()
    for i in (0, 7, 8, bh // 2, bh - 1):
        alone = torch.empty_like(o[i:i + 1])
        torch.ops.tilefusion.flash_attention_fwd(q[i:i + 1].contiguous(), k[i:i + 1].contiguous(), v[i:i + 1].contiguous(), alone,
                                                 d ** -0.5, True)
        assert torch.equal(o[i:i + 1], alone), i
    ref = torch.softmax((q.float() @ k.float().transpose(1, 2).contiguous() * d ** -0.5).masked_fill(
        torch.ones(lq, lq, dtype=torch.bool, device=DEV).triu(1), float("-inf")), -1) @ v.float()
    assert (o.float() - ref).norm() <= 1e-3 * ref.norm()


def test_scale_and_large_logits():
    # scale enters the logits; big logits need the running max (exp would overflow otherwise)
    q, k, v = _inputs(2, 128, 256, 128, 77)
    for scale in (1.0, 0.02, -0.1):
        o = c_attention(q.to(DEV), k.to(DEV), v.to(DEV), False, scale)
        ok, r, m = N.check_close(o, N.attention_ref(q, k, v, scale=scale))
        assert ok, f"scale={scale}: rel_l2={r:.3e} max_abs={m:.3e}"


@pytest.mark.parametrize("causal", [False, True])
def test_reference_maximum_moves_both_ways(causal):
    # The kernel starts every score at minus a lazily updated reference maximum.  Keys whose
    # scores are far below zero first, far above later (and the reverse) force the reference
    # down on the first tile and up by hundreds of log2 units afterwards; a stale reference
    # would underflow every weight to 0 (division by zero) or overflow fp16.
    g = torch.Generator().manual_seed(99)
    d, lq, lkv = 128, 256, 512
    q = torch.randn(1, lq, d, generator=g).half()
    k = torch.randn(1, lkv, d, generator=g).half()
    v = torch.randn(1, lkv, d, generator=g).half()
    q[..., 0] = 8.0                       # a strong common component ...
    ramp = torch.linspace(-6.0, 6.0, lkv)  # ... that the keys weight from very negative to very positive
    for direction in (1.0, -1.0):
        k2 = k.clone()
        k2[0, :, 0] = (direction * ramp).half()
        o = c_attention(q.to(DEV), k2.to(DEV), v.to(DEV), causal, 1.0)   # scale 1: logits span +-48
        assert not torch.isnan(o).any() and not torch.isinf(o).any()
        ok, r, m = N.check_close(o, N.attention_ref(q, k2, v, scale=1.0, causal=causal))
        assert ok, f"direction={direction}: rel_l2={r:.3e} max_abs={m:.3e}"


def test_invariants():
    q, k, v = _inputs(2, 256, 256, 128, 5)
    # causal row 0 sees only key 0
    o = c_attention(q.to(DEV), k.to(DEV), v.to(DEV), True)
    assert torch.equal(o[:, 0].cpu(), v[:, 0])
    # V = 1 -> every output is exactly 1 (weights sum to one)
    o = c_attention(q.to(DEV), k.to(DEV), torch.ones_like(v).to(DEV), False)
    assert (o.float() - 1).abs().max() < 2e-3
    # all keys equal -> mean of V
    keq = k[:, :1].expand(-1, 256, -1).contiguous()
    o = c_attention(q.to(DEV), keq.to(DEV), v.to(DEV), False)
    assert N.max_abs(o, v.float().mean(dim=1, keepdim=True).expand(-1, 256, -1)) < 2e-3


@pytest.mark.parametrize("causal", [False, True])
def test_c4_full_size(causal):
    # B2 H32 S4096 D128: all 64 slices on the GPU; the oracle runs on a sample of slices (a
    # 4096x4096 fp32 softmax each), every other slice is covered by the V = 1 property below
    q, k, v = oracle.make_c4_attention_inputs()
    qd, kd, vd = (t.reshape(64, 4096, 128).to(DEV) for t in (q, k, v))
    o = c_attention(qd, kd, vd, causal).cpu().reshape(2, 32, 4096, 128)
    assert not torch.isnan(o).any()
    for b, h in [(0, 0), (0, 17), (1, 5), (1, 31)]:
        ok, r, m = N.check_close(o[b, h], N.attention_ref(q[b, h], k[b, h], v[b, h], causal=causal))
        assert ok, f"slice ({b},{h}) causal={causal}: rel_l2={r:.3e} max_abs={m:.3e}"
    ones = c_attention(qd, kd, torch.ones_like(vd), causal)
    assert (ones.float() - 1).abs().max() < 2e-3


def test_large_scale_and_large_q_stay_finite():
    # The tuned kernels fold scale * log2(e) into an fp16 copy of Q.  |Q * scale * 1.4427| beyond
    # 65504 saturates instead of turning into inf / NaN scores; well inside the range (here up to
    # ~600) the result still matches the oracle, whose softmax is then nearly one-hot.
    g = torch.Generator().manual_seed(5)
    q = (torch.randn(2, 128, 128, generator=g) * 30).half()
    k = torch.randn(2, 256, 128, generator=g).half()
    v = torch.randn(2, 256, 128, generator=g).half()
    o = c_attention(q.to(DEV), k.to(DEV), v.to(DEV), scale=4.0)
    assert torch.isfinite(o).all()
    ref = N.attention_ref(q, k, v, 4.0)
    # rows whose winning key leads by a clear margin are that key's value row
    logits = (q.float() @ k.float().transpose(1, 2)) * 4.0
    top2 = logits.topk(2, dim=-1).values
    clear = (top2[..., 0] - top2[..., 1]) > 50
    assert clear.float().mean() > 0.5
    assert (o.float().cpu() - ref)[clear].abs().max() < 2e-2
    q_huge = (torch.randn(1, 64, 128, generator=g) * 3e4).half()
    o = c_attention(q_huge.to(DEV), k[:1].to(DEV), v[:1].to(DEV), scale=8.0)
    assert torch.isfinite(o).all()


# bf16 runs the same tuned kernels with the bf16 MFMA, bf16 softmax weights and bf16 output.  The
# oracle consumes the bf16-rounded inputs in fp32; what is left is the rounding of the weights and
# of the output to 8 mantissa bits: rel-L2 <= 4e-3, max-abs <= 4e-2.
@pytest.mark.parametrize("bh,lq,lkv,d,causal,vt", [
    (3, 256, 512, 128, False, False), (2, 384, 384, 128, True, False), (2, 200, 333, 128, False, False),
    (2, 100, 100, 128, True, False), (2, 256, 256, 64, True, False), (3, 130, 517, 64, False, False),
    (2, 256, 512, 128, False, True), (2, 320, 320, 64, True, True),
    (2, 256, 512, 96, False, False), (2, 384, 384, 96, True, False), (2, 130, 520, 96, False, True),
])
def test_bf16_tuned_kernels_match_the_oracle(bh, lq, lkv, d, causal, vt):
    g = torch.Generator().manual_seed(bh * 1000 + lq + lkv + d)
    q = torch.randn(bh, lq, d, generator=g).bfloat16()
    k = torch.randn(bh, lkv, d, generator=g).bfloat16()
    v = torch.randn(bh, lkv, d, generator=g).bfloat16()
    v_dev = v.transpose(1, 2).contiguous().to(DEV) if vt else v.to(DEV)
    o = c_attention(q.to(DEV), k.to(DEV), v_dev, causal=causal, v_transposed=vt)
    assert o.dtype == torch.bfloat16
    ref = N.attention_ref(q, k, v, 1.0 / math.sqrt(d), causal)
    assert N.rel_l2(o, ref) <= 4e-3 and N.max_abs(o, ref) <= 4e-2, (N.rel_l2(o, ref), N.max_abs(o, ref))


def test_bf16_and_fp16_kernels_agree_on_inputs_both_can_hold():
    # inputs with 3 significant bits are exact in both types: the two kernels then differ only in
    # how they round the softmax weights and the output
    g = torch.Generator().manual_seed(77)
    mk = lambda *shape: (torch.randint(-7, 8, shape, generator=g).float() / 4)
    q, k, v = mk(2, 256, 128), mk(2, 384, 128), mk(2, 384, 128)
    o16 = c_attention(q.half().to(DEV), k.half().to(DEV), v.half().to(DEV), causal=True, scale=0.05)
    ob = c_attention(q.bfloat16().to(DEV), k.bfloat16().to(DEV), v.bfloat16().to(DEV), causal=True, scale=0.05)
    ref = N.attention_ref(q, k, v, 0.05, True)
    assert N.rel_l2(o16, ref) <= 1e-3
    assert N.rel_l2(ob, ref) <= 4e-3
    assert N.rel_l2(ob.float(), o16.float().cpu()) <= 4e-3


def test_head_dimension_96_never_reads_the_padding_of_its_lds_rows():
    # Head dimension 96 is kept in 128-element LDS rows; the 32 elements of padding hold copies of
    # the row's last 8 columns (the requests re-fetch the last 16-byte chunk).  Those columns are
    # made to dominate the scores and the values: a fragment read that strayed into the padding
    # would count them more than once.
    g = torch.Generator().manual_seed(96)
    q = torch.randn(2, 256, 96, generator=g)
    k = torch.randn(2, 192, 96, generator=g)
    v = torch.randn(2, 192, 96, generator=g)
    q[..., 88:] *= 3.0
    k[..., 88:] *= 3.0
    v[..., 88:] += 4.0
    q, k, v = q.half(), k.half(), v.half()
    for causal in (False, True):
        for vt in (False, True):
            vd = v.transpose(1, 2).contiguous() if vt else v
            o = c_attention(q.to(DEV), k.to(DEV), vd.to(DEV), causal, None, vt)
            ok, r, m = N.check_close(o, N.attention_ref(q, k, v, causal=causal))
            assert ok, f"causal={causal} vt={vt}: rel_l2={r:.3e} max_abs={m:.3e}"


# Causal tiles end where the queries end where CUs get several: every workgroup size, with queries that fill the first tile but for one wavefront, by one
# row, by a key tile and not at all.  The rows are those of a call with as many queries as keys, bit for bit: only who computes them differs.
@pytest.mark.parametrize("rows,b,d", [(64, 3, 64), (64, 3, 128), (128, 130, 64), (256, 300, 128)])
@pytest.mark.parametrize("cut", [0, 1, 63, 64, 127, 129, 191, 192, 255])
def test_causal_tiles_end_with_the_queries(rows, b, d, cut):
    assert cut > 127 or _capi.load().tf_flash_attention_rows(b, 512 - cut, 512, d, 1) == rows
    q, k, v = (x.to(DEV) for x in _inputs(b, 512, 512, d, rows + d + cut))
    lq = 512 - cut
    o = c_attention(q[:, :lq].contiguous(), k, v, True)
    assert torch.equal(o, c_attention(q, k, v, True)[:, :lq])
    ok, r, m = N.check_close(o[-1:].cpu(), N.attention_ref(q[-1:, :lq].cpu(), k[-1:].cpu(), v[-1:].cpu(), causal=True))
    assert ok, f"rel_l2={r:.3e} max_abs={m:.3e}"


# Single causal tiles for no more than the CUs begin at the first query, up to 8 of a slice: (rows, slices, queries, D) with a last tile that is not
# full, up to 256 workgroups and 8 tiles and beyond.  The rows are those of a slice alone, bit for bit.
@pytest.mark.parametrize("rows,b,l,d", [(256, 95, 320, 128), (256, 101, 352, 128), (256, 128, 300, 128), (256, 42, 1290, 96), (128, 60, 311, 96),
                                        (128, 98, 176, 128), (128, 115, 174, 64), (128, 33, 827, 128), (128, 29, 949, 96),
                                        (128, 24, 1192, 128), (64, 129, 300, 128)])
def test_causal_tiles_of_one_round_begin_with_the_queries(rows, b, l, d):
    assert _capi.load().tf_flash_attention_rows(b, l, l, d, 1) == rows and not _capi.load().tf_flash_attention_pairs(b, l, l, d, 1)
    q, k, v = (x.to(DEV) for x in _inputs(b, l, l, d, rows + l))
    o = c_attention(q, k, v, True)
    for i in (0, b // 2, b - 1):
        assert torch.equal(o[i:i + 1], c_attention(q[i:i + 1], k[i:i + 1], v[i:i + 1], True)), i
    assert not torch.isnan(o).any()
    ok, r, m = N.check_close(o[-1:].cpu(), N.attention_ref(q[-1:].cpu(), k[-1:].cpu(), v[-1:].cpu(), causal=True))
    assert ok, f"rel_l2={r:.3e} max_abs={m:.3e}"


# Single causal tiles where two share a CU (rows, slices, queries, D): the second 256 workgroups come in the opposite order, by eights, up to 576 of
# them at D = 64 and 512 of wide heads; just beyond 256, where less than two eights are reordered, between, at the ends and beyond.
FOLDED = [(128, 88, 384, 64), (128, 89, 384, 64), (128, 90, 384, 64), (128, 97, 384, 64), (128, 121, 384, 56), (128, 169, 384, 64), (128, 176, 384, 56),
          (128, 192, 384, 64), (128, 192, 384, 56), (128, 200, 384, 64), (64, 32, 1024, 256), (64, 18, 1600, 256), (64, 9, 3584, 160), (64, 17, 1024, 192),
          (64, 33, 1024, 256)]
# ... and where a slice's stay on one XCD instead, or 64 rows are picked.
BY_XCD = [(128, 85, 384, 64), (64, 86, 384, 64), (128, 170, 384, 64), (128, 171, 384, 56), (128, 193, 384, 64)]


@pytest.mark.parametrize("rows,bh,l,d", FOLDED + BY_XCD)
def test_causal_second_round_of_workgroups(rows, bh, l, d):
    lib = _capi.load()
    if d > 128:
        assert lib.tf_flash_attention_wide_rows(bh, l, 1) == rows
    else:
        assert lib.tf_flash_attention_rows(bh, l, l, 64, 1) == rows and lib.tf_flash_attention_pairs(bh, l, l, 64, 1) == 0
    q, k, v = (x.to(DEV) for x in _inputs(bh, l, l, d, bh + d))
    o = torch.full_like(q, float("nan"))
    torch.ops.tilefusion.flash_attention_fwd(q, k, v, o, d ** -0.5, True)
    for i in range(0, bh, 3):   # every tile of a slice once, as alone
        alone = torch.empty_like(o[i:i + 1])
        torch.ops.tilefusion.flash_attention_fwd(q[i:i + 1].contiguous(), k[i:i + 1].contiguous(), v[i:i + 1].contiguous(), alone,
                                                 d ** -0.5, True)
        assert torch.equal(o[i:i + 1], alone), i
    assert not torch.isnan(o).any()
