"""The torch.ops.tilefusion.* / tilefusion_amd.ops path (binding -> C ABI -> HIP kernels),
restating the reference's op-level tests (tests/python/test_{gemm,fused_two_gemms,flash_attn}.py)
with fp32 CPU oracles.  Tolerance: rel-L2 <= 1e-3, max-abs <= 2e-2."""

import math

import pytest
import torch

import oracle
from oracle import numerics as N

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def test_gemm_op_reference_signature():
    from tilefusion_amd.ops import gemm
    a, b = oracle.make_c1_gemm_inputs(256, 256, 256)
    for dt in (torch.float32, torch.float16):
        c = torch.zeros(256, 256, device=DEV, dtype=dt)
        gemm(a.to(DEV), b.to(DEV), c, 64, 64, 64, 2, 1)
        ok, r, m = N.check_close(c, N.gemm_ref(a, b))
        assert ok, (r, m)
    with pytest.raises(RuntimeError, match="does not divide"):
        gemm(a.to(DEV), b.to(DEV), torch.zeros(256, 256, device=DEV), 96, 64, 64, 1, 0)
    with pytest.raises(RuntimeError, match="contiguous"):
        gemm(a.to(DEV).t(), b.to(DEV), torch.zeros(256, 256, device=DEV), 64, 64, 64, 1, 0)
    with pytest.raises(RuntimeError, match="float16"):
        gemm(a.to(DEV).float(), b.to(DEV), torch.zeros(256, 256, device=DEV), 64, 64, 64, 1, 0)


def test_fused_two_gemms_op():
    from tilefusion_amd.ops import fused_two_gemms
    a, b, c = oracle.make_c3_fused_inputs(256, 128, 64, 64)
    d = torch.zeros(256, 64, device=DEV, dtype=torch.float16)
    fused_two_gemms(a.to(DEV), b.to(DEV), c.to(DEV), d)  # default tiles 64
    ok, r, m = N.check_close(d, N.fused_two_gemms_ref(a, b, c))
    assert ok, (r, m)
    with pytest.raises(TypeError):
        fused_two_gemms(a.to(DEV).float(), b.to(DEV), c.to(DEV), d)


@pytest.mark.parametrize("lq,lkv,causal", [(64, 128, False), (128, 128, True)])
def test_flash_attention_op(lq, lkv, causal):
    # tests/python/test_flash_attn.py:173-199: query [Lq, D], key [D, Lkv], value [Lkv, Dv]
    from tilefusion_amd.ops import flash_attention
    torch.manual_seed(1234)
    q = torch.randn(lq, 128, dtype=torch.float16)
    k = torch.randn(128, lkv, dtype=torch.float16)
    v = torch.randn(lkv, 128, dtype=torch.float16)
    scale = 1.0 / math.sqrt(128)
    o = flash_attention(q.to(DEV), k.to(DEV), v.to(DEV), 64, 128, 128, 128, scale, causal)
    assert o.shape == (lq, 128)
    ok, r, m = N.check_close(o, N.attention_ref(q, k.t(), v, scale, causal))
    assert ok, (r, m)
    # the raw op keeps the reference contract: K [Lkv, D], V transposed [Dv, Lkv]
    o2 = torch.zeros_like(o)
    torch.ops.tilefusion.flash_attention(q.to(DEV), k.t().contiguous().to(DEV), v.t().contiguous().to(DEV), o2,
                                         64, 128, 128, 128, scale, causal)
    ok, r, m = N.check_close(o2, N.attention_ref(q, k.t(), v, scale, causal))
    assert ok, (r, m)


def test_flash_attention_batched_and_decode_ops():
    from tilefusion_amd.ops import flash_attention, flash_decode
    q, k, v = oracle.make_c4_attention_inputs(2, 3, 256, 128)
    o = flash_attention(q.to(DEV), k.transpose(-1, -2).contiguous().to(DEV), v.to(DEV), 64, 64, 128, 128,
                        1.0 / math.sqrt(128), True)
    ok, r, m = N.check_close(o, N.attention_ref(q, k, v, causal=True))
    assert ok, (r, m)
    qs, ks, vs = zip(*[oracle.make_c5_decode_slice(0, h, kv_len=3000) for h in range(6)])
    q, k, v = torch.stack(qs).view(2, 3, 1, 128), torch.stack(ks).view(2, 3, 3000, 128), torch.stack(vs).view(2, 3, 3000, 128)
    o = flash_decode(q.to(DEV), k.to(DEV), v.to(DEV), num_splits=8)
    assert o.shape == q.shape
    ok, r, m = N.check_close(o.view(6, 128), N.flash_decode_ref(q.view(6, 128), k.view(6, 3000, 128), v.view(6, 3000, 128)))
    assert ok, (r, m)


def test_flash_decode_op_takes_bf16_and_head_dimension_64():
    from tilefusion_amd.ops import flash_decode
    g = torch.Generator().manual_seed(31)
    q = torch.randn(2, 4, 1, 64, generator=g).bfloat16()
    k = torch.randn(2, 4, 1500, 64, generator=g).bfloat16()
    v = torch.randn(2, 4, 1500, 64, generator=g).bfloat16()
    o = flash_decode(q.to(DEV), k.to(DEV), v.to(DEV), num_splits=5)
    assert o.shape == q.shape and o.dtype == torch.bfloat16
    ref = N.flash_decode_ref(q.view(8, 64), k.view(8, 1500, 64), v.view(8, 1500, 64))
    # bf16 output: 8 mantissa bits
    assert N.rel_l2(o.view(8, 64), ref) <= 4e-3 and N.max_abs(o.view(8, 64), ref) <= 4e-2
    with pytest.raises(RuntimeError, match="same dtype"):
        flash_decode(q.to(DEV), k.half().to(DEV), v.to(DEV), num_splits=5)


def test_ops_run_on_the_current_stream():
    from tilefusion_amd.ops import gemm
    a, b = oracle.make_c1_gemm_inputs(512, 512, 512)
    ad, bd = a.to(DEV), b.to(DEV)
    s = torch.cuda.Stream()
    c = torch.zeros(512, 512, device=DEV)
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        for _ in range(3):
            gemm(ad, bd, c, 64, 64, 64, 1, 0)
    s.synchronize()
    ok, r, m = N.check_close(c, N.gemm_ref(a, b))
    assert ok, (r, m)


def test_smoke_entry():
    import __graft_entry__
    __graft_entry__.smoke()


# ---- shapes and element types without a tuned kernel: never an error for a legal call ---------------
# bf16 tolerance: the oracle consumes the bf16-rounded inputs in fp32; products are accumulated in
# fp32; what remains is the bf16 rounding (8 mantissa bits, 2^-9 relative) of the intermediate
# (fused: A*B, attention: the softmax weights) and of the output: rel-L2 <= 4e-3, max-abs <= 4e-2.

def _close_bf16(out, ref):
    return N.rel_l2(out, ref) <= 4e-3 and N.max_abs(out, ref) <= 4e-2 * max(1.0, float(ref.abs().max()))


@pytest.mark.parametrize("d,dv,lq,lkv,causal", [(64, 128, 128, 256, False), (96, 96, 128, 128, True),
                                                (48, 80, 64, 128, False), (128, 64, 40, 64, True),
                                                (48, 48, 200, 160, True), (32, 16, 64, 96, False)])
def test_flash_attention_ops_for_head_dims_without_a_tuned_kernel(d, dv, lq, lkv, causal):
    # Head dimensions up to 128 without a tuned kernel are zero-padded by the op to the next tuned
    # size ((48, 48) and (32, 16) -> 64, (48, 80) -> 96, mixed ones above that -> 128) and run the
    # tuned kernel, any Lq and Lkv; (96, 96) has a tuned kernel of its own.  Both op forms (natural
    # and transposed V).
    from tilefusion_amd.ops import flash_attention
    g = torch.Generator().manual_seed(d * 1000 + dv)
    q = torch.randn(2, lq, d, generator=g).half()
    k = torch.randn(2, lkv, d, generator=g).half()
    v = torch.randn(2, lkv, dv, generator=g).half()
    scale = 1.0 / math.sqrt(d)
    ref = N.attention_ref(q, k, v, scale, causal)
    o = flash_attention(q.to(DEV), k.transpose(1, 2).contiguous().to(DEV), v.to(DEV), 8, 32, d, dv, scale, causal)
    assert o.shape == (2, lq, dv)
    ok, r, m = N.check_close(o, ref)
    assert ok, (r, m)
    o2 = torch.full((2, lq, dv), float("nan"), dtype=torch.float16, device=DEV)
    torch.ops.tilefusion.flash_attention(q.to(DEV), k.to(DEV), v.transpose(1, 2).contiguous().to(DEV), o2,
                                         8, 32, d, dv, scale, causal)
    ok, r, m = N.check_close(o2, ref)
    assert ok, (r, m)


@pytest.mark.parametrize("d,dv,lq,lkv", [(160, 160, 48, 64), (192, 128, 40, 96)])
def test_flash_attention_ops_for_head_dims_above_128_run_the_header_kernel(d, dv, lq, lkv):
    # nothing to pad to, and no tuned kernel unless D == Dv and V is in its natural layout: compiled at run time
    # from the header kernel (query rows padded to whole MFMA tiles by the op).  Both layouts of V: with the
    # transposed one it is always the header kernel.
    g = torch.Generator().manual_seed(d + dv)
    q = torch.randn(1, lq, d, generator=g).half()
    k = torch.randn(1, lkv, d, generator=g).half()
    v = torch.randn(1, lkv, dv, generator=g).half()
    scale = 1.0 / math.sqrt(d)
    o = torch.full((1, lq, dv), float("nan"), dtype=torch.float16, device=DEV)
    torch.ops.tilefusion.flash_attention_fwd(q.to(DEV), k.to(DEV), v.to(DEV), o, scale, False)
    ok, r, m = N.check_close(o, N.attention_ref(q, k, v, scale, False))
    assert ok, (r, m)
    o.fill_(float("nan"))
    torch.ops.tilefusion.flash_attention(q.to(DEV), k.to(DEV), v.transpose(1, 2).contiguous().to(DEV), o, 8, 32, d, dv, scale, False)
    ok, r, m = N.check_close(o, N.attention_ref(q, k, v, scale, False))
    assert ok, (r, m)


@pytest.mark.parametrize("d,dv,lq,lkv,tq,tkv,causal", [(256, 256, 64, 128, 64, 64, False),
                                                         (512, 512, 64, 128, 64, 64, False),
                                                         (384, 384, 128, 256, 128, 128, True),
                                                         (512, 256, 48, 96, 48, 32, True)])
def test_flash_attention_ops_shrink_tiles_that_do_not_fit_the_lds(d, dv, lq, lkv, tq, tkv, causal):
    # Whole-head-dimension tiles of these shapes need more than a CU's 160 KiB of LDS (512 x 512
    # with 64 x 64 sequence tiles: 192 KiB; 384 x 384 with 128 x 128: 288 KiB).  The launcher cuts
    # the head dimension into chunks, then the sequence tiles, until they fit.
    from tilefusion_amd.ops import flash_attention
    g = torch.Generator().manual_seed(d * 7 + dv)
    q = torch.randn(2, lq, d, generator=g).half()
    k = torch.randn(2, lkv, d, generator=g).half()
    v = torch.randn(2, lkv, dv, generator=g).half()
    scale = 1.0 / math.sqrt(d)
    ref = N.attention_ref(q, k, v, scale, causal)
    o = flash_attention(q.to(DEV), k.transpose(1, 2).contiguous().to(DEV), v.to(DEV), tq, tkv, d, dv, scale, causal)
    assert o.shape == (2, lq, dv)
    ok, r, m = N.check_close(o, ref)
    assert ok, (r, m)
    # V transposed: the header kernel also where natural V has a tuned one (256)
    o = torch.full((2, lq, dv), float("nan"), dtype=torch.float16, device=DEV)
    torch.ops.tilefusion.flash_attention(q.to(DEV), k.to(DEV), v.transpose(1, 2).contiguous().to(DEV), o, tq, tkv, d, dv, scale, causal)
    ok, r, m = N.check_close(o, ref)
    assert ok, (r, m)


# Both workgroup sizes (64 queries; 128 where that saves a round of the 256 CUs), one key tile, fewer than
# the ring holds and more, rows that no tile divides, causal tiles heaviest first.
# Bounds: four times what the kernel shows against 64-bit sums (2.8e-4 fp16, 2.3e-3 bf16: the 16-bit weights
# and result).
@pytest.mark.parametrize("dtype,tol", [(torch.float16, 1.2e-3), (torch.bfloat16, 1e-2)])
@pytest.mark.parametrize("d", [160, 192, 256])
@pytest.mark.parametrize("bh,lq,lkv,causal", [(1, 1, 32, False), (2, 65, 96, False), (2, 130, 160, True), (2, 512, 512, True),
                                              (150, 129, 64, False), (80, 500, 512, True), (150, 384, 384, True),
                                              (100, 129, 64, False), (32, 1000, 1024, False)])
def test_flash_attention_wide_heads(bh, lq, lkv, causal, d, dtype, tol):
    g = torch.Generator().manual_seed(d + lq + lkv)
    q, k, v = (torch.randn(bh, n, d, generator=g).to(dtype) for n in (lq, lkv, lkv))
    scale = 1.0 / math.sqrt(d)
    o = torch.full((bh, lq, d), float("nan"), dtype=dtype, device=DEV)
    torch.ops.tilefusion.flash_attention_fwd(q.to(DEV), k.to(DEV), v.to(DEV), o, scale, causal)
    s = q.to(DEV).float() @ k.to(DEV).float().transpose(-1, -2).contiguous() * scale
    if causal:
        s.masked_fill_(torch.ones(lq, lkv, dtype=torch.bool, device=DEV).triu(1), -math.inf)
    ref = torch.softmax(s, -1) @ v.to(DEV).float()
    assert ((o.float() - ref).norm() / ref.norm()).item() < tol


@pytest.mark.parametrize("dtype,half_ulp", [(torch.float16, 2.0 ** -11), (torch.bfloat16, 2.0 ** -8)])
@pytest.mark.parametrize("d", [160, 192, 256])
@pytest.mark.parametrize("bh", [1, 300])
def test_flash_attention_wide_heads_round_no_error_into_the_largest_weight(bh, d, dtype, half_ulp):
    # Two keys count: one in the first key tile, and far behind it one whose weight is 1.5 + half_ulp times
    # as large, halfway between two 16-bit numbers.  Relative to the row's largest score the second weight
    # is 1 and the first one is never rounded in 16 bits other than as 1: what is left is the fp32 arithmetic,
    # which the values -1.5 and 1 let show as half_ulp / 2.5.  A weight of 1.5 + half_ulp kept against the
    # first score would be rounded to 1.5 or 1.5 + 2 half_ulp and give 0 or twice that.
    import tilefusion_amd.ops  # noqa: F401
    lq, lkv, far = 70, 512, 400
    q = torch.zeros(bh, lq, d); q[..., :3] = 1.0
    k = torch.zeros(bh, lkv, d); k[..., 0] = -60.0
    k[:, 3, 0] = 0.0
    score = torch.tensor(math.log(1.5 + half_ulp), dtype=torch.float64)
    for i in range(3):                                   # as a sum of three 16-bit numbers
        k[:, far, i] = score.to(dtype)
        score -= k[0, far, i].double()
    v = torch.zeros(bh, lkv, d); v[:, 3] = -1.5; v[:, far] = 1.0
    o = torch.full((bh, lq, d), float("nan"), dtype=dtype, device=DEV)
    torch.ops.tilefusion.flash_attention_fwd(*(x.to(dtype).to(DEV) for x in (q, k, v)), o, 1.0, False)
    want = half_ulp / (2.5 + half_ulp)
    # exp2, the score and the sums in fp32: a few 2^-23 of the two terms of 1.5 / 2.5; the result's own rounding
    assert (o.double() - want).abs().max().item() <= 16 * 2.0 ** -23 + half_ulp * want


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("d", [160, 192, 256])
def test_flash_attention_wide_heads_pass_infinite_values_on(d, dtype):
    # every weight is positive (key 90's is exact in 16 bits), so an infinite value makes its column that infinity
    import tilefusion_amd.ops  # noqa: F401
    g = torch.Generator().manual_seed(d)
    q, k, v = (torch.randn(3, n, d, generator=g).to(dtype) for n in (130, 160, 160))
    k[:, 90] = 0.0
    v[:, 5, 1], v[:, 90, 2], v[:, 150, d - 1] = math.inf, -math.inf, math.inf
    o = torch.full((3, 130, d), float("nan"), dtype=dtype, device=DEV)
    torch.ops.tilefusion.flash_attention_fwd(q.to(DEV), k.to(DEV), v.to(DEV), o, 0.1, False)
    ref = torch.softmax(q.float() @ k.float().transpose(1, 2) * 0.1, -1) @ v.float()
    assert torch.equal(o.isinf().cpu(), ref.isinf()) and not o.isnan().any()
    assert (o[..., 1] > 0).all() and (o[..., 2] < 0).all() and (o[..., d - 1] > 0).all()


def test_flash_attention_wide_heads_keep_rows_whose_first_scores_are_minus_infinity():
    # the first two key tiles score -inf: their weights are zero and the row's reference comes from the third
    g = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn(1, n, 256, generator=g).half() for n in (40, 128, 128))
    q[..., 0] = 1.0
    k[:, :64, 0] = -math.inf
    scale = 4.0
    o = torch.empty(1, 40, 256, dtype=torch.float16, device=DEV)
    torch.ops.tilefusion.flash_attention_fwd(q.to(DEV), k.to(DEV), v.to(DEV), o, scale, False)
    ref = torch.softmax(q.float() @ k.float().transpose(1, 2) * scale, -1) @ v.float()
    assert ((o.float().cpu() - ref).norm() / ref.norm()).item() < 1.2e-3


def test_flash_attention_key_length_that_cannot_be_padded_is_a_clear_error():
    # above 128 the key tiles are 32 wide, in the tuned kernels as in the header kernel
    q = torch.randn(16, 160, dtype=torch.float16, device=DEV)
    k = torch.randn(48, 160, dtype=torch.float16, device=DEV)
    v = torch.randn(48, 160, dtype=torch.float16, device=DEV)
    o = torch.zeros(16, 160, dtype=torch.float16, device=DEV)
    with pytest.raises(RuntimeError, match="multiple of 32"):
        torch.ops.tilefusion.flash_attention_fwd(q, k, v, o, 0.1, False)


@pytest.mark.parametrize("m,n,k,p", [(128, 64, 48, 64), (64, 48, 64, 32), (96, 80, 112, 48), (256, 128, 64, 72)])
def test_fused_two_gemms_op_pads_what_the_kernels_cannot_tile(m, n, k, p):
    # K = 48, N = 48 ...: legal for the reference's 16-wide base tiles, not whole 32-deep MFMAs
    from tilefusion_amd.ops import fused_two_gemms
    a, b, c = oracle.make_c3_fused_inputs(m, n, k, p)
    d = torch.full((m, p), float("nan"), device=DEV, dtype=torch.float16)
    fused_two_gemms(a.to(DEV), b.to(DEV), c.to(DEV), d, 16, 16, 16, 8)
    ok, r, mx = N.check_close(d, N.fused_two_gemms_ref(a, b, c))
    assert ok, (r, mx)


@pytest.mark.parametrize("m,n,k", [(256, 256, 128), (4096, 512, 256), (96, 160, 64), (128, 128, 96),
                                   (4096, 2048, 96), (32, 32, 32)])
def test_gemm_op_bf16(m, n, k):
    # every kernel of the GEMM is a template of the operand type; what runs here are split-K kernels and, at
    # 4096 x 2048 x 96, a ring kernel whose first k-tile is completed with zeros
    from tilefusion_amd.ops import gemm
    a, b = oracle.make_c1_gemm_inputs(m, n, k, seed=77)
    a, b = a.bfloat16(), b.bfloat16()
    ref = N.gemm_ref(a, b)
    c32 = torch.full((m, n), float("nan"), device=DEV)
    gemm(a.to(DEV), b.to(DEV), c32, 32, 32, 32, 2, 1)
    assert N.rel_l2(c32, ref) <= 1e-5, N.rel_l2(c32, ref)
    c16 = torch.full((m, n), float("nan"), device=DEV, dtype=torch.bfloat16)
    gemm(a.to(DEV), b.to(DEV), c16, 32, 32, 32, 3, 2)
    assert _close_bf16(c16, ref), (N.rel_l2(c16, ref), N.max_abs(c16, ref))
    # integer operands: exact
    g = torch.Generator().manual_seed(3)
    ai = torch.randint(-3, 4, (m, k), generator=g).bfloat16()
    bi = torch.randint(-3, 4, (n, k), generator=g).bfloat16()
    gemm(ai.to(DEV), bi.to(DEV), c32, 32, 32, 32, 1, 0)
    assert torch.equal(c32.cpu(), N.gemm_ref(ai, bi))
    with pytest.raises(RuntimeError, match="same dtype"):
        gemm(a.to(DEV), b.half().to(DEV), c32, 32, 32, 32, 1, 0)


def test_fused_two_gemms_and_flash_attention_ops_bf16():
    from tilefusion_amd.ops import flash_attention, fused_two_gemms
    a, b, c = [t.bfloat16() for t in oracle.make_c3_fused_inputs(256, 128, 64, 64)]
    d = torch.full((256, 64), float("nan"), device=DEV, dtype=torch.bfloat16)
    fused_two_gemms(a.to(DEV), b.to(DEV), c.to(DEV), d)
    ref = N.fused_two_gemms_ref(a, b, c)
    assert _close_bf16(d, ref), (N.rel_l2(d, ref), N.max_abs(d, ref))
    with pytest.raises(TypeError):
        fused_two_gemms(a.to(DEV), b.half().to(DEV), c.to(DEV), d)
    g = torch.Generator().manual_seed(9)
    q = torch.randn(128, 128, generator=g).bfloat16()
    k = torch.randn(256, 128, generator=g).bfloat16()
    v = torch.randn(256, 128, generator=g).bfloat16()
    for causal in (False, True):
        o = flash_attention(q.to(DEV), k.t().contiguous().to(DEV), v.to(DEV), 64, 64, 128, 128, 1 / math.sqrt(128), causal)
        assert o.dtype == torch.bfloat16
        ref = N.attention_ref(q, k, v, 1 / math.sqrt(128), causal)
        assert _close_bf16(o, ref), (causal, N.rel_l2(o, ref), N.max_abs(o, ref))


# Tile sizes that are not positive are refused whichever kernel the shape runs, the plain one, the streaming one or
# (operands off a 16-byte boundary) that on padded copies, and leave the output alone.
@pytest.mark.parametrize("k,n,p", [(64, 128, 64), (64, 320, 64), (48, 320, 64), (56, 136, 40), (24, 40, 40)])
@pytest.mark.parametrize("at", [0, 1, 2, 3])
@pytest.mark.parametrize("tile", [0, -1, -64])
def test_fused_two_gemms_refuses_tiles_that_are_not_positive(k, n, p, at, tile):
    from tilefusion_amd.ops import fused_two_gemms
    store = torch.ones(64 * k + 1, device=DEV, dtype=torch.float16)
    b, c = torch.ones(n, k, device=DEV, dtype=torch.float16), torch.ones(p, n, device=DEV, dtype=torch.float16)
    d = torch.full((64, p), 7.0, device=DEV, dtype=torch.float16)
    tiles = [1, 1, 1, 1]
    tiles[at] = tile
    for start in (0, 1):
        with pytest.raises(RuntimeError, match="tile sizes must be positive"):
            fused_two_gemms(store[start:start + 64 * k].view(64, k), b, c, d, *tiles)
    assert bool((d == 7.0).all())
    fused_two_gemms(store[:64 * k].view(64, k), b, c, d, 1, 1, 1, 1)
    assert bool((d == float(n * k)).all())


# The wrappers call the implementations directly where nothing is to see the call; a mode, a profiler, autocast, a gradient
# or a subclass gets the op itself.  Same results and same errors either way.
def test_direct_calls_and_ops_agree_and_observers_see_the_ops():
    from torch.utils._python_dispatch import TorchDispatchMode

    from tilefusion_amd import _direct, ops
    g = torch.Generator().manual_seed(3)
    a, b = (torch.randn(n, 96, generator=g).half().to(DEV) for n in (70, 40))
    c, c2 = (torch.empty(70, 40, device=DEV, dtype=torch.float32) for _ in range(2))
    q, k, v = (torch.randn(2, n, 64, generator=g).half().to(DEV) for n in (1, 200, 200))
    e, f = torch.randn(64, 40, generator=g).half().to(DEV), torch.empty(70, 64, device=DEV, dtype=torch.float16)
    idx, upd = torch.tensor([[1], [3], [1]], device=DEV), torch.ones(3, 8, device=DEV)
    data = torch.zeros(5, 8, device=DEV)
    calls = {
        "gemm": lambda: (ops.gemm(a, b, c2, 1, 1, 1, 1, 1), c2)[1],
        "fused_two_gemms": lambda: (ops.fused_two_gemms(a, b, e, f, 1, 1, 1, 1), f)[1],
        "flash_attention_fwd": lambda: ops.flash_attention(q, k.transpose(-1, -2), v, 1, 1, 64, 64, 0.125, False),
        "flash_attention_fwd_kt": lambda: ops.flash_attention(q, k.transpose(-1, -2).contiguous(), v, 1, 1, 64, 64, 0.125, False),
        "flash_decode": lambda: ops.flash_decode(q, k, v, 2),
        "scatter_nd": lambda: (data.zero_(), ops.scatter_nd(data, idx, upd), data)[2],
    }
    assert _direct.gemm(a, b, c, 1, 1, 1, 1, 1)
    seen = []

    class Log(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))
    for name, call in calls.items():
        direct = call().clone()
        with Log():
            through_op = call().clone()
        assert any(s.startswith(f"tilefusion.{name}.") for s in seen), (name, seen)
        assert torch.equal(direct, through_op), name
        with torch.autograd.profiler.profile() as prof:
            call()
        assert any(x.name == f"tilefusion::{name}" for x in prof.function_events), name
    ok, r, m = N.check_close(c, (a.float() @ b.float().T).cpu())
    assert ok
    with torch.autocast("cuda", dtype=torch.float16):
        assert not _direct.gemm(a, b, c, 1, 1, 1, 1, 1)
    assert not _direct.gemm(a.clone().requires_grad_(), b, c, 1, 1, 1, 1, 1)
    assert not _direct.gemm(a, b, c.cpu(), 1, 1, 1, 1, 1)
    assert not _direct.gemm(a, b, c, 1, 1, 1, 1, True) and not _direct.gemm(a, b, c, 1, 1, 1, 1)
    assert not torch.vmap(lambda x: torch.tensor(_direct.gemm(x, b, c, 1, 1, 1, 1, 1)))(torch.stack([a, a])).any()
    for bad in (lambda: ops.gemm(a.t(), b, c, 1, 1, 1, 1, 1), lambda: ops.gemm(a, b, c, 64, 64, 64, 1, 1),
                lambda: ops.gemm(a.float(), b, c, 1, 1, 1, 1, 1), lambda: ops.flash_decode(q, k, v[:1], 2),
                lambda: ops.flash_attention(q, k, v, 1, 1, 64, 64, 0.125, False), lambda: ops.scatter_nd(data, idx.int(), upd)):
        with pytest.raises(RuntimeError) as direct:
            bad()
        with Log(), pytest.raises(RuntimeError) as through_op:
            bad()
        assert str(direct.value).splitlines()[0] == str(through_op.value).splitlines()[0]


# What a program registers for an op is what the wrappers call: an implementation for the CUDA key in place of the library's, and
# a kernel under the autograd keys, which the op's own call goes through whether a gradient is wanted or not.
@pytest.mark.filterwarnings("ignore:Warning only once for all operators")
@pytest.mark.parametrize("key", ["CUDA", "AutogradCUDA", "Autograd"])
def test_registered_implementations_are_called(key):
    from tilefusion_amd import ops
    g = torch.Generator().manual_seed(4)
    a, b = (torch.randn(n, 96, generator=g).half().to(DEV) for n in (70, 40))
    c = torch.zeros(70, 40, device=DEV, dtype=torch.float32)
    q, k, v = (torch.randn(2, n, 64, generator=g).half().to(DEV) for n in (1, 200, 200))
    e, f = torch.randn(64, 40, generator=g).half().to(DEV), torch.zeros(70, 64, device=DEV, dtype=torch.float16)
    data, idx, upd = torch.zeros(5, 8, device=DEV), torch.tensor([[1], [3], [1]], device=DEV), torch.ones(3, 8, device=DEV)
    calls = {
        "gemm": lambda: ops.gemm(a, b, c, 1, 1, 1, 1, 1),
        "fused_two_gemms": lambda: ops.fused_two_gemms(a, b, e, f, 1, 1, 1, 1),
        "flash_attention_fwd": lambda: ops.flash_attention(q, k.transpose(-1, -2), v, 1, 1, 64, 64, 0.125, False),
        "flash_attention_fwd_kt": lambda: ops.flash_attention(q, k.transpose(-1, -2).contiguous(), v, 1, 1, 64, 64, 0.125, False),
        "flash_decode": lambda: ops.flash_decode(q, k, v, 2),
        "scatter_nd": lambda: ops.scatter_nd(data, idx, upd),
    }
    for name, call in calls.items():
        seen = []
        lib = torch.library.Library("tilefusion", "IMPL")
        try:
            lib.impl(name, lambda *args: seen.append(len(args)), key)
            call()
        finally:
            lib._destroy()
        assert len(seen) == 1, name
        call()                                                     # the library's own again
        assert len(seen) == 1, name
    assert bool(c.any()) and bool(f.any()) and bool(data.any())
