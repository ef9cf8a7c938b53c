"""GPU parity of the GEMM macro kernel through the C ABI against the fp32 CPU oracle.
Tolerance (benchmark contract): rel-L2 <= 1e-3 and max-abs <= 2e-2, fp16 in / fp32 accumulate."""

import pytest
import torch

import oracle
from oracle import numerics as N
from tests.gpu_util import DEV, c_gemm

pytestmark = pytest.mark.gpu


def _check(c, ref, what):
    ok, r, m = N.check_close(c, ref)
    assert ok, f"{what}: rel_l2={r:.3e} max_abs={m:.3e}"


def test_readme_single_tile_gemm_c1():
    # README example: A 128x256 row-major, B 256x64 col-major, C 128x64 fp32
    a, b = oracle.make_c1_gemm_inputs()
    c = c_gemm(a.to(DEV), b.to(DEV), torch.float32, (128, 64, 32))
    _check(c, N.gemm_ref(a, b), "C1")
    assert N.max_abs(c, N.gemm_ref(a, b)) < 1e-4  # fp32 output: only summation order differs


# tests/python/test_gemm.py:75-135: (128^3, 256^3, 512^3) x tile 64^3 x (stages, level)
@pytest.mark.parametrize("size,stages,level", [(128, 1, 0), (256, 1, 0), (256, 2, 1), (512, 2, 1), (512, 3, 2)])
def test_reference_op_cases(size, stages, level):
    g = torch.Generator().manual_seed(size + level)
    a = torch.randn(size, size, generator=g).half()
    b = torch.randn(size, size, generator=g).half()
    c = c_gemm(a.to(DEV), b.to(DEV), torch.float32, (64, 64, 64), stages, level)
    _check(c, N.gemm_ref(a, b), f"gemm {size}^3")


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.float16])
def test_large_gemm_c2(out_dtype):
    a, b = oracle.make_c2_gemm_inputs()
    c = c_gemm(a.to(DEV), b.to(DEV), out_dtype, (64, 128, 128), 2, 1)
    _check(c, N.gemm_ref(a, b), "C2 4096^3")


# shapes of tests/cpp/cell/test_gemm.cu:316-375 (M,N in 16..128, K in 32..256) plus ragged
# ones that exercise the bounds-checked path, non-square and mid-size direct-LDS tiles
@pytest.mark.parametrize("m,n,k", [(16, 16, 32), (32, 32, 64), (64, 64, 128), (128, 128, 256), (64, 128, 64),
                                   (100, 72, 40), (1, 1, 8), (33, 257, 136), (384, 128, 192), (256, 512, 64),
                                   (1024, 768, 320), (2048, 256, 64)])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.float16])
def test_shapes(m, n, k, out_dtype):
    g = torch.Generator().manual_seed(m * 131 + n * 17 + k)
    a = torch.rand(m, k, generator=g).half()
    b = torch.rand(n, k, generator=g).half()
    c = c_gemm(a.to(DEV), b.to(DEV), out_dtype)
    assert not torch.isnan(c).any()
    ref = N.gemm_ref(a, b)
    # U[0,1) inputs give outputs of size ~k/4: compare relative to that scale
    assert N.rel_l2(c, ref) <= 1e-3
    assert N.max_abs(c, ref) <= 2e-2 * max(1.0, float(ref.abs().max()))


def test_integer_inputs_are_exact():
    # products and sums of small integers are exact in fp32: bit-exact against the oracle
    g = torch.Generator().manual_seed(3)
    a = torch.randint(-3, 4, (512, 256), generator=g).half()
    b = torch.randint(-3, 4, (384, 256), generator=g).half()
    for dt in (torch.float32, torch.float16):
        c = c_gemm(a.to(DEV), b.to(DEV), dt)
        assert torch.equal(c.float().cpu(), N.gemm_ref(a, b))


# The 256x256x64 ring kernel (grids of more than 128 tiles of 256x256, K % 64 == 0): one k-tile,
# fewer k-tiles than ring units, counts that are not multiples of the ring length, non-square
# tile grids.
# Small integers make every product and partial sum exact, so the comparison is bit-exact and
# a single misplaced fragment, a stale ring unit or a missed wait cannot hide in a tolerance.
@pytest.mark.parametrize("m,n,k", [(4096, 3072, 64), (3072, 4096, 128), (4096, 4096, 192), (2304, 4096, 320),
                                   (6144, 2048, 448), (4096, 4096, 1088)])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.float16])
def test_ring_kernel_exact(m, n, k, out_dtype):
    g = torch.Generator(device=DEV).manual_seed(m + 3 * n + 7 * k)
    a = torch.randint(-2, 3, (m, k), generator=g, device=DEV).half()
    b = torch.randint(-2, 3, (n, k), generator=g, device=DEV).half()
    c = c_gemm(a, b, out_dtype)
    ref = torch.matmul(a.float(), b.float().T)  # exact in fp32 (|sum| < 2^24), any summation order
    if out_dtype == torch.float16:
        ref = ref.half()                        # |values| <= 4k <= 4352: exact or one correctly rounded step
    assert torch.equal(c, ref)
    # and against the CPU oracle on a sampled block (the oracle is the reference, torch only scales it up)
    blk = N.gemm_ref(a[256:384].cpu(), b[512:576].cpu())
    assert torch.equal(c[256:384, 512:576].float().cpu(), blk if out_dtype == torch.float32 else blk.half().float())


# The same ring kernel with 128x128 tiles (grids with fewer than 128 tiles of 256x256; a ring of
# 9 units, requests 4 tiles ahead): fewer k-tiles than the look-ahead, counts around the ring
# length, one tile, non-square grids.
@pytest.mark.parametrize("m,n,k", [(128, 128, 64), (128, 256, 128), (256, 128, 256), (384, 640, 320), (640, 384, 576),
                                   (1024, 1024, 1216), (2048, 2048, 2048),
                                   # more tiles than CUs: the 5-unit variant with two workgroups per CU
                                   (2048, 2176, 64), (2176, 2048, 192), (2048, 2304, 448), (3072, 2560, 704)])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.float16])
def test_ring_kernel_mid_tiles_exact(m, n, k, out_dtype):
    g = torch.Generator(device=DEV).manual_seed(m + 3 * n + 7 * k)
    a = torch.randint(-2, 3, (m, k), generator=g, device=DEV).half()
    b = torch.randint(-2, 3, (n, k), generator=g, device=DEV).half()
    c = c_gemm(a, b, out_dtype)
    ref = torch.matmul(a.float(), b.float().T)
    if out_dtype == torch.float16:
        ref = ref.half()   # |values| <= 4k = 8192 at most; sums of a few thousand terms of size <= 4 stay far below it
    assert torch.equal(c, ref)
    blk = N.gemm_ref(a[:128].cpu(), b[64:128].cpu())
    assert torch.equal(c[:128, 64:128].float().cpu(), blk if out_dtype == torch.float32 else blk.half().float())


def test_linearity_at_full_size():
    # size-independent property: (A1 + A2) B = A1 B + A2 B for integer-valued operands
    g = torch.Generator(device=DEV).manual_seed(5)
    a1 = torch.randint(-2, 3, (4096, 4096), generator=g, device=DEV).half()
    a2 = torch.randint(-2, 3, (4096, 4096), generator=g, device=DEV).half()
    b = torch.randint(-2, 3, (4096, 4096), generator=g, device=DEV).half()
    assert torch.equal(c_gemm(a1 + a2, b), c_gemm(a1, b) + c_gemm(a2, b))


def test_identity_operand():
    g = torch.Generator().manual_seed(9)
    a = torch.randn(256, 256, generator=g).half()
    eye = torch.eye(256).half()
    assert torch.equal(c_gemm(a.to(DEV), eye.to(DEV), torch.float16).cpu(), a)
    # B buffer is [N, K]: C = A @ B^T, so a non-symmetric B catches a transposed operand
    b = torch.randn(256, 256, generator=g).half()
    c = c_gemm(eye.to(DEV), b.to(DEV), torch.float16).cpu()
    assert torch.equal(c, b.T)


# Ragged problems for every kernel and tile that the dispatch can pick (for a 16-bit result; its position, see tf_gemm_kernel_index: m, n,
# k), at the edges where each can go wrong: fewer rows or columns than a tile, a last tile that overlaps its
# neighbour by all but one row, K that completes its first (ring kernels) or last (split-K kernels)
# 64-deep k-tile with 8 to 56 zeros, fewer k-tiles than wavefronts.  Small integers: exact in fp32, whatever the
# order of the sums.
EDGES = {
    0: [(1, 1, 8), (72, 1, 72), (17, 33, 8), (3, 577, 200)],                # 16 x 16, four wavefronts
    1: [(1, 264, 264), (15, 72, 4264), (33, 31, 1000), (44, 650, 1160)],    # 16 x 16, eight
    2: [(5390, 1, 200)],                                                    # 32 x 16
    3: [(33, 4449, 72), (131, 1433, 64), (925, 768, 64), (129, 4095, 120), (128, 6400, 64), (65, 6209, 8),
        (7000, 65, 24), (517, 3009, 64)],                                                    # 32 x 32, one
    4: [(17, 4561, 72), (257, 513, 328)],                                   # 32 x 32, four
    5: [(6426, 54, 4480), (165, 1765, 7616)],                               # 64 x 32
    6: [(3578, 101, 1000), (1088, 577, 1032), (50, 6432, 5688)],            # 64 x 64
    7: [(213, 5906, 448), (629, 2005, 448)],                                # 128 x 128, requests four tiles ahead
    8: [(2048, 2048, 136), (2177, 513, 136), (4939, 3091, 80), (1398, 5437, 72), (4929, 1741, 72),
        (4882, 2468, 72)],                                                  # 128 x 128, two ahead
    9: [(5216, 6236, 256)],                                                 # 128 x 128, two per CU
    10: [(2689, 1409, 136)],                                                # 192 x 128
    11: [(2305, 3265, 136), (1537, 4611, 152)],                             # 192 x 192
    12: [(6145, 897, 144)],                                                 # 256 x 128
    13: [(4097, 2305, 264), (5378, 1537, 144)],                             # 256 x 192
    14: [(4865, 2305, 136), (2305, 4867, 136)],                             # 256 x 256
    15: [(517, 3008, 64), (982, 5472, 72), (4097, 2305, 40), (3301, 2817, 8), (4794, 235, 72),
         (812, 4675, 72)],                                                  # bounds-checked
    16: [(205, 5613, 1904)],                                                # whole lines: 128 x 128
    17: [(819, 5552, 352), (2944, 2016, 1056)],                             # 192 x 128
    18: [(1555, 4613, 328)],                                                # 192 x 192
    19: [(3333, 2288, 1944)],                                               # 256 x 128
    20: [(2466, 1722, 256), (861, 5283, 384)],                              # 160 x 128, K a multiple of 64
    21: [(2999, 1544, 1032), (3657, 1390, 328)],                            # ... whole lines
}


@pytest.mark.parametrize("kernel,m,n,k", [(kernel, *mnk) for kernel, problems in EDGES.items() for mnk in problems])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_every_kernel_at_its_edges_is_exact(kernel, m, n, k, dtype):
    from tilefusion_amd import _capi
    lib = _capi.load()
    assert lib.tf_gemm_kernel_index(m, n, k, 0) == kernel
    g = torch.Generator().manual_seed(m + n + k)
    a = torch.randint(-2, 3, (m, k), generator=g).to(dtype).to(DEV)
    b = torch.randint(-2, 3, (n, k), generator=g).to(dtype).to(DEV)
    ref = a.float() @ b.float().t()                                      # exact: |sum| <= 4 k < 2^24
    for out_dtype in (torch.float32, dtype):
        buf = torch.full((m * n + 64,), 7.0, device=DEV, dtype=out_dtype)
        _capi.check(lib.tf_gemm(a.data_ptr(), b.data_ptr(), buf.data_ptr(), 2 if dtype == torch.bfloat16 else 1,
                                int(out_dtype == torch.float32), m, n, k, m, n, k, 1, 0,
                                torch.cuda.current_stream().cuda_stream), "tf_gemm")
        assert torch.equal(buf[:m * n].view(m, n), ref.to(out_dtype))
        assert bool((buf[m * n:] == 7.0).all())                          # nothing behind C is written


# Rows that start anywhere in a line (K % 64 != 0, from 328 on): the ring kernels fetch whole lines.  Every place in a line that
# rows 8 apart can start at (K), first rows at another (operands that start at 16 bytes, not at a line), last tiles that
# overlap their neighbours by any amount, few and many k-tiles; every tile that comes with whole lines (the position of
# what runs, as in EDGES), both operand types, both types of result.
LINES = [(16, 4875, 196, 520), (16, 300, 3476, 528), (16, 3802, 259, 536), (16, 4328, 232, 544), (16, 4432, 228, 552),
         (16, 1621, 647, 560), (16, 234, 4261, 568), (21, 770, 4610, 328), (21, 773, 4658, 336), (21, 4622, 776, 344),
         (21, 4659, 771, 352), (21, 776, 4619, 360), (21, 4705, 769, 368), (21, 786, 4615, 376), (18, 1555, 4613, 328),
         (18, 1539, 4624, 344), (18, 1542, 4633, 352), (18, 1559, 4653, 376), (19, 1159, 4639, 328), (19, 1155, 4609, 344),
         (19, 1155, 4680, 352), (19, 1157, 4648, 376), (16, 205, 5613, 1904), (21, 2999, 1544, 1032), (19, 3333, 2288, 1944),
         (17, 1028, 4632, 328), (17, 969, 4618, 336), (17, 3053, 1579, 344), (17, 3444, 1415, 352), (17, 1937, 2513, 360),
         (17, 1617, 2985, 368), (17, 1483, 3320, 376), (17, 2944, 2016, 1056)]


@pytest.mark.parametrize("kernel,m,n,k", LINES)
@pytest.mark.parametrize("start", [0, 8, 40])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_rows_that_start_anywhere_in_a_line(kernel, m, n, k, start, dtype):
    from tilefusion_amd import _capi
    lib = _capi.load()
    assert lib.tf_gemm_kernel_index(m, n, k, 0) == lib.tf_gemm_kernel_index(m, n, k, 1) == kernel
    g = torch.Generator(device=DEV).manual_seed(m + n + k)

    def inside(rows, at):   # between numbers that must not count
        buf = torch.full((rows * k + 128,), float("nan"), device=DEV, dtype=dtype)
        return buf[at:at + rows * k].view(rows, k).copy_(torch.randint(-2, 3, (rows, k), device=DEV, generator=g))

    a, b = inside(m, start), inside(n, 48 - start)
    ref = a.float() @ b.float().t()                                      # exact: |sum| <= 4 k < 2^24
    for out_dtype in (torch.float32, dtype):
        buf = torch.full((m * n + 64,), 7.0, device=DEV, dtype=out_dtype)
        _capi.check(lib.tf_gemm(a.data_ptr(), b.data_ptr(), buf.data_ptr(), 2 if dtype == torch.bfloat16 else 1,
                                int(out_dtype == torch.float32), m, n, k, m, n, k, 1, 0,
                                torch.cuda.current_stream().cuda_stream), "tf_gemm")
        assert torch.equal(buf[:m * n].view(m, n), ref.to(out_dtype))
        assert bool((buf[m * n:] == 7.0).all())                          # nothing behind C is written


# ... and the tile of 160 rows that takes the place of the pick where that leaves CUs idle or begins another round: an odd number
# of requests a wavefront and operand.
BETWEEN = [(3657, 1390, 328), (1895, 2281, 968), (1596, 2453, 464), (1661, 2930, 344), (2975, 1423, 984), (2642, 1847, 480),
           (2660, 1629, 360), (2501, 1657, 1000), (2315, 2084, 496), (1726, 2728, 376), (2643, 1708, 1016)]


@pytest.mark.parametrize("m,n,k", BETWEEN)
@pytest.mark.parametrize("start", [0, 8, 40])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_tile_of_160_rows(m, n, k, start, dtype):
    test_rows_that_start_anywhere_in_a_line(21, m, n, k, start, dtype)


# ... and with rows that start where lines do.
@pytest.mark.parametrize("m,n,k", [(2466, 1722, 256), (3003, 1494, 256), (1541, 2582, 448), (861, 5283, 384), (3073, 1373, 1984),
                                   (4224, 983, 256), (3182, 1397, 1152)])
@pytest.mark.parametrize("start", [0, 8])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_tile_of_160_rows_of_whole_lines(m, n, k, start, dtype):
    test_rows_that_start_anywhere_in_a_line(20, m, n, k, start, dtype)


def test_operands_without_16_byte_alignment():
    g = torch.Generator().manual_seed(5)
    a, b = (torch.randint(-2, 3, (1 + r * 264,), generator=g).half().to(DEV)[1:].view(r, 264) for r in (200, 150))
    assert a.data_ptr() % 16 != 0 and b.data_ptr() % 16 != 0
    assert torch.equal(c_gemm(a, b, torch.float32), a.float() @ b.float().t())
