"""CPU-only checks of the C ABI: the library loads, exports every symbol the header declares,
and rejects bad arguments before touching the device."""

import ctypes
import os
import re

import pytest

from tilefusion_amd import _capi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_symbols():
    text = open(os.path.join(ROOT, "include", "tilefusion_c.h")).read()
    return sorted(set(re.findall(r"TF_API\s+[\w\s\*]+?\b(tf_\w+)\s*\(", text)))


def test_header_symbols_are_exported_and_bound():
    names = _declared_symbols()
    assert len(names) >= 7
    lib = ctypes.CDLL(_capi.LIB_PATH)
    for n in names:
        assert hasattr(lib, n), f"{n} declared in tilefusion_c.h but not exported"
        assert n in _capi.SIGNATURES, f"{n} has no ctypes signature"
    assert sorted(_capi.SIGNATURES) == names


def test_version_and_error_string():
    lib = _capi.load()
    assert b"gfx950" in lib.tf_version()
    assert isinstance(lib.tf_last_error(), bytes)


def test_gemm_argument_validation():
    lib = _capi.load()
    p = 0x1000  # never dereferenced: validation fails first
    assert lib.tf_gemm_f16(None, p, p, 0, 128, 128, 128, 64, 64, 64, 1, 0, None) == _capi.TF_ERR_INVALID_ARG
    assert b"null" in lib.tf_last_error()
    assert lib.tf_gemm_f16(p, p, p, 0, 0, 128, 128, 64, 64, 64, 1, 0, None) == _capi.TF_ERR_INVALID_ARG
    assert lib.tf_gemm_f16(p, p, p, 0, 128, 128, 128, 48, 64, 64, 1, 0, None) == _capi.TF_ERR_INVALID_ARG
    assert b"does not divide" in lib.tf_last_error()
    assert lib.tf_gemm_f16(p, p, p, 0, 128, 128, 128, 64, 64, 64, 4, 0, None) == _capi.TF_ERR_INVALID_ARG
    assert lib.tf_gemm_f16(p, p, p, 0, 128, 128, 128, 64, 64, 64, 1, 3, None) == _capi.TF_ERR_INVALID_ARG
    assert lib.tf_gemm_f16(p, p, p, 0, 128, 128, 100, 64, 64, 100, 1, 0, None) == _capi.TF_ERR_UNSUPPORTED
    with pytest.raises(RuntimeError, match="multiple of 8"):
        _capi.check(_capi.TF_ERR_UNSUPPORTED, "tf_gemm_f16")


def test_fused_argument_validation():
    lib = _capi.load()
    p = 0x1000
    assert lib.tf_fused_two_gemms_f16(p, p, p, None, 1, 64, 64, 64, 64, 64, 64, 64, 64, None) == _capi.TF_ERR_INVALID_ARG
    assert lib.tf_fused_two_gemms_f16(p, p, p, p, 1, 64, 64, 64, 64, 48, 64, 64, 64, None) == _capi.TF_ERR_INVALID_ARG
    assert lib.tf_fused_two_gemms_f16(p, p, p, p, 1, 64, 48, 64, 64, 64, 48, 64, 64, None) == _capi.TF_ERR_UNSUPPORTED
    assert lib.tf_fused_two_gemms_f16(p, p, p, p, 0, 64, 64, 64, 64, 64, 64, 64, 64, None) == _capi.TF_ERR_INVALID_ARG


def test_attention_argument_validation():
    lib = _capi.load()
    p = 0x1000
    f = lib.tf_flash_attention_fwd_f16
    assert f(p, p, None, p, 1, 64, 64, 128, 128, 0, 64, 64, 128, 128, 0.1, 0, None) == _capi.TF_ERR_INVALID_ARG
    assert f(p, p, p, p, 1, 64, 64, 80, 80, 0, 64, 64, 80, 80, 0.1, 0, None) == _capi.TF_ERR_UNSUPPORTED
    assert f(p, p, p, p, 1, 64, 64, 128, 128, 0, 48, 64, 128, 128, 0.1, 0, None) == _capi.TF_ERR_INVALID_ARG
    assert f(p, p, p, p, 1, 64, 60, 128, 128, 1, 64, 60, 128, 128, 0.1, 0, None) == _capi.TF_ERR_UNSUPPORTED
    assert f(p, p, p, p, 1, 64, 64, 128, 128, 0, 64, 64, 128, 128, float("nan"), 0, None) == _capi.TF_ERR_INVALID_ARG


def test_decode_argument_validation_and_workspace():
    lib = _capi.load()
    p = 0x1000
    assert lib.tf_flash_decode_workspace_bytes(512, 128, 64) == 512 * 64 * 130 * 4
    assert lib.tf_flash_decode_workspace_bytes(0, 128, 64) == 0
    f = lib.tf_flash_decode_f16
    assert f(p, p, p, p, None, 0, 4, 128, 128, 4, 0.1, None) == _capi.TF_ERR_INVALID_ARG
    assert f(p, p, p, p, p, 16, 4, 128, 128, 4, 0.1, None) == _capi.TF_ERR_INVALID_ARG
    assert b"workspace" in lib.tf_last_error()
    assert f(p, p, p, p, p, 1 << 20, 4, 128, 96, 4, 0.1, None) == _capi.TF_ERR_UNSUPPORTED   # 128 and 64 only
    assert f(p, p, p, p, p, 1 << 20, 4, 0, 128, 4, 0.1, None) == _capi.TF_ERR_INVALID_ARG
    # without a workspace: only what is not cut
    f = lib.tf_flash_decode_uncut
    assert f(p, p, p, p, _capi.TF_DTYPE_F16, 8, 4096, 128, 64, 0.1, None) == _capi.TF_ERR_UNSUPPORTED
    assert f(p, p, p, p, _capi.TF_DTYPE_F32, 8, 64, 128, 64, 0.1, None) == _capi.TF_ERR_UNSUPPORTED
    assert f(p, p, p, p, _capi.TF_DTYPE_F16, 8, 64, 128, 0, 0.1, None) == _capi.TF_ERR_UNSUPPORTED
    assert f(p, None, p, p, _capi.TF_DTYPE_F16, 8, 64, 128, 64, 0.1, None) == _capi.TF_ERR_INVALID_ARG


# ---- what a call runs, decided on the host ------------------------------------------------------------
def test_gemm_edge_cases_reach_every_kernel_of_the_table():
    from tests.test_gpu_gemm import EDGES
    lib = _capi.load()
    for kernel, problems in EDGES.items():
        assert [lib.tf_gemm_kernel_index(*mnk, 0) for mnk in problems] == [kernel] * len(problems)
    text = open(os.path.join(ROOT, "tilefusion_amd", "csrc", "gemm.hip")).read()
    table = re.search(r"constexpr GemmKernel kGemmKernels\[\] = \{\n(.*?)\n\};", text, re.S).group(1)
    lines = re.search(r"constexpr LinesKernel kLinesKernels\[\] = \{\n(.*?)\n\};", text, re.S).group(1)
    # the table, the bounds-checked kernel, the tiles that come with whole lines too, both forms of the tile of 160 rows: all that
    # a call can run
    assert sorted(EDGES) == list(range(len(table.splitlines()) + 1 + len(lines.splitlines()) + 2))
    assert lib.tf_gemm_kernel_index(0, 64, 64, 0) == -1 and lib.tf_gemm_kernel_index(64, 64, 1 << 22, 0) == -1
    # the grid of the bounds-checked kernel ends at 65535 columns of tiles
    assert lib.tf_gemm_kernel_index(512, 65535 * 64, 8, 1) == 15 and lib.tf_gemm_kernel_index(512, 65535 * 64 + 1, 8, 1) != 15
    # the tile of 160 rows stands in for those of 128 columns, not for the larger ones
    assert [lib.tf_gemm_kernel_index(*mnk, 0) for mnk in ((2060, 7341, 816), (2073, 7409, 848), (2316, 6408, 904))] == [18, 18, 19]
    # nor do whole lines for 256 x 192 and 256 x 256
    assert [lib.tf_gemm_kernel_index(*mnk, 0) for mnk in ((5530, 3814, 1184), (7918, 1536, 1952), (7568, 5021, 1424))] == [13, 13, 14]
    # the split-K kernels' launches end at 2^35 elements of C
    assert lib.tf_gemm_kernel_index(1 << 25, 1 << 10, 8, 0) == 15


def _plan(bh, lkv, d, splits):
    waves = ctypes.c_int(0)
    return _capi.load().tf_flash_decode_plan(bh, lkv, d, splits, ctypes.byref(waves)), waves.value


def test_decode_cases_reach_every_way_to_cut():
    from tests.test_gpu_flash_decode import CUTS
    ways = {(_plan(*c)[0] > 1, _plan(*c)[1], c[2]) for c in CUTS}
    assert ways == {(cut, waves, d) for cut in (False, True) for waves in (4, 8) for d in (64, 128)}


def test_decode_cases_that_are_merged_by_the_last_workgroup():
    from tests.test_gpu_flash_decode import MERGED
    plans = [(_plan(*c), c) for c in MERGED]
    assert all(n > 1 and waves == 8 for (n, waves), _ in plans)
    assert {d for (n, _), (_, _, d, _) in plans if n > 8192 // d} == {64, 128}   # a second turn of the merging loop
    assert max(bh * n for (n, _), (bh, _, _, _) in plans) == 1023


def test_decode_plan():
    assert _plan(512, 32768, 128, 64) == (8, 4)      # ranges of 2 MiB
    assert _plan(512, 32768, 128, 3) == (3, 4)       # the caller's limit
    assert _plan(512, 32768, 128, 1) == (1, 4)
    assert _plan(512, 8192, 128, 64) == (1, 4)       # 4 MiB a slice: not cut
    assert _plan(768, 8193, 128, 64)[0] == 3         # beyond, and 2.75 GB together
    assert _plan(512, 10000, 128, 64) == (1, 4)      # less together
    assert _plan(0, 64, 128, 4)[0] == 0 and _plan(4, 64, 96, 4)[0] == 0
    for bh, lkv, d, splits in [(1, 1, 64, 64), (3, 100000, 128, 5), (65535, 7, 64, 9), (40, 40000, 128, 65536)]:
        n, waves = _plan(bh, lkv, d, splits)
        assert 1 <= n <= splits and waves in (4, 8)  # the workspace holds `splits` partials a slice


def _scatter_plan(n, targets, slice_, dtype):
    lane = ctypes.c_int(0)
    return _capi.load().tf_scatter_nd_plan(n, targets, slice_, dtype, ctypes.byref(lane)), lane.value


def test_scatter_plan():
    from tests.test_gpu_scatter_nd import FEW_WIDE
    for dtype, elems in ((0, 1), (1, 2), (2, 2)):
        for rows, words, n, chunk in FEW_WIDE:
            fewer = 0 if n <= 1024 else 16
            assert _scatter_plan(n, rows, words * elems, dtype) == ((1024 if n <= 1024 else 2048) if chunk else fewer, 1)
        # distinct targets are possible: a sort would be in the way
        for n, rows, words in ((407, 3872, 5048), (1000, 2732, 2248), (88, 2892, 32224), (560, 588, 3977)):
            assert _scatter_plan(n, rows, words * elems, dtype) == (0, 1)
        # a word a lane where that is a workgroup on every CU, with eight to a chunk or more
        for n, words, lane in ((4096, 2000, 1), (4097, 257, 1), (8192, 512, 1), (8193, 512, 2), (8192, 513, 2), (11264, 300, 1), (12886, 491, 2),
                               (9604, 696, 2), (5032, 581, 2), (19999, 2000, 2)):
            assert _scatter_plan(n, 32000, words * elems, dtype) == (2048, lane)
        assert _scatter_plan(20000, 32000, 512 * elems, dtype) == (4096, 2)
        assert [_scatter_plan(n, 32000, 100 * elems, dtype)[0] for n in (1024, 1280, 8192, 8193, 20000)] == [0, 16, 1024, 2048, 4096]
    # 16-bit updates of less than 2 Mi words are sorted by 16 up to 2048
    assert _scatter_plan(1791, 3285, 632, 0) == (2048, 1) and _scatter_plan(1791, 3285, 1264, 2) == (16, 1)
    assert _scatter_plan(2100, 300, 140000, 2) == (64, 1) and _scatter_plan(2401, 300, 140000, 2) == (128, 2)
    assert _scatter_plan(0, 64, 64, 0)[0] == -1 and _scatter_plan(64, 64, 64, 3)[0] == -1


def test_wide_attention_cases_reach_both_workgroup_sizes():
    import tests.test_gpu_ops as t
    marks = t.test_flash_attention_wide_heads.pytestmark
    cases = next(m.args[1] for m in marks if m.args[0] == "bh,lq,lkv,causal")
    lib = _capi.load()
    assert {(lib.tf_flash_attention_wide_rows(bh, lq, int(causal)), causal) for bh, lq, _, causal in cases} == {
        (rows, causal) for rows in (64, 128) for causal in (False, True)}


def test_attention_cases_of_a_second_round_reorder_workgroups():
    from tests.test_gpu_flash_attention import BY_XCD, FOLDED
    # (a slice's tiles stay on one XCD by their numbers, or where the XCDs get within 4% of the same number of slices)
    for cases, by_xcd in ((FOLDED, False), (BY_XCD, True)):
        assert {bh % 8 != 0 and (bh + 7) // 8 * 8 * 100 <= bh * 104 for _, bh, _, _ in cases} == {by_xcd}
    counts = {(d > 128, (l + rows - 1) // rows * bh) for rows, bh, l, d in FOLDED}
    assert {n for wide, n in counts if not wide} >= {264, 267, 291, 507, 576, 600} and {n for wide, n in counts if wide} >= {272, 450, 504, 512, 528}


def test_attention_cases_reach_every_workgroup_form():
    from tests.test_gpu_flash_attention import PAIR_CASES, RING_CASES, SINGLE_CASES
    lib = _capi.load()
    tuned = [(rows, d) for rows in (64, 128, 256) for d in (64, 96, 128)]
    for cases, paired in ((PAIR_CASES, 1), (SINGLE_CASES, 0)):
        for rows, b, lq, lkv, d in cases:
            assert lib.tf_flash_attention_rows(b, lq, lkv, d, 1) == rows and lib.tf_flash_attention_pairs(b, lq, lkv, d, 1) == paired
            assert lib.tf_flash_attention_pairs(1, lq, lkv, d, 1) == 0   # a slice alone
        assert {(c[0], c[4]) for c in cases} == set(tuned)
    for rows, b in RING_CASES:
        for lkv in (8, 64, 72, 128, 192, 200, 256, 320, 384, 448):
            assert {lib.tf_flash_attention_rows(b, 256, lkv, 128, causal) for causal in (0, 1)} == {rows}


def test_attention_with_few_keys_takes_large_workgroups():
    # several workgroups a CU that walk few key tiles: 256 rows where 128 took 1.05 to 1.3 times as long
    lib = _capi.load()
    for b, lq, lkv in [(869, 214, 8), (58, 1666, 32), (200, 440, 32), (57, 2781, 104), (503, 465, 208), (80, 2291, 280), (59, 2630, 840)]:
        assert lib.tf_flash_attention_rows(b, lq, lkv, 128, 0) == 256


def test_fused_cases_reach_every_streaming_instance():
    from tests.test_gpu_fused_two_gemms import STREAM_CASES
    lib = _capi.load()
    whole, cut = set(), set()
    for m, n, k, p in STREAM_CASES:
        size = lib.tf_fused_two_gemms_workspace_bytes(_capi.TF_DTYPE_F16, 1, m, n, k, p)
        rows = lib.tf_fused_two_gemms_rows(1, m, n, k, p, size)
        (cut if size else whole).add(((max(k, 64) + 31) // 32, 4 if p <= 64 else 6 if p <= 96 else 8, rows))
    assert whole == {(steps, blocks, rows) for steps in (2, 3, 4) for blocks in (4, 6, 8) for rows in (64, 128)}
    assert {x[:2] for x in cut} == {x[:2] for x in whole} and {x[2] for x in cut} == {64, 128}
    assert lib.tf_fused_two_gemms_rows(1, 16384, 128, 128, 128, 0) == 0     # one n-tile: the plain kernel
    assert lib.tf_fused_two_gemms_rows(1, 4000, 4096, 128, 128, 0) == 64    # no room for partial sums: other rows
    assert lib.tf_fused_two_gemms_workspace_bytes(_capi.TF_DTYPE_F32, 1, 70, 2056, 64, 64) == 0


def test_python_wrappers_validate_like_the_reference():
    # python/ops/fused_two_gemms.py:33-38: ValueError for a CPU tensor, TypeError for dtype
    import torch
    from tilefusion_amd import ops
    t = torch.zeros(64, 64, dtype=torch.float16)
    with pytest.raises(ValueError, match="must be a cuda tensor"):
        ops.fused_two_gemms(t, t, t, t)
    # CPU tensors never reach a kernel: the op exists only for the CUDA dispatch key
    with pytest.raises((NotImplementedError, RuntimeError)):
        ops.gemm(t, t, torch.zeros(64, 64), 64, 64, 64, 1, 0)
    assert sorted(ops.__all__) == ["FlashAttention", "flash_attention", "flash_decode", "fused_two_gemms", "gemm", "scatter_nd"]


def test_op_schemas_match_the_reference():
    # include/kernels/kernel_list.hpp:15-30
    import torch
    import tilefusion_amd  # noqa: F401
    want = {
        "scatter_nd": "tilefusion::scatter_nd(Tensor data, Tensor(a!) updates, Tensor indices) -> ()",
        "gemm": "tilefusion::gemm(Tensor A, Tensor B, Tensor(a!) C, int m, int n, int k, int num_stages, int pipeline_level) -> ()",
        "fused_two_gemms": "tilefusion::fused_two_gemms(Tensor A, Tensor B, Tensor C, Tensor(a!) D, int tm, int tn, int tk, int tp) -> ()",
        "flash_attention": "tilefusion::flash_attention(Tensor Q, Tensor K, Tensor V, Tensor(a!) O, int tile_length_q, int tile_length_kv, int tile_hidden_qk, int tile_hidden_v, float softmax_scale, bool causal) -> ()",
    }
    for name, schema in want.items():
        op = getattr(torch.ops.tilefusion, name).default
        assert str(op._schema) == schema


def test_reference_package_name_imports_the_same_modules():
    # callers written against the reference do `import tilefusion` / `from tilefusion.ops import gemm`
    import tilefusion
    import tilefusion_amd
    from tilefusion.ops import flash_attention, fused_two_gemms, gemm
    assert tilefusion.ops is tilefusion_amd.ops
    assert gemm is tilefusion_amd.ops.gemm and fused_two_gemms is tilefusion_amd.ops.fused_two_gemms
    assert flash_attention is tilefusion_amd.ops.flash_attention


def test_torch_binding_exports_the_reference_launcher_names():
    # TILEFUSION_EXPORT (include/kernel_registry.hpp:20-24, include/kernels/ops.hpp:36-58): the four host
    # launchers are C-linkage symbols of libtilefusion.so under the reference's names
    import ctypes
    import os

    import torch  # noqa: F401  (the binding links against libtorch)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    lib = ctypes.CDLL(os.path.join(root, "tilefusion_amd", "libtilefusion.so"))
    for name in ("gemm", "fused_two_gemms", "flash_attention", "scatter_nd"):
        assert hasattr(lib, name), name
