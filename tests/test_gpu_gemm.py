"""The model's projection GEMM against the oracle (oracle/gemm.py), on the
reference's own cases (tests/test_gemm.py of the reference: seeded shapes,
non-block-aligned shapes, empty dimensions, mismatched K) and on the
projection shapes of SmolLM2-360M and Llama-3.2-3B for one decoded token,
a few tokens (the hand-written streaming kernel, up to 8 rows) and prompts
(the hand-written MFMA kernel; the simple FMA kernel for rows that are not
16-byte aligned).  Tolerances: fp32 2e-3 max-abs (the reference's own
bar is allclose(rtol 1e-2, atol 5e-2)); 16-bit outputs within their
rounding, rtol 8e-3 + atol 1e-2.
"""

import ctypes
import time

import numpy as np
import pytest

from oracle import numerics as on
from oracle.gemm import gemm_ref
from tests import _helpers as H
from triton_llm import gpu
from triton_llm.kernels import gemm, gemm_grouped

pytestmark = pytest.mark.gpu


def gemm_cpu(a, b, dtype="float32"):
    return H.download(gemm(H.upload(a, dtype), H.upload(b, dtype)))


@pytest.mark.parametrize("M,K,N", [(64, 128, 32), (128, 256, 128), (256, 512, 256), (65, 130, 33), (100, 200, 150)])
def test_gemm_reference_cases(M, K, N):
    np.random.seed(42)
    a = np.random.randn(M, K).astype(np.float32)
    b = np.random.randn(K, N).astype(np.float32)
    out = gemm_cpu(a, b)
    assert np.allclose(out, a @ b, rtol=1e-2, atol=5e-2)
    err = H.max_abs(out, gemm_ref(a, b))
    H.report(f"gemm {M}x{K}@{K}x{N}", err, 2e-3)
    assert err <= 2e-3


@pytest.mark.parametrize("dtype", ["float32", "bfloat16", "float16"])
@pytest.mark.parametrize("M", [1, 3, 8, 37])
@pytest.mark.parametrize("K,N", [(960, 960), (960, 320), (960, 2560), (2560, 960), (3072, 1024), (8192, 3072)])
def test_gemm_projection_shapes(dtype, M, K, N):
    rng = np.random.default_rng(K * 7 + N + M)
    a = on.to_storage(rng.standard_normal((M, K), dtype=np.float32), dtype)
    b = on.to_storage(rng.standard_normal((K, N), dtype=np.float32) / np.sqrt(K), dtype)
    got = on.from_storage(gemm_cpu(a, b, dtype), dtype)
    exp = gemm_ref(on.from_storage(a, dtype), on.from_storage(b, dtype))
    if dtype == "float32":
        err = H.max_abs(got, exp)
        H.report(f"{dtype} {M}x{K}@{K}x{N}", err, 2e-3)
        assert err <= 2e-3
    else:
        np.testing.assert_allclose(got, exp, rtol=8e-3, atol=1e-2)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("M", [1, 4])
@pytest.mark.parametrize("K,N", [(960, 49152), (576, 49152), (1024, 65536), (1040, 65536)])
def test_gemm_lm_head_shapes(dtype, M, K, N):
    """The lm_head of a decoded token: so many column tiles that K is one
    slice (960, 576, 1024), stored straight to C with no reduce pass; 1040 just
    past one slice takes the reduce.  Also into a strided C (ldc > N)."""
    rng = np.random.default_rng(K + M)
    a = on.to_storage(rng.standard_normal((M, K), dtype=np.float32), dtype)
    b = on.to_storage(rng.standard_normal((K, N), dtype=np.float32) / np.sqrt(K), dtype)
    exp = gemm_ref(on.from_storage(a, dtype), on.from_storage(b, dtype))
    got = on.from_storage(gemm_cpu(a, b, dtype), dtype)
    tol = (2e-3, 0.0) if dtype == "float32" else (1e-2, 8e-3)
    np.testing.assert_allclose(got, exp, atol=tol[0], rtol=tol[1])
    # strided C through the C ABI: row stride N + 64, padding left untouched
    lib = gpu.runtime()
    code = gpu.dtype_code(H.GPU_DTYPES[dtype])
    ldc = N + 64
    pad = np.full((M, ldc), 7.0, np.float32)
    c_dev = H.upload(on.to_storage(pad, dtype), dtype)
    a_dev, b_dev = H.upload(a, dtype), H.upload(b, dtype)
    nws = lib.tl_gemm_workspace_bytes(M, N, K, code)
    ws = gpu.zeros((max(nws, 1),), np.uint8)
    assert lib.tl_gemm(a_dev.ptr, b_dev.ptr, c_dev.ptr, M, N, K, K, N, ldc, ws.ptr, nws, code, None) == 0
    c = on.from_storage(H.download(c_dev), dtype)
    np.testing.assert_allclose(c[:, :N], exp, atol=tol[0], rtol=tol[1])
    assert (c[:, N:] == 7.0).all()


@pytest.mark.parametrize("M,K,N", [(1, 130, 33), (2, 7, 40), (5, 1000, 100), (8, 4100, 260)])
def test_gemm_few_rows_odd_shapes(M, K, N):
    """Few-row products on shapes the streaming kernel handles partly (a
    ragged last K-slice or column tile) or not at all (N not a multiple of
    the 16-byte chunk: the simple FMA kernel), against the oracle."""
    rng = np.random.default_rng(M * 1000 + K + N)
    a = rng.standard_normal((M, K), dtype=np.float32)
    b = rng.standard_normal((K, N), dtype=np.float32)
    err = H.max_abs(gemm_cpu(a, b), gemm_ref(a, b))
    H.report(f"few rows {M}x{K}@{K}x{N}", err, 2e-3)
    assert err <= 2e-3


def test_gemm_edge_cases():
    # K = 0: zeros of shape (M, N) (the reference only checks the shape)
    out = gemm_cpu(np.zeros((10, 0), np.float32), np.zeros((0, 10), np.float32))
    assert out.shape == (10, 10) and not out.any()
    assert gemm_cpu(np.zeros((0, 20), np.float32), np.ones((20, 10), np.float32)).shape == (0, 10)
    assert gemm_cpu(np.ones((10, 20), np.float32), np.zeros((20, 0), np.float32)).shape == (10, 0)
    with pytest.raises(AssertionError):
        gemm(gpu.to_device(np.ones((10, 20), np.float32)), gpu.to_device(np.ones((30, 10), np.float32)))
    with pytest.raises(AssertionError):
        gemm(gpu.to_device(np.ones((10, 20), np.float32)), gpu.to_device(np.ones((20, 10), np.float32)),
             out_dev=gpu.allocate((10, 11), np.float32))
    # a given output is written in place
    a, b = np.random.randn(33, 17).astype(np.float32), np.random.randn(17, 5).astype(np.float32)
    out = gpu.allocate((33, 5), np.float32)
    assert gemm(gpu.to_device(a), gpu.to_device(b), out_dev=out) is out
    assert H.max_abs(H.download(out), gemm_ref(a, b)) <= 2e-3


def test_gemm_reference_performance_bound():
    """The reference's performance test: 512x1024 @ 1024x512 under 50 ms
    per call including the copies."""
    a = np.random.randn(512, 1024).astype(np.float32)
    b = np.random.randn(1024, 512).astype(np.float32)
    for _ in range(3):
        gemm_cpu(a, b)
    t0 = time.perf_counter()
    for _ in range(10):
        gemm_cpu(a, b)
    assert (time.perf_counter() - t0) / 10 * 1e3 < 50


@pytest.mark.parametrize("dtype", ["float32", "bfloat16", "float16"])
@pytest.mark.parametrize("M,K,N", [(128, 3072, 1024), (300, 960, 2560), (517, 2560, 960), (2048, 3072, 3072),
                                   (64, 8192, 3072), (9, 136, 200)])
def test_gemm_prompt_shapes_mfma(dtype, M, K, N):
    """Prompt-sized products on the matrix-core kernel: the models' projection
    shapes, ragged tiles in M and N, K not a multiple of the LDS stage."""
    print(f"[case] gemm mfma {dtype} {M}x{K}@{K}x{N}", flush=True)
    rng = np.random.default_rng(M + 3 * K + 7 * N)
    a = on.to_storage(rng.standard_normal((M, K), dtype=np.float32), dtype)
    b = on.to_storage(rng.standard_normal((K, N), dtype=np.float32) / np.sqrt(K), dtype)
    got = on.from_storage(gemm_cpu(a, b, dtype), dtype)
    exp = gemm_ref(on.from_storage(a, dtype), on.from_storage(b, dtype))
    if dtype == "float32":
        err = H.max_abs(got, exp)
        H.report(f"mfma {dtype} {M}x{K}@{K}x{N}", err, 2e-3)
        assert err <= 2e-3
    else:
        np.testing.assert_allclose(got, exp, rtol=8e-3, atol=1e-2)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("M,K,Ns", [(1900, 136, (16456,)), (2048, 264, (16384,)), (2000, 72, (8192, 8200))])
def test_gemm_prompt_huge_tiles(dtype, M, K, Ns):
    """Large 16-bit products (520, 512 and 520 tiles of 256 x 256 here): ragged M
    and N, K tails inside a 32-k stage, and the grouped form."""
    print(f"[case] gemm huge {dtype} {M}x{K} -> {Ns}", flush=True)
    rng = np.random.default_rng(M + K + sum(Ns))
    a = on.to_storage(rng.standard_normal((M, K), dtype=np.float32), dtype)
    bs = [on.to_storage(rng.standard_normal((K, n), dtype=np.float32) / np.sqrt(K), dtype) for n in Ns]
    a_dev = H.upload(a, dtype)
    if len(Ns) == 1:
        outs = [gemm(a_dev, H.upload(bs[0], dtype))]
    else:
        outs = gemm_grouped(a_dev, [H.upload(b, dtype) for b in bs])
    for b, o in zip(bs, outs):
        got = on.from_storage(H.download(o), dtype)
        exp = gemm_ref(on.from_storage(a, dtype), on.from_storage(b, dtype))
        np.testing.assert_allclose(got, exp, rtol=8e-3, atol=1e-2)


@pytest.mark.parametrize("dtype,M,K,Ns", [("float32", 2048, 3072, (3072,)), ("float32", 1900, 3000, (3000,)),
                                          ("float32", 300, 3072, (3072, 1024, 1024)), ("float32", 2048, 8200, (3068,))])
def test_gemm_prompt_split_k(dtype, M, K, Ns):
    """fp32 products whose whole tiles would leave some CUs a tile more than
    others run K in slices (fp32 partials, one reduce pass): ragged M and N,
    a K tail in the last slice, the grouped form.  The workspace query
    reports the partials, so these shapes do take the split path."""
    print(f"[case] gemm split-k {dtype} {M}x{K} -> {Ns}", flush=True)
    lib = gpu.runtime()
    code = gpu.dtype_code(H.GPU_DTYPES[dtype])
    n_arr = (ctypes.c_int * len(Ns))(*Ns)
    assert lib.tl_gemm_grouped_workspace_bytes(M, K, len(Ns), n_arr, code) >= 2 * M * sum(Ns) * 4
    rng = np.random.default_rng(M + K + sum(Ns))
    a = on.to_storage(rng.standard_normal((M, K), dtype=np.float32), dtype)
    bs = [on.to_storage(rng.standard_normal((K, n), dtype=np.float32) / np.sqrt(K), dtype) for n in Ns]
    a_dev = H.upload(a, dtype)
    if len(Ns) == 1:
        outs = [gemm(a_dev, H.upload(bs[0], dtype))]
    else:
        outs = gemm_grouped(a_dev, [H.upload(b, dtype) for b in bs])
    for b, o in zip(bs, outs):
        got = on.from_storage(H.download(o), dtype)
        exp = gemm_ref(on.from_storage(a, dtype), on.from_storage(b, dtype))
        if dtype == "float32":
            err = H.max_abs(got, exp)
            H.report(f"split-k {dtype} {M}x{K}@{K}x{b.shape[1]}", err, 2e-3)
            assert err <= 2e-3
        else:
            np.testing.assert_allclose(got, exp, rtol=8e-3, atol=1e-2)


@pytest.mark.parametrize("M,K,Ns", [(2048, 960, (960, 320, 320)), (2048, 960, (960,)), (2048, 960, (320,)),
                                   (2000, 2560, (960,)), (1999, 964, (2560, 2560)), (1600, 960, (2560,)),
                                   (1999, 964, (648,))])
def test_gemm_prompt_fp32_plans(M, K, Ns):
    """fp32 prompt products of SmolLM2-360M's projections at about 2048 tokens:
    128- and 64-row tiles, whole-K and with K split (test_gemm_plans.py checks
    that both are reached): the grouped q/k/v, o / down with their splits, ragged
    M and a K tail inside a 32-k stage."""
    print(f"[case] gemm fp32 prompt {M}x{K} -> {Ns}", flush=True)
    rng = np.random.default_rng(M + 5 * K + sum(Ns))
    a = rng.standard_normal((M, K), dtype=np.float32)
    bs = [rng.standard_normal((K, n), dtype=np.float32) / np.float32(np.sqrt(K)) for n in Ns]
    a_dev = gpu.to_device(a)
    if len(Ns) == 1:
        outs = [gemm(a_dev, gpu.to_device(bs[0]))]
    else:
        outs = gemm_grouped(a_dev, [gpu.to_device(b) for b in bs])
    for b, o in zip(bs, outs):
        err = H.max_abs(H.download(o), gemm_ref(a, b))
        H.report(f"fp32 prompt {M}x{K}@{K}x{b.shape[1]}", err, 2e-3)
        assert err <= 2e-3


@pytest.mark.parametrize("dtype", ["bfloat16", "float16", "float32"])
@pytest.mark.parametrize("M,K,Ns", [(9, 3072, (3072,)), (33, 3072, (3072, 1024, 1024)), (64, 8192, (3072,)),
                                    (130, 3072, (3072, 1024)), (17, 3000, (3000,))])
def test_gemm_few_rows_split_k(dtype, M, K, Ns):
    """A batch of decoded tokens (9 to a few hundred rows): the MFMA product
    has only a few dozen tiles of C, so K is split until about one item per
    CU runs, two for fp32 (fp32 partials in the workspace, one reduce pass rounding to the
    output type); ragged M, a K tail, slices past K, the grouped form.  The
    workspace query reports the partials, so these shapes take the split path."""
    print(f"[case] gemm few-rows split-k {dtype} {M}x{K} -> {Ns}", flush=True)
    lib = gpu.runtime()
    code = gpu.dtype_code(H.GPU_DTYPES[dtype])
    n_arr = (ctypes.c_int * len(Ns))(*Ns)
    assert lib.tl_gemm_grouped_workspace_bytes(M, K, len(Ns), n_arr, code) >= 2 * M * sum(Ns) * 4
    rng = np.random.default_rng(M + K + sum(Ns))
    a = on.to_storage(rng.standard_normal((M, K), dtype=np.float32), dtype)
    bs = [on.to_storage(rng.standard_normal((K, n), dtype=np.float32) / np.sqrt(K), dtype) for n in Ns]
    a_dev = H.upload(a, dtype)
    if len(Ns) == 1:
        outs = [gemm(a_dev, H.upload(bs[0], dtype))]
    else:
        outs = gemm_grouped(a_dev, [H.upload(b, dtype) for b in bs])
    for b, o in zip(bs, outs):
        got = on.from_storage(H.download(o), dtype)
        exp = gemm_ref(on.from_storage(a, dtype), on.from_storage(b, dtype))
        if dtype == "float32":
            err = H.max_abs(got, exp)
            H.report(f"few-rows split-k {dtype} {M}x{K}@{K}x{b.shape[1]}", err, 2e-3)
            assert err <= 2e-3
        else:
            np.testing.assert_allclose(got, exp, rtol=8e-3, atol=1e-2)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16", "float32"])
@pytest.mark.parametrize("M", [9, 63, 64, 65])
def test_gemm_row_tile_boundaries(dtype, M):
    """Around the end of a 64-row tile (64 / 65 rows: one and two of them), with a K
    tail (1000 = 31 stages of 32 k + 8) and column counts that are not whole tiles,
    grouped and single."""
    print(f"[case] gemm row-tile boundary {dtype} M={M}", flush=True)
    K, Ns = 1000, (1000, 200)
    rng = np.random.default_rng(M)
    a = on.to_storage(rng.standard_normal((M, K), dtype=np.float32), dtype)
    bs = [on.to_storage(rng.standard_normal((K, n), dtype=np.float32) / np.sqrt(K), dtype) for n in Ns]
    a_dev = H.upload(a, dtype)
    outs = gemm_grouped(a_dev, [H.upload(b, dtype) for b in bs]) + [gemm(a_dev, H.upload(bs[1], dtype))]
    for b, o in zip(bs + [bs[1]], outs):
        got = on.from_storage(H.download(o), dtype)
        exp = gemm_ref(on.from_storage(a, dtype), on.from_storage(b, dtype))
        if dtype == "float32":
            err = H.max_abs(got, exp)
            H.report(f"row-tile boundary {dtype} {M}x{K}@{K}x{b.shape[1]}", err, 2e-3)
            assert err <= 2e-3
        else:
            assert np.all(np.isfinite(got))
            np.testing.assert_allclose(got, exp, rtol=8e-3, atol=1e-2)


@pytest.mark.parametrize("dtype,M", [("float32", 2048), ("float32", 40), ("bfloat16", 64)])
def test_gemm_prompt_split_k_without_workspace_runs_whole(dtype, M):
    """The C ABI with no workspace for a shape its plan would split: the
    product runs with whole-K tiles instead (no failure, same result)."""
    lib = gpu.runtime()
    K, N = 3072, 3072
    code = gpu.dtype_code(H.GPU_DTYPES[dtype])
    assert lib.tl_gemm_workspace_bytes(M, N, K, code) > 0
    rng = np.random.default_rng(5 + M)
    a = on.to_storage(rng.standard_normal((M, K), dtype=np.float32), dtype)
    b = on.to_storage(rng.standard_normal((K, N), dtype=np.float32) / np.sqrt(K), dtype)
    a_dev, b_dev = H.upload(a, dtype), H.upload(b, dtype)
    c_dev = gpu.allocate((M, N), H.GPU_DTYPES[dtype])
    assert lib.tl_gemm(a_dev.ptr, b_dev.ptr, c_dev.ptr, M, N, K, K, N, N, None, 0, code, None) == 0
    got = on.from_storage(H.download(c_dev), dtype)
    exp = gemm_ref(on.from_storage(a, dtype), on.from_storage(b, dtype))
    if dtype == "float32":
        err = H.max_abs(got, exp)
        H.report(f"split-k shape {M} rows, no workspace", err, 2e-3)
        assert err <= 2e-3
    else:
        np.testing.assert_allclose(got, exp, rtol=8e-3, atol=1e-2)


@pytest.mark.parametrize("dtype,K", [("bfloat16", 136), ("float16", 72), ("float32", 132), ("float32", 20)])
def test_gemm_strided_operands_keep_padding_out(dtype, K):
    """Row strides past the logical sizes, with NaN in every padding element:
    lda = K + 8 (the last LDS stage reads past K into the padding, which must
    not reach C), ldb = N + 8, ldc = N + 4 (padding of C left untouched)."""
    M, N = 150, 200
    print(f"[case] gemm strided {dtype} K={K}", flush=True)
    rng = np.random.default_rng(K)
    a = rng.standard_normal((M, K), dtype=np.float32)
    b = rng.standard_normal((K, N), dtype=np.float32) / np.sqrt(K)
    a_pad = np.full((M, K + 8), np.nan, np.float32)
    a_pad[:, :K] = a
    b_pad = np.full((K, N + 8), np.nan, np.float32)
    b_pad[:, :N] = b
    a_s, b_s = on.to_storage(a_pad, dtype), on.to_storage(b_pad, dtype)
    ldc = N + 4
    c_dev = H.upload(on.to_storage(np.full((M, ldc), 3.0, np.float32), dtype), dtype)
    lib = gpu.runtime()
    code = gpu.dtype_code(H.GPU_DTYPES[dtype])
    st = lib.tl_gemm(H.upload(a_s, dtype).ptr, H.upload(b_s, dtype).ptr, c_dev.ptr, M, N, K, K + 8, N + 8, ldc,
                     None, 0, code, None)
    assert st == 0
    c = on.from_storage(H.download(c_dev), dtype)
    exp = gemm_ref(on.from_storage(a_s, dtype)[:, :K], on.from_storage(b_s, dtype)[:, :N])
    if dtype == "float32":
        err = H.max_abs(c[:, :N], exp)
        H.report(f"strided {dtype} K={K}", err, 2e-3)
        assert err <= 2e-3
    else:  # output rounding of 16-bit C; NaN anywhere fails
        np.testing.assert_allclose(c[:, :N], exp, rtol=8e-3, atol=1e-2)
    assert (c[:, N:] == 3.0).all()


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("M", [1, 3, 8, 37, 300])
@pytest.mark.parametrize("K,Ns", [(3072, (3072, 1024, 1024)), (960, (2560, 2560)), (576, (576, 192, 192)),
                                  (100, (40, 0, 24))])
def test_gemm_grouped_matches_each_product(dtype, M, K, Ns):
    """q/k/v (and gate/up) in one launch: every output against the oracle.
    Few-row products share one K-slice plan and one reduce; prompts share one
    MFMA tile space; a zero-width group is skipped; (100, (40, 0, 24)) has
    rows that are not 16-byte aligned (the simple kernel, one grid layer per
    group)."""
    print(f"[case] gemm_grouped {dtype} M={M} K={K} N={Ns}", flush=True)
    rng = np.random.default_rng(M + K + sum(Ns))
    a = on.to_storage(rng.standard_normal((M, K), dtype=np.float32), dtype)
    bs = [on.to_storage(rng.standard_normal((K, n), dtype=np.float32) / np.sqrt(K), dtype) for n in Ns]
    outs = gemm_grouped(H.upload(a, dtype), [H.upload(b, dtype) for b in bs])
    for b, o in zip(bs, outs):
        got = on.from_storage(H.download(o), dtype)
        exp = gemm_ref(on.from_storage(a, dtype), on.from_storage(b, dtype))
        assert got.shape == exp.shape
        if dtype == "float32":
            err = H.max_abs(got, exp)
            H.report(f"grouped {dtype} {M}x{K}@{K}x{b.shape[1]}", err, 2e-3)
            assert err <= 2e-3
        else:
            np.testing.assert_allclose(got, exp, rtol=8e-3, atol=1e-2)


def test_gemm_few_rows_mixed_shapes_share_workspace():
    """Few-row products of different tilings, one after another and repeated,
    through the one module-wide workspace: each comes out right whatever ran
    before it."""
    rng = np.random.default_rng(5)
    shapes = [(1, 3072, 5120), (4, 8192, 3072), (1, 3072, 5120), (2, 3072, 16384), (8, 1000, 100), (1, 8192, 3072)]
    cases = []
    for M, K, N in shapes:
        a = rng.standard_normal((M, K), dtype=np.float32)
        b = (rng.standard_normal((K, N), dtype=np.float32) / np.sqrt(K)).astype(np.float32)
        cases.append((gpu.to_device(a), gpu.to_device(b), gemm_ref(a, b)))
    for rep in range(3):
        outs = [gemm(a, b) for a, b, _ in cases]
        for (M, K, N), out, (_, _, exp) in zip(shapes, outs, cases):
            err = H.max_abs(out.to_numpy(), exp)
            H.report(f"mixed shapes rep {rep} {M}x{K}@{K}x{N}", err, 2e-3)
            assert err <= 2e-3


def test_gemm_zero_k_strided_output_keeps_padding():
    """K = 0 writes zeros into the (M, N) view only: a strided C (ldc > N)
    keeps its padding columns, through the C ABI, for the single and the
    grouped entry points."""
    lib = gpu.runtime()
    M, N, ldc = 5, 40, 56
    print("[case] gemm K=0 strided", flush=True)
    c_dev = gpu.to_device(np.full((M, ldc), 7.0, np.float32))
    a_dev = gpu.allocate((M, 1), np.float32)
    b_dev = gpu.allocate((1, N), np.float32)
    assert lib.tl_gemm(a_dev.ptr, b_dev.ptr, c_dev.ptr, M, N, 0, 1, N, ldc, None, 0, 0, None) == 0
    c = c_dev.to_numpy()
    assert not c[:, :N].any() and (c[:, N:] == 7.0).all()
    c2 = gpu.to_device(np.full((M, ldc), 7.0, np.float32))
    ns = (ctypes.c_int * 2)(N, 8)
    bs = (ctypes.c_void_p * 2)(b_dev.ptr.value, b_dev.ptr.value)
    cs = (ctypes.c_void_p * 2)(c_dev.ptr.value, c2.ptr.value)
    lds_b = (ctypes.c_int64 * 2)(N, 8)
    lds_c = (ctypes.c_int64 * 2)(ldc, ldc)
    c_dev.from_numpy(np.full((M, ldc), 7.0, np.float32))
    assert lib.tl_gemm_grouped(a_dev.ptr, M, 0, 1, 2, bs, cs, ns, lds_b, lds_c, None, 0, 0, None) == 0
    c, c2h = c_dev.to_numpy(), c2.to_numpy()
    assert not c[:, :N].any() and (c[:, N:] == 7.0).all()
    assert not c2h[:, :8].any() and (c2h[:, 8:] == 7.0).all()


# The 16-bit prompt kernel's tiles (64 x 128 to 256 x 256), each reached, whole and
# with K split, by capping the CUs the plan counts rounds for
# (test_gemm_plans.py checks that they are): ragged last rows and columns, odd
# and even counts of 32-k stages, k tails of 8, 16 and 24, one stage, groups; NaN
# past k in A's padding, past n in B's. Tolerance as above: the output's rounding.
@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("M,K,Ns,cus", [
    (300, 136, (584,), 1), (300, 136, (584,), 3), (300, 136, (584,), 4), (300, 136, (584,), 6), (300, 136, (584,), 8),
    (300, 136, (584,), 16), (300, 136, (584, 200), 5), (193, 1000, (400,), 1), (193, 1000, (400,), 2),
    (130, 264, (328,), 4),
    (449, 72, (776,), 3), (449, 72, (776,), 256), (257, 24, (264,), 1), (65, 32, (8,), 256), (16, 8, (136,), 256),
    (1025, 64, (256,), 2), (300, 136, (584,), 5), (300, 136, (584,), 9),
    # with K split, every tile again
    (193, 2000, (400,), 6), (130, 1000, (400,), 4), (193, 2000, (400,), 12), (130, 2000, (328,), 16),
    (130, 2000, (328,), 12), (130, 1000, (328,), 24)])
def test_gemm_wide_tiles(monkeypatch, dtype, M, K, Ns, cus):
    print(f"[case] gemm wide {dtype} {M}x{K} -> {Ns} cus {cus}", flush=True)
    H.set_override(monkeypatch, "TRITON_LLM_HIP_MAX_CUS", cus)
    rng = np.random.default_rng(M + K + cus)
    pad = lambda x, w: np.concatenate([x, np.full((x.shape[0], w), np.nan, np.float32)], 1)  # noqa: E731
    a = on.to_storage(pad(rng.standard_normal((M, K), dtype=np.float32), 8), dtype)
    bs = [on.to_storage(pad(rng.standard_normal((K, n), dtype=np.float32) / np.float32(np.sqrt(K)), 8), dtype)
          for n in Ns]
    lib, code, n_g = gpu.runtime(), gpu.dtype_code(H.GPU_DTYPES[dtype]), len(Ns)
    for extra in (0, 4, 1):  # rows of C that take 16-byte stores, shorter runs, single elements
        a_dev, b_dev = H.upload(a, dtype), [H.upload(b, dtype) for b in bs]
        c_dev = [H.upload(on.to_storage(np.full((M, n + extra), 3.0, np.float32), dtype), dtype) for n in Ns]
        ws = gpu.allocate((max(1, lib.tl_gemm_grouped_workspace_bytes(M, K, n_g, (ctypes.c_int * n_g)(*Ns), code)),),
                          np.uint8)
        st = lib.tl_gemm_grouped(a_dev.ptr, M, K, K + 8, n_g, (ctypes.c_void_p * n_g)(*[b.data_ptr() for b in b_dev]),
                                 (ctypes.c_void_p * n_g)(*[c.data_ptr() for c in c_dev]), (ctypes.c_int * n_g)(*Ns),
                                 (ctypes.c_int64 * n_g)(*[n + 8 for n in Ns]),
                                 (ctypes.c_int64 * n_g)(*[n + extra for n in Ns]), ws.ptr, ws.nbytes, code, None)
        assert st == 0
        for b, c, n in zip(bs, c_dev, Ns):
            got = on.from_storage(H.download(c), dtype)
            exp = gemm_ref(on.from_storage(a, dtype)[:, :K], on.from_storage(b, dtype)[:, :n])
            np.testing.assert_allclose(got[:, :n], exp, rtol=8e-3, atol=1e-2)
            assert (got[:, n:] == 3.0).all()


# fp32 products split into bf16 parts: tile edges, k tails, both tile heights, K
# slices, rows of C that take scalar stores. Tolerance: six fp32 roundings a
# 32-k stage, each 2^-24 of the sum's magnitude bound |a| . |b|.
@pytest.mark.parametrize("M,K,Ns,cus", [(9, 4, (4,), 256), (65, 36, (132, 8), 256), (128, 32, (128,), 1),
                                        (129, 100, (260,), 2), (200, 1000, (196,), 4), (300, 2560, (264,), 256),
                                        (1100, 64, (516,), 8)])
def test_gemm_fp32_parts_tiles(monkeypatch, M, K, Ns, cus):
    print(f"[case] gemm fp32 parts {M}x{K} -> {Ns} cus {cus}", flush=True)
    H.set_override(monkeypatch, "TRITON_LLM_HIP_MAX_CUS", cus)
    rng = np.random.default_rng(M + K)
    a = rng.standard_normal((M, K), dtype=np.float32)
    bs = [rng.standard_normal((K, n), dtype=np.float32) for n in Ns]
    outs = gemm_grouped(gpu.to_device(a), [gpu.to_device(b) for b in bs])
    lib = gpu.runtime()
    c1 = gpu.to_device(np.full((M, Ns[0] + 1), 3.0, np.float32))
    a_d, b_d = gpu.to_device(a), gpu.to_device(bs[0])
    assert lib.tl_gemm(a_d.ptr, b_d.ptr, c1.ptr, M, Ns[0], K, K, Ns[0], Ns[0] + 1, None, 0, 0, None) == 0
    got1 = H.download(c1)
    assert (got1[:, Ns[0]:] == 3.0).all()
    for b, got in list(zip(bs, map(H.download, outs))) + [(bs[0], got1[:, :Ns[0]])]:
        exact = a.astype(np.float64) @ b.astype(np.float64)
        bound = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
        assert (np.abs(got - exact) <= 6 * (K / 32 + 1) * 2.0 ** -24 * bound + 1e-30).all()


def test_gemm_fp32_parts_whole_range():
    """Values whose parts do not cover them -- NaN, infinities, magnitudes near
    the ends of fp32 -- give what fp32 multiply-adds give, in their rows and
    columns and nowhere else; zeros and mixed magnitudes stay exact enough."""
    M, K, N = 150, 96, 200
    rng = np.random.default_rng(3)
    for what in ("nan", "inf", "inf0", "huge", "tiny-row", "tiny-column", "zero-row", "mixed"):
        a = rng.standard_normal((M, K), dtype=np.float32)
        b = rng.standard_normal((K, N), dtype=np.float32)
        if what == "nan":
            a[3, 5], b[7, 131] = np.nan, np.nan
        elif what == "inf":
            a[140, 95], b[0, 0] = np.inf, -np.inf
            b[95, :4] = 1.5  # exact in one part: infinity times the other parts' zeros must not appear
        elif what == "inf0":
            a[2, 2] = np.inf
            b[2, 9] = 0.0
        elif what == "huge":
            a[17, :] = np.float32(3e38) * np.sign(a[17])
            b *= np.float32(1e-3)
        elif what == "tiny-row":
            a[10] *= np.float32(1e-35)
        elif what == "tiny-column":
            b[:, 199] *= np.float32(1e-35)
        elif what == "zero-row":
            a[5], b[:, 6] = 0.0, 0.0
        else:
            a[:, ::3] *= np.float32(1e-12)
            b[1::2] *= np.float32(1e10)
        print(f"[case] gemm fp32 whole range {what}", flush=True)
        got = H.download(gemm(gpu.to_device(a), gpu.to_device(b)))
        with np.errstate(all="ignore"):
            ref = (a[:, :, None] * b[None]).astype(np.float32).sum(1, dtype=np.float64)
            bound = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
        # an fp32 chain may overflow where the sum stays finite; elsewhere the patterns are the same
        sure = np.abs(ref) < 3e38
        np.testing.assert_array_equal(np.isnan(got)[~np.isfinite(ref)], np.isnan(ref)[~np.isfinite(ref)])
        inf = np.isinf(ref) & ~np.isnan(got)
        np.testing.assert_array_equal(got[inf], ref[inf].astype(np.float32))
        ok = np.isfinite(ref) & sure & (bound < 1e38)
        assert (np.abs(got[ok] - ref[ok]) <= (K + 4) * 2.0 ** -24 * bound[ok] + 1e-45).all(), what


@pytest.mark.parametrize("dtype,K,lda", [("bfloat16", 130, 136), ("float16", 1001, 1008), ("float32", 131, 136),
                                         ("float32", 998, 1000)])
@pytest.mark.parametrize("M", [40, 150])
def test_gemm_partial_k_chunk(dtype, K, lda, M):
    """Aligned rows whose k ends inside a 16-byte chunk, NaN behind it (the
    kernel for such k, whole and with K slices)."""
    N = 136
    print(f"[case] gemm partial k chunk {dtype} {M}x{K}", flush=True)
    rng = np.random.default_rng(K + M)
    a = np.full((M, lda), np.nan, np.float32)
    a[:, :K] = rng.standard_normal((M, K), dtype=np.float32)
    b = rng.standard_normal((K, N), dtype=np.float32) / np.float32(np.sqrt(K))
    a_s, b_s = on.to_storage(a, dtype), on.to_storage(b, dtype)
    lib, code = gpu.runtime(), gpu.dtype_code(H.GPU_DTYPES[dtype])
    a_d, b_d, c_d = H.upload(a_s, dtype), H.upload(b_s, dtype), gpu.allocate((M, N), H.GPU_DTYPES[dtype])
    exp = gemm_ref(on.from_storage(a_s, dtype)[:, :K], on.from_storage(b_s, dtype))
    need = lib.tl_gemm_workspace_bytes(M, N, K, code)
    ws = gpu.allocate((max(1, need),), np.uint8)
    for ptr, size in ((None, 0), (ws.ptr, ws.nbytes)):
        assert lib.tl_gemm(a_d.ptr, b_d.ptr, c_d.ptr, M, N, K, lda, N, N, ptr, size, code, None) == 0
        got = on.from_storage(H.download(c_d), dtype)
        np.testing.assert_allclose(got, exp, rtol=1e-4 if dtype == "float32" else 8e-3,
                                   atol=1e-4 if dtype == "float32" else 1e-2)


# One and two tokens on the whole-K kernel: its largest K and one past it, its
# largest tile count and one past it, ragged columns, groups, few rows of K.
@pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("M,K,Ns", [(1, 1024, (8, 520)), (1, 1025, (520,)), (2, 1024, (264, 8)), (1, 1, (8,)),
                                    (1, 130, (8192,)), (1, 130, (8200,)), (2, 500, (2048,)), (2, 500, (2056,)),
                                    (1, 64, (16392,))])
def test_gemm_one_token_whole_k(dtype, M, K, Ns):
    print(f"[case] gemm whole-k {dtype} {M}x{K} -> {Ns}", flush=True)
    rng = np.random.default_rng(M + K + sum(Ns))
    a = on.to_storage(rng.standard_normal((M, K), dtype=np.float32), dtype)
    bs = [on.to_storage(rng.standard_normal((K, n), dtype=np.float32) / np.float32(np.sqrt(K)), dtype) for n in Ns]
    outs = gemm_grouped(H.upload(a, dtype), [H.upload(b, dtype) for b in bs])
    for b, o in zip(bs, outs):
        exp = gemm_ref(on.from_storage(a, dtype), on.from_storage(b, dtype))
        np.testing.assert_allclose(on.from_storage(H.download(o), dtype), exp, rtol=1e-4 if dtype == "float32" else 8e-3,
                                   atol=1e-4 if dtype == "float32" else 1e-2)


# Operands that are the first rows and columns of larger ones, NaN in every other
# element: the ring's loads past a slice's last row, and a ragged last tile's past
# the last column, come from inside the allocation here and must read as zeros.
@pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("M,K,N", [(150, 136, 200), (300, 96, 584), (40, 1000, 136), (260, 1000, 264)])
def test_gemm_views_of_larger_operands(dtype, M, K, N):
    print(f"[case] gemm view {dtype} {M}x{K}x{N}", flush=True)
    rng = np.random.default_rng(M + K + N)
    a, b = np.full((M + 400, K + 8), np.nan, np.float32), np.full((K + 1200, N + 264), np.nan, np.float32)
    a[:M, :K] = rng.standard_normal((M, K))
    b[:K, :N] = rng.standard_normal((K, N)) / np.sqrt(K)
    a_s, b_s = on.to_storage(a, dtype), on.to_storage(b, dtype)
    exp = gemm_ref(on.from_storage(a_s, dtype)[:M, :K], on.from_storage(b_s, dtype)[:K, :N])
    lib, code = gpu.runtime(), gpu.dtype_code(H.GPU_DTYPES[dtype])
    a_d, b_d, c_d = H.upload(a_s, dtype), H.upload(b_s, dtype), gpu.allocate((M, N), H.GPU_DTYPES[dtype])
    ws = gpu.allocate((max(1, lib.tl_gemm_workspace_bytes(M, N, K, code)),), np.uint8)
    for ptr, size in ((None, 0), (ws.ptr, ws.nbytes)):
        assert lib.tl_gemm(a_d.ptr, b_d.ptr, c_d.ptr, M, N, K, K + 8, N + 264, N, ptr, size, code, None) == 0
        got = on.from_storage(H.download(c_d), dtype)
        np.testing.assert_allclose(got, exp, rtol=1e-4 if dtype == "float32" else 8e-3,
                                   atol=1e-4 if dtype == "float32" else 1e-2)


def test_gemm_one_token_adds_its_waves_by_halves():
    """The sixteen waves' sums of the whole-K kernel, rows 8 w .. 8 w + 7 each:
    one of them is 1, the others 0.99 * 2^-24, which a chain that starts at 1
    would drop one by one (15 * 2^-24 in all).  By halves each of the four levels
    rounds once, and the first drops one of the small sums."""
    K, N = 1024, 64
    b = np.zeros((K, N), np.float32)
    b[8:128:8] = 0.99 * 2.0 ** -24
    b[0] = 1.0
    a = np.ones((1, K), np.float32)
    exact = a.astype(np.float64) @ b.astype(np.float64)
    got = H.download(gemm(gpu.to_device(a), gpu.to_device(b)))
    assert (np.abs(got - exact) <= 5 * 2.0 ** -24).all(), got[0, 0] - exact[0, 0]


@pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("M,N", [(1, 520), (2, 960), (2, 1024), (12, 136), (20, 456), (16, 3072), (64, 1024),
                                 (100, 1024)])
def test_gemm_output_over_its_input(dtype, M, N):
    """C = A in memory, where K is split: every workgroup's operands are read
    before the reduce pass writes.  At 12 and 20 rows a C of its
    own takes whole K."""
    print(f"[case] gemm in place {dtype} {M}x{N}", flush=True)
    rng = np.random.default_rng(M + N)
    a = on.to_storage(rng.standard_normal((M, N), dtype=np.float32), dtype)
    b = on.to_storage(rng.standard_normal((N, N), dtype=np.float32) / np.float32(np.sqrt(N)), dtype)
    lib, code = gpu.runtime(), gpu.dtype_code(H.GPU_DTYPES[dtype])
    need = lib.tl_gemm_workspace_bytes(M, N, N, code)
    assert need > 0
    exp = gemm_ref(on.from_storage(a, dtype), on.from_storage(b, dtype))
    b_d, ws = H.upload(b, dtype), gpu.allocate((need,), np.uint8)
    for _ in range(3):
        a_d = H.upload(a, dtype)
        assert lib.tl_gemm(a_d.ptr, b_d.ptr, a_d.ptr, M, N, N, N, N, N, ws.ptr, need, code, None) == 0
        np.testing.assert_allclose(on.from_storage(H.download(a_d), dtype), exp, rtol=1e-4 if dtype == "float32" else 8e-3,
                                   atol=1e-4 if dtype == "float32" else 1e-2)


# fp32 products whose parts do not cover an operand, on both tile heights, whole,
# with K in slices (the outlier in one of them) and in a group, rows of C that take
# vector and scalar stores: the tile comes from the fp32 MFMA, its rows and
# columns without an outlier unchanged in value.  Bound as for the parts.
@pytest.mark.parametrize("M,K,Ns,cus", [(150, 96, (200,), 256), (200, 1000, (196,), 4), (128, 68, (128, 40), 1),
                                        (300, 2560, (264,), 256)])
@pytest.mark.parametrize("what", ["nan", "inf", "huge", "tiny row", "tiny column", "tiny entries"])
def test_gemm_fp32_outliers(monkeypatch, M, K, Ns, cus, what):
    print(f"[case] gemm fp32 outliers {what} {M}x{K} -> {Ns} cus {cus}", flush=True)
    H.set_override(monkeypatch, "TRITON_LLM_HIP_MAX_CUS", cus)
    rng = np.random.default_rng(M + K)
    a = rng.standard_normal((M, K), dtype=np.float32)
    bs = [rng.standard_normal((K, n), dtype=np.float32) for n in Ns]
    if what == "nan":
        a[M // 2, K - 1], bs[0][0, 3] = np.nan, np.nan
    elif what == "inf":
        a[3, K - 1] = np.inf
        bs[0][K - 1, ::2] = 0.0
    elif what == "huge":
        a[M - 1, K // 2] = 1e30
        bs[0][K // 2] = 1e-3
    elif what == "tiny row":
        a[5] *= np.float32(1e-20)
    elif what == "tiny column":
        bs[0][:, 7] *= np.float32(1e-20)
    else:  # below 2^-102 beside ones, against columns that are zero where the ones are
        a[9, : K // 2] *= np.float32(1e-33)
        bs[0][K // 2:, : Ns[0] // 2] = 0.0
    lib, n_g = gpu.runtime(), len(Ns)
    a_d, b_d = gpu.to_device(a), [gpu.to_device(b) for b in bs]
    ns = (ctypes.c_int * n_g)(*Ns)
    ws = gpu.allocate((max(1, lib.tl_gemm_grouped_workspace_bytes(M, K, n_g, ns, 0)),), np.uint8)
    for extra in (0, 1):
        c_d = [gpu.to_device(np.full((M, n + extra), 3.0, np.float32)) for n in Ns]
        st = lib.tl_gemm_grouped(a_d.ptr, M, K, K, n_g, (ctypes.c_void_p * n_g)(*[b.data_ptr() for b in b_d]),
                                 (ctypes.c_void_p * n_g)(*[c.data_ptr() for c in c_d]), ns,
                                 (ctypes.c_int64 * n_g)(*Ns), (ctypes.c_int64 * n_g)(*[n + extra for n in Ns]),
                                 ws.ptr, ws.nbytes, 0, None)
        assert st == 0
        for b, c, n in zip(bs, c_d, Ns):
            got = H.download(c)
            assert (got[:, n:] == 3.0).all()
            with np.errstate(all="ignore"):
                exact = a.astype(np.float64) @ b.astype(np.float64)
                bound = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
            ok = np.isfinite(exact)
            np.testing.assert_array_equal(np.isnan(got[:, :n]), np.isnan(exact))
            np.testing.assert_array_equal(got[:, :n][np.isinf(exact)], exact[np.isinf(exact)].astype(np.float32))
            assert (np.abs(got[:, :n][ok] - exact[ok]) <= (K + 4) * 2.0 ** -24 * bound[ok] + 1e-44).all()


# Aligned rows whose k ends inside a 16-byte chunk, on the tiles and K slices that
# whole chunks take: every remainder, fewer k than a chunk, NaN in A's padding and
# behind B's last row, groups, each way C is stored.
@pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("M,K,Ns,cus", [(9, 1, (8,), 256), (9, 7, (136,), 256), (65, 33, (264, 8), 256),
                                        (130, 1002, (328,), 256), (40, 3069, (256,), 256), (300, 135, (584,), 1),
                                        (300, 134, (584,), 4), (300, 138, (584, 200), 16), (300, 1003, (200,), 256)])
def test_gemm_ragged_k(monkeypatch, dtype, M, K, Ns, cus):
    print(f"[case] gemm ragged k {dtype} {M}x{K} -> {Ns} cus {cus}", flush=True)
    H.set_override(monkeypatch, "TRITON_LLM_HIP_MAX_CUS", cus)
    rng = np.random.default_rng(M + K + cus)
    lda = (K + 7) // 8 * 8
    a = np.full((M, lda), np.nan, np.float32)
    a[:, :K] = rng.standard_normal((M, K))
    bs = [np.full((K + 2, n), np.nan, np.float32) for n in Ns]
    for b in bs:
        b[:K] = rng.standard_normal((K, b.shape[1])) / np.sqrt(K)
    a, bs = on.to_storage(a, dtype), [on.to_storage(b, dtype) for b in bs]
    lib, code, n_g = gpu.runtime(), gpu.dtype_code(H.GPU_DTYPES[dtype]), len(Ns)
    a_d, b_d, ns = H.upload(a, dtype), [H.upload(b, dtype) for b in bs], (ctypes.c_int * n_g)(*Ns)
    ws = gpu.allocate((max(1, lib.tl_gemm_grouped_workspace_bytes(M, K, n_g, ns, code)),), np.uint8)
    for extra, ptr, size in ((0, ws.ptr, ws.nbytes), (4, None, 0), (1, ws.ptr, ws.nbytes)):
        c_d = [H.upload(on.to_storage(np.full((M, n + extra), 3.0, np.float32), dtype), dtype) for n in Ns]
        st = lib.tl_gemm_grouped(a_d.ptr, M, K, lda, n_g, (ctypes.c_void_p * n_g)(*[b.data_ptr() for b in b_d]),
                                 (ctypes.c_void_p * n_g)(*[c.data_ptr() for c in c_d]), ns,
                                 (ctypes.c_int64 * n_g)(*Ns), (ctypes.c_int64 * n_g)(*[n + extra for n in Ns]),
                                 ptr, size, code, None)
        assert st == 0
        for b, c, n in zip(bs, c_d, Ns):
            got = on.from_storage(H.download(c), dtype)
            exp = gemm_ref(on.from_storage(a, dtype)[:, :K], on.from_storage(b, dtype)[:K])
            np.testing.assert_allclose(got[:, :n], exp, rtol=1e-4 if dtype == "float32" else 8e-3,
                                       atol=1e-4 if dtype == "float32" else 1e-2)
            assert (got[:, n:] == 3.0).all()


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("lda,ldb", [((1 << 22) + 8, 24), (80, 1 << 24)])
def test_gemm_long_strides(dtype, lda, ldb):
    """Row strides whose tiles and stages, counted past the operands' ends, come near
    or past 32 bits."""
    M, K, N = 9, 9, 24
    if dtype == "float32":
        ldb = min(ldb, 1 << 23)
    print(f"[case] gemm long strides {dtype} lda {lda} ldb {ldb}", flush=True)
    rng = np.random.default_rng(lda)
    a, b = np.zeros((M, lda), np.float32), np.zeros((K, ldb), np.float32)
    a[:, :K], b[:, :N] = rng.standard_normal((M, K)), rng.standard_normal((K, N))
    a[:, K:K + 8] = np.nan
    a_s, b_s = on.to_storage(a, dtype), on.to_storage(b, dtype)
    exp = gemm_ref(on.from_storage(a_s[:, :K], dtype), on.from_storage(b_s[:, :N], dtype))
    lib, code = gpu.runtime(), gpu.dtype_code(H.GPU_DTYPES[dtype])
    a_d, b_d, c_d = H.upload(a_s, dtype), H.upload(b_s, dtype), gpu.allocate((M, N), H.GPU_DTYPES[dtype])
    assert lib.tl_gemm(a_d.ptr, b_d.ptr, c_d.ptr, M, N, K, lda, ldb, N, None, 0, code, None) == 0
    got = on.from_storage(H.download(c_d), dtype)
    np.testing.assert_allclose(got, exp, rtol=1e-4 if dtype == "float32" else 8e-3,
                               atol=1e-4 if dtype == "float32" else 1e-2)
