"""GPU parity of the dense path (dequantize, GEMV, small-M, tile GEMM) against
the CPU oracle, through the C ABI.

The first half replays the reference's own test cases for this path
(src/ops/transformer.rs qk_tests / q6_k_tests, src/diffusion/tests.rs:716-761)
with its closed-form inputs and its tolerances; the second half applies the
benchmark's bars (dequant bit-exact; max relative error 1e-3 and relative L2
1e-5 with f32 accumulation) at the benchmark shapes on seeded synthetic blocks.
"""
import ctypes
import functools

import numpy as np
import pytest

import ferrum_fixtures as fx
import oracle
from helpers import assert_matmul_parity, bits, few_rows, fma_gemv, oracle_columns, rel_l2
from ferrum_amd import synth

pytestmark = pytest.mark.gpu

Q4_K, Q6_K = 12, 14


@pytest.fixture(scope="module")
def api():
    from ferrum_amd import api as module
    return module


@pytest.fixture(scope="module")
def d(api):
    return api.Device.new()


def qm(api, d, ggml, rows, cols, packed):
    fmt = api.QuantizationFormat(ggml)
    return api.QuantizedMatrix.from_reader(d, rows, cols, fmt, lambda dst: np.copyto(dst, packed))


# ------------------------------------------------------------- dequantize

@pytest.mark.parametrize("ggml,rows,cols", [(Q4_K, 5, 512), (Q6_K, 5, 512), (Q4_K, 133, 2560),
                                            (Q6_K, 133, 2560)])
def test_dequantize_is_bit_exact_on_reference_fixtures(api, d, ggml, rows, cols):
    packed = fx.q4k_packed(rows, cols) if ggml == Q4_K else fx.q6k_packed(rows, cols)
    w = qm(api, d, ggml, rows, cols, packed)
    assert w.byte_size() == rows * (cols // 256) * (144 if ggml == Q4_K else 210)
    got = d.dequantize(w).to_f32()
    assert np.array_equal(bits(got), bits(oracle.dequantize(ggml, packed, rows, cols)))


@pytest.mark.parametrize("ggml", [Q4_K, Q6_K])
def test_dequantize_is_bit_exact_on_synthetic_blocks_in_every_dtype(api, d, ggml):
    rows, cols = 257, 5120
    packed = synth.matrix(ggml, rows, cols, seed=1234)
    w = qm(api, d, ggml, rows, cols, packed)
    want = oracle.dequantize(ggml, packed, rows, cols)
    assert np.array_equal(bits(d.dequantize(w).to_f32()), bits(want))
    for dtype, code in ((api.DType.F16, oracle.F16), (api.DType.BF16, oracle.BF16)):
        got = d.dequantize(w, dtype).to_f32()
        assert np.array_equal(bits(got), bits(oracle.round_storage(want, code).reshape(rows, cols)))


def test_embedding_gather_decodes_selected_rows(api, d):
    # src/ops/transformer.rs:3307-3329 and :4351-4369: bitwise after BF16 rounding
    for ggml, packed in ((Q4_K, fx.q4k_packed(5, 512)), (Q6_K, fx.q6k_packed(5, 512))):
        w = qm(api, d, ggml, 5, 512, packed)
        ids = [4, 0, 3]
        out = d.embedding_gather_quantized(w, ids, api.DType.BF16)
        assert out.operation == ("embedding_gather_q4_k" if ggml == Q4_K else "embedding_gather_q6_k")
        dense = oracle.dequantize(ggml, packed, 5, 512)
        want = oracle.round_storage(dense[ids], oracle.BF16).reshape(3, 512)
        assert np.array_equal(bits(out.tensor.to_f32()), bits(want))
        with pytest.raises(api.TokenError):
            d.embedding_gather_quantized(w, [5], api.DType.BF16)


# ---------------------------------------------- the reference's GEMV / GEMM cases

def test_q4_k_gemv_gemm_cover_blocks_and_batch_tails(api, d):
    # src/ops/transformer.rs:2982-3002
    n, k = 5, 512
    packed = fx.q4k_packed(n, k)
    w = qm(api, d, Q4_K, n, k, packed)
    for m in (1, 2, 3, 4, 5, 7):
        values = fx.q4k_input(m, k)
        x = api.Tensor.from_f32(d, (m, k), api.DType.F32, values)
        actual = d.project_quantized(x, w).tensor.to_f32()
        reference = oracle.project(Q4_K, packed, n, k, values)
        assert np.abs(actual - reference).max() <= 2.0e-4, m


def test_q6_k_gemv_gemm_cover_superblock_and_batch_tails(api, d):
    # src/ops/transformer.rs:4251-4269
    n, k = 5, 512
    packed = fx.q6k_packed(n, k)
    w = qm(api, d, Q6_K, n, k, packed)
    for m in (1, 2, 3, 4, 5, 7):
        values = fx.q6k_input(m, k)
        x = api.Tensor.from_f32(d, (m, k), api.DType.F32, values)
        actual = d.project_quantized(x, w).tensor.to_f32()
        reference = oracle.project(Q6_K, packed, n, k, values)
        assert np.abs(actual - reference).max() <= 0.02, m
        # far tighter than the reference asks: f32 parity
        assert np.abs(actual - reference).max() <= 1e-4 * max(1.0, np.abs(reference).max())


@pytest.mark.parametrize("ggml", [Q4_K, Q6_K])
def test_gemv_ksplit_covers_row_and_block_tails(api, d, ggml):
    # src/ops/transformer.rs:3004-3029 and :4190-4214: 133 rows leave a partial
    # row tile; 10 and 19 super-blocks leave partial strides for every split.
    with pytest.raises(api.ParameterError):
        d.set_k_quant_gemv_ksplit(3)
    try:
        for n, k in ((133, 2560), (6, 4864)):
            packed = fx.q4k_packed(n, k) if ggml == Q4_K else fx.q6k_packed(n, k)
            values = fx.q4k_input(1, k) if ggml == Q4_K else fx.q6k_input(1, k)
            w = qm(api, d, ggml, n, k, packed)
            x = api.Tensor.from_f32(d, (1, k), api.DType.F32, values)
            reference = oracle.project(ggml, packed, n, k, values)
            outputs = []
            for simds in (1, 2, 4, 8):
                d.set_k_quant_gemv_ksplit(simds)
                out = d.project_quantized(x, w)
                name = "q4_k" if ggml == Q4_K else "q6_k"
                assert out.operation == (f"{name}_gemv_ksplit" if simds > 1 else f"{name}_gemv_factored")
                actual = out.tensor.to_f32()
                assert np.all(np.abs(actual - reference) <= 1.0e-3 * np.maximum(np.abs(reference), 1.0)), \
                    (n, k, simds)
                # segments meet in a fixed order: a second launch gives the same bits
                again = d.project_quantized(x, w).tensor.to_f32()
                assert np.array_equal(bits(actual), bits(again))
                outputs.append(actual)
    finally:
        d.set_k_quant_gemv_ksplit(0)


@pytest.mark.parametrize("dtype_name", ["F16", "BF16"])
def test_gemv_accepts_half_precision_activations(api, d, dtype_name):
    n, k = 133, 1024
    dtype = api.DType[dtype_name]
    code = oracle.F16 if dtype_name == "F16" else oracle.BF16
    for ggml in (Q4_K, Q6_K):
        packed = fx.q4k_packed(n, k) if ggml == Q4_K else fx.q6k_packed(n, k)
        w = qm(api, d, ggml, n, k, packed)
        values = fx.q4k_input(1, k)
        x = api.Tensor.from_f32(d, (1, k), dtype, values)
        rounded = x.to_f32()
        assert np.array_equal(rounded, oracle.round_storage(values, code).reshape(1, k))
        out = d.project_quantized(x, w)                      # output dtype = input dtype
        want = oracle.project(ggml, packed, n, k, rounded, accumulate="f64")
        assert np.array_equal(out.tensor.to_f32(), oracle.round_storage(out.tensor.to_f32(), code).reshape(1, n))
        assert rel_l2(out.tensor.to_f32(), want) <= (1e-3 if dtype_name == "F16" else 6e-3)
        out32 = d.project_quantized(x, w, out_dtype=api.DType.F32).tensor.to_f32()
        assert_matmul_parity(out32, want, f"{dtype_name} gemv")


def test_k_quant_gemms_match_the_cpu_dequant(api, d):
    # src/diffusion/tests.rs:716-761: F16 activations, M=200, K=512, N=100,
    # f64-accumulated CPU dequant, worst error <= 2e-3 * max|ref|.
    m, k, n = 200, 512, 100
    x = oracle.round_storage(fx.xorshift_uniform(m * k, 31), oracle.F16).reshape(m, k)
    for ggml in (Q4_K, Q6_K):
        packed = fx.xorshift_blocks(ggml, n * k // 256)
        w = qm(api, d, ggml, n, k, packed)
        xt = api.Tensor.from_f32(d, (m, k), api.DType.F16, x)
        out = d.project_quantized(xt, w, out_dtype=api.DType.F32)
        assert out.operation.startswith("q4_k_gemm_mfma" if ggml == Q4_K else "q6_k_gemm_mfma")
        got = out.tensor.to_f32()
        want = oracle.project(ggml, packed, n, k, x, accumulate="f64")
        scale = np.abs(want).max()
        assert scale > 0.1, "reference is vacuous"
        assert np.abs(got - want).max() <= 2e-3 * scale
        # against the tile-dtype oracle (weights rounded to f16 first) the
        # result is f32-accumulation accurate
        tile = oracle.project(ggml, packed, n, k, x, accumulate="f64", weight_round=oracle.F16)
        assert_matmul_parity(got, tile, "f16 tile gemm")


def test_bf16_tile_gemm_covers_row_output_and_group_tails(api, d):
    # src/ops/transformer.rs:3115-3175: (N, K) = (65, 512), M in {4, 8, 15, 35},
    # BF16 activations, weights rounded to BF16, result stored as BF16, abs <= 0.04.
    n, k = 65, 512
    for ggml, tol in ((Q4_K, 0.04), (Q6_K, 0.12)):
        packed = fx.q4k_packed(n, k) if ggml == Q4_K else fx.q6k_packed(n, k)
        w = qm(api, d, ggml, n, k, packed)
        for m in (4, 8, 15, 35):
            values = fx.q4k_input(m, k) if ggml == Q4_K else fx.q6k_input(m, k)
            x = api.Tensor.from_f32(d, (m, k), api.DType.BF16, values)
            rounded = x.to_f32()
            expected = oracle.project(ggml, packed, n, k, rounded, weight_round=oracle.BF16,
                                      out_round=oracle.BF16)
            out = d.project_quantized(x, w)
            assert "gemm_mfma" in out.operation
            assert np.abs(out.tensor.to_f32() - expected).max() <= tol, (ggml, m)


@pytest.mark.parametrize("ggml,dtype_name", [(Q4_K, "F16"), (Q6_K, "BF16")])
def test_tile_gemm_both_tile_sizes_match_the_f16_tile_oracle(api, d, ggml, dtype_name):
    # M = 130 rows: N = 16000 takes 128 x 128 tiles (250 workgroups), N = 1000 takes
    # 64 x 64 tiles; both have ragged last tiles in M and N.  Oracle on sampled columns.
    k, m = 512, 130
    dtype = api.DType[dtype_name]
    code = oracle.F16 if dtype_name == "F16" else oracle.BF16
    x = oracle.round_storage(synth.activations(m, k, seed=91), code).reshape(m, k)
    xt = api.Tensor.from_f32(d, x.shape, dtype, x)
    for n in (16000, 1000):
        packed = synth.matrix(ggml, n, k, seed=92 + n)
        w = qm(api, d, ggml, n, k, packed)
        d.set_tuning("gemm_resident", 0)   # rows this short would otherwise stay in LDS (tested below),
        d.set_tuning("gemm_wide_shape", 0) # and the 128-row tiles of the 32x32x16 form would take 16000 columns
        try:
            out = d.project_quantized(xt, w, out_dtype=api.DType.F32)
        finally:
            d.set_tuning("gemm_resident", 1)
            d.set_tuning("gemm_wide_shape", 1)
        assert out.operation == ("q4_k_gemm_mfma" if ggml == Q4_K else "q6_k_gemm_mfma")
        got = out.tensor.to_f32()
        rows = np.unique(np.concatenate([np.arange(0, 130), np.arange(n - 70, n),
                                         synth.rng(93).integers(0, n, 64)]))
        want = oracle_columns(ggml, packed, n, k, rows, x, weight_round=code, accumulate="f64")
        assert_matmul_parity(got[:, rows], want, f"tile gemm n={n}")


@pytest.mark.parametrize("ggml,dtype_name", [(Q4_K, "F16"), (Q4_K, "BF16"), (synth.Q5_K, "F16"),
                                             (synth.Q5_K, "BF16"), (Q6_K, "F16"), (Q6_K, "BF16")])
def test_register_dequant_gemm_up_to_64_rows(api, d, ggml, dtype_name):
    # 33..64 rows stay on the kernel that dequantises in registers (four 16-row MFMA
    # operands per wave); 65 is the first row count on the 256-row tile.  N = 1100 leaves
    # a ragged last row group.
    n, k = 1100, 1280
    dtype = api.DType[dtype_name]
    code = oracle.F16 if dtype_name == "F16" else oracle.BF16
    packed = synth.matrix(ggml, n, k, seed=131)
    w = qm(api, d, ggml, n, k, packed)
    for m in (32, 33, 49, 64, 65):
        x = oracle.round_storage(synth.activations(m, k, seed=132 + m), code).reshape(m, k)
        d.set_tuning("gemm_resident", 0)   # rows too long for LDS take these kernels; these would fit
        try:
            out = d.project_quantized(api.Tensor.from_f32(d, x.shape, dtype, x), w, out_dtype=api.DType.F32)
        finally:
            d.set_tuning("gemm_resident", 1)
        assert out.operation.endswith("_skinny") == (m <= 64), (m, out.operation)
        want = oracle.project(ggml, packed, n, k, x, weight_round=code, accumulate="f64")
        assert_matmul_parity(out.tensor.to_f32(), want, f"{dtype_name} m={m}")


@pytest.mark.parametrize("ggml", [Q4_K, Q6_K])
def test_f32_activations_take_the_tile_kernels_from_a_chosen_row_count(api, d, ggml):
    # HybridModel::project (src/hybrid/engine.rs:3407-3500) sends f32 activations to f16
    # tiles from 5 rows on; here that is opt-in, and below the threshold (or with the key at
    # 0) every row keeps exact f32 weights.
    n, k = 1100, 1024
    packed = synth.matrix(ggml, n, k, seed=121)
    w = qm(api, d, ggml, n, k, packed)
    d.set_tuning("gemm_f32_min_rows", 5)
    try:
        for m in (4, 5, 16, 40, 130):
            x = synth.activations(m, k, seed=122 + m)
            out = d.project_quantized(api.Tensor.from_f32(d, x.shape, api.DType.F32, x), w)
            assert out.tensor.dtype == api.DType.F32
            if m < 5:
                assert out.operation.endswith("_gemm") and "mfma" not in out.operation
                want = oracle.project(ggml, packed, n, k, x, accumulate="f64")
            else:
                assert "gemm_mfma" in out.operation
                want = oracle.project(ggml, packed, n, k, oracle.round_storage(x, oracle.F16).reshape(m, k),
                                      weight_round=oracle.F16, accumulate="f64")
            assert_matmul_parity(out.tensor.to_f32(), want, f"f32 activations m={m}")
    finally:
        d.set_tuning("gemm_f32_min_rows", 0)
    x = synth.activations(16, k, seed=123)
    exact = d.project_quantized(api.Tensor.from_f32(d, x.shape, api.DType.F32, x), w)
    assert "mfma" not in exact.operation
    assert_matmul_parity(exact.tensor.to_f32(), oracle.project(ggml, packed, n, k, x, accumulate="f64"), "exact f32")
    with pytest.raises(api.ParameterError):
        d.set_tuning("gemm_f32_min_rows", 1)


# ------------------------------------------------------- benchmark shapes

def check_gemv(api, d, ggml, n, k, seed, l2_tol=1e-5):
    packed = synth.matrix(ggml, n, k, seed)
    x = synth.activations(1, k, seed)
    w = qm(api, d, ggml, n, k, packed)
    xt = api.Tensor.from_f32(d, (1, k), api.DType.F32, x)
    got = d.project_quantized(xt, w).tensor.to_f32()
    want64 = oracle.project(ggml, packed, n, k, x, accumulate="f64", threads=8)
    want32 = oracle.project(ggml, packed, n, k, x, accumulate="f32", threads=8)
    l2, mr = assert_matmul_parity(got, want64, f"gemv {ggml} {n}x{k} vs f64", l2_tol=l2_tol)
    # the reference's sequential-f32 answer, whose own rounding error grows with K
    assert_matmul_parity(got, want32, f"gemv {ggml} {n}x{k} vs f32seq", l2_tol=l2_tol)
    assert l2 <= rel_l2(want32, want64) * 1.5 + 1e-7, "GPU is less accurate than the sequential CPU sum"


# The streamed matrix-core GEMV (dense Q4_K and Q6_K): row lengths on both sides of its per-wave
# block budgets, tile heights 1..16, every activation dtype, batched rows; rows too long for one
# tile (more than 48 super-blocks, or 16 rows of them past 64 KB) are cut into 2 to 6 K segments.
# Q6_K rows take it when they hold an even number of super-blocks (their 210-byte blocks then start
# on a dword).
STREAM_SHAPES = [(Q4_K, n, k) for n, k in [(37, 256), (133, 2560), (300, 4864), (1100, 5120), (4100, 2048), (70, 6144),
                                           (33, 8192), (20, 12288), (100, 12544), (777, 14336), (530, 17408),
                                           (64, 34816)]]
STREAM_SHAPES += [(Q6_K, n, k) for n, k in [(37, 512), (133, 2560), (300, 4608), (1100, 5120), (4100, 2048), (70, 6144),
                                            (33, 8192), (200, 9728), (20, 12288), (100, 12800), (777, 14336),
                                            (530, 17408), (64, 34816)]]


@pytest.mark.parametrize("ggml,n,k", STREAM_SHAPES)
@pytest.mark.parametrize("dtype", ["F32", "F16", "BF16"])
def test_streamed_gemv_matches_the_oracle(api, d, ggml, n, k, dtype):
    code = {"F32": oracle.F32, "F16": oracle.F16, "BF16": oracle.BF16}[dtype]
    name = "q4_k" if ggml == Q4_K else "q6_k"
    packed = synth.matrix(ggml, n, k, seed=n + k)
    w = qm(api, d, ggml, n, k, packed)
    d.set_tuning("gemv_stream", 2)   # also where the matrix is small enough for the FMA kernel to win
    for m in ((1, 3) if dtype == "F32" else (1,)):   # 16-bit rows beyond the first take the tile kernels
        x = oracle.round_storage(synth.activations(m, k, seed=7 * n + m), code).reshape(m, k)
        xt = api.Tensor.from_f32(d, (m, k), getattr(api.DType, dtype), x)
        out = d.project_quantized(xt, w, out_dtype=api.DType.F32)
        if m > 1:
            assert out.operation == name + "_gemm"
        elif ggml == Q4_K:
            assert out.operation == ("q4_k_gemv_ksplit" if k > 12288 else "q4_k_gemv_factored")
        else:
            assert out.operation in ("q6_k_gemv_ksplit", "q6_k_gemv_factored")
            assert k <= 12288 or out.operation == "q6_k_gemv_ksplit"
        segmented = out.operation.endswith("ksplit")
        want = oracle.project(ggml, packed, n, k, x, accumulate="f64")
        assert_matmul_parity(out.tensor.to_f32(), want, f"streamed gemv {name} {n}x{k} {dtype} m={m}")
        if segmented:   # the segments are added in a fixed order
            again = d.project_quantized(xt, w, out_dtype=api.DType.F32).tensor.to_f32()
            assert np.array_equal(bits(again), bits(out.tensor.to_f32()))
        with fma_gemv(d):
            other = d.project_quantized(xt, w, out_dtype=api.DType.F32).tensor.to_f32()
        assert rel_l2(out.tensor.to_f32(), other) <= 1e-5 and not np.array_equal(bits(out.tensor.to_f32()), bits(other))
        # tiles of up to 14 rows are loaded block by block by the waves that multiply them, taller
        # ones row by row by all waves: the same arithmetic either way
        d.set_tuning("gemv_stream_own_loads", 0)
        try:
            by_rows = d.project_quantized(xt, w, out_dtype=api.DType.F32).tensor.to_f32()
        finally:
            d.set_tuning("gemv_stream_own_loads", 1)
        assert np.array_equal(bits(by_rows), bits(out.tensor.to_f32()))
    d.set_tuning("gemv_stream", 1)


@pytest.mark.parametrize("n,k", [(5, 256), (37, 4096), (4113, 4352), (100, 6144), (8209, 2560), (77, 6400), (2100, 12544), (200, 34816)])
@pytest.mark.parametrize("dtype", ["F32", "F16", "BF16"])
def test_ring_gemv_matches_the_oracle(api, d, n, k, dtype):
    # one tile and fewer, a workgroup's second and third tile, one and two super-blocks a wave, two to six K segments;
    # the operands are those of the kernel that gives every tile a workgroup, only the waves' sums are cut otherwise:
    # some 2 sqrt(nb) more roundings of 2^-24 / sqrt(3)
    code = {"F32": oracle.F32, "F16": oracle.F16, "BF16": oracle.BF16}[dtype]
    packed = synth.matrix(Q4_K, n, k, seed=n + k)
    w = qm(api, d, Q4_K, n, k, packed)
    x = oracle.round_storage(synth.activations(1, k, seed=7 * n + 1), code).reshape(1, k)
    xt = api.Tensor.from_f32(d, (1, k), getattr(api.DType, dtype), x)
    d.set_tuning("gemv_stream", 2)
    try:
        d.set_tuning("gemv_ring", 0)
        tiles = d.project_quantized(xt, w, out_dtype=api.DType.F32).tensor.to_f32()
        d.set_tuning("gemv_ring", 2)
        out = d.project_quantized(xt, w, out_dtype=api.DType.F32)
        again = d.project_quantized(xt, w, out_dtype=api.DType.F32).tensor.to_f32()
    finally:
        d.set_tuning("gemv_ring", 1)
        d.set_tuning("gemv_stream", 1)
    assert out.operation == ("q4_k_gemv_ksplit" if k > 6144 else "q4_k_gemv_factored")
    got = out.tensor.to_f32()
    assert np.array_equal(bits(got), bits(again))
    assert_matmul_parity(got, oracle.project(Q4_K, packed, n, k, x, accumulate="f64"), f"ring {n}x{k} {dtype}")
    assert rel_l2(got, tiles) <= 2 * np.sqrt(k / 256) * 2.0 ** -24 / np.sqrt(3) + 2.0 ** -24


def test_large_q4_k_matrices_take_the_ring_by_themselves(api, d):
    n, k = 34010, 5120      # 680,200 super-blocks
    base = synth.matrix(Q4_K, 1790, k, seed=31).reshape(1790, -1)
    w = qm(api, d, Q4_K, n, k, np.tile(base, (n // 1790, 1)).reshape(-1))
    xt = api.Tensor.from_f32(d, (1, k), api.DType.F32, synth.activations(1, k, seed=32))
    got = d.project_quantized(xt, w).tensor.to_f32()
    d.set_tuning("gemv_ring", 2)
    try:
        forced = d.project_quantized(xt, w).tensor.to_f32()
        d.set_tuning("gemv_ring", 0)
        tiles = d.project_quantized(xt, w).tensor.to_f32()
    finally:
        d.set_tuning("gemv_ring", 1)
    assert np.array_equal(bits(got), bits(forced)) and not np.array_equal(bits(got), bits(tiles))
    assert rel_l2(got, tiles) <= 6e-7 and np.array_equal(bits(got[0, :1790]), bits(got[0, -1790:]))


@pytest.mark.parametrize("n,k,streamed", [(22000, 3072, True), (31250, 2048, True), (6300, 10240, True), (31200, 2048, False),
                                          (9000, 6144, False), (50000, 1536, False)])
def test_large_q6_k_matrices_of_long_rows_are_streamed(api, d, n, k, streamed):
    # from 250,000 super-blocks in rows of eight on, whole rows and cut ones, an f32 row alone takes the streamed kernel
    base = synth.matrix(Q6_K, 50, k, seed=k).reshape(50, -1)
    w = qm(api, d, Q6_K, n, k, np.resize(base, (n, base.shape[1])).reshape(-1))
    x = synth.activations(1, k, seed=k + 1).reshape(1, k)
    xt = api.Tensor.from_f32(d, (1, k), api.DType.F32, x)
    got = d.project_quantized(xt, w).tensor.to_f32()
    other = {}
    for mode in (0, 2):
        d.set_tuning("gemv_stream", mode)
        try:
            other[mode] = d.project_quantized(xt, w).tensor.to_f32()
        finally:
            d.set_tuning("gemv_stream", 1)
    assert np.array_equal(bits(got), bits(other[2 if streamed else 0])) and not np.array_equal(bits(other[0]), bits(other[2]))
    assert_matmul_parity(got[:, :50], oracle.project(Q6_K, base.reshape(-1), 50, k, x, accumulate="f64"), f"{n} x {k}")
    assert np.array_equal(bits(got), bits(got[:, np.arange(n) % 50]))


@pytest.mark.parametrize("n,k,fma", [(16400, 256, True), (4200, 1024, True), (3300, 1280, False), (20000, 1280, True), (12400, 2048, False),
                                     (12512, 2048, True), (11200, 2304, False)])
def test_short_q4_k_rows_take_the_fma_kernel(api, d, n, k, fma):
    # every size above 16384 super-blocks in rows of up to four, from 100,000 on in rows of five to eight; batches as before
    packed = synth.matrix(Q4_K, n, k, seed=33)
    w = qm(api, d, Q4_K, n, k, packed)
    for m in (1, 2):
        x = synth.activations(m, k, seed=34).reshape(m, k)
        xt = api.Tensor.from_f32(d, (m, k), api.DType.F32, x)
        got = d.project_quantized(xt, w).tensor.to_f32()
        d.set_tuning("gemv_stream", 0)
        try:
            other = d.project_quantized(xt, w).tensor.to_f32()
        finally:
            d.set_tuning("gemv_stream", 1)
        assert np.array_equal(bits(got), bits(other)) == (fma and m == 1)
        rows = np.unique(np.concatenate([np.arange(20), np.arange(n - 20, n)]))
        assert_matmul_parity(got[:, rows], oracle_columns(Q4_K, packed, n, k, rows, x, accumulate="f64"), f"{n}x{k} m={m}")


def test_large_q6_k_output_matrix_streams_in_uncut_sixteen_row_tiles(api, d):
    # a million super-blocks in rows the FMA kernel cannot cut evenly over its block slots (20 per row):
    # sixteen rows of 5120 Q6_K weights are a 67 KB tile
    n, k = 52000, 5120
    base = synth.matrix(Q6_K, 2000, k, seed=97).reshape(2000, -1)
    packed = np.tile(base, (n // 2000, 1)).reshape(-1)
    w = qm(api, d, Q6_K, n, k, packed)
    for dtype, code in (("F32", oracle.F32), ("F16", oracle.F16)):
        x = oracle.round_storage(synth.activations(1, k, seed=98), code).reshape(1, k)
        xt = api.Tensor.from_f32(d, (1, k), getattr(api.DType, dtype), x)
        out = d.project_quantized(xt, w, out_dtype=api.DType.F32)
        assert out.operation == "q6_k_gemv_factored"
        got = out.tensor.to_f32()
        rows = np.unique(np.concatenate([np.arange(0, 40), np.arange(n - 40, n), synth.rng(99).integers(0, n, 120)]))
        want = oracle_columns(Q6_K, packed, n, k, rows, x, accumulate="f64")
        assert_matmul_parity(got[:, rows], want, f"streamed q6_k {n}x{k} {dtype}")
        with fma_gemv(d):
            other = d.project_quantized(xt, w, out_dtype=api.DType.F32).tensor.to_f32()
        # another kernel, another order of summation: equal to the tolerance and not to the bit
        assert rel_l2(got, other) <= 1e-5 and not np.array_equal(bits(got), bits(other))
        assert np.array_equal(bits(got[0, :2000]), bits(got[0, 2000:4000]))   # the rows repeat


@pytest.mark.parametrize("n,k,dtype", [(37, 512, "F32"), (16, 1024, "F16"), (133, 5120, "F32"), (65, 5632, "BF16"),
                                       (50, 12800, "F16"), (40, 17408, "F32")])
def test_streamed_q6_k_sums_digits_of_the_activations_exactly(api, d, n, k, dtype):
    # An activation is 30 bits of its 16-weight group's largest, its products with the quants are summed as integers;
    # what rounds is two conversions and the scales per group, up to six super-blocks of a lane, the waves and the
    # segments: some 30 roundings of at most 2^-24, uniform, 2^-24 / sqrt(3) * sqrt(30) = 1.9e-7 in the mean square.
    packed = synth.matrix(Q6_K, n, k, seed=93)
    w = qm(api, d, Q6_K, n, k, packed)
    weights = oracle.dequantize(Q6_K, packed, n, k).reshape(n, k).astype(np.float64)
    x = synth.activations(1, k, seed=94).reshape(1, k)
    x[0, ::7] *= np.float32(2.0 ** -9)     # within a group, too
    x[0, 16:32] = 0
    x[0, 32:48] = np.float32(-1.0)         # every digit of a power of two
    x[0, 48:64] = np.float32(1.9999999)    # the largest mantissa carries through all digits
    xt = api.Tensor.from_f32(d, (1, k), getattr(api.DType, dtype), x)
    want = xt.to_f32().astype(np.float64) @ weights.T
    d.set_tuning("gemv_stream", 2)
    try:
        got = d.project_quantized(xt, w, out_dtype=api.DType.F32)
        assert rel_l2(got.tensor.to_f32(), want) <= 3e-7
        for value in (np.inf, -np.inf, np.nan):     # none of the row's sums is finite, as on the FMA kernel
            x[0, k - 5] = value
            xt = api.Tensor.from_f32(d, (1, k), getattr(api.DType, dtype), x)
            assert np.isnan(d.project_quantized(xt, w, out_dtype=api.DType.F32).tensor.to_f32()).all()
    finally:
        d.set_tuning("gemv_stream", 1)


@pytest.mark.parametrize("rows", ["normal", "gated", "outliers", "spread"])
@pytest.mark.parametrize("n,k", [(1000, 5120), (700, 17408)])
def test_streamed_q6_k_rows_are_no_farther_from_64_bits_than_on_the_fma_kernel(api, d, n, k, rows):
    # also where a group's largest activation leaves the others few of its 30 bits: a channel in 250 a thousand times the
    # others, magnitudes spread over 2^20
    packed = synth.matrix(Q6_K, n, k, seed=95)
    w = qm(api, d, Q6_K, n, k, packed)
    g = synth.rng(96)
    x = g.standard_normal((1, k))
    if rows == "gated":
        x = 3 * x / (1 + np.exp(-3 * x)) * g.standard_normal((1, k))
    elif rows == "outliers":
        x = x * np.where(g.random((1, k)) < 0.004, 1000.0, 1.0)
    elif rows == "spread":
        x = x * 2.0 ** g.uniform(-20, 0, (1, k))
    x = x.astype(np.float32)
    xt = api.Tensor.from_f32(d, (1, k), api.DType.F32, x)
    d.set_tuning("gemv_stream", 2)
    try:
        got = d.project_quantized(xt, w).tensor.to_f32()
    finally:
        d.set_tuning("gemv_stream", 1)
    with fma_gemv(d):
        other = d.project_quantized(xt, w).tensor.to_f32()
    assert not np.array_equal(bits(got), bits(other))
    want = x.astype(np.float64) @ oracle.dequantize(Q6_K, packed, n, k).reshape(n, k).astype(np.float64).T
    assert rel_l2(got, want) <= rel_l2(other, want)


def test_only_f32_rows_stream_q6_k_matrices_below_a_million_super_blocks(api, d):
    n, k = 32000, 5120     # 640,000 super-blocks, sixteen-row tiles
    base = synth.matrix(Q6_K, 2000, k, seed=35).reshape(2000, -1)
    w = qm(api, d, Q6_K, n, k, np.tile(base, (n // 2000, 1)).reshape(-1))
    for dtype, streamed in (("F32", True), ("F16", False), ("BF16", False)):
        xt = api.Tensor.from_f32(d, (1, k), getattr(api.DType, dtype), synth.activations(1, k, seed=36))
        got = d.project_quantized(xt, w, out_dtype=api.DType.F32).tensor.to_f32()
        with fma_gemv(d):
            other = d.project_quantized(xt, w, out_dtype=api.DType.F32).tensor.to_f32()
        assert np.array_equal(bits(got), bits(other)) == (not streamed)
        assert rel_l2(got, other) <= 7e-7


@pytest.mark.parametrize("m", [2, 3])
def test_two_or_three_f32_rows_of_such_a_matrix_stay_on_the_fma_kernel(api, d, m):
    n, k = 32000, 5120
    base = synth.matrix(Q6_K, 2000, k, seed=35).reshape(2000, -1)
    w = qm(api, d, Q6_K, n, k, np.tile(base, (n // 2000, 1)).reshape(-1))
    xt = api.Tensor.from_f32(d, (m, k), api.DType.F32, synth.activations(m, k, seed=37))
    got = d.project_quantized(xt, w).tensor.to_f32()
    with fma_gemv(d):
        assert np.array_equal(bits(got), bits(d.project_quantized(xt, w).tensor.to_f32()))
    want = xt.to_f32().reshape(m, k).astype(np.float64) @ oracle.dequantize(Q6_K, base.reshape(-1), 2000, k).reshape(2000, k).astype(np.float64).T
    assert rel_l2(got[:, :2000], want) <= 4e-7


def test_one_activated_f32_row_of_a_large_q6_k_matrix_takes_the_streamed_kernel(api, d):
    # 3000 x 17408: 204,000 super-blocks; the bits of the separate calls, and the tolerance of the test above
    n, k = 3000, 17408
    base = synth.matrix(Q6_K, 300, k, seed=95).reshape(300, -1)
    w = qm(api, d, Q6_K, n, k, np.tile(base, (n // 300, 1)).reshape(-1))
    packed = api.Tensor.from_f32(d, (1, 2 * k), api.DType.F32, synth.activations(1, 2 * k, seed=96))
    fused = d.project_quantized(packed, w, silu_mul=True)
    activated = d.expert_silu_mul(packed, k)
    assert fused.operation == "q6_k_gemv_ksplit"
    assert np.array_equal(bits(fused.tensor.to_f32()), bits(d.project_quantized(activated, w).tensor.to_f32()))
    with fma_gemv(d):
        other = d.project_quantized(packed, w, silu_mul=True).tensor.to_f32()
    weights = oracle.dequantize(Q6_K, base.reshape(-1), 300, k).reshape(300, k).astype(np.float64)
    want = np.tile(activated.to_f32().astype(np.float64) @ weights.T, (1, n // 300))
    assert rel_l2(fused.tensor.to_f32(), want) <= 3e-7
    assert rel_l2(other, want) <= 4e-7 and not np.array_equal(bits(other), bits(fused.tensor.to_f32()))


@pytest.mark.parametrize("ggml", [Q4_K, Q6_K])
def test_streamed_gemv_scales_every_chunk_by_itself(api, d, ggml):
    # activations whose 64-value chunks differ by dozens of orders of magnitude, zero chunks, one
    # value per chunk: the power-of-two scale of a chunk (Q6_K: of a 16-weight group) keeps 22 bits
    # of each
    n, k = 64, 2048
    packed = synth.matrix(ggml, n, k, seed=91)
    w = qm(api, d, ggml, n, k, packed)
    d.set_tuning("gemv_stream", 2)
    x = synth.activations(1, k, seed=92).reshape(k // 64, 64)
    x *= np.float32(10.0) ** np.linspace(-30, 30, k // 64, dtype=np.float32)[:, None]
    x[3] = 0
    x[5, 1:] = 0
    x = x.reshape(1, k)
    got = d.project_quantized(api.Tensor.from_f32(d, (1, k), api.DType.F32, x), w).tensor.to_f32()
    want = oracle.project(ggml, packed, n, k, x, accumulate="f64")
    assert rel_l2(got, want) <= 1e-5
    # each chunk alone: what the huge chunks would hide
    for chunk in (0, 5, 16, 31):
        part = np.zeros_like(x).reshape(k // 64, 64)
        part[chunk] = x.reshape(k // 64, 64)[chunk]
        part = part.reshape(1, k)
        got = d.project_quantized(api.Tensor.from_f32(d, (1, k), api.DType.F32, part), w).tensor.to_f32()
        want = oracle.project(ggml, packed, n, k, part, accumulate="f64")
        assert rel_l2(got, want) <= 1e-5, chunk
    if ggml == Q6_K:
        # sixteen-value groups of one chunk that differ as much: each has a scale of its own
        part = np.zeros((k // 16, 16), np.float32)
        part[8:12] = synth.activations(1, 64, seed=93).reshape(4, 16) * np.float32(10.0) ** np.array([-20, 0, 11, 25], np.float32)[:, None]
        part = part.reshape(1, k)
        got = d.project_quantized(api.Tensor.from_f32(d, (1, k), api.DType.F32, part), w).tensor.to_f32()
        for group in range(8, 12):
            alone = np.zeros((k // 16, 16), np.float32)
            alone[group] = part.reshape(k // 16, 16)[group]
            one = d.project_quantized(api.Tensor.from_f32(d, (1, k), api.DType.F32, alone.reshape(1, k)), w).tensor.to_f32()
            assert rel_l2(one, oracle.project(ggml, packed, n, k, alone.reshape(1, k), accumulate="f64")) <= 1e-5, group
        assert rel_l2(got, oracle.project(ggml, packed, n, k, part, accumulate="f64")) <= 1e-5
    # non-finite activations reach the rows they touch
    bad = x.copy()
    bad[0, 7] = np.inf
    got = d.project_quantized(api.Tensor.from_f32(d, (1, k), api.DType.F32, bad), w).tensor.to_f32()
    assert not np.isfinite(got).any()
    d.set_tuning("gemv_stream", 1)


def test_config0_q4_k_gemv_4096(api, d):
    check_gemv(api, d, Q4_K, 4096, 4096, seed=1)


@pytest.mark.parametrize("n,k", [(5120, 5120), (17408, 5120), (5120, 17408)])
def test_config1_q4_k_decode_shapes(api, d, n, k):
    check_gemv(api, d, Q4_K, n, k, seed=2)


@pytest.mark.parametrize("n,k", [(5120, 17408), (151936, 5120)])
def test_config2_q6_k_gemv(api, d, n, k):
    check_gemv(api, d, Q6_K, n, k, seed=3)


@pytest.mark.parametrize("m", [8, 16, 128, 512])
def test_config3_q4_k_gemm_5120_17408(api, d, m):
    n, k = 17408, 5120
    packed = synth.matrix(Q4_K, n, k, seed=4)
    x = synth.activations(m, k, seed=4, f16=True)
    w = qm(api, d, Q4_K, n, k, packed)
    xt = api.Tensor.from_f32(d, (m, k), api.DType.F16, x)
    full = d.project_quantized(xt, w, out_dtype=api.DType.F32)
    got = full.tensor.to_f32()
    rows = np.sort(synth.rng(4, 77).choice(n, size=192, replace=False))
    rows[:4] = [0, 1, 2, 3]
    rows[-2:] = [n - 2, n - 1]
    rows = np.unique(rows)
    tile = oracle_columns(Q4_K, packed, n, k, rows, x, accumulate="f64", weight_round=oracle.F16,
                          threads=8)
    assert_matmul_parity(got[:, rows], tile, f"gemm M={m} vs f16-tile oracle")
    plain = oracle_columns(Q4_K, packed, n, k, rows, x, accumulate="f64", threads=8)
    # distance to the unrounded CPU reference: only the f16 tile rounding
    assert rel_l2(got[:, rows], plain) <= 4e-4
    # linearity in M: row i of the product depends only on row i of X.  The 256-row tile has two
    # forms that sum in different orders and are chosen by shape, so each is held fixed in turn.
    if m >= 16:
        xt2 = api.Tensor.from_f32(d, (m // 2, k), api.DType.F16, x[: m // 2])
        before = d.get_tuning("gemm_wide_shape")
        try:
            for shape in (0, 2):
                d.set_tuning("gemm_wide_shape", shape)
                whole = d.project_quantized(xt, w, out_dtype=api.DType.F32)
                half = d.project_quantized(xt2, w, out_dtype=api.DType.F32)
                if half.operation == whole.operation:
                    assert np.array_equal(half.tensor.to_f32(), whole.tensor.to_f32()[: m // 2])
                else:  # another kernel, another summation order
                    assert_matmul_parity(half.tensor.to_f32(), got[: m // 2], f"gemm M={m // 2} vs M={m}")
                assert_matmul_parity(whole.tensor.to_f32()[:, rows], tile, f"gemm M={m}, tile form {shape}")
        finally:
            d.set_tuning("gemm_wide_shape", before)


@pytest.mark.parametrize("m", [8, 512])
def test_config3_every_column_against_a_closed_form(api, d, m):
    # All 17408 columns, which a sample of columns cannot vouch for: row n keeps one super-block,
    # number n % 20, and zero blocks (d = dmin = 0) elsewhere, so y[:, n] is a 256-term product the
    # host evaluates for every column.
    n, k = 17408, 5120
    nb = k // 256
    blocks = synth.matrix(Q4_K, n, 256, seed=401).reshape(n, 144)
    packed = np.zeros((n, nb, 144), np.uint8)
    keep = np.arange(n) % nb
    packed[np.arange(n), keep] = blocks
    x = synth.activations(m, k, seed=402, f16=True)
    w = qm(api, d, Q4_K, n, k, packed.reshape(-1))
    out = d.project_quantized(api.Tensor.from_f32(d, (m, k), api.DType.F16, x), w, out_dtype=api.DType.F32)
    got = out.tensor.to_f32()
    dense = oracle.round_storage(oracle.dequantize(Q4_K, blocks.reshape(-1), n, 256), oracle.F16).astype(np.float64)
    want = np.empty((m, n), np.float64)
    for b in range(nb):
        rows = np.nonzero(keep == b)[0]
        want[:, rows] = x[:, 256 * b:256 * (b + 1)].astype(np.float64) @ dense[rows].T
    assert_matmul_parity(got, want, f"every column at M={m} ({out.operation})")
    worst = np.abs(got - want).max(axis=0)
    assert worst.max() <= 1e-3 * np.abs(want).max(), int(worst.argmax())


# ------------------------------------------------------------ error behaviour

def test_project_rejects_bad_geometry_and_foreign_buffers(api, d):
    packed = fx.q4k_packed(5, 512)
    w = qm(api, d, Q4_K, 5, 512, packed)
    with pytest.raises(api.ShapeError):
        d.project_quantized(api.Tensor.zeros(d, (1, 256), api.DType.F32), w)
    with pytest.raises(api.ShapeError):
        d.project_quantized(api.Tensor.zeros(d, (512,), api.DType.F32), w)
    other = api.Device.new()
    foreign = api.Tensor.zeros(other, (1, 512), api.DType.F32)
    with pytest.raises(api.DeviceMismatch):
        d.project_quantized(foreign, w)
    x = api.Tensor.zeros(d, (2, 512), api.DType.F32)
    with pytest.raises(api.RangeError):
        d.project_quantized(x.view(0, (1, 512)), w, out=x.view(0, (1, 5)))     # aliasing
    with pytest.raises(api.RangeError):
        d.project_quantized(x.view(1, (1, 512)), w)                            # misaligned view


def test_quantized_matrix_validation(api, d):
    # src/quantization.rs:93-103, :212-261 and qk_tests "reject partial blocks"
    fmt = api.QuantizationFormat.Q4_K
    with pytest.raises(api.ShapeError):
        api.QuantizedMatrix.from_reader(d, 3, 255, fmt, lambda dst: None)
    with pytest.raises(api.ShapeError):
        api.QuantizedMatrix.from_reader(d, 0, 256, fmt, lambda dst: None)
    good = fx.q4k_packed(2, 256)
    with pytest.raises(api.GgufError):
        api.QuantizedMatrix.from_bytes(d, 2, 256, fmt, good[:-1])
    with pytest.raises(api.ShapeError):
        api.QuantizedMatrix.from_bytes(d, 3, 256, fmt, good)
    bad = good.copy()
    bad[146:148] = np.frombuffer(np.float16(np.nan).tobytes(), np.uint8)
    with pytest.raises(api.WeightError):
        api.QuantizedMatrix.from_bytes(d, 2, 256, fmt, bad)
    bad6 = fx.q6k_packed(2, 256)
    bad6[208:210] = np.frombuffer(np.float16(np.inf).tobytes(), np.uint8)
    with pytest.raises(api.WeightError):
        api.QuantizedMatrix.from_bytes(d, 2, 256, api.QuantizationFormat.Q6_K, bad6)
    with pytest.raises(api.GgufError):
        api.QuantizationFormat.from_ggml_type(5)
    assert api.QuantizationFormat.from_ggml_type(12).block_bytes() == 144
    assert api.QuantizationFormat.from_ggml_type(14).block_bytes() == 210


# ------------------------------------------------------------ executions

def test_recorded_execution_replays_bitwise_with_eager_work_in_between(api, d):
    # Execution (src/metal/mod.rs:263-278): calls recorded once, replayed many times
    n, k = 1024, 2048
    w = qm(api, d, Q4_K, n, k, synth.matrix(Q4_K, n, k, seed=101))
    x = api.Tensor.from_f32(d, (1, k), api.DType.F32, synth.activations(1, k, seed=102))
    x8 = api.Tensor.from_f32(d, (8, k), api.DType.F16, synth.activations(8, k, seed=103, f16=True))
    y, y8 = api.Tensor.zeros(d, (1, n), api.DType.F32), api.Tensor.zeros(d, (8, n), api.DType.F32)
    eager = d.project_quantized(x, w).tensor.raw()
    eager8 = d.project_quantized(x8, w, out_dtype=api.DType.F32).tensor.raw()
    with d.execution() as ex:
        d.project_quantized(x, w, out=y)
        d.project_quantized(x8, w, out=y8)
        with pytest.raises(api.Error):
            api.Tensor.zeros(d, (4,), api.DType.F32)          # allocation is refused while recording
        with pytest.raises(api.Error):
            y.to_f32()                                         # so is a download
    for _ in range(3):
        ex.graph.launch()
        assert np.array_equal(y.raw(), eager) and np.array_equal(y8.raw(), eager8)
        y.buffer.upload(0, np.zeros(n, np.float32))            # eager work between the replays
        d.project_quantized(x8, w)
        d.synchronize()


def test_a_recorded_execution_survives_the_growth_of_the_scratch(api, d):
    # a recorded long-K GEMV carries the address of the device scratch (partial sums, counters);
    # an eager call that outgrows the scratch afterwards must not take that memory away
    n, k = 2048, 17408
    w = qm(api, d, Q4_K, n, k, synth.matrix(Q4_K, n, k, seed=121))
    x = api.Tensor.from_f32(d, (1, k), api.DType.F32, synth.activations(1, k, seed=122))
    y = api.Tensor.zeros(d, (1, n), api.DType.F32)
    eager = d.project_quantized(x, w)
    assert eager.operation == "q4_k_gemv_ksplit"
    with d.execution() as ex:
        d.project_quantized(x, w, out=y)
    ex.graph.launch()
    assert np.array_equal(y.raw(), eager.tensor.raw())
    # 3000 x 5120 f32 rows rounded to f16 in the scratch: 30 MB, beyond the 16 MB it starts with
    kb, nbig, mb = 5120, 256, 3000
    wb = qm(api, d, Q4_K, nbig, kb, synth.matrix(Q4_K, nbig, kb, seed=123))
    xb = api.Tensor.from_f32(d, (mb, kb), api.DType.F32, synth.activations(mb, kb, seed=124))
    d.set_tuning("gemm_f32_min_rows", 2)
    try:
        big = d.project_quantized(xb, wb)
    finally:
        d.set_tuning("gemm_f32_min_rows", 0)
    assert "mfma" in big.operation
    for _ in range(2):
        y.buffer.upload(0, np.zeros(n, np.float32))
        ex.graph.launch()
        assert np.array_equal(y.raw(), eager.tensor.raw())
        d.project_quantized(x, w)          # eager work on the new scratch in between
        d.synchronize()


def test_f32_batches_of_any_size_run_through_the_long_k_gemv(api, d):
    # q4_k_gemm accepts any M (src/metal/shaders/ops.metal:1102-1121): on the GEMV, which has these batches where
    # the few-rows kernel is switched off, a long-K projection of 110 f32 rows needs more row-tile counters
    # than one launch has, so the batch is cut into runs
    n, k, m = 5120, 17408, 110
    packed = synth.matrix(Q4_K, n, k, seed=131)
    w = qm(api, d, Q4_K, n, k, packed)
    x = synth.activations(m, k, seed=132)
    with few_rows(d, 0):
        out = d.project_quantized(api.Tensor.from_f32(d, (m, k), api.DType.F32, x), w)
        assert out.operation == "q4_k_gemm" and d.get_tuning("last_rows_plan") == 0
        got = out.tensor.to_f32()
        first = d.project_quantized(api.Tensor.from_f32(d, (60, k), api.DType.F32, x[:60]), w).tensor.to_f32()
        last = d.project_quantized(api.Tensor.from_f32(d, (50, k), api.DType.F32, x[60:]), w).tensor.to_f32()
    assert np.array_equal(bits(got[:60]), bits(first)) and np.array_equal(bits(got[60:]), bits(last))
    rows = np.unique(synth.rng(133).integers(0, n, 48))
    picked = [0, 59, 60, 101, 102, 103, 109]
    want = oracle_columns(Q4_K, packed, n, k, rows, x[picked], accumulate="f64")
    assert_matmul_parity(got[picked][:, rows], want, "f32 batch through the K-split GEMV")


def test_wide_gemm_covers_every_column_of_its_tiles(api, d):
    # 300 rows x 36864 columns: the 256-row tile kernel with 136 columns per workgroup; the last
    # columns of a workgroup's tile (the ninth MFMA column tile) are the ones checked
    n, k, m = 36864, 512, 300
    packed = synth.matrix(Q4_K, n, k, seed=141)
    w = qm(api, d, Q4_K, n, k, packed)
    x = synth.activations(m, k, seed=142, f16=True)
    d.set_tuning("gemm_wide_shape", 0)     # the 16x16x32 form, whose tiles have the ninth column tile
    try:
        out = d.project_quantized(api.Tensor.from_f32(d, (m, k), api.DType.F16, x), w, out_dtype=api.DType.F32)
    finally:
        d.set_tuning("gemm_wide_shape", 1)
    assert out.operation == "q4_k_gemm_mfma_m256"
    got = out.tensor.to_f32()
    for width in (128, 136, 144):      # whichever width the plan chose, its tiles' last 16 columns
        rows = np.concatenate([np.arange(t * width + width - 16, t * width + width) for t in (0, 1, 100, n // width - 1)])
        rows = rows[rows < n]
        want = oracle_columns(Q4_K, packed, n, k, rows, x, accumulate="f64", weight_round=oracle.F16)
        assert_matmul_parity(got[:, rows], want, f"columns at the end of {width}-wide tiles")
    rows = np.arange(n - 40, n)
    want = oracle_columns(Q4_K, packed, n, k, rows, x, accumulate="f64", weight_round=oracle.F16)
    assert_matmul_parity(got[:, rows], want, "last columns")


@pytest.mark.parametrize("ggml", [12, 13, 14, 23, 8], ids=["q4_k", "q5_k", "q6_k", "iq4_xs", "q8_0"])
@pytest.mark.parametrize("dtype", ["F16", "BF16"])
def test_wide_gemm_on_the_32x32x16_instruction(api, d, ggml, dtype):
    # the tiles built on v_mfma_f32_32x32x16, each forced in turn: 256 rows x 160 / 128 columns and
    # 128 rows x 160 / 128 / 64 columns.  300 rows leave the last row tile 44 rows, 8072 columns
    # leave the last workgroup 72, 8 or 8 of its columns.  Every output of the first is checked
    # against the oracle; the others add the same products in the same order, so they must give
    # its bits, and so must whichever tile the library picks by itself.
    n, k, m = 8072, 512, 300
    packed = synth.matrix(ggml, n, k, seed=171)
    w = qm(api, d, ggml, n, k, packed)
    code = oracle.F16 if dtype == "F16" else oracle.BF16
    x = oracle.round_storage(synth.activations(m, k, seed=172), code).reshape(m, k)
    xt = api.Tensor.from_f32(d, (m, k), getattr(api.DType, dtype), x)
    shape, tile = d.get_tuning("gemm_wide_shape"), d.get_tuning("gemm_wide32_tile")
    results = {}
    try:
        d.set_tuning("gemm_wide_shape", 2)
        for forced in (25, 24, 15, 14, 12, 0):
            d.set_tuning("gemm_wide32_tile", forced)
            out = d.project_quantized(xt, w, out_dtype=api.DType.F32)
            assert out.operation.endswith("_gemm_mfma_m256")
            results[forced] = out.tensor.to_f32()
        d.set_tuning("gemm_wide_shape", 0)
        other = d.project_quantized(xt, w, out_dtype=api.DType.F32)
        assert other.operation.endswith("_gemm_mfma_m256")
    finally:
        d.set_tuning("gemm_wide_shape", shape)
        d.set_tuning("gemm_wide32_tile", tile)
    want = oracle.project(ggml, packed, n, k, x, accumulate="f64", weight_round=code, threads=8)
    assert_matmul_parity(results[25], want, "every output of the 256 x 160 tiles")
    for forced, got in results.items():
        assert np.array_equal(bits(got), bits(results[25])), f"tile {forced} against 256 x 160"
    assert_matmul_parity(results[25], other.tensor.to_f32(), "against the 16x16x32 tiles", l2_tol=2e-6)


@pytest.mark.parametrize("ggml,m,n,k,segments", [
    (12, 33, 4090, 16 * 256, 4), (14, 129, 1003, 17 * 256, 4), (13, 257, 600, 9 * 256, 2), (23, 128, 96, 32 * 256, 8),
    (8, 300, 333, 13 * 256, 3), (12, 511, 1021, 33 * 256, 7)])
@pytest.mark.parametrize("dtype,out", [("F16", "F32"), ("BF16", "BF16")])
def test_tiles_whose_k_is_cut_into_segments(api, d, ggml, m, n, k, segments, dtype, out):
    # every 32x32x16 tile with that many segments (the last one shorter), ragged rows and columns, outputs whose count
    # is no multiple of four; against the tile-rounded oracle, and repeated with the same bits
    packed = synth.matrix(ggml, n, k, seed=177)
    w = qm(api, d, ggml, n, k, packed)
    code = oracle.F16 if dtype == "F16" else oracle.BF16
    x = oracle.round_storage(synth.activations(m, k, seed=178 + m), code).reshape(m, k)
    xt = api.Tensor.from_f32(d, (m, k), getattr(api.DType, dtype), x)
    rows = np.unique(np.concatenate([np.arange(0, 40), np.arange(n // 2, n // 2 + 30), np.arange(n - 40, n)]))
    want = oracle_columns(ggml, packed, n, k, rows, x, weight_round=code, accumulate="f64")
    try:
        d.set_tuning("gemm_wide32_segments", segments)
        for tile in (12, 13, 14, 15, 24, 25):
            d.set_tuning("gemm_wide32_tile", tile)
            got = d.project_quantized(xt, w, out_dtype=api.DType.F32)
            assert got.operation.endswith("_gemm_mfma_m256")
            assert_matmul_parity(got.tensor.to_f32()[:, rows], want, f"tile {tile}")
            again = d.project_quantized(xt, w, out_dtype=getattr(api.DType, out)).tensor.to_f32()
            stored = got.tensor.to_f32() if out == "F32" else oracle.round_storage(got.tensor.to_f32(), code).reshape(m, n)
            assert np.array_equal(bits(again), bits(stored))
    finally:
        d.set_tuning("gemm_wide32_segments", 0)
        d.set_tuning("gemm_wide32_tile", 0)


@pytest.mark.parametrize("m,n,blocks,segments,last", [(40, 131, 21, 5, 17), (65, 70, 36, 8, 32), (129, 96, 32, 7, 28), (33, 64, 17, 4, 13)])
def test_segments_of_tiles_differ_by_one_super_block_at_most(api, d, m, n, blocks, segments, last):
    # 21 super-blocks in five segments are 5 4 4 4 4 and not 5 5 5 5 1.  Where the last segment begins shows in what
    # cancels: big values of opposite sign in the super-blocks before and at its first one meet after the segments' own sums,
    # so a small value behind the second of them is lost there, and kept if both lie in one segment.
    k = blocks * 256
    packed = synth.matrix(Q4_K, n, k, seed=183)
    w = qm(api, d, Q4_K, n, k, packed)
    x = oracle.round_storage(synth.activations(m, k, seed=184), oracle.F16).reshape(m, k)
    weights = oracle.round_storage(oracle.dequantize(Q4_K, packed, n, k), oracle.F16).reshape(n, k)
    split = np.zeros((m, k), dtype=np.float32)
    split[0, (last + 1) * 256 - 1] = 2.0 ** -14
    kept = split[0] @ weights.T
    at = (last - 1) * 256 + 255, last * 256      # neighbours on either side of the boundary
    split[0, at[0]], split[0, at[1]] = -16384.0, 16384.0
    try:
        d.set_tuning("gemm_wide32_segments", segments)
        for tile in (12, 15, 24):
            d.set_tuning("gemm_wide32_tile", tile)
            got = d.project_quantized(api.Tensor.from_f32(d, (m, k), api.DType.F16, x), w, out_dtype=api.DType.F32).tensor.to_f32()
            assert_matmul_parity(got, x.astype(np.float64) @ weights.T.astype(np.float64), f"tile {tile}")
            got = d.project_quantized(api.Tensor.from_f32(d, (m, k), api.DType.F16, split), w, out_dtype=api.DType.F32).tensor.to_f32()
            # plane `segments - 1` is fl(16384 w + small), the one before it -16384 w' exactly
            want = (np.float32(-16384.0) * weights[:, at[0]]) + (np.float32(16384.0) * weights[:, at[1]] + kept).astype(np.float32)
            assert np.array_equal(got[0], want.astype(np.float32)), tile
    finally:
        d.set_tuning("gemm_wide32_segments", 0)
        d.set_tuning("gemm_wide32_tile", 0)


def test_partial_sums_of_tiles_take_only_the_room_there_is(api):
    # 512 x 5120 x 17408 in four segments: 42 MB of sums, which the scratch of a new device does not hold.  While it
    # records the device takes another kernel; a plain call grows the scratch, and the recording stays what it was.
    dev = api.Device.new()
    m, n, k = 512, 5120, 17408
    w = qm(api, dev, Q4_K, n, k, synth.matrix(Q4_K, n, k, seed=179))
    x = api.Tensor.from_f32(dev, (m, k), api.DType.F16, synth.activations(m, k, seed=180, f16=True))
    recorded = api.Tensor.zeros(dev, (m, n), api.DType.F32)
    dev.synchronize()
    held = dev.get_tuning("held_scratch_bytes")
    with dev.execution() as ex:
        dev.project_quantized(x, w, out=recorded)
    ex.graph.launch()
    dev.synchronize()
    assert dev.get_tuning("held_scratch_bytes") == held
    first = recorded.to_f32()
    direct = dev.project_quantized(x, w, out_dtype=api.DType.F32).tensor.to_f32()
    assert held < dev.get_tuning("held_scratch_bytes") <= 64 << 20
    assert rel_l2(first, direct) <= 1e-5
    for _ in range(2):
        ex.graph.launch()
        dev.synchronize()
        assert np.array_equal(bits(recorded.to_f32()), bits(first))
    again = api.Tensor.zeros(dev, (m, n), api.DType.F32)
    with dev.execution() as cut:
        dev.project_quantized(x, w, out=again)
    for _ in range(3):
        cut.graph.launch()
        dev.synchronize()
        assert np.array_equal(bits(again.to_f32()), bits(direct))


@pytest.mark.parametrize("live_graph", [False, True])
@pytest.mark.parametrize("ggml,m,n,k,wanted", [(Q4_K, 512, 5120, 17408, 42), (Q6_K, 1500, 8192, 4096, 67)])
def test_products_run_without_the_scratch_they_would_like(api, live_graph, ggml, m, n, k, wanted):
    # planes of partial sums and a panel of decoded weights, on a GPU that has no room for them: a limit on single
    # allocations makes the request a real one that fails.  No error, no block changes hands, and the GPU is not asked again
    # on every call; once there is room, the scratch grows to what is asked for.
    dev = api.Device.new()
    base = synth.matrix(ggml, 64, k, seed=185)
    w = qm(api, dev, ggml, n, k, np.resize(base, base.size // 64 * n))
    x = api.Tensor.from_f32(dev, (m, k), api.DType.F16, synth.activations(m, k, seed=186, f16=True))
    y, held = api.Tensor.zeros(dev, (m, n), api.DType.F32), dev.get_tuning("held_scratch_bytes")
    graph = None
    if live_graph:
        with dev.execution() as ex:
            dev.project_quantized(x, w, out=y)
        graph = ex.graph
    dev.set_tuning("allocation_limit_bytes", 20 << 20)
    dev.project_quantized(x, w, out=y)
    first = y.to_f32()
    for _ in range(3):
        dev.project_quantized(x, w, out=y)
        assert dev.get_tuning("held_scratch_bytes") == held and dev.get_tuning("retired_scratch_blocks") == 0
    assert np.array_equal(bits(y.to_f32()), bits(first))
    dev.set_tuning("allocation_limit_bytes", 0)
    dev.project_quantized(x, w, out=y)
    assert dev.get_tuning("held_scratch_bytes") == held      # one that failed just now is not asked for again
    for _ in range(600):      # ... before 256 calls have done without (a product may try two sizes)
        dev.project_quantized(x, w, out=y)
    dev.synchronize()
    grown = dev.get_tuning("held_scratch_bytes")
    assert wanted * 10 ** 6 <= grown <= (wanted + 1) * 10 ** 6 + (1 << 20)
    assert dev.get_tuning("retired_scratch_blocks") == (1 if live_graph else 0)
    if ggml == Q6_K:      # panels, and in their place the uncut tiles of the 32x32x16 form: the same sums
        assert dev.get_tuning("last_decoded_tile") != 0 and np.array_equal(bits(y.to_f32()), bits(first))
    else:
        assert rel_l2(y.to_f32(), first) <= 1e-5
    dev.set_tuning("held_scratch_bytes", 0)
    assert dev.get_tuning("held_scratch_bytes") == (grown if live_graph else held)
    if live_graph:
        graph.launch()
        dev.synchronize()
        assert np.array_equal(bits(y.to_f32()), bits(first))
        ex.graph = graph = None
        assert dev.get_tuning("retired_scratch_blocks") == 0
        dev.set_tuning("held_scratch_bytes", 0)
        assert dev.get_tuning("held_scratch_bytes") == held
    dev.project_quantized(x, w, out=y)
    assert rel_l2(y.to_f32(), first) <= 1e-5


def test_a_required_scratch_that_cannot_grow_is_an_error_and_nothing_is_lost(api):
    dev = api.Device.new()
    n, k, m = 96, 8192, 3000        # f32 rows rounded into the scratch: 49 MB
    packed = synth.matrix(Q4_K, n, k, seed=187)
    w = qm(api, dev, Q4_K, n, k, packed)
    x = api.Tensor.from_f32(dev, (m, k), api.DType.F32, synth.activations(m, k, seed=188))
    few = api.Tensor.from_f32(dev, (8, k), api.DType.F32, synth.activations(8, k, seed=189))
    dev.set_tuning("gemm_f32_min_rows", 5)
    before = dev.project_quantized(few, w).tensor.to_f32()
    dev.set_tuning("allocation_limit_bytes", 20 << 20)
    for _ in range(2):
        with pytest.raises(Exception, match="hipMalloc"):
            dev.project_quantized(x, w)
        assert np.array_equal(bits(dev.project_quantized(few, w).tensor.to_f32()), bits(before))
    dev.set_tuning("allocation_limit_bytes", 0)
    out = dev.project_quantized(x, w).tensor.to_f32()
    rows = np.arange(n)
    rounded = oracle.round_storage(x.to_f32()[:8], oracle.F16).reshape(8, k)
    assert_matmul_parity(out[:8], oracle_columns(Q4_K, packed, n, k, rows, rounded, weight_round=oracle.F16, accumulate="f64"), "grown")


@pytest.mark.parametrize("m", [80, 128, 200, 330, 512])
def test_the_tile_picked_by_row_count_gives_the_bits_of_the_largest(api, d, m):
    # 17000 columns at every row count that changes the tile (128 x 68 of the 96-column tile up to
    # 128 rows, 128 x 160 up to 256, 128 x 128 up to 384, 256 x 160 beyond); the pick and the forced
    # 128 x 64 and 128 x 96 tiles against the forced 256 x 160 tile.
    n, k = 17000, 2816
    w = qm(api, d, Q4_K, n, k, synth.matrix(Q4_K, n, k, seed=173))
    x = synth.activations(m, k, seed=174, f16=True)
    xt = api.Tensor.from_f32(d, (m, k), api.DType.F16, x)
    tile, resident, shape = d.get_tuning("gemm_wide32_tile"), d.get_tuning("gemm_resident"), d.get_tuning("gemm_wide_shape")
    try:
        d.set_tuning("gemm_resident", 0)      # at 80 rows its estimate is close to the tile's,
        d.set_tuning("gemm_wide_shape", 2)    # at 512 the 16x16x32 form's, whose bits differ
        picked = d.project_quantized(xt, w, out_dtype=api.DType.F32)
        d.set_tuning("gemm_wide32_tile", 25)
        largest = d.project_quantized(xt, w, out_dtype=api.DType.F32)
        for forced in (12, 13):
            d.set_tuning("gemm_wide32_tile", forced)
            assert np.array_equal(d.project_quantized(xt, w, out_dtype=api.DType.F32).tensor.raw(), largest.tensor.raw())
    finally:
        d.set_tuning("gemm_wide32_tile", tile)
        d.set_tuning("gemm_resident", resident)
        d.set_tuning("gemm_wide_shape", shape)
    assert picked.operation == largest.operation == "q4_k_gemm_mfma_m256"
    assert np.array_equal(picked.tensor.raw(), largest.tensor.raw())


@pytest.mark.parametrize("ggml,m,n,k", [(8, 512, 17408, 5120), (8, 400, 34816, 4096)])
def test_the_32x32x16_form_is_taken_where_the_forms_are_close(api, d, ggml, m, n, k):
    base = synth.matrix(ggml, 11, k, seed=191)
    w = qm(api, d, ggml, n, k, np.resize(base, base.size // 11 * n))
    xt = api.Tensor.from_f32(d, (m, k), api.DType.F16, synth.activations(m, k, seed=192, f16=True))
    out, results = api.Tensor.zeros(d, (m, n), api.DType.F32), {}
    try:
        for name, key, value in (("default", "gemm_wide_shape", 1), ("32", "gemm_wide32_tile", 25), ("16", "gemm_wide_shape", 0)):
            d.set_tuning(key, value)
            d.project_quantized(xt, w, out=out)
            assert d.get_tuning("last_decoded_tile") == 0
            results[name] = out.raw()
            d.set_tuning("gemm_wide_shape", 1)
            d.set_tuning("gemm_wide32_tile", 0)
    finally:
        d.set_tuning("gemm_wide_shape", 1)
        d.set_tuning("gemm_wide32_tile", 0)
    assert np.array_equal(results["default"], results["32"]) and not np.array_equal(results["default"], results["16"])


@pytest.mark.parametrize("n,k", [(5120, 17408), (17000, 2816), (2560, 8192)])
def test_rows_of_the_default_kernels_agree_at_every_row_count(api, d, n, k):
    # Which kernel, tile and K segments take a product follows from its row count, and with them the order of a row's sums, not
    # its bits.  An instruction brings at least the eight products of a lane group into an f32 accumulator, so at most k / 8
    # sums follow each other there, each off by 2^-24 at most, uniform: 2^-24 / sqrt(3) * sqrt(k / 16) in the mean square
    # from 64 bits on the rounded weights, on either side of a comparison.
    w = qm(api, d, Q4_K, n, k, synth.matrix(Q4_K, n, k, seed=175))
    x = synth.activations(512, k, seed=176, f16=True).reshape(512, k)
    bound = 2.0 ** -24 / np.sqrt(3) * np.sqrt(k / 16)
    cols = np.unique(np.concatenate([np.arange(0, 60), np.arange(n - 60, n)]))
    want = oracle_columns(Q4_K, synth.matrix(Q4_K, n, k, seed=175), n, k, cols, x[:33], weight_round=oracle.F16, accumulate="f64")
    last = None
    for m in (33, 64, 80, 128, 200, 256, 330, 512):
        got = d.project_quantized(api.Tensor.from_f32(d, (m, k), api.DType.F16, x[:m]), w, out_dtype=api.DType.F32).tensor.to_f32()
        assert rel_l2(got[:33][:, cols], want) <= bound, m
        if last is not None:
            assert rel_l2(got[: len(last)], last) <= np.sqrt(2) * bound, m
        last = got


@pytest.mark.parametrize("ggml", [12, 13, 14, 23, 8], ids=["q4_k", "q5_k", "q6_k", "iq4_xs", "q8_0"])
@pytest.mark.parametrize("m,n,k,dtype", [(2, 17000, 5120, "F16"), (9, 4100, 5120, "BF16"), (16, 17000, 4096, "F16"),
                                         (8, 1000, 2048, "F16"), (16, 20000, 768, "BF16")])
def test_few_rows_deal_a_tiles_super_blocks_over_the_waves(api, d, ggml, m, n, k, dtype):
    # up to 16 rows and at most five 16-row weight tiles per compute unit: every wave of the
    # workgroup takes some super-blocks of every tile and the partial sums meet in LDS.  Rows of 1 -
    # 20 super-blocks (8 and 16 waves), one to five tiles per workgroup, a ragged last tile, every
    # format; against the tile-rounded oracle on sampled columns and against the kernel that
    # gives a wave whole tiles (the same products, added in another order).
    packed = synth.matrix(ggml, n, k, seed=181 + m)
    w = qm(api, d, ggml, n, k, packed)
    code = oracle.F16 if dtype == "F16" else oracle.BF16
    x = oracle.round_storage(synth.activations(m, k, seed=182), code).reshape(m, k)
    xt = api.Tensor.from_f32(d, (m, k), getattr(api.DType, dtype), x)
    with few_rows(d, 2):
        out = d.project_quantized(xt, w, out_dtype=api.DType.F32)
    # (both kernels report the name the rows-resident one has always had)
    assert out.operation.endswith("_gemm_mfma_resident") and d.get_tuning("last_rows_plan") // 1000 == 16
    with few_rows(d, 0):
        whole = d.project_quantized(xt, w, out_dtype=api.DType.F32)
    assert whole.operation == out.operation and d.get_tuning("last_rows_plan") == 0
    got = out.tensor.to_f32()
    rows = np.unique(np.concatenate([np.arange(0, 40), np.arange(n - 40, n), synth.rng(183).integers(0, n, 80)]))
    want = oracle_columns(ggml, packed, n, k, rows, x, weight_round=code, accumulate="f64")
    assert_matmul_parity(got[:, rows], want, "dealt super-blocks against the tile-rounded oracle")
    assert_matmul_parity(got, whole.tensor.to_f32(), "against whole tiles per wave", l2_tol=2e-6)
    assert not np.array_equal(got, np.zeros_like(got))
    with few_rows(d, 2):
        half = d.project_quantized(xt, w, out_dtype=getattr(api.DType, dtype))      # 16-bit output: the scalar stores
    assert np.array_equal(half.tensor.to_f32(), oracle.round_storage(got, code).reshape(m, n))


# Edges of the few-rows kernel: rows of 1, 2, 4, 9 and 17 super-blocks (1, 2, 4 or 8 waves along K, a
# wave without a block, an odd block out), rows whose K is cut into segments, ragged last tiles and row
# groups of 16 and 32, exact f32 rows.  16-bit rows against the tile-rounded oracle, f32 rows against
# the exact one, both at the matmul bar; the same bits on a second call (the sums have one order).
@pytest.mark.parametrize("ggml", [12, 13, 14, 23, 8], ids=["q4_k", "q5_k", "q6_k", "iq4_xs", "q8_0"])
@pytest.mark.parametrize("m,n,k,dtype", [
    (2, 70, 256, "F16"), (17, 100, 512, "BF16"), (32, 301, 1024, "F16"), (5, 1003, 2304, "BF16"), (33, 533, 4352, "F16"),
    (64, 48, 2048, "BF16"), (16, 1030, 17408, "F16"), (100, 96, 17408, "BF16"), (3, 20, 9216, "F16"),
    (6, 61, 256, "F32"), (17, 333, 1280, "F32"), (40, 19, 4352, "F32"), (7, 1030, 17408, "F32")])
def test_few_rows_on_the_edges_of_the_kernel(api, d, ggml, m, n, k, dtype):
    packed = synth.matrix(ggml, n, k, seed=251 + n)
    w = qm(api, d, ggml, n, k, packed)
    code = {"F32": oracle.F32, "F16": oracle.F16, "BF16": oracle.BF16}[dtype]
    x = oracle.round_storage(synth.activations(m, k, seed=252 + m), code).reshape(m, k)
    xt = api.Tensor.from_f32(d, (m, k), getattr(api.DType, dtype), x)
    with few_rows(d, 2):
        out = d.project_quantized(xt, w, out_dtype=api.DType.F32)
        assert out.operation.endswith("_gemm" if dtype == "F32" else "_skinny" if k > 5120 and m <= 64 else "_resident")
        assert d.get_tuning("last_rows_plan") // 1000 == (32 if dtype != "F32" and m > 16 else 16)
        got = out.tensor.to_f32()
        want = oracle.project(ggml, packed, n, k, x, accumulate="f64", weight_round=code, threads=8)
        assert_matmul_parity(got, want, f"few rows {m}x{n}x{k} {dtype}")
        again = d.project_quantized(xt, w, out_dtype=api.DType.F32).tensor.to_f32()
        assert np.array_equal(bits(again), bits(got))
        if dtype == "F32" and m > 5:    # a row's sums do not depend on the rows beside it
            part = d.project_quantized(api.Tensor.from_f32(d, (m - 1, k), api.DType.F32, x[:-1]), w).tensor.to_f32()
            assert np.array_equal(bits(part), bits(got[:-1]))
        stored = d.project_quantized(xt, w).tensor.to_f32()      # 16-bit results: the packed stores
        assert np.array_equal(bits(stored), bits(oracle.round_storage(got, code).reshape(m, n)))


@functools.lru_cache(maxsize=1)
def _sixteen_thousand_rows(ggml, k):
    return synth.matrix(ggml, 16750, k, seed=291)


# Two to five weight tiles per wave (n picks them: one round of the chip), the ragged last tile and the packed and
# element stores, in the 32-row, 16-row and f32 forms of every format; and four tiles with K cut in three.
@pytest.mark.parametrize("ggml", [12, 13, 14, 23, 8], ids=["q4_k", "q5_k", "q6_k", "iq4_xs", "q8_0"])
@pytest.mark.parametrize("tiles,n", [(2, 4150), (3, 8200), (4, 12700), (5, 16750)])
def test_few_rows_with_several_tiles_per_wave(api, d, ggml, tiles, n):
    k = 2048
    packed = _sixteen_thousand_rows(ggml, k).reshape(16750, -1)[:n].reshape(-1)
    w = qm(api, d, ggml, n, k, packed)
    rows = np.unique(np.concatenate([np.arange(0, 24), np.arange(n - 40, n), synth.rng(292).integers(0, n, 40)]))
    for m, dtype in ((9, "F32"), (13, "F16"), (20, "F16"), (33, "BF16")):
        code = {"F32": oracle.F32, "F16": oracle.F16, "BF16": oracle.BF16}[dtype]
        x = oracle.round_storage(synth.activations(m, k, seed=293 + m), code).reshape(m, k)
        with few_rows(d, 2):
            got = d.project_quantized(api.Tensor.from_f32(d, x.shape, getattr(api.DType, dtype), x), w,
                                      out_dtype=api.DType.F32).tensor.to_f32()
        assert d.get_tuning("last_rows_plan") == (32000 if m > 16 else 16000) + 100 * tiles + 1
        want = oracle_columns(ggml, packed, n, k, rows, x, accumulate="f64", weight_round=code)
        assert_matmul_parity(got[:, rows], want, f"{tiles} tiles, {m} {dtype} rows")


@pytest.mark.parametrize("ggml", [12, 13, 14, 23, 8], ids=["q4_k", "q5_k", "q6_k", "iq4_xs", "q8_0"])
def test_few_rows_with_four_tiles_and_three_segments(api, d, ggml):
    n, k = 5120, 17408
    tile = synth.matrix(ggml, 80, k, seed=295)      # five tiles, over and over: a wave's four are different
    w = qm(api, d, ggml, n, k, np.tile(tile, n // 80))
    for m, dtype in ((7, "F32"), (19, "F16")):
        code = oracle.F32 if dtype == "F32" else oracle.F16
        x = oracle.round_storage(synth.activations(m, k, seed=296 + m), code).reshape(m, k)
        with few_rows(d, 2):
            got = d.project_quantized(api.Tensor.from_f32(d, x.shape, getattr(api.DType, dtype), x), w,
                                      out_dtype=api.DType.F32).tensor.to_f32()
        plan = d.get_tuning("last_rows_plan")
        assert plan == (32403 if dtype == "F16" else 16403), plan
        want = oracle.project(ggml, tile, 80, k, x, accumulate="f64", weight_round=code, threads=8)
        assert_matmul_parity(got[:, :80], want, f"{m} {dtype} rows")
        assert np.array_equal(bits(got), bits(np.tile(got[:, :80], n // 80)))


# A row's sums do not depend on how many rows come with it, on either side of the line between row groups of 16 and 32 either: rows
# of a number of super-blocks that eight waves share unevenly (9, 20, 12) and evenly, several tiles a wave, a ragged last tile.
@pytest.mark.parametrize("ggml", [12, 13, 14, 23, 8], ids=["q4_k", "q5_k", "q6_k", "iq4_xs", "q8_0"])
@pytest.mark.parametrize("n,k", [(28001, 2304), (34816, 5120), (24131, 3072), (16750, 2048)])
def test_few_rows_sums_do_not_depend_on_the_rows_beside_them(api, d, ggml, n, k):
    block = synth.matrix(ggml, 61, k, seed=301).reshape(61, -1)      # over and over: neighbouring tiles are different
    w = qm(api, d, ggml, n, k, np.resize(block, (n, block.shape[1])).reshape(-1))
    for dtype, code in (("F16", oracle.F16), ("BF16", oracle.BF16)):
        x = oracle.round_storage(synth.activations(33, k, seed=302), code).reshape(33, k)
        want = oracle.project(ggml, block.reshape(-1), 61, k, x, accumulate="f64", weight_round=code, threads=8)
        first = None
        for m in (2, 9, 16, 17, 33):
            with few_rows(d, 2):
                got = d.project_quantized(api.Tensor.from_f32(d, (m, k), getattr(api.DType, dtype), x[:m]), w,
                                          out_dtype=api.DType.F32).tensor.to_f32()
            assert d.get_tuning("last_rows_plan") // 1000 == (32 if m > 16 else 16)
            assert_matmul_parity(got[:, :61], want[:m], f"{m} {dtype} rows")
            assert np.array_equal(bits(got), bits(got[:, np.arange(n) % 61]))
            first = got[:2] if first is None else first
            assert np.array_equal(bits(got[:2]), bits(first)), (m, dtype)


@pytest.mark.parametrize("ggml,m,n,k,few", [(13, 8, 151936, 2048, False), (12, 8, 28672, 4096, False), (13, 16, 28672, 4096, False),
                                            (12, 8, 17408, 5120, True), (12, 32, 34816, 5120, True), (12, 80, 17408, 5120, True)])
def test_16_bit_rows_take_the_faster_of_two_kernels(api, d, ggml, m, n, k, few):
    """Where the few-rows kernel's rounds are many or not whole the rows-resident kernel is ahead: 66 against 91 us for
    Q5_K's vocabulary matrix, 24 against 26.5 and 33 against 36 at 28672 x 4096; it is behind in the other three, 18
    against 24, 42 against 50 and 50 against 59.  The two multiply the same rounded weights."""
    tile = synth.matrix(ggml, 64, k, seed=271)
    w = qm(api, d, ggml, n, k, np.tile(tile, n // 64))
    x = api.Tensor.from_f32(d, (m, k), api.DType.F16, synth.activations(m, k, seed=272))
    got = d.project_quantized(x, w, out_dtype=api.DType.F32).tensor.to_f32()
    assert (d.get_tuning("last_rows_plan") != 0) == few
    want = oracle.project(ggml, tile, 64, k, x.to_f32(), accumulate="f64", weight_round=oracle.F16, threads=8)
    assert_matmul_parity(got[:, :64], want, "first rows")
    assert np.array_equal(bits(got), bits(np.tile(got[:, :64], n // 64)))


def taken_by(api, d, ggml, m, n, k):
    """Which kernel takes m f16 rows: "rows" (few-rows), "resident" or "m256" (the tiles)."""
    base = synth.matrix(ggml, 251, k, seed=760).reshape(251, -1)
    w = qm(api, d, ggml, n, k, np.resize(base, (n, base.shape[1])).reshape(-1))
    xt = api.Tensor.from_f32(d, (m, k), api.DType.F16, synth.activations(m, k, seed=761))
    got = d.project_quantized(xt, w)
    return "rows" if d.get_tuning("last_rows_plan") else got.operation.split("_")[-1]


@pytest.mark.parametrize("m,n", [(43, 27495), (42, 59617), (70, 41115)])
def test_a_tile_that_is_not_taken_keeps_no_call_from_the_few_rows_kernel(api, d, m, n):
    # rows of 256 are the resident kernel's where the few-rows kernel does not take them, whatever a tile would cost
    assert taken_by(api, d, Q6_K, m, n, 256) == "rows"


@pytest.mark.parametrize("ggml,m,n,k,kernel", [(23, 67, 13035, 3328, "m256"), (8, 102, 2271, 2816, "resident"),
                                               (8, 92, 8535, 2304, "resident")])
def test_uneven_shares_of_a_row_count_against_the_few_rows_kernel(api, d, ggml, m, n, k, kernel):
    assert taken_by(api, d, ggml, m, n, k) == kernel


def test_a_last_round_behind_one_of_pairs_counts_against_the_tiles(api, d):
    assert taken_by(api, d, Q4_K, 41, 96877, 1536) == "resident"


@pytest.mark.parametrize("ggml,m,n,k", [(14, 45, 22548, 1280), (8, 73, 23033, 1792)])
def test_the_96_column_tile_takes_rows_of_a_few_super_blocks(api, d, ggml, m, n, k):
    assert taken_by(api, d, ggml, m, n, k) == "m256"


@pytest.mark.parametrize("ggml", [12, 13, 14, 23, 8], ids=["q4_k", "q5_k", "q6_k", "iq4_xs", "q8_0"])
@pytest.mark.parametrize("m,n,k", [(16, 256, 256), (48, 100, 512), (8, 1024, 1024), (6, 4096, 4096), (40, 4100, 1024)])
def test_small_f32_batches_stay_on_the_gemv(api, d, ggml, m, n, k):
    """Q4_K and Q5_K batches take the few-rows kernel where it is the faster one, the other formats, whose GEMV is
    farther from 64 bits, always; both multiply exact weights by exact rows.  The GEMV's chains are up to 64 products
    (2.0e-7 in the mean square, 2^-24 / sqrt(3) * sqrt(64 / 2)), the other kernel's 16 and 24 adds (1.6e-7)."""
    w = qm(api, d, ggml, n, k, synth.matrix(ggml, n, k, seed=261))
    x = api.Tensor.from_f32(d, (m, k), api.DType.F32, synth.activations(m, k, seed=262))
    got = d.project_quantized(x, w).tensor.to_f32()
    small = m * n * (k // 256) < 80000 and ggml in (12, 13)
    assert (d.get_tuning("last_rows_plan") == 0) == small
    with few_rows(d, 0), fma_gemv(d):
        gemv = d.project_quantized(x, w).tensor.to_f32()
        assert d.get_tuning("last_rows_plan") == 0
    with few_rows(d, 2):
        rows = d.project_quantized(x, w).tensor.to_f32()
        assert d.get_tuning("last_rows_plan") != 0
    assert np.array_equal(got, gemv if small else rows)
    assert rel_l2(rows, gemv) <= 2.6e-7     # the two in the mean square


@pytest.mark.parametrize("ggml,m,dtype", [(12, 130, "F16"), (12, 300, "BF16"), (14, 200, "F16"), (8, 130, "F16")],
                         ids=["q4_k-130", "q4_k-300-bf16", "q6_k-200", "q8_0-130"])
def test_rows_too_long_for_lds_take_the_128_row_tiles(api, d, ggml, m, dtype):
    # K = 17408 (the 27B model's down projection): no 16 rows of it fit LDS, so from 65 rows on the
    # choice is between the tiles only.  5120 columns are too few for 256-row tiles to fill the chip
    # and enough for 128 x 64 ones (160 or 240 workgroups), the default; the square tiles
    # (tuning gemm_wide_shape 0) give the reference bits of the same products in another order.
    n, k = 5120, 17408
    packed = synth.matrix(ggml, n, k, seed=191)
    w = qm(api, d, ggml, n, k, packed)
    code = oracle.F16 if dtype == "F16" else oracle.BF16
    x = oracle.round_storage(synth.activations(m, k, seed=192), code).reshape(m, k)
    xt = api.Tensor.from_f32(d, (m, k), getattr(api.DType, dtype), x)
    out = d.project_quantized(xt, w, out_dtype=api.DType.F32)
    d.set_tuning("gemm_wide_shape", 0)
    try:
        square = d.project_quantized(xt, w, out_dtype=api.DType.F32)
    finally:
        d.set_tuning("gemm_wide_shape", 1)
    assert out.operation.endswith("_gemm_mfma_m256") == (m > 128) and square.operation.endswith("_gemm_mfma")
    got = out.tensor.to_f32()
    rows = np.unique(np.concatenate([np.arange(0, 70), np.arange(n - 70, n), synth.rng(193).integers(0, n, 60)]))
    want = oracle_columns(ggml, packed, n, k, rows, x, weight_round=code, accumulate="f64")
    assert_matmul_parity(got[:, rows], want, "rows of 17408 on the tiles")
    assert_matmul_parity(got, square.tensor.to_f32(), "against the square tiles", l2_tol=2e-6)


def test_objects_may_outlive_their_device(api):
    # buffers, matrices and recorded executions hold the device object: releasing them after
    # fh_device_destroy (any order a garbage collector may pick) is safe
    import gc
    dev = api.Device.new()
    n, k = 64, 512
    w = qm(api, dev, Q4_K, n, k, synth.matrix(Q4_K, n, k, seed=151))
    x = api.Tensor.from_f32(dev, (1, k), api.DType.F32, synth.activations(1, k, seed=152))
    y = api.Tensor.zeros(dev, (1, n), api.DType.F32)
    with dev.execution() as ex:
        dev.project_quantized(x, w, out=y)
    ex.graph.launch()
    want = y.to_f32().copy()
    handle, dev._handle = dev._handle, None
    api._lib.fh_device_destroy(handle)
    with pytest.raises(api.Error):
        y.to_f32()                                  # the device is gone: a clear error, not a crash
    with pytest.raises(api.Error):
        ex.graph.launch()
    del ex, w, x, y
    gc.collect()
    assert np.abs(want).max() > 0


def test_releases_asked_for_while_recording_wait_for_its_end(api, d):
    import gc
    n, k = 512, 1024
    packed = synth.matrix(Q4_K, n, k, seed=111)
    w = qm(api, d, Q4_K, n, k, packed)
    x = api.Tensor.from_f32(d, (1, k), api.DType.F32, synth.activations(1, k, seed=112))
    y = api.Tensor.zeros(d, (1, n), api.DType.F32)
    want = d.project_quantized(x, w).tensor.raw()
    with d.execution() as old:
        d.project_quantized(x, w, out=y)
    old.graph.launch()
    spare_w = qm(api, d, Q4_K, n, k, packed)
    spare_t = api.Tensor.zeros(d, (64, 64), api.DType.F32)
    with d.execution() as ex:
        d.project_quantized(x, w, out=y)
        # dropping a graph, a matrix and a tensor here must not disturb the recording
        del old, spare_w, spare_t
        gc.collect()
        d.project_quantized(x, w, out=y)
    y.buffer.upload(0, np.zeros(n, np.float32))
    ex.graph.launch()
    assert np.array_equal(y.raw(), want)
    assert np.array_equal(d.project_quantized(x, w).tensor.raw(), want)


@pytest.mark.parametrize("nbytes", [4, 4096, 40_000, 1_000_000, 64 << 20, (64 << 20) + 4])
def test_a_buffer_is_zero_whatever_held_its_memory_before(api, d, nbytes):
    # the block of a freed buffer serves the next one of its size class behind the work already enqueued
    for size in (nbytes, nbytes, max(nbytes - 4, 4)):
        t = api.Tensor.zeros(d, (size // 4,), api.DType.F32)
        assert not t.raw().any()
        t.buffer.upload(0, np.full(size // 4, 7, np.uint32))
        del t


def test_a_full_pool_makes_room_and_an_exposed_address_is_not_handed_on(api):
    dev = api.Device.new()
    kept = lambda: dev.get_tuning("held_pool_bytes")
    seen = []
    for step in range(12):
        held = [api.Buffer(dev, (40 << 20) + step * (1 << 20), zeroed=False) for _ in range(4)]
        del held
        seen.append(kept())
    assert 4 * 40 << 20 <= max(seen) <= 256 << 20 and sum(b < a for a, b in zip(seen, seen[1:])) > 1   # emptied more than once
    dev.set_tuning("held_pool_bytes", 0)
    assert kept() == 0
    b = api.Buffer(dev, 3 << 20)
    del b
    assert kept() == 3 << 20
    b = api.Buffer(dev, (3 << 20) - 100)      # of the same size class
    assert kept() == 0
    assert b.device_ptr()
    del b
    assert kept() == 0                        # its address has left the library
    big = api.Buffer(dev, (64 << 20) + 4)
    del big
    assert kept() == 0
    x = api.Tensor.zeros(dev, (8, 1024), api.DType.F16)
    assert not x.raw().any()
    with pytest.raises(api.Error):
        dev.set_tuning("held_pool_bytes", 1)


def test_blocks_whose_address_has_left_wait_for_all_work_on_the_gpu(api):
    dev, size, steps = api.Device.new(), 4 << 20, 40     # more than wait together
    kept, waiting = lambda: dev.get_tuning("held_pool_bytes"), lambda: dev.get_tuning("waiting_pool_bytes")
    hip, other = api._lib, ctypes.c_void_p()             # (the runtime the library is linked with)
    assert hip.hipStreamCreateWithFlags(ctypes.byref(other), 1) == 0
    copy = lambda to, source, count: hip.hipMemcpyAsync(ctypes.c_void_p(to), ctypes.c_void_p(source), ctypes.c_size_t(count), 3, other)
    busy, copies, reused = api.Buffer(dev, 512 << 20), api.Buffer(dev, steps * size), False
    dev.synchronize()
    for step in range(steps):
        b = api.Buffer(dev, size)
        b.upload(0, np.full(size // 4, step + 1, np.uint32))
        # its last use, on a stream of the caller's, is far from done when the buffer is dropped
        for _ in range(2):
            assert copy(busy.device_ptr(), busy.device_ptr() + (256 << 20), 256 << 20) == 0
        assert copy(copies.device_ptr() + step * size, b.device_ptr(), size) == 0
        before = kept()
        del b
        assert kept() <= 64 << 20 and waiting() < 64 << 20
        reused = reused or kept() > before
        fresh = api.Buffer(dev, size)                    # may get its block, and clears it at once
        del fresh
    assert hip.hipStreamSynchronize(other) == 0 and hip.hipStreamDestroy(other) == 0
    for step in range(steps):
        assert np.all(copies.download(step * size, size).view(np.uint32) == step + 1), step
    assert reused
    b = api.Buffer(dev, 1 << 20)
    assert b.device_ptr()
    before = waiting()
    del b
    assert waiting() == before + (1 << 20)
    dev.set_tuning("held_pool_bytes", 0)
    assert kept() == waiting() == 0
    small = [api.Buffer(dev, 4096) for _ in range(600)]     # and no more blocks than that, however small
    assert all(x.device_ptr() for x in small)
    small.clear()
    assert kept() == 511 * 4096 and waiting() == 88 * 4096     # 512 of them, of which one has gone back
    dev.set_tuning("held_pool_bytes", 0)
    assert kept() == waiting() == 0


def test_one_device_object_gives_back_what_another_on_the_gpu_keeps(api):
    # what an allocation that finds no memory does before it tries once more
    first, second = api.Device.new(), api.Device.new()
    w = qm(api, first, Q4_K, 64, 512, synth.matrix(Q4_K, 64, 512, seed=161))
    x = api.Tensor.from_f32(first, (1, 512), api.DType.F32, synth.activations(1, 512, seed=162))
    y = api.Tensor.zeros(first, (1, 64), api.DType.F32)
    want = first.project_quantized(x, w).tensor.raw()
    assert first.get_tuning("held_pool_bytes") > 0      # that result is gone again
    with first.execution() as recorded:
        first.project_quantized(x, w, out=y)
        before = first.get_tuning("held_pool_bytes")
        second.set_tuning("held_pool_bytes", 0)         # a device that is recording is left alone
        assert first.get_tuning("held_pool_bytes") == before > 0
    second.set_tuning("held_pool_bytes", 0)
    assert first.get_tuning("held_pool_bytes") == 0
    recorded.graph.launch()
    assert np.array_equal(y.raw(), want)
    handle, first._handle = first._handle, None
    api._lib.fh_device_destroy(handle)
    second.set_tuning("held_pool_bytes", 0)             # the other one is no longer looked at
    assert second.get_tuning("held_pool_bytes") == 0


# ------------------------------------------------------------- greedy selection

@pytest.mark.parametrize("dtype_name", ["F32", "F16", "BF16"])
def test_argmax_rows_matches_the_oracle(api, d, dtype_name):
    dtype = api.DType[dtype_name]
    code = {"F32": oracle.F32, "F16": oracle.F16, "BF16": oracle.BF16}[dtype_name]
    rng = synth.rng(131)
    for rows, width in ((1, 1), (3, 33), (4, 1024), (5, 4099), (2, 151936)):
        x = oracle.round_storage(rng.standard_normal((rows, width)).astype(np.float32), code).reshape(rows, width)
        if width > 40:
            x[0, 5] = x[0, width - 3] = 9.0
            if rows > 2:
                x[1, 9] = np.inf
                x[2, 0] = np.nan
            if rows > 3:
                x[3, 2047 % width] = np.nan
        got = d.argmax_rows(api.Tensor.from_f32(d, x.shape, dtype, x))
        assert d.last_operation() == "argmax_rows"
        want = oracle.argmax_rows(x)
        assert np.array_equal(got.raw().view(np.uint32).reshape(rows, 2), want), (rows, width)
    with pytest.raises(api.ShapeError):
        d.argmax_rows(api.Tensor.zeros(d, (4,), dtype))


@pytest.mark.parametrize("width", [8192, 8193, 16385, 30000])
def test_argmax_of_rows_cut_into_pieces(api, d, width):
    # rows of more than 8192 columns are searched piece by piece: ties across pieces, the maximum in a last
    # piece of one column, rows of -inf, signed zeros, and NaN where the reference's schedule starts a
    # thread's scan (columns below 1024) and where it does not
    x = synth.rng(137).standard_normal((8, width)).astype(np.float32)
    x[0, 7] = x[0, width - 1] = 9.0
    x[1, width - 1] = 9.0
    x[2, :] = -np.inf
    x[3, :] = -1.0
    x[3, 5000] = -0.0
    x[3, width - 2] = 0.0
    x[4, 9] = np.nan
    x[5, 4000] = np.nan
    x[5, 4001] = np.inf
    x[6, :1024] = np.nan
    x[7, width - 1] = np.nan
    for _ in range(2):     # the counters are left at zero
        got = d.argmax_rows(api.Tensor.from_f32(d, x.shape, api.DType.F32, x))
        assert np.array_equal(got.raw().view(np.uint32).reshape(8, 2), oracle.argmax_rows(x))


def test_argmax_of_a_row_alone_and_among_many(api, d):
    # many rows fill the chip with a workgroup each, a few are cut into pieces: the same answers
    rows, width = 150, 16385
    x = synth.rng(139).integers(0, 50, (rows, width)).astype(np.float32)     # ties all along every row
    x[3, 9000] = np.nan
    x[77, 16384] = np.inf
    want = oracle.argmax_rows(x)
    t = api.Tensor.from_f32(d, x.shape, api.DType.F32, x)
    assert np.array_equal(d.argmax_rows(t).raw().view(np.uint32).reshape(rows, 2), want)
    for at in (0, 3, 77, 149):
        one = api.Tensor.from_f32(d, (1, width), api.DType.F32, x[at])
        assert np.array_equal(d.argmax_rows(one).raw().view(np.uint32).reshape(2), want[at])


@pytest.mark.parametrize("ggml,n,k,dtype", [
    (Q6_K, 700, 17408, "F32"), (Q6_K, 700, 17408, "BF16"), (Q4_K, 4200, 1024, "F16"), (Q4_K, 1100, 17408, "F32"),
    (Q4_K, 300, 512, "F16"), (Q6_K, 1300, 17408, "F32"), (Q4_K, 1300, 17408, "BF16"), (Q4_K, 20500, 1024, "F16"),
    (Q4_K, 20480, 1024, "F32"), (Q4_K, 20479, 1024, "F32")])
def test_one_activated_row_has_the_bits_of_the_separate_calls(api, d, ggml, n, k, dtype):
    # Large matrices (81920 super-blocks) have the activated row written out first, small ones activate it in place;
    # both multiply on the FMA kernel.  A lane of it chains up to 3 x 64 products: roundings of at most 2^-24, uniform,
    # make 2^-24 / sqrt(3) * sqrt(192 / 2) = 3.4e-7 in the mean square, the tree over the lanes and segments some
    # 1e-7 more.
    packed_w = synth.matrix(ggml, n, k, seed=138)
    w = qm(api, d, ggml, n, k, packed_w)
    dt = getattr(api.DType, dtype)
    packed = api.Tensor.from_f32(d, (1, 2 * k), dt, synth.activations(1, 2 * k, seed=139))
    fused = d.project_quantized(packed, w, silu_mul=True)
    activated = d.expert_silu_mul(packed, k)
    with fma_gemv(d):
        separate = d.project_quantized(activated, w)
    assert np.array_equal(fused.tensor.raw(), separate.tensor.raw())
    assert np.abs(fused.tensor.to_f32()).max() > 1e-3
    exact = d.project_quantized(packed, w, out_dtype=api.DType.F32, silu_mul=True).tensor.to_f32()
    weights = oracle.dequantize(ggml, packed_w, n, k).reshape(n, k).astype(np.float64)
    assert rel_l2(exact, activated.to_f32().astype(np.float64) @ weights.T) <= 4e-7


def test_lm_head_projection_then_argmax_picks_the_oracle_token(api, d):
    n, k = 4096, 1024
    packed = synth.matrix(Q6_K, n, k, seed=141)
    w = qm(api, d, Q6_K, n, k, packed)
    x = synth.activations(1, k, seed=142)
    logits = d.project_quantized(api.Tensor.from_f32(d, x.shape, api.DType.F32, x), w).tensor
    picked = d.argmax_rows(logits).raw().view(np.uint32)
    want = oracle.project(Q6_K, packed, n, k, x, accumulate="f64")
    assert picked[1] == 0 and picked[0] == int(np.argmax(logits.to_f32()))
    top2 = np.sort(want[0])[-2:]
    if top2[1] - top2[0] > 1e-3 * abs(top2[1]):      # unambiguous in the oracle too
        assert picked[0] == int(np.argmax(want))


# ----------------------------------------------------------------------- Q5_K

Q5_K = 13


def test_q5_k_dequantize_and_gather_are_bit_exact(api, d):
    for rows, cols, packed in ((5, 512, fx.q5k_packed(5, 512)), (133, 2560, fx.q5k_packed(133, 2560)),
                               (257, 1024, synth.matrix(Q5_K, 257, 1024, seed=181))):
        w = qm(api, d, Q5_K, rows, cols, packed)
        assert w.byte_size() == rows * (cols // 256) * 176
        want = oracle.dequantize(Q5_K, packed, rows, cols)
        assert np.array_equal(bits(d.dequantize(w).to_f32()), bits(want))
        assert np.array_equal(bits(d.dequantize(w, api.DType.BF16).to_f32()),
                              bits(oracle.round_storage(want, oracle.BF16).reshape(rows, cols)))
        ids = [rows - 1, 0, 3]
        got = d.embedding_gather_quantized(w, ids, api.DType.F32)
        assert got.operation == "embedding_gather_q5_k"
        assert np.array_equal(bits(got.tensor.to_f32()), bits(want[ids]))


def test_q5_k_gemv_and_small_batches_replay_the_reference_cases(api, d):
    # q4_k_and_q5_k_gemv_gemm_cover_blocks_and_batch_tails (src/ops/transformer.rs:2982-3002):
    # (N, K) = (5, 512), M in 1..7 except 6, f32, abs <= 2e-4 against the f32-sequential sum
    n, k = 5, 512
    packed = fx.q5k_packed(n, k)
    w = qm(api, d, Q5_K, n, k, packed)
    for m in (1, 2, 3, 4, 5, 7):
        x = fx.q4k_input(m, k)
        out = d.project_quantized(api.Tensor.from_f32(d, x.shape, api.DType.F32, x), w)
        assert out.operation == ("q5_k_gemv_factored" if m == 1 else "q5_k_gemm")
        want = oracle.project(Q5_K, packed, n, k, x, accumulate="f32")
        assert np.abs(out.tensor.to_f32() - want).max() <= 2e-4, m


@pytest.mark.parametrize("n,k,m,dtype_name", [(4099, 5120, 1, "F32"), (1003, 4864, 1, "F32"), (5120, 17408, 1, "F32"),
                                              (515, 1280, 3, "F32"), (515, 1280, 1, "F16"), (515, 1280, 4, "BF16")])
def test_q5_k_projection_matches_the_f64_oracle(api, d, n, k, m, dtype_name):
    dtype = api.DType[dtype_name]
    code = {"F32": oracle.F32, "F16": oracle.F16, "BF16": oracle.BF16}[dtype_name]
    packed = synth.matrix(Q5_K, n, k, seed=n + k)
    w = qm(api, d, Q5_K, n, k, packed)
    x = oracle.round_storage(synth.activations(m, k, seed=11), code).reshape(m, k)
    out = d.project_quantized(api.Tensor.from_f32(d, x.shape, dtype, x), w, out_dtype=api.DType.F32)
    rows = np.unique(np.concatenate([np.arange(0, 40), np.arange(n - 40, n), synth.rng(12).integers(0, n, 64)]))
    tiles = m > 1 and dtype_name != "F32"            # 16-bit batches take the tile kernels: weights rounded once
    want = oracle_columns(Q5_K, packed, n, k, rows, x, accumulate="f64", **({"weight_round": code} if tiles else {}))
    assert_matmul_parity(out.tensor.to_f32()[:, rows], want, f"q5_k {n}x{k} m={m} {dtype_name}")
    if k == 17408:
        assert out.operation == "q5_k_gemv_ksplit"


@pytest.mark.parametrize("m,n,dtype_name", [(8, 1100, "F16"), (20, 1100, "BF16"), (130, 1000, "F16"),
                                            (130, 16000, "BF16"), (300, 33000, "F16")])
def test_q5_k_tile_kernels_match_the_rounded_weight_oracle(api, d, m, n, dtype_name):
    # skinny (M <= 32), 64- and 128-wide tiles, and the 256-row tile (33000 columns x 2 row tiles)
    k = 512
    dtype = api.DType[dtype_name]
    code = oracle.F16 if dtype_name == "F16" else oracle.BF16
    packed = synth.matrix(Q5_K, n, k, seed=201 + n)
    w = qm(api, d, Q5_K, n, k, packed)
    x = oracle.round_storage(synth.activations(m, k, seed=202), code).reshape(m, k)
    d.set_tuning("gemm_resident", 0)       # the square tiles, which rows longer than LDS still take
    d.set_tuning("gemm_wide_shape", 0)     # where too few 256-row tiles would fill the chip (128-row ones do)
    try:
        out = d.project_quantized(api.Tensor.from_f32(d, x.shape, dtype, x), w, out_dtype=api.DType.F32)
    finally:
        d.set_tuning("gemm_resident", 1)
        d.set_tuning("gemm_wide_shape", 1)
    want_name = {8: "q5_k_gemm_mfma_skinny", 20: "q5_k_gemm_mfma_skinny", 130: "q5_k_gemm_mfma",
                 300: "q5_k_gemm_mfma_m256"}[m]
    assert out.operation == want_name
    rows = np.unique(np.concatenate([np.arange(0, 140), np.arange(n - 80, n), synth.rng(203).integers(0, n, 64)]))
    want = oracle_columns(Q5_K, packed, n, k, rows, x, weight_round=code, accumulate="f64")
    assert_matmul_parity(out.tensor.to_f32()[:, rows], want, f"q5_k tile m={m} n={n}")
    # the bf16 reference case: result stored in the activation dtype
    if m == 20:
        stored = d.project_quantized(api.Tensor.from_f32(d, x.shape, dtype, x), w).tensor.to_f32()
        assert np.array_equal(bits(stored), bits(oracle.round_storage(out.tensor.to_f32(), code).reshape(m, n)))


def test_q5_k_expert_projection_and_validation(api, d):
    experts, rows, cols, a = 4, 40, 768, 9
    packed = synth.matrix(Q5_K, experts * rows, cols, seed=191)
    w = api.QuantizedExpertMatrix.new(d, packed, api.QuantizationFormat(Q5_K), experts, rows, cols)
    meta = np.zeros((a, 3), dtype=np.uint32)
    meta[:, 0] = [0, 3, 1, 1, 2, 7, 0, 3, 2]          # 7 does not exist: a zero row
    meta[:, 1] = np.arange(a)
    meta[:, 2] = np.float32(1.0).view(np.uint32)
    x = synth.activations(a, cols, seed=192)
    got = d.expert_project_quantized(api.Tensor.from_f32(d, x.shape, api.DType.F32, x),
                                     api.Tensor.from_bits(d, meta.shape, meta), w, cols, experts)
    assert d.last_operation() == "expert_project_q5_k_factored"
    got = got.to_f32()
    safe = meta.copy(); safe[5, 0] = 0
    want = oracle.expert_project(Q5_K, packed, experts, rows, cols, x, safe.view(np.float32), accumulate="f64")
    valid = np.arange(a) != 5
    assert np.all(got[5] == 0)
    assert_matmul_parity(got[valid], want[valid], "q5_k expert projection")
    bad = packed.copy()
    bad[1] = 0x7c                                       # d = +inf in the first block
    with pytest.raises(api.WeightError):
        api.QuantizedMatrix.from_bytes(d, experts * rows, cols, api.QuantizationFormat(Q5_K), bad)
    with pytest.raises(api.Error):
        api.QuantizedMatrix.from_bytes(d, experts * rows, cols, api.QuantizationFormat(Q5_K), packed[:-1])


IQ4_XS, Q8_0 = 23, 8


# Rows that fit LDS for their whole length (K <= 2560 for groups of 32 rows, K <= 5120 for groups
# of 16), two rows or more: the kernel that keeps a group of rows resident and streams the
# weights past them.  Ragged row groups, ragged row tiles, more pieces than compute units, both
# group sizes, every format, both 16-bit dtypes.
@pytest.mark.parametrize("ggml,m,n,k,dtype_name", [
    (Q4_K, 70, 1000, 768, "F16"), (Q4_K, 200, 50, 4096, "BF16"), (Q4_K, 2000, 1000, 256, "F16"),
    (Q4_K, 40, 300, 5120, "F16"), (Q4_K, 2, 1000, 768, "F16"), (Q4_K, 16, 100, 4096, "BF16"), (Q6_K, 17, 530, 1024, "F16"), (Q5_K, 64, 1000, 512, "F16"),
    (Q5_K, 130, 1000, 512, "BF16"), (Q6_K, 97, 530, 1024, "F16"), (Q6_K, 65, 40, 2560, "F16"),
    (IQ4_XS, 300, 300, 512, "F16"), (Q8_0, 129, 260, 1280, "BF16")])
def test_rows_resident_gemm_matches_the_rounded_weight_oracle(api, d, ggml, m, n, k, dtype_name):
    dtype = api.DType[dtype_name]
    code = oracle.F16 if dtype_name == "F16" else oracle.BF16
    packed = synth.matrix(ggml, n, k, seed=301 + n + m)
    w = qm(api, d, ggml, n, k, packed)
    x = oracle.round_storage(synth.activations(m, k, seed=302 + m), code).reshape(m, k)
    xt = api.Tensor.from_f32(d, x.shape, dtype, x)
    with few_rows(d, 0):      # (up to 128 rows the few-rows kernel may take the call under the same name)
        out = d.project_quantized(xt, w, out_dtype=api.DType.F32)
    assert out.operation.endswith("_gemm_mfma_resident") and d.get_tuning("last_rows_plan") == 0
    rows = np.unique(np.concatenate([np.arange(0, min(n, 48)), np.arange(max(0, n - 40), n),
                                     synth.rng(303).integers(0, n, 32)]))
    want = oracle_columns(ggml, packed, n, k, rows, x, weight_round=code, accumulate="f64")
    got = out.tensor.to_f32()
    assert_matmul_parity(got[:, rows], want, f"rows-resident m={m} n={n} k={k}")
    # stored in the activation dtype (packed stores where rows allow, element stores on ragged ones)
    with few_rows(d, 0):
        stored = d.project_quantized(xt, w)
    assert stored.operation == out.operation
    assert np.array_equal(bits(stored.tensor.to_f32()), bits(oracle.round_storage(got, code).reshape(m, n)))
    # every row group and tile was written: the square tiles give the same product
    d.set_tuning("gemm_resident", 0)
    try:
        tiles = d.project_quantized(xt, w, out_dtype=api.DType.F32)
    finally:
        d.set_tuning("gemm_resident", 1)
    assert not tiles.operation.endswith("_resident")
    assert rel_l2(got, tiles.tensor.to_f32()) <= 1e-5


@pytest.mark.parametrize("m,n,k,rounded", [(320, 5120, 17408, False), (128, 2500, 31744, True)])
def test_a_batch_whose_partial_sums_outgrow_the_scratch_can_be_recorded_first(api, m, n, k, rounded):
    """Partial sums of K segments save time only.  Exact f32 rows run in launches whose sums fit the scratch a new
    device has.  Rows that are rounded to f16 have 7.8 MiB of it for that, and 9.8 MiB of sums no longer fit: while
    it records the device takes a kernel that needs none, and replays are that kernel's results."""
    dev = api.Device.new()
    dev.set_tuning("gemm_few_tiles_split", 2)
    dev.set_tuning("gemm_f32_min_rows", 2 if rounded else 0)
    w = qm(api, dev, Q4_K, n, k, synth.matrix(Q4_K, n, k, seed=711))
    x = api.Tensor.from_f32(dev, (m, k), api.DType.F32, synth.activations(m, k, seed=712))
    recorded = api.Tensor.zeros(dev, (m, n), api.DType.F32)
    dev.synchronize()
    with dev.execution() as ex:
        dev.project_quantized(x, w, out=recorded)
    assert (dev.get_tuning("last_rows_plan") == 0) == rounded
    ex.graph.launch()
    dev.synchronize()
    held = dev.get_tuning("held_scratch_bytes")
    direct = dev.project_quantized(x, w, out_dtype=api.DType.F32).tensor.to_f32()   # the scratch may grow here
    assert dev.get_tuning("last_rows_plan") != 0
    assert (dev.get_tuning("held_scratch_bytes") > held) == rounded
    for _ in range(2):
        ex.graph.launch()
        dev.synchronize()
        if rounded:
            assert rel_l2(recorded.to_f32(), direct) <= 1e-5
        else:
            assert np.array_equal(bits(recorded.to_f32()), bits(direct))


@pytest.mark.parametrize("ggml,m,n,k", [(Q4_K, 1000, 5120, 17408), (Q6_K, 1800, 1030, 17408)])
def test_an_f32_batch_of_any_size_leaves_the_scratch_as_it_is(api, ggml, m, n, k):
    """Rows this long are cut into three K segments, whose partial sums for all of the batch would be 58 and 21 MiB;
    the batch runs in launches whose sums fit the 16 MiB a device always has, so it needs no memory of its own.
    A row's bits do not depend on the launch it is in."""
    dev = api.Device.new()
    packed = synth.matrix(ggml, n, k, seed=731)
    w = qm(api, dev, ggml, n, k, packed)
    x = np.resize(synth.activations(97, k, seed=732), (m, k)).astype(np.float32)    # 97: no row at the same place in two launches
    held = dev.get_tuning("held_scratch_bytes")
    got = dev.project_quantized(api.Tensor.from_f32(dev, (m, k), api.DType.F32, x), w).tensor.to_f32()
    assert dev.get_tuning("held_scratch_bytes") == held
    assert np.array_equal(bits(got), bits(np.resize(got[:97], (m, n))))
    rows = np.unique(np.concatenate([np.arange(0, 40), np.arange(n - 40, n)]))
    want = oracle_columns(ggml, packed, n, k, rows, x[:97], accumulate="f64")
    assert_matmul_parity(got[:97][:, rows], want, "f32 batch in several launches")
    part = dev.project_quantized(api.Tensor.from_f32(dev, (7, k), api.DType.F32, x[m - 7:]), w).tensor.to_f32()
    assert np.array_equal(bits(part), bits(got[m - 7:]))


@pytest.mark.parametrize("ggml,m,n,k", [(Q4_K, 5, 200, 256), (Q4_K, 16, 1024, 1024), (Q6_K, 24, 530, 2048), (Q5_K, 64, 777, 5120),
                                        (IQ4_XS, 12, 300, 4096), (Q8_0, 9, 400, 4352), (Q6_K, 6, 1030, 17408), (Q8_0, 7, 1030, 17408),
                                        (IQ4_XS, 5, 1030, 14336), (Q4_K, 6, 1030, 17408)])
def test_a_batch_of_f32_rows_is_as_close_to_64_bits_as_its_chains_are_short(api, d, ggml, m, n, k):
    """Sixteen products follow each other in one accumulator, the rest is added in pairs and over eight waves.
    A chain of L roundings of at most 2^-24, uniform, is off by 2^-24 / sqrt(3) * sqrt(L / 2) in the mean square:
    1.0e-7 for 16, 1.6e-7 with the adds behind it counted as another 24; all 256 of a super-block in one
    chain give 3.9e-7."""
    packed = synth.matrix(ggml, n, k, seed=721)
    w = qm(api, d, ggml, n, k, packed)
    x = np.asarray(synth.activations(m, k, seed=722), dtype=np.float32).reshape(m, k)
    xt = api.Tensor.from_f32(d, x.shape, api.DType.F32, x)
    with few_rows(d, 2):
        got = d.project_quantized(xt, w).tensor.to_f32()
        assert d.get_tuning("last_rows_plan") != 0
    weights = oracle.dequantize(ggml, packed, n, k).reshape(n, k).astype(np.float64)
    exact = x.astype(np.float64) @ weights.T
    assert rel_l2(got, exact) <= 1.6e-7
    # the default is this kernel or, for Q4_K and Q5_K, a GEMV that is as close
    assert rel_l2(d.project_quantized(xt, w).tensor.to_f32(), exact) <= 1.6e-7


@pytest.mark.parametrize("ggml", [12, 13, 14, 23], ids=["q4_k", "q5_k", "q6_k", "iq4_xs"])
@pytest.mark.parametrize("m,n,k", [(17, 65601, 256), (20, 33000, 512), (32, 22003, 768), (33, 26315, 1280), (65, 2573, 6912), (49, 4099, 4352)])
def test_f32_batches_as_pairs_of_f16(api, d, ggml, m, n, k):
    """Rows of 1, 2, 3, 5, 17 and 27 super-blocks (a K half without one, an odd one out, K segments with a short last one),
    ragged tiles and groups of rows, rows of very different magnitudes.  Against 64 bits: chains of at most eight matrix
    steps and the adds behind them, which with the half unit an operand pair loses stay within the 1.6e-7 of the kernel
    on the f32 instruction."""
    packed = synth.matrix(ggml, n, k, seed=741)
    w = qm(api, d, ggml, n, k, packed)
    x = np.asarray(synth.activations(m, k, seed=742), dtype=np.float32).reshape(m, k)
    x[1] *= 1e-25
    x[2] *= 1e25
    x[3, ::7] *= 1e4
    x[4] = 0
    x[5, : k // 2] = 0
    xt = api.Tensor.from_f32(d, x.shape, api.DType.F32, x)
    got = d.project_quantized(xt, w)
    assert d.get_tuning("last_rows_plan") // 1000 == 32 or (33 <= m <= 48 and ggml == 14)
    rows = np.unique(np.concatenate([np.arange(0, 160), np.arange(n - 160, n), synth.rng(743).integers(0, n, 200)]))
    row_bytes = packed.size // n
    weights = oracle.dequantize(ggml, np.ascontiguousarray(packed.reshape(n, row_bytes)[rows]).reshape(-1), len(rows), k)
    want = x.astype(np.float64) @ weights.reshape(len(rows), k).astype(np.float64).T
    out = got.tensor.to_f32()[:, rows]
    assert not out[4].any()
    for r in range(m):
        if r != 4:
            assert rel_l2(out[r], want[r]) <= 2.4e-7, r     # one row: the mean square over fewer outputs
    live = [r for r in range(m) if r != 4]
    size = np.linalg.norm(want[live], axis=1, keepdims=True)
    assert rel_l2(out[live] / size, want[live] / size) <= 1.6e-7
    assert np.array_equal(bits(d.project_quantized(xt, w).tensor.to_f32()), bits(got.tensor.to_f32()))
    if d.get_tuning("last_rows_plan") // 1000 == 32 and not 33 <= m - 1 <= 48 and m > 17:    # a row's sums are its own
        part = d.project_quantized(api.Tensor.from_f32(d, (m - 1, k), api.DType.F32, x[1:]), w).tensor.to_f32()
        assert np.array_equal(bits(part), bits(got.tensor.to_f32()[1:]))
    half = api.Tensor.zeros(d, (m, n), api.DType.F16)
    d.project_quantized(xt, w, out=half)
    assert np.array_equal(bits(half.to_f32()), bits(oracle.round_storage(got.tensor.to_f32(), oracle.F16).reshape(m, n)))


@pytest.mark.parametrize("ggml", [12, 13, 14, 23], ids=["q4_k", "q5_k", "q6_k", "iq4_xs"])
@pytest.mark.parametrize("rows", ["normal", "gated", "outliers"])
def test_f32_batches_as_pairs_are_no_farther_from_64_bits_than_on_the_f32_instruction(api, d, ggml, rows):
    # also where few elements carry a sum: what SiLU and a product make of normal values, and rows with a few channels
    # a thousand times the others
    m, n, k = 24, 2573, 17408
    packed = synth.matrix(ggml, n, k, seed=745)
    w = qm(api, d, ggml, n, k, packed)
    g = synth.rng(746)
    x = g.standard_normal((m, k))
    if rows == "gated":
        x = 3 * x / (1 + np.exp(-3 * x)) * g.standard_normal((m, k))
    elif rows == "outliers":
        x = x * np.where(g.random((1, k)) < 0.004, 1000.0, 1.0)
    x = x.astype(np.float32)
    xt = api.Tensor.from_f32(d, (m, k), api.DType.F32, x)
    got = d.project_quantized(xt, w).tensor.to_f32()
    assert d.get_tuning("last_rows_plan") // 1000 == 32
    with few_rows(d, 2):
        other = d.project_quantized(xt, w).tensor.to_f32()
        assert d.get_tuning("last_rows_plan") // 1000 == 16
    want = x.astype(np.float64) @ oracle.dequantize(ggml, packed, n, k).reshape(n, k).astype(np.float64).T
    assert rel_l2(got, want) <= rel_l2(other, want)


@pytest.mark.parametrize("ggml,n,k,pairs", [(12, 7147, 4352, True), (13, 7147, 4352, False), (13, 6144, 6144, True), (12, 7000, 4352, False),
                                             (12, 126084, 256, False), (13, 76728, 512, False), (12, 50643, 768, True)])
def test_up_to_sixteen_f32_rows_take_pairs_by_format_and_size(api, d, ggml, n, k, pairs):
    base = synth.matrix(ggml, 7, k, seed=759)
    w = qm(api, d, ggml, n, k, np.resize(base, base.size // 7 * n))
    x = api.Tensor.from_f32(d, (16, k), api.DType.F32, synth.activations(16, k, seed=760))
    got = d.project_quantized(x, w).tensor.to_f32()
    assert d.get_tuning("last_rows_plan") // 1000 == (32 if pairs else 16)
    want = x.to_f32().reshape(16, k).astype(np.float64) @ oracle.dequantize(ggml, base, 7, k).reshape(7, k).astype(np.float64).T
    assert rel_l2(got[:, :7], want) <= 1.8e-7    # (1.6e-7 over many outputs, as above; here 112)


def test_f32_batches_without_room_for_pairs_take_the_f32_instruction(api):
    # 43000 x 4352: the operands of 32 rows and their sums of three K segments are 17.1 MB, more than the scratch of a
    # new device holds while it records
    dev = api.Device.new()
    m, n, k = 32, 43000, 4352
    base = synth.matrix(Q4_K, 100, k, seed=747)
    w = qm(api, dev, Q4_K, n, k, np.resize(base, base.size // 100 * n))
    x = synth.activations(m, k, seed=748).reshape(m, k)
    xt = api.Tensor.from_f32(dev, (m, k), api.DType.F32, x)
    recorded = api.Tensor.zeros(dev, (m, n), api.DType.F32)
    with dev.execution() as ex:
        dev.project_quantized(xt, w, out=recorded)
    assert dev.get_tuning("last_rows_plan") // 1000 == 16
    with few_rows(dev, 2):
        other = dev.project_quantized(xt, w).tensor.to_f32()
    got = dev.project_quantized(xt, w).tensor.to_f32()
    assert dev.get_tuning("last_rows_plan") // 1000 == 32
    for _ in range(2):
        ex.graph.launch()
        dev.synchronize()
        assert np.array_equal(bits(recorded.to_f32()), bits(other))
    assert rel_l2(got, other) <= 2.6e-7 and np.array_equal(bits(got[:, :100]), bits(got[:, 42900:]))


@pytest.mark.parametrize("ggml", [12, 14], ids=["q4_k", "q6_k"])
def test_f32_batches_with_infinities_and_nan(api, d, ggml):
    # they reach the outputs that the products of the row as it is written give: the same ones as on the f32 instruction
    m, n, k = 20, 2600, 6912
    w = qm(api, d, ggml, n, k, synth.matrix(ggml, n, k, seed=751))
    x = np.asarray(synth.activations(m, k, seed=752), dtype=np.float32).reshape(m, k)
    x[2, 77], x[5, 900], x[7, 3], x[7, 6900], x[9, 4] = np.inf, np.nan, -np.inf, np.inf, 3e38
    xt = api.Tensor.from_f32(d, x.shape, api.DType.F32, x)
    got = d.project_quantized(xt, w).tensor.to_f32()
    assert d.get_tuning("last_rows_plan") // 1000 == 32
    with few_rows(d, 2):
        want = d.project_quantized(xt, w).tensor.to_f32()
        assert d.get_tuning("last_rows_plan") // 1000 == 16
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.isnan(want[5]).all()
    inf = np.isinf(want)
    assert np.array_equal(np.isinf(got), inf) and np.array_equal(got[inf], want[inf]) and inf[2].any()
    fine = [r for r in range(m) if r not in (2, 5, 7, 9)]
    assert rel_l2(got[fine], want[fine]) <= 2.6e-7


@pytest.mark.parametrize("ggml", [12, 13, 14, 23], ids=["q4_k", "q5_k", "q6_k", "iq4_xs"])
@pytest.mark.parametrize("m,n,k", [(20, 33000, 512), (60, 2573, 17408)])
def test_infinities_in_f32_batches_are_the_products_of_the_infinite_values(api, d, ggml, m, n, k):
    # one and several K segments; infinities of one sign and of both, in one super-block and in many, in many rows at once,
    # beside a NaN
    packed = synth.matrix(ggml, n, k, seed=755)
    w = qm(api, d, ggml, n, k, packed)
    x = np.asarray(synth.activations(m, k, seed=756), dtype=np.float32).reshape(m, k)
    x[0, k - 1] = np.inf
    x[1, 3], x[1, 4] = np.inf, -np.inf
    x[2, ::97] = -np.inf
    x[3] = np.inf
    x[4], x[4, 5] = np.inf, np.nan
    x[5, 255], x[5, 256] = -np.inf, -np.inf
    x[6] = np.nan
    x[m - 1, k // 2 + 1] = np.nan
    x[m - 9:m - 2, 40] = np.inf
    xt = api.Tensor.from_f32(d, x.shape, api.DType.F32, x)
    got = d.project_quantized(xt, w).tensor.to_f32()
    assert d.get_tuning("last_rows_plan") // 1000 == 32
    rows = np.unique(np.concatenate([np.arange(0, 130), np.arange(n - 130, n)]))
    row_bytes = packed.size // n
    weights = oracle.dequantize(ggml, np.ascontiguousarray(packed.reshape(n, row_bytes)[rows]).reshape(-1), len(rows), k)
    with np.errstate(invalid="ignore"):
        want = x.astype(np.float64) @ weights.reshape(len(rows), k).astype(np.float64).T
    out = got[:, rows]
    assert np.array_equal(np.isnan(out), np.isnan(want)) and np.isnan(got[[4, 6, m - 1]]).all()
    inf = np.isinf(want)
    assert np.array_equal(np.isinf(out), inf) and np.array_equal(out[inf], want[inf]) and inf[0].any() and inf[m - 5].any()
    fine = [r for r in range(7, m - 9)]
    assert rel_l2(out[fine], want[fine]) <= 1.6e-7


@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_values_that_are_not_finite_do_not_multiply_the_time_of_a_batch(api, d, value):
    # some 40 us with finite rows; 60 ms when every output was multiplied out again
    m, n, k = 24, 2573, 17408
    w = qm(api, d, Q6_K, n, k, synth.matrix(Q6_K, n, k, seed=757))
    x = np.asarray(synth.activations(m, k, seed=758), dtype=np.float32).reshape(m, k)
    x[:, 77] = value
    xt, y = api.Tensor.from_f32(d, (m, k), api.DType.F32, x), api.Tensor.zeros(d, (m, n), api.DType.F32)
    d.project_quantized(xt, w, out=y)
    start, end = api.Event(d), api.Event(d)
    start.record()
    d.project_quantized(xt, w, out=y)
    end.record()
    d.synchronize()
    assert start.elapsed_ms(end) < 3.0


@pytest.mark.parametrize("ggml", [12, 13, 14, 23, 8], ids=["q4_k", "q5_k", "q6_k", "iq4_xs", "q8_0"])
@pytest.mark.parametrize("m,n,k,dtype", [(257, 33, 256, "F16"), (300, 1000, 512, "BF16"), (513, 2571, 1280, "F16"), (700, 517, 2304, "BF16")])
def test_weights_decoded_first_give_the_bits_of_the_fused_tiles(api, d, ggml, m, n, k, dtype):
    # one to nine super-blocks, ragged rows and columns, every tile of the product; and the fused tiles against the oracle
    packed = synth.matrix(ggml, n, k, seed=761)
    w = qm(api, d, ggml, n, k, packed)
    code = oracle.F16 if dtype == "F16" else oracle.BF16
    x = oracle.round_storage(synth.activations(m, k, seed=762), code).reshape(m, k)
    xt = api.Tensor.from_f32(d, (m, k), getattr(api.DType, dtype), x)
    try:
        d.set_tuning("gemm_wide32_tile", 25)
        want = d.project_quantized(xt, w, out_dtype=api.DType.F32)
        d.set_tuning("gemm_wide32_tile", 0)
        d.set_tuning("gemm_decoded_min_rows", 2)
        for tile in (192, 256, 320):
            d.set_tuning("gemm_decoded_tile", tile)
            got = d.project_quantized(xt, w, out_dtype=api.DType.F32)
            assert got.operation == want.operation
            assert np.array_equal(bits(got.tensor.to_f32()), bits(want.tensor.to_f32())), tile
            stored = d.project_quantized(xt, w).tensor.to_f32()
            assert np.array_equal(bits(stored), bits(oracle.round_storage(got.tensor.to_f32(), code).reshape(m, n)))
    finally:
        d.set_tuning("gemm_wide32_tile", 0)
        d.set_tuning("gemm_decoded_min_rows", 1)
        d.set_tuning("gemm_decoded_tile", 0)
    rows = np.unique(np.concatenate([np.arange(0, 20), np.arange(n - 20, n)]))
    assert_matmul_parity(want.tensor.to_f32()[:, rows], oracle_columns(ggml, packed, n, k, rows, x, weight_round=code, accumulate="f64"),
                         "fused tiles")


@pytest.mark.parametrize("ggml,m,n,k,dtype", [(12, 257, 33, 512, "F16"), (14, 300, 1000, 768, "BF16"), (8, 513, 2572, 1280, "F16"),
                                              (23, 700, 517, 2304, "BF16"), (13, 1025, 644, 4352, "F16"), (12, 2048, 1280, 2048, "BF16")])
def test_decoded_products_with_k_cut_in_two(api, d, ggml, m, n, k, dtype):
    # two super-blocks to seventeen, even and odd, ragged rows and columns, rows that are whole fours and rows that are not, one
    # tile and several rows of them.  At most k / 8 sums follow each other on either side, each off by 2^-24 at most, uniform.
    packed = synth.matrix(ggml, n, k, seed=771)
    w = qm(api, d, ggml, n, k, packed)
    code = oracle.F16 if dtype == "F16" else oracle.BF16
    x = oracle.round_storage(synth.activations(m, k, seed=772), code).reshape(m, k)
    xt = api.Tensor.from_f32(d, (m, k), getattr(api.DType, dtype), x)
    rows = np.unique(np.concatenate([np.arange(0, 20), np.arange(n - 20, n)]))
    want = oracle_columns(ggml, packed, n, k, rows, x, weight_round=code, accumulate="f64")
    bound = 2.0 ** -24 / np.sqrt(3) * np.sqrt(k / 16)
    try:
        d.set_tuning("gemm_decoded_min_rows", 2)
        for tile in (192, 256, 320):
            d.set_tuning("gemm_decoded_tile", tile)
            d.set_tuning("gemm_decoded_segments", 1)
            whole = d.project_quantized(xt, w, out_dtype=api.DType.F32).tensor.to_f32()
            assert (d.get_tuning("last_decoded_tile"), d.get_tuning("last_decoded_cut")) == (tile, 0)
            d.set_tuning("gemm_decoded_segments", 2)
            got = d.project_quantized(xt, w, out_dtype=api.DType.F32).tensor.to_f32()
            assert (d.get_tuning("last_decoded_tile"), d.get_tuning("last_decoded_cut")) == (0, tile)
            assert rel_l2(got[:, rows], want) <= bound and rel_l2(got, whole) <= np.sqrt(2) * bound
            stored = api.Tensor.zeros(d, (m, n), getattr(api.DType, dtype))
            with d.execution() as recording:       # whichever segment ends first, the same bits; also replayed
                d.project_quantized(xt, w, out=stored)
            for _ in range(3):
                recording.graph.launch()
                d.synchronize()
                assert np.array_equal(bits(stored.to_f32()), bits(oracle.round_storage(got, code).reshape(m, n)))
                assert np.array_equal(bits(d.project_quantized(xt, w, out_dtype=api.DType.F32).tensor.to_f32()), bits(got))
    finally:
        d.set_tuning("gemm_decoded_min_rows", 1)
        d.set_tuning("gemm_decoded_tile", 0)
        d.set_tuning("gemm_decoded_segments", 0)


@pytest.mark.parametrize("m,n,count", [(300, 57344, 1), (300, 57001, 1), (520, 34816, 1), (600, 24000, 1), (1300, 14336, 1),
                                       (1025, 52844, 2), (1025, 54838, 2), (1300, 43871, 2), (2047, 32904, 2), (2047, 52845, 2)])
def test_runs_of_several_decoded_tiles_give_the_bits_of_one(api, d, m, n, count):
    # columns of more than a round of the chip, in one run of tiles or whole rounds of one tile and the rest on another (320 first and
    # 256 first, the second run ragged, rows that are whole fours and rows that are not): every column comes from one of them
    k = 512
    base = synth.matrix(Q4_K, 251, k, seed=775).reshape(251, -1)
    w = qm(api, d, Q4_K, n, k, np.resize(base, (n, base.shape[1])).reshape(-1))
    xt = api.Tensor.from_f32(d, (m, k), api.DType.F16, synth.activations(m, k, seed=776))
    out = api.Tensor.zeros(d, (m, n), api.DType.F16)
    try:
        d.set_tuning("gemm_decoded_min_rows", 2)
        d.project_quantized(xt, w, out=out)
        runs = out.raw()
        assert d.get_tuning("last_decoded_tile") != 0 and d.get_tuning("last_decoded_runs") == count
        for tile in (192, 256, 320):
            d.set_tuning("gemm_decoded_tile", tile)
            d.project_quantized(xt, w, out=out)
            assert (d.get_tuning("last_decoded_tile"), d.get_tuning("last_decoded_runs")) == (tile, 1)
            assert np.array_equal(out.raw(), runs), tile
    finally:
        d.set_tuning("gemm_decoded_min_rows", 1)
        d.set_tuning("gemm_decoded_tile", 0)


@pytest.mark.parametrize("ggml,m,n,k,tile", [(14, 1024, 12288, 4096, 192), (8, 1999, 7147, 4352, 256), (14, 1500, 8192, 8192, 256),
                                             (14, 1999, 17408, 5120, 320), (12, 1999, 17408, 5120, 320),
                                             (14, 741, 19548, 1024, 256), (13, 1030, 14387, 2048, 320)])
def test_the_fastest_of_the_decoded_tiles_is_taken(api, d, ggml, m, n, k, tile):
    # shapes where one tile is the fastest of three by 5% to 30%, all of them faster than the fused tiles; also where the
    # caller asks for panels and leaves the tile open
    base = synth.matrix(ggml, 7, k, seed=781)
    w = qm(api, d, ggml, n, k, np.resize(base, base.size // 7 * n))
    xt = api.Tensor.from_f32(d, (m, k), api.DType.BF16, synth.activations(m, k, seed=782))
    out = api.Tensor.zeros(d, (m, n), api.DType.BF16)
    d.project_quantized(xt, w, out=out)
    assert d.get_tuning("last_decoded_tile") == tile
    first = out.raw()
    try:
        d.set_tuning("gemm_decoded_min_rows", m)
        d.project_quantized(xt, w, out=out)
        assert d.get_tuning("last_decoded_tile") == tile and np.array_equal(out.raw(), first)
        d.set_tuning("gemm_decoded_tile", 192 if tile == 256 else 256)
        d.project_quantized(xt, w, out=out)
        assert d.get_tuning("last_decoded_tile") == (192 if tile == 256 else 256) and np.array_equal(out.raw(), first)
        d.set_tuning("gemm_decoded_min_rows", 0)
        d.project_quantized(xt, w, out=out)
        assert d.get_tuning("last_decoded_tile") == 0
    finally:
        d.set_tuning("gemm_decoded_min_rows", 1)
        d.set_tuning("gemm_decoded_tile", 0)


@pytest.mark.parametrize("ggml,m,n,k", [(14, 768, 28672, 4096), (12, 1999, 5120, 17408), (8, 512, 17408, 5120),
                                         (13, 786, 144422, 256)])
def test_products_that_the_fused_tiles_run_faster_are_not_decoded(api, d, ggml, m, n, k):
    # us, fused / the best panel: 245 / 271, 352 / 403, 141 / 170, 178 / 222
    base = synth.matrix(ggml, 3, k, seed=787)
    w = qm(api, d, ggml, n, k, np.resize(base, base.size // 3 * n))
    xt = api.Tensor.from_f32(d, (m, k), api.DType.BF16, synth.activations(m, k, seed=788))
    d.project_quantized(xt, w, out=api.Tensor.zeros(d, (m, n), api.DType.BF16))
    assert d.get_tuning("last_decoded_tile") == 0


@pytest.mark.parametrize("ggml", [12, 13, 14, 23, 8], ids=["q4_k", "q5_k", "q6_k", "iq4_xs", "q8_0"])
@pytest.mark.parametrize("m,n,k", [(300, 512, 4096), (384, 512, 5120), (267, 580, 2816), (512, 256, 7168)])
def test_products_with_few_columns_stay_on_the_square_tiles(api, d, ggml, m, n, k):
    packed = synth.matrix(ggml, n, k, seed=783)
    w = qm(api, d, ggml, n, k, packed)
    x = oracle.round_storage(synth.activations(m, k, seed=784), oracle.F16).reshape(m, k)
    out = d.project_quantized(api.Tensor.from_f32(d, (m, k), api.DType.F16, x), w, out_dtype=api.DType.F32)
    assert out.operation.endswith("_gemm_mfma") and d.get_tuning("last_decoded_tile") == 0
    rows = np.unique(np.concatenate([np.arange(0, 20), np.arange(n - 20, n)]))
    assert_matmul_parity(out.tensor.to_f32()[:, rows], oracle_columns(ggml, packed, n, k, rows, x, weight_round=oracle.F16, accumulate="f64"),
                         "square tiles")


def test_the_switches_of_segments_and_panels_take_only_what_they_mean(api, d):
    for key, good, bad in (("gemm_wide32_segments", (0, 1, 8), (-1, 9, 1 << 32)),
                           ("gemm_decoded_min_rows", (0, 1, 2, 300, 2 ** 31 - 1), (-1, 2 ** 31, 1 << 32)),
                           ("gemm_decoded_tile", (0, 192, 256, 320), (-192, 100, 128, (1 << 32) + 192)),
                           ("gemm_decoded_segments", (0, 1, 2), (-1, 3, 1 << 32))):
        before = d.get_tuning(key)
        try:
            for value in good:
                d.set_tuning(key, value)
                assert d.get_tuning(key) == value
            for value in bad:
                with pytest.raises(Exception, match="out of range"):
                    d.set_tuning(key, value)
                assert d.get_tuning(key) == good[-1]
        finally:
            d.set_tuning(key, before)
    # a row count asked for is the line, also where the estimate would decode below it
    m, n, k = 1024, 12288, 4096
    base = synth.matrix(Q6_K, 3, k, seed=785)
    w = qm(api, d, Q6_K, n, k, np.resize(base, base.size // 3 * n))
    xt = api.Tensor.from_f32(d, (m, k), api.DType.F16, synth.activations(m, k, seed=786))
    out = api.Tensor.zeros(d, (m, n), api.DType.F16)
    taken = []
    try:
        for rows in (1, 1025, 1024):
            d.set_tuning("gemm_decoded_min_rows", rows)
            d.project_quantized(xt, w, out=out)
            taken.append(d.get_tuning("last_decoded_tile"))
    finally:
        d.set_tuning("gemm_decoded_min_rows", 1)
    assert taken == [192, 0, 192]


def test_decoded_panels_take_only_the_room_there_is(api):
    # 1100 x 70000 x 2048 is two panels of at most 256 MiB.  A new device that records has no room for one and takes the
    # fused tiles (f16 outputs of sums that may be of another order); once a plain call has made room, a recording decodes too.
    dev = api.Device.new()
    m, n, k = 1100, 70000, 2048
    tile = synth.matrix(Q6_K, 80, k, seed=771)
    w = qm(api, dev, Q6_K, n, k, np.tile(tile, n // 80))
    x = api.Tensor.from_f32(dev, (m, k), api.DType.F16, synth.activations(m, k, seed=772, f16=True))
    recorded = api.Tensor.zeros(dev, (m, n), api.DType.F16)
    dev.synchronize()
    held = dev.get_tuning("held_scratch_bytes")
    with dev.execution() as ex:
        dev.project_quantized(x, w, out=recorded)
    ex.graph.launch()
    dev.synchronize()
    assert dev.get_tuning("held_scratch_bytes") == held
    first = recorded.raw()
    direct = dev.project_quantized(x, w)
    assert 100 << 20 < dev.get_tuning("held_scratch_bytes") <= 257 << 20
    assert rel_l2(direct.tensor.to_f32(), recorded.to_f32()) <= 1e-4
    again = api.Tensor.zeros(dev, (m, n), api.DType.F16)
    with dev.execution() as decoded:
        dev.project_quantized(x, w, out=again)
    for _ in range(3):
        decoded.graph.launch()
        ex.graph.launch()
        dev.synchronize()
        assert np.array_equal(again.raw(), direct.tensor.raw()) and np.array_equal(recorded.raw(), first)
    got = direct.tensor.to_f32()
    assert np.array_equal(bits(got[:, :80]), bits(got[:, -80:])) and np.array_equal(bits(got[:, :80]), bits(got[:, 35200:35280]))
