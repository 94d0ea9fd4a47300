"""LayerNorm, Cast and MatMul: the oracle against the reference's own C files (CPU), and
the HIP operators against the oracle (GPU), including an FP16 chain through the graph
(Cast -> LayerNorm -> MatMul + bias -> Cast) that stays on the device.

Tolerances: FP32 <= 1e-4 absolute (LayerNorm outputs are O(1); MatMul sums are scaled so
the outputs are O(1)), FP16 <= 2e-2 with fp32 accumulation; Cast is exact.
"""

import ctypes

import numpy as np
import pytest

import oracle as O
from helpers import dev, gemm_plan, max_abs

TOL32, TOL16 = 1e-4, 2e-2
needs_ref = pytest.mark.skipif(not O.ref_available(), reason="reference build not available")


def _ln_inputs(N, D, seed):
    x = O.normal((N, D), seed)
    g = O.normal((D,), seed + 1, 1.0, 0.1)
    b = O.normal((D,), seed + 2, 0.0, 0.1)
    return x, g, b


# --------------------------------------------------------------------- plans (CPU) ---

@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("M", [1, 16, 300])
def test_very_wide_products_keep_64_bit_indexing(native, M, f16):
    """The DMA products step over W (K, N) by 32 or 64 rows in 32 bits, which wraps from 2^25
    columns on (a step of 0 there in FP32): such a product, alone or as one of the three side
    by side, keeps the kernels that index in 64 bits.  W (N, K) steps along k and is not meant."""
    wide = 1 << 25
    assert gemm_plan(native, M, wide - 64, 64, f16)[0] > 0
    for n in (wide, wide + 64, 1 << 26, (1 << 31) - 64):
        plan, _, mix_ok = gemm_plan(native, M, n, 64, f16)
        assert plan == -1 and not mix_ok
    if f16:
        assert gemm_plan(native, M, [64, wide, 64], 64, f16)[0] == -1
    assert gemm_plan(native, M, wide, 64, f16, nk=True)[0] > 0


# ------------------------------------------------------------------ oracle (CPU) ---

@needs_ref
@pytest.mark.parametrize("N,D", [(33, 768), (5, 1000), (2, 1), (3, 4098)])
def test_oracle_layernorm_matches_reference_build(N, D):
    x, g, b = _ln_inputs(N, D, N + D)
    assert np.array_equal(O.layernorm(x, g, b, 1e-5), O.layernorm(x, g, b, 1e-5, use_ref=True))


def test_oracle_layernorm_constant_rows_give_beta():
    x = np.full((3, 64), 2.5, np.float32)
    g = O.normal((64,), 5)
    b = O.normal((64,), 6)
    assert np.array_equal(O.layernorm(x, g, b), np.broadcast_to(b, x.shape))


@needs_ref
@pytest.mark.parametrize("ta,tb,batch,bias", [(False, False, 1, True), (True, False, 1, False), (False, True, 3, True),
                                              (True, True, 2, True)])
def test_oracle_matmul_matches_reference_build(ta, tb, batch, bias):
    M, N, K = 7, 5, 9
    A = O.normal((batch, M * K), 1)
    B = O.normal((batch, K * N), 2)
    bb = O.normal((N,), 3) if bias else None
    kw = dict(transpose_a=ta, transpose_b=tb, batch=batch, stride_a=M * K, stride_b=K * N, stride_c=M * N)
    assert np.array_equal(O.matmul(A, B, bb, M, N, K, **kw), O.matmul(A, B, bb, M, N, K, use_ref=True, **kw))


def test_oracle_matmul_identity():
    A = O.normal((6, 6), 4)
    assert np.array_equal(O.matmul(A, np.eye(6, dtype=np.float32), None, 6, 6, 6).reshape(6, 6), A)


@needs_ref
def test_reference_cast_agrees_with_ieee_where_its_cuda_op_does():
    """cast.c's FLOAT16 -> FLOAT and INT64 <-> FLOAT match IEEE conversions (numpy); its
    FLOAT -> FLOAT16 truncates (cast.c:8-16), which only agrees with the CUDA op's
    round-to-nearest on exactly representable values."""
    h = O.to_f16(O.normal((1000,), 7))
    assert np.array_equal(O.cast_ref(h, O.ONNX_FLOAT16, O.ONNX_FLOAT), h.astype(np.float32))
    i = np.arange(-500, 500, dtype=np.int64) * 12345
    assert np.array_equal(O.cast_ref(i, O.ONNX_INT64, O.ONNX_FLOAT), i.astype(np.float32))
    f = O.normal((1000,), 8) * 1000
    assert np.array_equal(O.cast_ref(f, O.ONNX_FLOAT, O.ONNX_INT64), f.astype(np.int64))
    exact = h.astype(np.float32)
    assert np.array_equal(O.cast_ref(exact, O.ONNX_FLOAT, O.ONNX_FLOAT16), h)


# ------------------------------------------------------------------ HIP (GPU) ---

def _ln_gpu(x, g, b, eps, f16, in_place=False):
    import cudaforge_amd as cf
    N, D = x.shape
    bx, bg, bb = dev(x, f16), dev(g, f16), dev(b, f16)
    out = bx if in_place else cf.DeviceBuffer.empty(x.shape, np.float16 if f16 else np.float32)
    p = O.LayerNormParams(N, D, eps)
    assert cf.call_op("layernorm_f16_cuda" if f16 else "layernorm_f32_cuda", [bx, bg, bb], [out], p) == 0
    return out.download().astype(np.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("N,D,eps", [(4096, 768, 1e-12), (7, 1000, 1e-5), (3, 4098, 1e-5), (2, 8192, 1e-5),
                                     (5, 64, 1e-5)])
def test_layernorm_f32_cuda(gpu, N, D, eps):
    x, g, b = _ln_inputs(N, D, N * 7 + D)
    assert max_abs(O.layernorm(x, g, b, eps), _ln_gpu(x, g, b, eps, False)) <= TOL32


@pytest.mark.gpu
@pytest.mark.parametrize("N,D", [(4096, 768), (9, 1024), (3, 4098)])
def test_layernorm_f16_cuda(gpu, N, D):
    x, g, b = (O.round_f16(a) for a in _ln_inputs(N, D, N + 3 * D))
    want = O.layernorm(x, g, b, 1e-5)
    assert max_abs(want, _ln_gpu(x, g, b, 1e-5, True)) <= TOL16
    assert max_abs(want, _ln_gpu(x, g, b, 1e-5, True, in_place=True)) <= TOL16


@pytest.mark.gpu
@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("N", [3, 700])
@pytest.mark.parametrize("D", [4, 256, 260, 772, 1028, 1536, 2052, 4096, 4100, 8192, 8196])
def test_layernorm_row_widths(gpu, f16, N, D):
    """Each count of 4-element groups per lane, full and cut short, with one wave and four
    waves per row (few and many rows), in place."""
    x, g, b = _ln_inputs(N, D, N + 3 * D)
    if f16:
        x, g, b = (O.round_f16(a) for a in (x, g, b))
    got = _ln_gpu(x, g, b, 1e-5, f16, in_place=True)
    assert max_abs(O.layernorm(x, g, b, 1e-5), got) <= (TOL16 if f16 else TOL32)


@pytest.mark.gpu
@pytest.mark.parametrize("N", [65535, 65536, 65537, 131075])
def test_layernorm_many_long_rows(gpu, native, N):
    """Rows that a whole workgroup takes, more of them than the grid has along x: the first,
    the last and those around its end against the oracle, in place, and nothing written behind."""
    import cudaforge_amd as cf
    D = 2052
    x = cf.DeviceBuffer.normal((N + 1, D), np.float16, 17)
    g, b = O.round_f16(O.normal((D,), 18, 1.0, 0.1)), O.round_f16(O.normal((D,), 19, 0.0, 0.1))
    before = x.download()
    assert cf.call_op("layernorm_f16_cuda", [x, dev(g, True), dev(b, True)], [x], cf.LayerNormParams(N, D, 1e-5)) == 0
    after = x.download()
    rows = sorted({0, 1, 65534, N - 2, N - 1} | ({65535, 65536} & set(range(N))))
    want = O.layernorm(before[rows].astype(np.float32), g, b, 1e-5)
    assert max_abs(want, after[rows].astype(np.float32)) <= TOL16
    assert np.array_equal(after[N], before[N])
    assert np.all(after[:N].std(axis=1, dtype=np.float32) > 0.5)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 7, 2047, 2048, 2049, 6151])
@pytest.mark.parametrize("skew_in,skew_out", [(0, 0), (1, 0), (0, 1), (1, 1), (3, 5)])
def test_cast_f16_misaligned(gpu, native, n, skew_in, skew_out):
    """f32 <-> f16 with either end off its 16-byte alignment, around the 2048 elements of a
    workgroup: nearest even and exact, and nothing written past the n elements."""
    import cudaforge_amd as cf
    x = O.normal((n + 8,), n, 0.0, 3.0)
    x[::5] *= np.float32(1e-6)                                 # subnormal halves
    for src, dst, a, b in ((O.ONNX_FLOAT, O.ONNX_FLOAT16, x, np.full(n + 16, 7.0, np.float16)),
                           (O.ONNX_FLOAT16, O.ONNX_FLOAT, x.astype(np.float16), np.full(n + 16, 7.0, np.float32))):
        A, B = cf.DeviceBuffer.from_numpy(a), cf.DeviceBuffer.from_numpy(b)
        ins = (ctypes.c_void_p * 1)(A.ptr + skew_in * a.itemsize)
        outs = (ctypes.c_void_p * 1)(B.ptr + skew_out * b.itemsize)
        p = O.CastParams(src, dst, n)
        assert cf.find_op("cast_f32_cuda").func(ctypes.cast(ins, ctypes.POINTER(ctypes.c_void_p)),
                                                ctypes.cast(outs, ctypes.POINTER(ctypes.c_void_p)),
                                                ctypes.cast(ctypes.pointer(p), ctypes.c_void_p), None) == 0
        want = b.copy()
        want[skew_out:skew_out + n] = a[skew_in:skew_in + n].astype(b.dtype)
        assert np.array_equal(B.download(), want)


@pytest.mark.gpu
def test_cast_f32_cuda_all_pairs(gpu):
    import cudaforge_amd as cf

    def run(arr, src, dst, out_dtype):
        i = cf.DeviceBuffer.from_numpy(np.ascontiguousarray(arr))
        o = cf.DeviceBuffer.empty(arr.shape, out_dtype)
        assert cf.call_op("cast_f32_cuda", [i], [o], O.CastParams(src, dst, arr.size)) == 0
        return o.download()

    f = np.concatenate([O.normal((5000,), 9) * 100, np.float32([0.0, -0.0, 1e-7, -3e-6, 65504.0, 70000.0, 6.1e-5])])
    with np.errstate(over="ignore"):                                         # 70000 -> inf on purpose
        want16 = f.astype(np.float16).view(np.uint16)
    assert np.array_equal(run(f, O.ONNX_FLOAT, O.ONNX_FLOAT16, np.float16).view(np.uint16),
                          want16)                                            # RNE, subnormals, overflow
    h = O.to_f16(O.normal((5000,), 10))
    assert np.array_equal(run(h, O.ONNX_FLOAT16, O.ONNX_FLOAT, np.float32), h.astype(np.float32))
    i = (np.arange(-2500, 2500, dtype=np.int64) * 987654321)
    assert np.array_equal(run(i, O.ONNX_INT64, O.ONNX_FLOAT, np.float32), i.astype(np.float32))
    g = O.normal((5000,), 11) * 1e6
    assert np.array_equal(run(g, O.ONNX_FLOAT, O.ONNX_INT64, np.int64), g.astype(np.int64))
    assert np.array_equal(run(g, O.ONNX_FLOAT, O.ONNX_FLOAT, np.float32), g)    # other pairs copy


def _mm_gpu(A, B, bias, M, N, K, f16, **kw):
    import cudaforge_amd as cf
    dt = np.float16 if f16 else np.float32
    batch = kw.get("batch", 1)
    C = cf.DeviceBuffer.empty(((batch - 1) * kw.get("stride_c", 0) + M * N,), dt)
    p = O.MatmulParams(M, N, K, kw.get("transpose_a", False), kw.get("transpose_b", False), batch,
                       kw.get("stride_a", 0), kw.get("stride_b", 0), kw.get("stride_c", 0), 0)
    slots = [dev(A, f16), dev(B, f16), None if bias is None else dev(bias, f16)]
    name = "matmul_f16_cuda" if f16 else "matmul_f32_cuda"
    assert cf.call_op(name, slots, [C], p) == 0
    return C.download().astype(np.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("M,N,K", [(33, 70, 17), (128, 256, 64), (256, 3072, 768)])
def test_matmul_cuda(gpu, f16, M, N, K):
    r = O.round_f16 if f16 else (lambda a: a)
    A = r(O.normal((M, K), M + N))
    B = r(O.normal((K, N), K + 1, 0.0, 1.0 / np.sqrt(K)))
    bias = r(O.normal((N,), 5, 0.0, 0.1))
    want = A.astype(np.float64) @ B.astype(np.float64) + bias
    if M * N * K <= 1 << 20:
        want = O.matmul(A, B, bias, M, N, K).reshape(M, N)
    got = _mm_gpu(A, B, bias, M, N, K, f16).reshape(M, N)
    assert max_abs(want, got) <= (TOL16 if f16 else TOL32)


@pytest.mark.gpu
@pytest.mark.parametrize("bm,bn", [(256, 48), (128, 96), (64, 64), (64, 128)])
@pytest.mark.parametrize("M,N,K", [(1, 8, 64), (65, 200, 128), (129, 72, 192), (300, 328, 64)])
def test_matmul_f16_tile_ends(gpu, native, bm, bn, M, N, K):
    """The wave-specialised GEMM with its last row and column tiles cut short: values at the
    ends and nothing written past the M x N result."""
    import cudaforge_amd as cf
    A = O.round_f16(O.normal((M, K), M + N))
    B = O.round_f16(O.normal((K, N), K + 1, 0.0, 1.0 / np.sqrt(K)))
    bias = O.round_f16(O.normal((N,), 5, 0.0, 0.1))
    want = A.astype(np.float64) @ B.astype(np.float64) + bias
    guard = 1024
    C = cf.DeviceBuffer.from_numpy(np.full(M * N + guard, 7.0, np.float16))
    try:
        native.cf_gemm_set_ws_shape(bm, bn)
        p = cf.MatmulParams(M, N, K, False, False, 1, 0, 0, 0, 0)
        assert cf.call_op("matmul_f16_cuda", [dev(A, True), dev(B, True), dev(bias, True)], [C], p) == 0
        got = C.download().astype(np.float32)
    finally:
        native.cf_gemm_set_ws_shape(0, 0)
    assert max_abs(want, got[:M * N].reshape(M, N)) <= TOL16
    assert np.all(got[M * N:] == 7.0)


@pytest.mark.gpu
@pytest.mark.parametrize("nk", [False, True])
@pytest.mark.parametrize("M,N,K,bm,bn,ks", [
    (1, 72, 1024, 64, 64, 8), (16, 200, 1088, 64, 128, 3), (65, 64, 640, 64, 64, 5), (130, 328, 512, 128, 96, 2),
    (17, 136, 4096, 64, 64, 16), (300, 264, 192, 256, 64, 1), (130, 72, 192, 64, 128, 1)])
def test_matmul_f16_k_ranges(gpu, native, nk, M, N, K, bm, bn, ks):
    """Split sums over ranges of k (uneven last ranges, cut row and column tiles) and W
    given as (N, K), forced tile by tile, against float64 and, without a forced tile, for
    the cost model's choice; nothing written past the result."""
    import cudaforge_amd as cf
    A = O.round_f16(O.normal((M, K), M + N))
    B = O.round_f16(O.normal((K, N), K + 1, 0.0, 1.0 / np.sqrt(K)))
    bias = O.round_f16(O.normal((N,), 5, 0.0, 0.1))
    want = A.astype(np.float64) @ B.astype(np.float64) + bias
    p = cf.MatmulParams(M, N, K, False, nk, 1, 0, 0, 0, 0)
    for force in (True, False):
        C = cf.DeviceBuffer.from_numpy(np.full(M * N + 1024, 7.0, np.float16))
        try:
            if force:
                native.cf_gemm_set_ws_shape(bm, bn)
                native.cf_gemm_set_ws_ksplit(ks)
            assert cf.call_op("matmul_f16_cuda", [dev(A, True), dev(B.T if nk else B, True), dev(bias, True)], [C], p) == 0
            got = C.download().astype(np.float32)
        finally:
            native.cf_gemm_set_ws_shape(0, 0)
            native.cf_gemm_set_ws_ksplit(0)
        assert max_abs(want, got[:M * N].reshape(M, N)) <= 4e-3      # one fp16 rounding of values below 8
        assert np.all(got[M * N:] == 7.0)


def _mm_f32_run(native, A, B, bias, nk, kernel, bm, bn, ks):
    """One FP32 product, forced onto "x3" (bf16 MFMA on split operands) or "f32" (the few-row
    fp32 MFMA kernel) at a tile and number of k ranges; nothing may be written past it."""
    import cudaforge_amd as cf
    (M, K), N = A.shape, B.shape[1]
    C = cf.DeviceBuffer.from_numpy(np.full(M * N + 1024, 7.0, np.float32))
    p = cf.MatmulParams(M, N, K, False, nk, 1, 0, 0, 0, 0)
    try:
        if kernel == "x3":
            native.cf_gemm_set_x3(2, bm, bn, ks)
        elif kernel == "f32":
            native.cf_gemm_set_x3(1, 0, 0, 0)
            native.cf_gemm_set_f32(0, bm, bn, ks)
        elif kernel == "general":
            native.cf_gemm_set_x3(1, 0, 0, 0)
            native.cf_gemm_set_f32(1, 0, 0, 0)
        slots = [dev(A), dev(B.T if nk else B), None if bias is None else dev(bias)]
        assert cf.call_op("matmul_f32_cuda", slots, [C], p) == 0
        got = C.download()
    finally:
        native.cf_gemm_set_x3(0, 0, 0, 0)
        native.cf_gemm_set_f32(0, 0, 0, 0)
    assert np.all(got[M * N:] == 7.0)
    return got[:M * N].reshape(M, N)


X3_TILES = [(256, 160), (256, 144), (256, 128), (256, 96), (256, 64), (128, 192), (128, 128), (128, 96), (128, 64),
            (64, 64)]
F32_TILES = [(16, 64), (32, 64), (64, 64), (32, 32), (128, 64), (16, 128)]


@pytest.mark.gpu
@pytest.mark.parametrize("nk", [False, True])
@pytest.mark.parametrize("kernel,bm,bn", [("x3", *t) for t in X3_TILES] + [("f32", *t) for t in F32_TILES])
def test_matmul_f32_tiles(gpu, native, nk, kernel, bm, bn):
    """Each FP32 tile with its last rows and columns cut, one and several ranges of k (the
    last one shorter), W in both layouts, against float64.  Bound per element: K products rounded
    once per step at most, by 2^-24 of |a b| and of the sum so far, independently of one another:
    sqrt(K) * 2^-24 * sum |a b|, ten times what is seen."""
    for M, N, K, ks in ((1, 16, 32, 1), (130, 208, 352, 1), (277, 176, 3104, 3), (64, 64, 4096, 4)):
        A, B = O.normal((M, K), M + N), O.normal((K, N), K + 1, 0.0, 1.0 / np.sqrt(K))
        bias = O.normal((N,), 5, 0.0, 0.1)
        want = A.astype(np.float64) @ B.astype(np.float64) + bias
        bound = np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64) * (K ** 0.5 * 2.0 ** -24) + 2.0 ** -22
        got = _mm_f32_run(native, A, B, bias, nk, kernel, bm, bn, ks)
        assert np.all(np.abs(got - want) <= bound)


@pytest.mark.gpu
def test_matmul_f32_split_operands_keep_precision_and_range(gpu, native):
    """The bf16-MFMA product is no further from float64 than the general fp32 kernel, also
    for operands spread over 40 binary orders, at the largest and smallest exponents and
    with exact cancellation; infinities and NaN give what the fp32 kernel gives."""
    rng = np.random.default_rng(3)

    def err(y, want):
        return float(np.linalg.norm(y - want) / np.linalg.norm(want))

    M, N, K = 320, 192, 768
    a, b = rng.standard_normal((M, K)).astype(np.float32), rng.standard_normal((K, N)).astype(np.float32)
    # A running sum of one sign, long enough for a bias of the accumulation to show.
    long_a, long_b = rng.standard_normal((M, 4096)).astype(np.float32), rng.standard_normal((4096, N)).astype(np.float32)
    spread = np.exp2(rng.integers(-20, 20, (M, K))).astype(np.float32)
    for A, B in ((a, b), (np.abs(a), np.abs(b)), (a * spread, b), (a * np.float32(2.0 ** 100), b * np.float32(2.0 ** -90)),
                 (a * np.float32(1e-30), b * np.float32(1e-4)), (np.concatenate([a, -a], 1), np.concatenate([b, b], 0)),
                 (np.abs(long_a), np.abs(long_b))):
        want = A.astype(np.float64) @ B.astype(np.float64)
        x3 = _mm_f32_run(native, A, B, None, False, "x3", 0, 0, 0)
        if not want.any():
            assert np.abs(x3).max() <= 1e-3                    # the cancelled sums' rounding
            continue
        assert err(x3, want) <= max(1.2 * err(_mm_f32_run(native, A, B, None, False, "general", 0, 0, 0), want), 2e-7)
    A, B = a.copy(), b.copy()
    A[5, 7], A[300, 100], B[3, 9] = np.inf, np.nan, -np.inf
    for nk in (False, True):
        x3, ref = (_mm_f32_run(native, A, B, None, nk, k, 0, 0, 0) for k in ("x3", "general"))
        assert np.array_equal(np.isnan(x3), np.isnan(ref)) and np.array_equal(np.isinf(x3), np.isinf(ref))
        ok = np.isfinite(ref)
        assert np.array_equal(np.sign(x3[np.isinf(ref)]), np.sign(ref[np.isinf(ref)]))
        assert max_abs(x3[ok], ref[ok]) <= 1e-3
    # The next call is finite again.
    assert err(_mm_f32_run(native, a, b, None, False, "x3", 0, 0, 0), a.astype(np.float64) @ b.astype(np.float64)) <= 1e-6


@pytest.mark.gpu
def test_matmul_f32_split_operands_single_products(gpu, native):
    """FP32 products on split operands, element by element against float64, with one term per
    sum (a diagonal A): random ones, the mantissas whose dropped terms are largest, and results
    at the end of the finite numbers whose rounded first parts multiply to more than that.
    Bound: h and m are the nearest of 8 bits, so |m| <= 2^-8 |x| and |l| <= 2^-17 |x|, and the three
    dropped terms are below 2 * 2^-25 + 2^-34 of |a b|; the MFMAs cut their sums at 2^-23, of |a b|
    the last, of 2^-8 |a b| and less the others."""
    rng = np.random.default_rng(8)
    n = 512
    one = 1 + 2.0 ** -7 - 2.0 ** -23                           # all bits after the first seven zeros
    tie = 1 + 2.0 ** -8 + 2.0 ** -17 + 2.0 ** -23                # h and m next to ties
    for d, B in ((rng.standard_normal(n), rng.standard_normal((n, 64)) * 0.02), (np.full(n, one), np.full((n, 64), one)),
                 (np.full(n, tie), np.full((n, 64), tie)), (np.full(n, 3.4e38), rng.uniform(-1, 1, (n, 64))),
                 (np.full(n, 2.0 ** 65 * (1 - 2.0 ** -24)), np.full((n, 64), 2.0 ** 63 * (1 - 2.0 ** -10)))):
        A, B = np.diag(d.astype(np.float32)), B.astype(np.float32)
        want = A.astype(np.float64) @ B.astype(np.float64)
        got = _mm_f32_run(native, A, B, None, False, "x3", 64, 64, 0)
        assert np.all(np.abs(got - want) <= np.abs(want) * (2.0 ** -24 + 2.0 ** -34 + 1.01 * 2.0 ** -23))


@pytest.mark.gpu
@pytest.mark.parametrize("ks", [1, 3])
def test_matmul_f32_split_operands_have_no_bias(gpu, native, ks):
    """The mean error of the FP32 product on split operands: sums of one sign are off by no
    more than 2^-26 on average (cut instead of rounded parts lose 2^-24.6, all the same way), and
    the columns' means of sums of both signs, where a bias of the matrix core's sums would
    stay while the elements' own errors average out, by no more than the fp32 kernel's.  An even
    and an odd number of stages, and ranges of k of which the last is shorter."""
    rng = np.random.default_rng(9)
    for K in (768, 800):
        A, B = rng.uniform(1, 2, (256, K)).astype(np.float32), rng.uniform(1, 2, (K, 64)).astype(np.float32)
        want = A.astype(np.float64) @ B.astype(np.float64)
        assert abs(((_mm_f32_run(native, A, B, None, False, "x3", 64, 64, ks) - want) / want).mean()) <= 2.0 ** -26
        A, B = rng.standard_normal((4096, K)).astype(np.float32), rng.standard_normal((K, 64)).astype(np.float32)
        want = A.astype(np.float64) @ B.astype(np.float64)
        x3, general = (np.linalg.norm((_mm_f32_run(native, A, B, None, False, k, 64, 64, ks) - want).mean(0))
                       for k in ("x3", "general"))
        assert x3 <= general


@pytest.mark.gpu
@pytest.mark.parametrize("nk", [False, True])
def test_matmul_f32_split_operands_very_small_numbers(gpu, native, nk):
    """FP32 products on split operands whose parts would be subnormal (the bf16 MFMA takes those
    as zero): operands down to the smallest normal numbers, on either side, in some rows only
    and beside zeros and ordinary numbers.  Bound per element: each of the K products rounded
    once per step (test_matmul_f32_tiles), and beside a number of 2^-95 or more what is lost is
    below 2^-126 per element; subnormal operands give what the general kernel gives."""
    rng = np.random.default_rng(10)
    M, N, K = 80, 64, 96
    a, b = rng.standard_normal((M, K)), rng.standard_normal((K, N))
    tiny, some = np.ones((M, 1)), a.copy()
    tiny[10:30] = 1e-37
    some[:, 1:] *= 1e-37
    sparse = np.where(rng.random((M, K)) < 0.1, a * 1e-36, 0.0)
    for A, B in ((a * 1e-37, b * 1e5), (a * 1e5, b * 1e-37), (a * tiny, b * 1e5), (a * 1e-32, b * 1e-3),
                 (sparse, b * 1e5), (some, b), (a * 2.0 ** -90, b), (a * 2.0 ** -94, b), (a * 2.0 ** -100, b)):
        A, B = A.astype(np.float32), B.astype(np.float32)
        want = A.astype(np.float64) @ B.astype(np.float64)
        bound = np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64) * (K ** 0.5 * 2.0 ** -24) + 2.0 ** -126 * K
        got = _mm_f32_run(native, A, B, None, nk, "x3", 64, 64, 1)
        assert np.all(np.abs(got - want) <= np.where(np.abs(want) < 1e-20, bound - 2.0 ** -126 * K, bound))
    A = (a * 1e-40).astype(np.float32)
    x3, general = (_mm_f32_run(native, A, (b * 1e8).astype(np.float32), None, nk, k, 64, 64, 1) for k in ("x3", "general"))
    assert np.array_equal(x3, general)


@pytest.mark.gpu
@pytest.mark.parametrize("bm,bn,ks", [(64, 64, 1), (256, 144, 1), (128, 64, 3)])
def test_matmul_f32_non_finite_operands_stay_where_they_are(gpu, native, bm, bn, ks):
    """FP32 products on split operands: an infinity in one row changes the results' path in
    the tiles of that row only (rows of other tiles keep the bits of the finite product), and
    leaves nothing behind in a recording, whose next replay with finite operands has the bits
    it had before."""
    import cudaforge_amd as cf
    M, N, K = 512, 288, 768
    A, B = O.normal((M, K), 11), O.normal((K, N), 12, 0.0, 1.0 / np.sqrt(K))
    bad = A.copy()
    bad[3, 5], bad[3, 6], bad[7, 40] = np.inf, -np.inf, np.nan
    clean = _mm_f32_run(native, A, B, None, False, "x3", bm, bn, ks)
    got = _mm_f32_run(native, bad, B, None, False, "x3", bm, bn, ks)
    assert np.array_equal(got[256:], clean[256:])
    assert not np.isfinite(got[3]).any() and np.isnan(got[7]).all()
    rest = np.setdiff1d(np.arange(256), [3, 7])
    assert max_abs(got[rest], clean[rest]) <= 1e-5
    dA, dB, C = dev(A), dev(B), cf.DeviceBuffer.empty((M, N), np.float32)
    p, st, ex = cf.MatmulParams(M, N, K, False, False, 1, 0, 0, 0, 0), cf.Stream(), ctypes.c_void_p()
    try:
        native.cf_gemm_set_x3(2, bm, bn, ks)
        assert cf.call_op("matmul_f32_cuda", [dA, dB, None], [C], p, st) == 0        # the workspace
        st.synchronize()
        assert native.gpu_capture_begin(st.handle) == 0
        rc = cf.call_op("matmul_f32_cuda", [dA, dB, None], [C], p, st)
        assert native.gpu_capture_end(st.handle, ctypes.byref(ex)) == 0 and rc == 0
        for a, want in ((A, clean), (bad, got), (A, clean), (A, clean)):
            dA.upload(a, st)
            assert native.gpu_graph_launch(ex, st.handle) == 0
            assert np.array_equal(C.download(st), want, equal_nan=True)
    finally:
        native.cf_gemm_set_x3(0, 0, 0, 0)
        st.synchronize()
        if ex:
            native.gpu_graph_exec_destroy(ex)


@pytest.mark.gpu
@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("ta,tb", [(True, False), (False, True), (True, True)])
def test_matmul_cuda_transposed_batched(gpu, f16, ta, tb):
    r = O.round_f16 if f16 else (lambda a: a)
    M, N, K, batch = 40, 72, 48, 3
    sa, sb, sc = M * K + 5, K * N + 3, M * N + 7          # padded slices: strides are honoured
    A = r(O.normal(((batch - 1) * sa + M * K,), 21))
    B = r(O.normal(((batch - 1) * sb + K * N,), 22, 0.0, 0.2))
    bias = r(O.normal((N,), 23))
    kw = dict(transpose_a=ta, transpose_b=tb, batch=batch, stride_a=sa, stride_b=sb, stride_c=sc)
    want = O.matmul(A, B, bias, M, N, K, **kw)
    got = _mm_gpu(A, B, bias, M, N, K, f16, **kw)
    for bi in range(batch):
        sl = slice(bi * sc, bi * sc + M * N)
        assert max_abs(want[sl], got[sl]) <= (TOL16 if f16 else TOL32)


@pytest.mark.gpu
def test_fp16_layer_chain_through_the_graph(gpu, native):
    """X (F32) -> Cast -> F16 -> LayerNorm -> MatMul (+ bias, slot 2) -> Cast -> F32, every
    node resolved to a HIP operator by the graph's name rule and run on the device."""
    from helpers import DT_F16, DT_F32, OP_INPUT, OP_OUTPUT, Graph
    OP_MATMUL, OP_LAYERNORM, OP_CAST = 3, 21, 26
    S, D, F = 64, 256, 512
    x = O.normal((S, D), 31)
    g16, b16 = O.to_f16(O.normal((D,), 32, 1.0, 0.1)), O.to_f16(O.normal((D,), 33, 0.0, 0.1))
    W16 = O.to_f16(O.normal((D, F), 34, 0.0, 1.0 / np.sqrt(D)))
    bias16 = O.to_f16(O.normal((F,), 35, 0.0, 0.1))
    gr = Graph(native)
    try:
        tX, iX = gr.tensor(x)
        _, iXh = gr.tensor(np.zeros((S, D), np.float16), DT_F16)
        _, iL = gr.tensor(np.zeros((S, D), np.float16), DT_F16)
        _, iM = gr.tensor(np.zeros((S, F), np.float16), DT_F16)
        tY, iY = gr.tensor(np.zeros((S, F), np.float32))
        tg = gr.tensor(g16, DT_F16)[0]
        tb = gr.tensor(b16, DT_F16)[0]
        tW = gr.tensor(W16, DT_F16)[0]
        tbias = gr.tensor(bias16, DT_F16)[0]
        names = []
        buf = ctypes.create_string_buffer(64)
        n1 = gr.node(OP_CAST, [iX], [iXh], (), O.CastParams(O.ONNX_FLOAT, O.ONNX_FLOAT16, S * D))
        n2 = gr.node(OP_LAYERNORM, [iXh], [iL], (tg, tb), O.LayerNormParams(S, D, 1e-5))
        n3 = gr.node(OP_MATMUL, [iL], [iM], (tW, tbias), O.MatmulParams(S, F, D, False, False, 1, 0, 0, 0, 0))
        n4 = gr.node(OP_CAST, [iM], [iY], (), O.CastParams(O.ONNX_FLOAT16, O.ONNX_FLOAT, S * F))
        native.graph_set_input(gr.g, gr.node(OP_INPUT, [], [iX]))
        native.graph_set_output(gr.g, gr.node(OP_OUTPUT, [iY], []))
        assert native.graph_build(gr.g) == 0
        for n in (n1, n2, n3, n4):
            assert native.graph_resolve_op(gr.g, n, True, buf, 64)
            names.append(buf.value)
        assert names == [b"cast_f32_cuda", b"layernorm_f16_cuda", b"matmul_f16_cuda", b"cast_f32_cuda"]
        ins, outs = (ctypes.c_void_p * 1)(tX), (ctypes.c_void_p * 1)(tY)
        assert native.graph_execute(gr.g, ins, outs, True) == 0
        got = gr.read(tY, (S, F))
        xh = O.round_f16(x)
        ln = O.round_f16(O.layernorm(xh, g16.astype(np.float32), b16.astype(np.float32), 1e-5))
        want = O.matmul(ln, W16.astype(np.float32), bias16.astype(np.float32), S, F, D).reshape(S, F)
        assert max_abs(want, got) <= TOL16
    finally:
        gr.destroy()


@pytest.mark.gpu
@pytest.mark.parametrize("f16,M,N,K", [(True, 16, 768, 3072), (False, 16, 768, 4096), (False, 512, 2304, 768)])
def test_matmul_in_a_callers_own_recording_holds_the_callers_pointers(gpu, native, f16, M, N, K):
    """A MatMul without transposes captured by the caller through HIP itself, with a workspace
    there that its plan would use: one launch, of the caller's buffers only (with partial sums
    or split operands in the workspace there are two and more), so growing the workspace cannot
    take anything from under the recording.  A capture through gpu_capture_begin, whose caller
    watches the buffer generation, uses the workspace as an eager call does."""
    import cudaforge_amd as cf
    hip = ctypes.CDLL("libamdhip64.so")
    r = O.round_f16 if f16 else (lambda a: a)
    A, B = r(O.normal((M, K), M + N)), r(O.normal((K, N), K + 1, 0.0, 1.0 / np.sqrt(K)))
    want = A.astype(np.float64) @ B.astype(np.float64)
    ins, C = [dev(A, f16), dev(B, f16), None], cf.DeviceBuffer.empty((M, N), np.float16 if f16 else np.float32)
    p, st = cf.MatmulParams(M, N, K, False, False, 1, 0, 0, 0, 0), cf.Stream()
    name, tol = ("matmul_f16_cuda", TOL16) if f16 else ("matmul_f32_cuda", 1e-4)
    assert cf.call_op(name, ins, [C], p, st) == 0              # the workspace
    st.synchronize()
    assert native.gpu_workspace_size() > 0
    handle, graph, ex, n = st.handle, ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_size_t()
    assert hip.hipStreamBeginCapture(handle, 1) == 0           # thread-local mode
    rc = cf.call_op(name, ins, [C], p, st)
    assert hip.hipStreamEndCapture(handle, ctypes.byref(graph)) == 0 and rc == 0
    assert hip.hipGraphGetNodes(graph, None, ctypes.byref(n)) == 0 and n.value == 1
    assert hip.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, ctypes.c_size_t(0)) == 0
    for _ in range(3):
        C.fill_zero()
        native.gpu_device_synchronize()
        assert hip.hipGraphLaunch(ex, handle) == 0
        assert max_abs(want, C.download(st).astype(np.float64)) <= tol
    hip.hipGraphExecDestroy(ex)
    hip.hipGraphDestroy(graph)
    assert native.gpu_capture_begin(st.handle) == 0
    assert native.gpu_capture_foreign(handle) == 0
    assert native.gpu_capture_end(st.handle, ctypes.byref(ex)) == 0
    native.gpu_graph_exec_destroy(ex)


@pytest.mark.gpu
def test_workspace_request_of_all_it_holds_inside_a_recording(gpu, native):
    """A buffer grown by a quarter, asked for down to its last byte and for one byte more while
    its stream is captured: the first is given as it is, the second refused, and neither frees
    anything (the buffer generation stays) or breaks the recording."""
    import cudaforge_amd as cf
    native.gpu_buffer_generation.restype = ctypes.c_uint64
    st, ex = cf.Stream(), ctypes.c_void_p()
    native.gpu_device_synchronize()
    native.gpu_workspace_release()
    base = native.gpu_workspace_get_stream(st.handle, (64 << 20) + 257)
    held, gen = native.gpu_workspace_size(), native.gpu_buffer_generation()
    assert base and held > 64 << 20
    assert native.gpu_capture_begin(st.handle) == 0
    got = [native.gpu_workspace_try_stream(st.handle, held + more) for more in (-1, 0, 1)]
    assert native.gpu_capture_end(st.handle, ctypes.byref(ex)) == 0
    native.gpu_graph_exec_destroy(ex)
    assert got == [base, base, None]
    assert (native.gpu_workspace_size(), native.gpu_buffer_generation()) == (held, gen)


@pytest.mark.gpu
def test_workspace_stays_where_optional_scratch_finds_no_memory(gpu, native):
    """An operator with a buffer of its own (the FP32 prefill) whose products could use more
    than memory allows, call after call: the buffer it has stays, so nothing is freed and
    recordings stay valid (the buffer generation), and the result is that of the products that
    need no scratch."""
    import cudaforge_amd as cf
    from helpers import FusedCase
    native.gpu_buffer_generation.restype = ctypes.c_uint64
    B, S, D = 8, 512, 768
    c = FusedCase(B, S, 12, 12, 64, seed=5, residual=True, bias_std=0.02)
    ins, p = [dev(x) for x in c.arrays()], c.params(cf.MhaFusedParams)
    Y = cf.DeviceBuffer.empty((B, S, D), np.float32)

    def run():
        assert cf.call_op("mha_fused_f32_cuda", ins, [Y], p) == 0
        return Y.download()

    own = 4 * B * S * D * 4                                    # q, k, v and the attention output
    native.gpu_device_synchronize()
    native.gpu_workspace_release()
    want = run()
    assert native.gpu_workspace_size() > 64 << 20              # with all the scratch
    native.gpu_workspace_release()
    base = native.gpu_workspace_get(own)                       # the least it allocates, 64 MiB
    before = native.gpu_workspace_size(), native.gpu_buffer_generation()
    for _ in range(3):
        native.gpu_inject_alloc_failures(1)
        try:
            got = run()
        finally:
            native.gpu_inject_alloc_failures(0)
        assert (native.gpu_workspace_size(), native.gpu_buffer_generation()) == before
        assert max_abs(got, want) <= 1e-5
    assert native.gpu_workspace_get(own) == base
    run()                                                      # memory again: it grows
    assert native.gpu_workspace_size() > before[0]


@pytest.mark.gpu
@pytest.mark.parametrize("f16,nk,M,N,K", [(True, False, 16, 768, 3072), (True, True, 16, 768, 3072),
                                          (False, False, 16, 768, 4096), (False, False, 512, 2304, 768),
                                          (False, True, 512, 2304, 768), (False, True, 2048, 2304, 768)])
@pytest.mark.parametrize("how", ["capture", "memory"])
def test_matmul_without_room_for_partial_sums(gpu, native, f16, nk, M, N, K, how):
    """Products whose plan wants a workspace, where there is none to have: first called while
    a stream is captured, or with the allocation failing.  They still run, and the recording
    gives the result on every replay.  Where a transposed B has to be copied first and there is
    no memory for the copy either, the call returns -1 and records nothing, and the same call
    works on that stream afterwards."""
    import cudaforge_amd as cf
    r = O.round_f16 if f16 else (lambda a: a)
    A, B = r(O.normal((M, K), M + N)), r(O.normal((K, N), K + 1, 0.0, 1.0 / np.sqrt(K)))
    want = A.astype(np.float64) @ B.astype(np.float64)
    ins = [dev(A, f16), dev(B.T if nk else B, f16), None]
    C = cf.DeviceBuffer.from_numpy(np.full((M, N), 7.0, np.float16 if f16 else np.float32))
    p = cf.MatmulParams(M, N, K, False, nk, 1, 0, 0, 0, 0)
    name, tol = ("matmul_f16_cuda", TOL16) if f16 else ("matmul_f32_cuda", 1e-5)
    # A transposed B is copied where the plan that reads it as it is cannot run without room.
    copies = nk and (f16 or gemm_plan(native, M, N, K, f16, nk)[0] < 2000)
    st = cf.Stream()
    native.gpu_device_synchronize()
    native.gpu_workspace_release()
    if how == "memory":
        native.gpu_inject_alloc_failures(2)
        try:
            rc = cf.call_op(name, ins, [C], p, st)
        finally:
            native.gpu_inject_alloc_failures(0)
        assert rc == (-1 if copies else 0)
        if rc != 0:
            assert cf.call_op(name, ins, [C], p, st) == 0
        assert max_abs(want, C.download(st).astype(np.float64)) <= tol
    else:
        ex = ctypes.c_void_p()
        assert native.gpu_capture_begin(st.handle) == 0
        rc = cf.call_op(name, ins, [C], p, st)
        assert native.gpu_capture_end(st.handle, ctypes.byref(ex)) == 0
        assert rc == (-1 if copies else 0)
        for _ in range(3):
            C.fill_zero()
            native.gpu_device_synchronize()
            assert (cf.call_op(name, ins, [C], p, st) if copies else native.gpu_graph_launch(ex, st.handle)) == 0
            assert max_abs(want, C.download(st).astype(np.float64)) <= tol
        native.gpu_graph_exec_destroy(ex)
    st.synchronize()
