"""GPU checks of the MFMA GEMM engine against numpy (float64 reference products).

FP64 tolerance: |C - C_ref| <= 1e-13 * (|A| |op(B)| + |beta C|) elementwise-bound scale; FP32:
2e-5 relative to the same scale, widened in proportion to K beyond 700 (sums of K products of
O(1) numbers).  Shapes cover the direct kernel, both tile sizes of the slice kernels (128-row
tiles: TILES_128), ragged M, N and K (K not a multiple of the 8-deep slice), and transb = 0, 1
and 2 (symmetric B read from its lower triangle).
"""
import numpy as np
import pytest

from moao_amd.device import DeviceArray
from moao_amd.reconstructor import dgemm_dev, sgemm_dev

pytestmark = pytest.mark.gpu

CASES = [(128, 128, 16, 1, 0.0), (130, 77, 33, 1, 1.0), (300, 129, 200, 0, -1.0),
         (1, 1, 1, 0, 0.5), (257, 383, 700, 1, 1.0), (64, 500, 5, 0, 0.0),
         # more than 512 tiles of 128 rows, which run as 64-row tiles
         (4133, 3900, 300, 1, 1.0), (4133, 3900, 301, 0, -1.0), (4133, 2100, 301, 0, 1.0),
         # symmetric B (K == N)
         (50, 300, 300, 2, 1.0), (257, 129, 129, 2, 0.0), (7, 16, 16, 2, 1.0),
         (200, 77, 77, 2, -1.0), (4133, 2100, 2100, 2, 0.5)]


def sym_lower(B, K):
    L = np.tril(B[:K, :K].astype(np.float64))
    return L + np.tril(L, -1).T


def op_b(B, transb, N, K):
    if transb == 1:
        return B[:N].T.astype(np.float64)
    if transb == 0:
        return B[:K].astype(np.float64)
    return sym_lower(B, K)


@pytest.mark.parametrize("M,N,K,transb,beta", CASES)
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_gemm_matches_numpy(M, N, K, transb, beta, dtype):
    print(f"[gemm] {dtype.__name__} M={M} N={N} K={K} transb={transb} beta={beta}", flush=True)
    rng = np.random.default_rng(M * 7 + N * 3 + K)
    lda, ldb, ldc = M + 3, (N if transb == 1 else K) + 5, M + 1
    A = np.asfortranarray(rng.standard_normal((lda, K)).astype(dtype))
    B = np.asfortranarray(rng.standard_normal((ldb, N if transb == 0 else K)).astype(dtype))
    C = np.asfortranarray(rng.standard_normal((ldc, N)).astype(dtype))
    alpha = -0.75
    dA, dB, dC = DeviceArray.from_host(A), DeviceArray.from_host(B), DeviceArray.from_host(C)
    f = dgemm_dev if dtype == np.float64 else sgemm_dev
    f(transb, M, N, K, alpha, dA.ptr, lda, dB.ptr, ldb, beta, dC.ptr, ldc)
    out = dC.to_host()
    a = A[:M].astype(np.float64)
    b = op_b(B, transb, N, K)
    ref = alpha * a @ b + beta * C[:M].astype(np.float64)
    scale = np.abs(alpha) * np.abs(a) @ np.abs(b) + abs(beta) * np.abs(C[:M])
    tol = 1e-13 if dtype == np.float64 else 2e-5 * max(1.0, K / 700.0)
    assert np.all(np.abs(out[:M] - ref) <= tol * (scale + 1e-30))
    # rows beyond M (padding of ldc) untouched
    assert np.array_equal(out[M:], C[M:])


@pytest.mark.parametrize("M,N,K,transb", [(4133, 3900, 300, 1), (4133, 2100, 301, 0),
                                          (4133, 2100, 2100, 2), (300, 129, 203, 1),
                                          (300, 129, 203, 0), (200, 77, 77, 2)])
def test_gemm_reads_only_the_operands(M, N, K, transb):
    """NaN in every element the product must not read -- the leading-dimension padding of A
    and B, and for symmetric B its strict upper triangle -- leaves C bit-identical to the run
    on clean operands: row/column edges, the K tail of the last slice and the symmetric
    diagonal blocks stay inside the operands."""
    print(f"[gemm-nan] M={M} N={N} K={K} transb={transb}", flush=True)
    rng = np.random.default_rng(11 + transb)
    lda, ldb, ldc = M + 3, (N if transb == 1 else K) + 5, M
    A = np.asfortranarray(rng.standard_normal((lda, K)))
    B = np.asfortranarray(rng.standard_normal((ldb, N if transb == 0 else K)))
    C = np.asfortranarray(rng.standard_normal((ldc, N)))
    An, Bn = A.copy(order="F"), B.copy(order="F")
    An[M:] = np.nan
    Bn[(N if transb == 1 else K):] = np.nan
    if transb == 2:
        Bn[np.triu_indices(K, 1)] = np.nan
    outs = []
    for a_, b_ in ((A, B), (An, Bn)):
        dA, dB, dC = DeviceArray.from_host(a_), DeviceArray.from_host(b_), DeviceArray.from_host(C)
        dgemm_dev(transb, M, N, K, 0.5, dA.ptr, lda, dB.ptr, ldb, 1.0, dC.ptr, ldc)
        outs.append(dC.to_host())
    assert np.all(np.isfinite(outs[1]))
    assert np.array_equal(outs[0], outs[1])
    ref = 0.5 * A[:M] @ op_b(B, transb, N, K) + C
    assert np.allclose(outs[0], ref, rtol=0, atol=1e-12 * np.abs(ref).max())


SPLIT_CASES = [(128, 128, 32, 1, 0.0), (130, 77, 33, 1, 1.0), (300, 129, 200, 0, -1.0),
               (1, 1, 1, 0, 0.5), (257, 383, 700, 1, 1.0), (64, 500, 5, 0, 0.0),
               (4133, 3900, 300, 1, 1.0), (4133, 3900, 301, 0, -1.0), (4133, 2100, 3001, 1, 1.0)]


@pytest.mark.parametrize("M,N,K,transb,beta", SPLIT_CASES)
def test_split_bf16_gemm_matches_numpy(M, N, K, transb, beta):
    """The split-BF16 product (hi*hi + hi*lo + lo*hi on BF16 MFMA, FP32 accumulation): each
    product carries a relative error of at most ~3 * 2^-16 (the dropped lo*lo term and the
    residue of the two-term split), so |C - C_ref| <= 1e-4 (|A||op(B)| + |beta C|) elementwise
    plus the FP32 accumulation bound; and the relative Frobenius error of the product stays
    below 1e-4, where one BF16 term per operand would give ~2e-3.  NaN planted in the
    leading-dimension padding must not reach C."""
    from moao_amd.reconstructor import sgemm_bf16x3_dev
    print(f"[gemm-bf16x3] M={M} N={N} K={K} transb={transb} beta={beta}", flush=True)
    rng = np.random.default_rng(M * 5 + N * 3 + K)
    lda, ldb, ldc = M + 3, (N if transb == 1 else K) + 5, M + 1
    A = np.asfortranarray(rng.standard_normal((lda, K)).astype(np.float32))
    B = np.asfortranarray(rng.standard_normal((ldb, N if transb == 0 else K)).astype(np.float32))
    C = np.asfortranarray(rng.standard_normal((ldc, N)).astype(np.float32))
    A[M:] = np.nan
    B[(N if transb == 1 else K):] = np.nan
    alpha = -0.75
    dA, dB, dC = DeviceArray.from_host(A), DeviceArray.from_host(B), DeviceArray.from_host(C)
    sgemm_bf16x3_dev(transb, M, N, K, alpha, dA.ptr, lda, dB.ptr, ldb, beta, dC.ptr, ldc)
    out = dC.to_host()
    a = A[:M].astype(np.float64)
    b = op_b(B, transb, N, K)
    prod = alpha * a @ b
    ref = prod + beta * C[:M].astype(np.float64)
    scale = np.abs(alpha) * np.abs(a) @ np.abs(b) + abs(beta) * np.abs(C[:M])
    tol = 1e-4 + 2e-5 * max(1.0, K / 700.0)
    err = np.abs(out[:M] - ref)
    assert np.all(np.isfinite(out[:M]))
    assert np.all(err <= tol * (scale + 1e-30)), float(np.max(err / (scale + 1e-30)))
    rel = np.linalg.norm(out[:M] - ref) / np.linalg.norm(prod)
    print(f"    max normalised error {np.max(err / (scale + 1e-30)):.2e}, "
          f"relative Frobenius {rel:.2e}", flush=True)
    assert rel <= 1e-4
    assert np.array_equal(out[M:], C[M:])


@pytest.mark.parametrize("transb", [0, 1])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_few_rows_equal_the_rows_of_a_large_product(transb, dtype):
    """Launches that leave most of the chip idle run on the direct kernel (16 or 32 rows per
    workgroup), large ones on the slice kernels; both take every product in the same k order, so
    a product of the first r rows has the bits of those rows in a product of 52,000: edges of the
    16- and 32-row blocks, ragged columns, K below, at and past whole 16-k chunks, beta = 0 and 1."""
    f = dgemm_dev if dtype == np.float64 else sgemm_dev
    rng = np.random.default_rng(3 + transb)
    big = 52000
    for N, K in [(128, 128), (97, 131), (128, 7)]:
        lda, ldb = big + 3, (N if transb == 1 else K) + 1
        A = np.asfortranarray(rng.standard_normal((lda, K)).astype(dtype))
        B = np.asfortranarray(rng.standard_normal((ldb, N if transb == 0 else K)).astype(dtype))
        C = np.asfortranarray(rng.standard_normal((big, N)).astype(dtype))
        dA, dB = DeviceArray.from_host(A), DeviceArray.from_host(B)
        for beta in (0.0, 1.0):
            dC = DeviceArray.from_host(C)
            f(transb, big, N, K, -1.25, dA.ptr, lda, dB.ptr, ldb, beta, dC.ptr, big)
            want = dC.to_host()
            for r in (1, 15, 16, 17, 33, 300, 4097, 9000):
                print(f"[gemm-direct] {dtype.__name__} transb={transb} N={N} K={K} rows={r}",
                      flush=True)
                dC = DeviceArray.from_host(C)
                f(transb, r, N, K, -1.25, dA.ptr, lda, dB.ptr, ldb, beta, dC.ptr, big)
                got = dC.to_host()
                assert np.array_equal(got[:r], want[:r])
                assert np.array_equal(got[r:], C[r:])


def test_direct_in_place_panel():
    """C == A with N <= 128 (the panel solve of a leaf): every row is read before it is written."""
    rng = np.random.default_rng(9)
    for M, N in [(1, 1), (40, 128), (333, 128), (9001, 77)]:
        A = np.asfortranarray(rng.standard_normal((M, N)))
        B = np.asfortranarray(rng.standard_normal((N, N)))
        dA, dB, dC = DeviceArray.from_host(A), DeviceArray.from_host(B), DeviceArray((M, N))
        for transb in (0, 1):
            dgemm_dev(transb, M, N, N, 1.0, dA.ptr, M, dB.ptr, N, 0.0, dC.ptr, M)
            want = dC.to_host()
            dX = DeviceArray.from_host(A)
            dgemm_dev(transb, M, N, N, 1.0, dX.ptr, M, dB.ptr, N, 0.0, dX.ptr, M)
            assert np.array_equal(dX.to_host(), want), (M, N, transb)


@pytest.mark.parametrize("M,N,K", [(3073, 2945, 257), (3103, 3009, 260), (3105, 2943, 8),
                                   (3136, 2977, 7), (3137, 3041, 264), (3199, 3039, 129)])
def test_tiles_at_the_edge(M, N, K):
    """op(B) = B^T launches of 64-row tiles whose last 128 rows and columns hold 1, 31, 33, 64, 65 or 127
    of them (waves that leave out their MFMAs) and whose K ends inside a slice.
    Tolerance: K products of values below 1, each rounded once and added once."""
    print(f"[gemm] edge tiles {M} x {N} x {K}", flush=True)
    rng = np.random.default_rng(M)
    A, B, C = (np.asfortranarray(rng.uniform(-1, 1, s)) for s in ((M, K), (N, K), (M, N)))
    dA, dB, dC = (DeviceArray.from_host(x) for x in (A, B, C))
    dgemm_dev(1, M, N, K, 0.5, dA.ptr, M, dB.ptr, N, 1.0, dC.ptr, M)
    err = np.max(np.abs(dC.to_host() - (0.5 * (A @ B.T) + C)))
    assert err <= 2 * K * 2.0 ** -52


@pytest.mark.parametrize("M", [1, 130, 447, 448, 1000])
@pytest.mark.parametrize("K", [1, 63, 65, 128, 700])
def test_symmetric_operand_from_its_lower_triangle(M, K):
    """The symmetric operand written out in full (448 rows and more) or read in place (fewer); its
    upper triangle holds NaN, so nothing may be read from there.  Tolerance as above."""
    print(f"[gemm] symmetric B {M} x {K}", flush=True)
    rng = np.random.default_rng(M + K)
    A = np.asfortranarray(rng.uniform(-1, 1, (M, K)))
    S = rng.uniform(-1, 1, (K, K))
    S = S + S.T
    low = np.asfortranarray(np.where(np.tri(K, dtype=bool), S, np.nan))
    dA, dB, dC = DeviceArray.from_host(A), DeviceArray.from_host(low), \
        DeviceArray.from_host(np.zeros((M, K), order="F"))
    dgemm_dev(2, M, K, K, 1.0, dA.ptr, M, dB.ptr, K, 0.0, dC.ptr, M)
    assert np.max(np.abs(dC.to_host() - A @ S)) <= 2 * K * 2.0 ** -52 * 2


@pytest.mark.parametrize("transb", [0, 1])
def test_few_rows_of_the_split_bf16_product(transb):
    """The split-BF16 product of few rows (16- or 32-row workgroups without LDS) has the bits of those
    rows in a product large enough for the staged kernel: K below, at and past whole chunks of 32
    and flushes of 256, ragged columns, beta = 0 and 1."""
    from moao_amd.reconstructor import sgemm_bf16x3_dev
    rng = np.random.default_rng(30 + transb)
    big = 16000
    for N, K in [(128, 128), (131, 300), (97, 31), (128, 600)]:
        ldb = N if transb == 1 else K
        A = np.asfortranarray(rng.standard_normal((big, K)).astype(np.float32))
        B = np.asfortranarray(rng.standard_normal((ldb, N if transb == 0 else K)).astype(np.float32))
        C = np.asfortranarray(rng.standard_normal((big, N)).astype(np.float32))
        dA, dB = DeviceArray.from_host(A), DeviceArray.from_host(B)
        for beta in (0.0, 1.0):
            dC = DeviceArray.from_host(C)
            sgemm_bf16x3_dev(transb, big, N, K, -1.25, dA.ptr, big, dB.ptr, ldb, beta, dC.ptr, big)
            want = dC.to_host()
            for r in (1, 16, 17, 300, 2049, 4097, 5000):
                print(f"[split-direct] transb={transb} N={N} K={K} rows={r}", flush=True)
                dC = DeviceArray.from_host(C)
                sgemm_bf16x3_dev(transb, r, N, K, -1.25, dA.ptr, big, dB.ptr, ldb, beta, dC.ptr, big)
                got = dC.to_host()
                assert np.array_equal(got[:r], want[:r])
                assert np.array_equal(got[r:], C[r:])


@pytest.mark.parametrize("dtype,transb,lda,ldb", [
    (np.float64, 1, 179_000_000, 20), (np.float64, 0, 179_000_000, 20),
    (np.float64, 1, 20, 179_000_000), (np.float32, 1, 358_000_000, 21)])
def test_small_product_of_very_tall_buffers(dtype, transb, lda, ldb):
    """20 x 20 x 5 products whose operands are the first rows of buffers so tall that 3 columns span
    more than 4 GiB: offsets of 32 bits would read other rows.  Tolerance: K products of values
    below 1, each rounded once and added once."""
    from moao_amd.lib import check, lib
    import ctypes
    print(f"[gemm-tall] {dtype.__name__} transb={transb} lda={lda} ldb={ldb}", flush=True)
    rng = np.random.default_rng(5)
    M = N = 20
    K = 5

    def tall(rows, cols, ld):
        a = np.asfortranarray(rng.uniform(-1, 1, (rows, cols)).astype(dtype))
        d = DeviceArray((ld, cols), dtype)
        for c in range(cols):
            check(lib().moao_hip_memcpy_h2d(ctypes.c_void_p(d.ptr + c * ld * a.itemsize),
                                            a[:, c].copy().ctypes.data, rows * a.itemsize), "h2d")
        return a, d
    A, dA = tall(M, K, lda)
    B, dB = tall(N if transb == 1 else K, K if transb == 1 else N, ldb)
    dC = DeviceArray.from_host(np.zeros((M, N), dtype, order="F"))
    f = dgemm_dev if dtype == np.float64 else sgemm_dev
    f(transb, M, N, K, 1.0, dA.ptr, lda, dB.ptr, ldb, 0.0, dC.ptr, M)
    ref = A.astype(np.float64) @ (B.T if transb == 1 else B).astype(np.float64)
    assert np.max(np.abs(dC.to_host() - ref)) <= 2 * K * np.finfo(dtype).eps
    dA.free()
    dB.free()


@pytest.mark.parametrize("K", [1, 127, 129, 700, 2000])
def test_symmetric_operand_in_full_and_in_place_give_the_same_bits(K):
    """1000 rows multiply the symmetric matrix written out in full, 447 read it in place through its
    diagonal blocks: the k order is the same, so which of them a call has room for does not show."""
    print(f"[gemm] symmetric B, K = {K}, both forms", flush=True)
    rng = np.random.default_rng(K)
    A = np.asfortranarray(rng.uniform(-1, 1, (1000, K)))
    low = np.asfortranarray(np.tril(rng.uniform(-1, 1, (K, K))))
    dA, dB = DeviceArray.from_host(A), DeviceArray.from_host(low)
    out = []
    for M in (1000, 447):
        dC = DeviceArray.from_host(np.zeros((M, K), order="F"))
        dgemm_dev(2, M, K, K, 1.0, dA.ptr, 1000, dB.ptr, K, 0.0, dC.ptr, M)
        out.append(dC.to_host())
    assert np.array_equal(out[0][:447], out[1])


# Launches of 128-row tiles (tests/test_host_paths.py holds them to that; the shapes of CASES and of
# test_tiles_at_the_edge run on 64-row tiles): as (type, transb, M, N, K).
TILES_128 = [(np.float64, 1, 4609 + d, 4737 - d, 2056 + k) for d, k in
             ((0, 0), (30, 1), (32, 7), (63, 3), (64, 5), (126, 4))] + \
            [(np.float64, 0, 7425, 7423, 8195), (np.float64, 0, 7551, 7393, 8200),
             (np.float32, 1, 5921, 5889, 520), (np.float32, 1, 5951, 5999, 525),
             (np.float32, 0, 4673, 4735, 2049), (np.float32, 0, 4735, 4673, 2061)]


@pytest.mark.parametrize("dtype,transb,M,N,K", TILES_128)
def test_128_row_tiles_at_the_edge(dtype, transb, M, N, K):
    """128-row tiles whose last row and column tiles hold 1 to 127 rows and columns (waves that leave
    out half or all of their MFMAs) and whose K ends inside a slice or with one.  The first and the
    last rows and some between against numpy in 64 bits; tolerance: K products of values below 1,
    each rounded once and added once, and the two operations of alpha and beta."""
    print(f"[gemm-128] {dtype.__name__} transb={transb} {M} x {N} x {K}", flush=True)
    rng = np.random.default_rng(M)

    def uniform(r, c):
        return np.asfortranarray(rng.uniform(-1, 1, (r, c)).astype(dtype))
    A, C = uniform(M, K), uniform(M, N)
    B = uniform(N, K) if transb == 1 else uniform(K, N)
    dA, dB, dC = (DeviceArray.from_host(x) for x in (A, B, C))
    f = dgemm_dev if dtype == np.float64 else sgemm_dev
    f(transb, M, N, K, 0.5, dA.ptr, M, dB.ptr, B.shape[0], 1.0, dC.ptr, M)
    rows = np.unique(np.r_[:3, 60:68, 126:131, M // 2:M // 2 + 3, M - 130:M])
    op = (B.T if transb == 1 else B).astype(np.float64)
    ref = 0.5 * (A[rows].astype(np.float64) @ op) + C[rows]
    err = np.max(np.abs(dC.to_host()[rows] - ref))
    assert err <= 2 * (K + 2) * np.finfo(dtype).eps


# Products of few rows and of so many that the slice kernels take them, with ragged columns and a K
# that ends past whole chunks of the direct kernel (checked there too).
RAGGED, RAGGED_ROWS = (97, 131), (1, 15, 16, 17, 33, 300, 4097, 9000, 66000)


@pytest.mark.parametrize("transb", [0, 1])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_few_ragged_rows_equal_the_rows_of_a_slice_product(transb, dtype):
    """The direct kernel's rows have the bits of the slice kernel's."""
    print(f"[gemm-direct] {dtype.__name__} transb={transb} ragged", flush=True)
    f = dgemm_dev if dtype == np.float64 else sgemm_dev
    rng = np.random.default_rng(17 + transb)
    N, K = RAGGED
    big = RAGGED_ROWS[-1]
    ldb = (N if transb == 1 else K) + 1
    A = np.asfortranarray(rng.standard_normal((big, K)).astype(dtype))
    B = np.asfortranarray(rng.standard_normal((ldb, N if transb == 0 else K)).astype(dtype))
    C = np.asfortranarray(rng.standard_normal((big, N)).astype(dtype))
    dA, dB = DeviceArray.from_host(A), DeviceArray.from_host(B)
    for beta in (0.0, 1.0):
        dC = DeviceArray.from_host(C)
        f(transb, big, N, K, -1.25, dA.ptr, big, dB.ptr, ldb, beta, dC.ptr, big)
        want = dC.to_host()
        for r in RAGGED_ROWS[:-1]:
            dC = DeviceArray.from_host(C)
            f(transb, r, N, K, -1.25, dA.ptr, big, dB.ptr, ldb, beta, dC.ptr, big)
            got = dC.to_host()
            assert np.array_equal(got[:r], want[:r])
            assert np.array_equal(got[r:], C[r:])
