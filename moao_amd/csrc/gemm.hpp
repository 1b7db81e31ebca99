// MFMA GEMM engine shared by the reconstructor and Cee/Cvv stages.
//
//   C_g[M_g x N] = alpha * A_g[M_g x K] * op(B) + beta * C_g       for each segment g
//
// Column-major, explicit leading dimensions.  op(B) = B^T with B stored N x K (transb = 1),
// op(B) = B with B stored K x N (transb = 0), or op(B) = B for a symmetric K x K matrix of which
// only the lower triangle is read (transb = 2, the B operand of dsymm(Right, Lower)).
// Up to kMaxSeg row segments share one B and one
// launch (grid.z = segment): the reconstructor uses this to update the Cmm rows and the Ctm
// rows of every target with a single launch.  A segment may bring its own B of the same shape
// (GemmSeg::B: a batch of independent products in one launch, e.g. one per target).  Segment 0
// (every segment with tri_all) may be restricted to its lower trapezoid (row + tri_off >= col):
// tiles wholly above that line are skipped and elements above it are not written.
//
// In-place use: when C_g == A_g and N <= the kernel's N tile (one column tile), each workgroup
// reads its whole row block of A before it writes C, and no other workgroup touches those rows,
// so C := A * op(B) in place is well defined (used for the triangular-inverse panel solves).
#pragma once

#include <hip/hip_runtime.h>

namespace moao {

constexpr int kMaxSeg = 8;

// Split-BF16 planes of an FP32 matrix region: the hi term of element (row, k) at
// hi[row * ld + k], the lo term at hi[ps + row * ld + k] (k contiguous within a row; ld a
// multiple of 8 and at least the row's last chunk of 32 k).
struct Planes {
    const unsigned short* hi;
    long ld;
    long ps;
};

template <typename T>
struct GemmSeg {
    const T* A;
    T* C;
    long lda, ldc;
    int M;
    Planes ap;  // split = 2: A's planes (row = row of this segment)
    const T* B;  // optional: this segment's own B (same shape and ldb), else GemmArgs::B
    // FP32, split = 0, optional: the planes of C, written with it (element (r, c) as plane row r,
    // k = c, at cp[r * cpl.ld + c]; 4 * N bytes aligned to 8)
    unsigned short* cp;
    Planes cpl;  // ld and ps of cp
};

template <typename T>
struct GemmArgs {
    GemmSeg<T> seg[kMaxSeg];
    int nseg;
    const T* B;
    long ldb;
    int N, K;
    int transb;
    int tri;      // segment 0 lower-trapezoid restriction
    int tri_off;
    int tri_all;  // with tri: every segment restricted, not only segment 0
    T alpha, beta;
    // transb = 2 only, optional: full symmetric copies of B's 128 x 128 diagonal blocks (gemm_sym);
    // with it the launch runs on the direct-to-LDS kernel.
    const T* symdiag;
    // FP32 only: 2 = run the product on BF16 MFMA from split-BF16 planes of the operands
    // (hi = bf16(a), lo = bf16(a - hi); hi*hi + hi*lo + lo*hi accumulated in FP32; A from
    // seg[].ap, op(B) element (k, n) from bp row n); 0 = FP32 MFMA.
    int split;
    Planes bp;  // split = 2: B's planes (row = column n of op(B))
    // Optional device status word: when it is non-zero at launch time the whole launch is a
    // no-op.  The factorization points it at its dpotrf info, so the updates and solves queued
    // after a failing pivot do nothing and no host synchronisation is needed to stop them.
    const int* skip_if;
};

// Scratch for products with a symmetric operand.  From kSymRows rows on it holds the matrix written
// out in full, so that they run on the kernel for op(B) = B^T; with fewer, full copies of its 128 x
// 128 diagonal blocks, with which a kernel reads the lower triangle in place, columns above the
// diagonal and rows below it.  K = 18,688, in place -> in full: 256 rows 4.1 -> 5.3 ms, 512 rows
// 9.8 -> 7.6, 8 x 2,336 rows 213 -> 187.  For one matrix and one caller's scope; stream-ordered
// (sym_alloc) or in the caller's memory (sym_place).
constexpr long kSymRows = 448;
struct SymWork {
    double* p = nullptr;
    hipStream_t s = nullptr;
    bool own = false;   // from sym_alloc
    int cols = 0;       // columns written out at a time; 0: diagonal blocks
    bool held = false;  // the whole matrix, or its blocks, are there
    SymWork() = default;
    SymWork(const SymWork&) = delete;
    SymWork& operator=(const SymWork&) = delete;
    ~SymWork();
};
// Allocates for products of `rows` rows with a K x K matrix: the first that the pool has of the
// matrix in full and its blocks; leaves w empty where it has neither.
void sym_alloc(SymWork& w, long rows, long K, hipStream_t s);
// Bytes that serve products of `rows` rows best, and the least that serve them (the blocks).
size_t sym_bytes(long rows, long K);
inline size_t sym_least_bytes(long K) { return sym_bytes(1, K); }
// The same in `bytes` of device memory at mem, at least sym_least_bytes(K), for work on one stream.
void sym_place(SymWork& w, long rows, long K, void* mem, size_t bytes);
// The transb = 2 product, through w where it has room, else on the fallback kernel.
int gemm_sym(const GemmArgs<double>& a, SymWork& w, hipStream_t stream);

// Planes of an FP32 column-major region (rows x cols at A, leading dimension lda):
// transposed = 1 writes element (r, c) as plane row r, k = c (hi[r * ld + c]); transposed = 0 as
// plane row c, k = r (hi[c * ld + r]).
int split_planes(const float* A, long lda, int rows, int cols, unsigned short* hi, long ld,
                 long ps, int transposed, hipStream_t stream);

// Launches on `stream`; returns a MOAO_* status (argument checks only, launch is async).
int gemm_f64(const GemmArgs<double>& a, hipStream_t stream);
int gemm_f32(const GemmArgs<float>& a, hipStream_t stream);

inline int gemm(const GemmArgs<double>& a, hipStream_t s) { return gemm_f64(a, s); }
inline int gemm(const GemmArgs<float>& a, hipStream_t s) { return gemm_f32(a, s); }

// Convenience for a single segment.
template <typename T>
inline GemmArgs<T> gemm_args(int M, int N, int K, T alpha, const T* A, long lda, const T* B,
                             long ldb, int transb, T beta, T* C, long ldc) {
    GemmArgs<T> g{};
    g.seg[0] = {A, C, lda, ldc, M};
    g.nseg = 1;
    g.B = B;
    g.ldb = ldb;
    g.N = N;
    g.K = K;
    g.transb = transb;
    g.tri = 0;
    g.tri_off = 0;
    g.tri_all = 0;
    g.alpha = alpha;
    g.beta = beta;
    g.symdiag = nullptr;
    g.split = 0;
    g.bp = Planes{nullptr, 0, 0};
    g.skip_if = nullptr;
    return g;
}

}  // namespace moao
