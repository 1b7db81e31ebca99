// Mixed-precision reconstructor: R = Ctm * Cmm^{-1} to a stated tolerance with the O(n^3)
// factorization and the O(m n^2) solves in low precision and the residuals in FP64.  Two modes:
// MOAO_MIXED_FP32 runs the updates on FP32 MFMA; MOAO_MIXED_BF16 on BF16 MFMA with each FP32
// operand split into two BF16 terms (split-BF16 planes of every finished column of L and of the
// right-hand sides are written as the recursion goes, and of L by columns before the second
// solve), FP32 accumulation; the leaves are FP64 in both.
//
// Cmm carries an exact low-rank term: the reference adds lgs_cst to every entry of each LGS
// xx and yy block (common/kernels/matcov_kernels.cpp:320-321), i.e. Cmm = C0 + c U U^T with U
// the n x p indicator matrix of those 2*nlgs index ranges.  That term makes Cmm
// ill-conditioned (its eigenvalues c*Nsubap sit 4-6 decades above the noise floor; FP32
// Cholesky of Cmm loses definiteness by n ~ 1e4) while C0 stays well conditioned, so:
//   1. C0 (FP32) = Cmm - c U U^T, converted in one pass;
//   2. tall factorization of C0 (FP32 storage) with [Ctm; U^T] riding along, then the second
//      solve: Y = Ctm C0^{-1}, W = U^T C0^{-1}   (low-precision updates, FP64 leaves);
//   3. Woodbury in FP64: S = I/c + W U (p x p, host), R = Y - (Y U) S^{-1} W;
//   4. refinement: E = Ctm - R Cmm (FP64 GEMM on the full Cmm, lower triangle read);
//      stop when ||E||_F <= tol ||Ctm||_F, else D = E C0^{-1} (low-precision solves) corrected
//      by Woodbury, R += D.
// Without a low-rank description (p = 0) the same loop runs on Cmm itself.
// With the environment variable MOAO_DEBUG set, the norms of the intermediate terms and the
// residual of every refinement step are printed to stderr (synchronising after each).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <string>
#include <vector>

#include "common.hpp"
#include "gemm.hpp"
#include "leaf.hpp"
#include "profile.hpp"
#include "recon.hpp"
#include "stages.hpp"

namespace moao {
namespace {

// C0[r,c] = Cmm[r,c] - c*[r,c in the same low-rank range], lower triangle, to FP32.
__global__ void cmm_to_c0_f32(const double* __restrict__ A, long lda, float* __restrict__ B,
                              long ldb, int n, const int* __restrict__ rid, double cst) {
    const int r = blockIdx.x * 64 + (threadIdx.x & 63);
    const int c = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (r >= n || c >= n || r < c) return;
    double v = A[r + (long)c * lda];
    const int a = rid[r];
    if (a >= 0 && a == rid[c]) v -= cst;
    B[r + (long)c * ldb] = (float)v;
}

__global__ void cvt_f64_f32(const double* __restrict__ a, long lda, float* __restrict__ b,
                            long ldb, int rows, int cols) {
    const int r = blockIdx.x * 64 + (threadIdx.x & 63);
    const int c = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (r < rows && c < cols) b[r + (long)c * ldb] = (float)a[r + (long)c * lda];
}

__global__ void cvt_f32_f64(const float* __restrict__ a, long lda, double* __restrict__ b,
                            long ldb, int rows, int cols) {
    const int r = blockIdx.x * 64 + (threadIdx.x & 63);
    const int c = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (r < rows && c < cols) b[r + (long)c * ldb] = (double)a[r + (long)c * lda];
}

// b += a (FP64)
__global__ void add_f64(const double* __restrict__ a, long lda, double* __restrict__ b, long ldb,
                        int rows, int cols) {
    const int r = blockIdx.x * 64 + (threadIdx.x & 63);
    const int c = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (r < rows && c < cols) b[r + (long)c * ldb] += a[r + (long)c * lda];
}

// Per-workgroup partial sums of squares of a rows x cols matrix (one column strip per group).
__global__ void sumsq_partial(const double* __restrict__ a, long lda, int rows, int cols,
                              double* __restrict__ part) {
    __shared__ double red[256];
    double acc = 0.0;
    const long total = (long)rows * cols;
    for (long e = (long)blockIdx.x * 256 + threadIdx.x; e < total; e += (long)gridDim.x * 256) {
        const long c = e / rows, r = e - c * rows;
        const double v = a[r + c * lda];
        acc += v * v;
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// rid[k] = the range that holds index k (-1: none) and the columns k of U^T (p x n, leading
// dimension ldt), U the indicator of the ranges [ends[2q], ends[2q + 1]).
__global__ void lowrank_init(const int* __restrict__ ends, int p, int n, int* __restrict__ rid,
                             float* __restrict__ Ut, long ldt) {
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= n) return;
    int r = -1;
    for (int q = 0; q < p; ++q) {
        const bool in = k >= ends[2 * q] && k < ends[2 * q + 1];
        if (in) r = q;
        Ut[q + (long)k * ldt] = in ? 1.0f : 0.0f;
    }
    rid[k] = r;
}

// Z = X U for the indicator U: Z[r, q] = sum of X[r, k] over the columns k of range q.  The range's
// columns are cut into gridDim.z parts summed apart (part [.][r, q] in P) and added by
// range_sums_add in part order.  A workgroup sums 64 rows, its four waves every fourth column.
// Bound by the one read of X: as a K x N product this was one 128-column tile with 2 nlgs of its
// columns in use (n = 9,632, m = 1,376: 515 -> 30 us).
__global__ void range_sums(const double* __restrict__ X, long ldx, int rows,
                           const int* __restrict__ ends, double* __restrict__ P, int p) {
    __shared__ double red[4][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, q = blockIdx.y;
    const int r = blockIdx.x * 64 + lane;
    const int k0 = ends[2 * q], len = ends[2 * q + 1] - k0;
    const int b = k0 + (int)((long)len * blockIdx.z / gridDim.z);
    const int e = k0 + (int)((long)len * (blockIdx.z + 1) / gridDim.z);
    double acc = 0.0;
    if (r < rows) {
        double a[4] = {0, 0, 0, 0};
        int k = b + wave;
        for (; k + 12 < e; k += 16)
#pragma unroll
            for (int u = 0; u < 4; ++u) a[u] += X[r + (long)(k + 4 * u) * ldx];
        for (; k < e; k += 4) a[0] += X[r + (long)k * ldx];
        acc = (a[0] + a[1]) + (a[2] + a[3]);
    }
    red[wave][lane] = acc;
    __syncthreads();
    if (wave == 0 && r < rows)
        P[(long)blockIdx.z * rows * p + r + (long)q * rows] =
            (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]);
}

__global__ void range_sums_add(const double* __restrict__ P, long cells, int parts,
                               double* __restrict__ Z) {
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= cells) return;
    double acc = P[i];
    for (int z = 1; z < parts; ++z) acc += P[z * cells + i];
    Z[i] = acc;
}

constexpr int kNormBlocks = 1024;
constexpr int kSumParts = 8;    // parts of a range in range_sums

dim3 grid2(int rows, int cols) { return dim3((rows + 63) / 64, (cols + 3) / 4); }

struct Ranges {
    std::vector<long> start, len;
    double cst = 0.0;
    int p() const { return (int)start.size(); }
};

Ranges lowrank_ranges(const moao_tomo_view* t, long n) {
    Ranges R;
    if (!t || t->lgs_cst == 0.0) return R;
    R.cst = t->lgs_cst;
    long off = 0;
    for (int w = 0; w < t->Nw - 1; ++w) {
        const long ns = t->Nsubap[w];
        if (w < t->nlgs) {
            R.start.push_back(2 * off);
            R.len.push_back(ns);
            R.start.push_back(2 * off + ns);
            R.len.push_back(ns);
        }
        off += ns;
    }
    if (2 * off != n) R.start.clear(), R.len.clear();  // view does not describe this Cmm
    return R;
}

// Inverse of the p x p matrix S (column-major) by Gauss-Jordan with partial pivoting; false if
// singular.  S = I/c + W U is used exactly as computed (not symmetrised): the Woodbury identity
// reproduces the inverse of C0_low + c U U^T only when S is formed from the same W that is
// applied, and W from low-precision solves makes W U symmetric only to ~1e-5.
bool small_inverse(const std::vector<double>& S, int p, std::vector<double>& inv) {
    std::vector<double> a(S);
    inv.assign((size_t)p * p, 0.0);
    for (int i = 0; i < p; ++i) inv[i + i * p] = 1.0;
    for (int c = 0; c < p; ++c) {
        int piv = c;
        for (int r = c + 1; r < p; ++r)
            if (std::fabs(a[r + c * p]) > std::fabs(a[piv + c * p])) piv = r;
        if (!(std::fabs(a[piv + c * p]) > 0)) return false;
        if (piv != c)
            for (int k = 0; k < p; ++k) {
                std::swap(a[c + k * p], a[piv + k * p]);
                std::swap(inv[c + k * p], inv[piv + k * p]);
            }
        const double d = a[c + c * p];
        for (int k = 0; k < p; ++k) {
            a[c + k * p] /= d;
            inv[c + k * p] /= d;
        }
        for (int r = 0; r < p; ++r) {
            if (r == c) continue;
            const double f = a[r + c * p];
            if (f == 0.0) continue;
            for (int k = 0; k < p; ++k) {
                a[r + k * p] -= f * a[c + k * p];
                inv[r + k * p] -= f * inv[c + k * p];
            }
        }
    }
    return true;
}

struct MixedWs {
    float* C0;     // n x n
    float* X32;    // (m + p) x n: rows [0,m) right-hand sides, rows [m, m+p) U^T
    float* invL;   // leaves
    double* E;     // m x n residual / correction
    double* Ctm0;  // m x n copy of the right-hand side for the residuals
    double* W;     // p x n
    double* Z;     // m x p
    double* Z2;    // m x p
    double* Sinv;  // p x p
    double* WU;    // p x p
    double* part;  // norm partial sums
    int* rid;      // n range ids
    int* info;
    int* ends;     // p ranges: first index, one past the last
};

}  // namespace

// Leading dimension of the split-BF16 planes of an order-n solve.
static long plane_ld(long n) { return (n + 63) / 64 * 64; }

// Byte offsets of the workspace pieces (MixedWs order, then for the BF16 mode the planes of L in
// both orientations and of the right-hand sides, last the scratch of the residuals' symmetric
// operand, which may be longer) and the least total size.
static size_t mixed_layout(long n, long m, int p, int mode, std::vector<size_t>* offs) {
    const long xr = m + p;
    const long q = std::max(p, 1);
    auto al = [](size_t b) { return (b + 255) & ~size_t(255); };
    size_t off = 0;
    auto take = [&](size_t bytes) {
        if (offs) offs->push_back(off);
        off += al(bytes);
    };
    take(sizeof(float) * n * n);
    take(sizeof(float) * xr * n);
    take(sizeof(float) * recon_invl_doubles(n));
    take(sizeof(double) * m * n);
    take(sizeof(double) * m * n);
    take(sizeof(double) * q * n);
    take(sizeof(double) * m * q);
    take(sizeof(double) * m * q);
    take(sizeof(double) * q * q);
    take(sizeof(double) * q * q);
    take(sizeof(double) * kNormBlocks);
    take(sizeof(int) * n);
    take(sizeof(int) * 4);
    take(sizeof(int) * 2 * q);
    if (mode == MOAO_MIXED_BF16) {
        const long ld = plane_ld(n);
        take(sizeof(unsigned short) * 2 * n * ld);   // L, plane row = row
        take(sizeof(unsigned short) * 2 * n * ld);   // L, plane row = column
        take(sizeof(unsigned short) * 2 * xr * ld);  // right-hand sides
    }
    take(sym_least_bytes(n));
    return off;
}

size_t mixed_workspace_bytes(long n, long m, const moao_tomo_view* lowrank, int mode) {
    return mixed_layout(n, m, lowrank_ranges(lowrank, n).p(), mode, nullptr);
}

size_t mixed_spare_bytes(long n, long m) {
    const size_t best = sym_bytes(m, n), least = sym_least_bytes(n);
    return best > least ? best - least : 0;
}

int reconstructor_mixed_dev(long n, long m, const double* Cmm, long ldCmm, double* Ctm, long ldCtm,
                            const moao_tomo_view* lowrank, int mode, double tol, int max_iter,
                            double* resid_out, int* iters_out, void* ws, size_t ws_bytes,
                            hipStream_t s) {
    if (n < 1 || m < 1 || ldCmm < n || ldCtm < m || !Cmm || !Ctm || max_iter < 0 ||
        n >= (1L << 31) || m >= (1L << 31) ||
        (mode != MOAO_MIXED_FP32 && mode != MOAO_MIXED_BF16)) {
        set_error("reconstructor_mixed: invalid arguments");
        return MOAO_ERR_ARG;
    }
    const int split = mode == MOAO_MIXED_BF16 ? 1 : 0;
    const bool debug = std::getenv("MOAO_DEBUG") != nullptr;
    const Ranges rg = lowrank_ranges(lowrank, n);
    const int p = rg.p();
    const long xr = m + p;  // rows of the FP32 right-hand-side block
    std::vector<size_t> offs;
    const size_t total = mixed_layout(n, m, p, mode, &offs);
    if (!ws || ws_bytes < total) {
        set_error("reconstructor_mixed: workspace too small");
        return MOAO_ERR_ARG;
    }
    char* b = static_cast<char*>(ws);
    MixedWs w{(float*)(b + offs[0]), (float*)(b + offs[1]), (float*)(b + offs[2]),
              (double*)(b + offs[3]), (double*)(b + offs[4]), (double*)(b + offs[5]),
              (double*)(b + offs[6]), (double*)(b + offs[7]), (double*)(b + offs[8]),
              (double*)(b + offs[9]), (double*)(b + offs[10]), (int*)(b + offs[11]),
              (int*)(b + offs[12]), (int*)(b + offs[13])};
    const int N = (int)n, M = (int)m;
    SplitWs sw{};
    const SplitWs* swp = nullptr;
    if (split) {
        const long ld = plane_ld(n);
        sw = SplitWs{(unsigned short*)(b + offs[14]), (unsigned short*)(b + offs[15]),
                     (unsigned short*)(b + offs[16]), ld, n * ld, n * ld, xr * ld};
        swp = &sw;
    }

    auto norm = [&](const double* a, long lda, int rows, int cols, double* out) -> int {
        hipLaunchKernelGGL(sumsq_partial, dim3(kNormBlocks), dim3(256), 0, s, a, lda, rows, cols,
                           w.part);
        MOAO_HIP_TRY(hipGetLastError());
        std::vector<double> h(kNormBlocks);
        MOAO_HIP_TRY(hipMemcpyAsync(h.data(), w.part, sizeof(double) * kNormBlocks,
                                    hipMemcpyDeviceToHost, s));
        MOAO_HIP_TRY(hipStreamSynchronize(s));
        double acc = 0;
        for (double v : h) acc += v;
        *out = std::sqrt(acc);
        return MOAO_OK;
    };

    // --- range ids and U^T (rows m .. m+p-1 of X32), written on the device from the ranges
    if (p) {
        std::vector<int> ends(2 * (size_t)p);
        for (int q = 0; q < p; ++q) {
            ends[2 * q] = (int)rg.start[q];
            ends[2 * q + 1] = (int)(rg.start[q] + rg.len[q]);
        }
        MOAO_HIP_TRY(hipMemcpyAsync(w.ends, ends.data(), sizeof(int) * 2 * p,
                                    hipMemcpyHostToDevice, s));
        MOAO_HIP_TRY(hipStreamSynchronize(s));  // the host vector goes out of scope
    }
    hipLaunchKernelGGL(lowrank_init, dim3((N + 255) / 256), dim3(256), 0, s, w.ends, p, N, w.rid,
                       w.X32 + m, xr);
    MOAO_HIP_TRY(hipGetLastError());

    // --- 1. C0 in FP32; right-hand sides Ctm in FP32
    {
        ProfScope ps(kProfConvert, 12.0 * n * (n + 1) / 2, s);
        hipLaunchKernelGGL(cmm_to_c0_f32, grid2(N, N), dim3(256), 0, s, Cmm, ldCmm, w.C0, n, N,
                           w.rid, rg.cst);
        hipLaunchKernelGGL(cvt_f64_f32, grid2(M, N), dim3(256), 0, s, Ctm, ldCtm, w.X32, xr, M, N);
        MOAO_HIP_TRY(hipGetLastError());
    }
    double ctm_norm = 0;
    if (int rc = norm(Ctm, ldCtm, M, N, &ctm_norm)) return rc;
    // keep the original Ctm for the residuals
    MOAO_HIP_TRY(hipMemcpy2DAsync(w.Ctm0, m * sizeof(double), Ctm, ldCtm * sizeof(double),
                                  m * sizeof(double), n, hipMemcpyDeviceToDevice, s));

    // --- 2. FP32 factorization with [Ctm; U^T] riding along, second solve
    std::vector<RowGroup<float>> all{{w.X32, xr, (int)xr}};
    if (int rc = potrf_tall<float>(n, w.C0, n, all, w.invL, w.info, s, swp)) return rc;
    int hinfo = 0;
    MOAO_HIP_TRY(hipMemcpyAsync(&hinfo, w.info, sizeof(int), hipMemcpyDeviceToHost, s));
    MOAO_HIP_TRY(hipStreamSynchronize(s));
    if (hinfo) {
        set_error("reconstructor_mixed: FP32 factorization of C0 failed");
        return hinfo;
    }
    // the second solve reads L by columns: its planes with plane row = column of L
    if (split)
        if (int rc = split_planes(w.C0, n, N, N, sw.lq, sw.ld, sw.lqs, 0, s)) return rc;
    if (int rc = trsm_right_lower_notrans<float>(n, w.C0, n, w.invL, all, s, nullptr, swp))
        return rc;

    // Z = X U (rows x p, leading dimension rows); the parts' sums in `room` bytes at P, memory of the
    // workspace that is free meanwhile, as many parts as it holds
    auto times_u = [&](const double* X, long ldx, int rows, double* Z, void* P, size_t room) -> int {
        const long cells = (long)rows * p;
        const int parts = (int)std::min<size_t>(kSumParts, room / (sizeof(double) * cells));
        double* to = parts > 1 ? static_cast<double*>(P) : Z;
        hipLaunchKernelGGL(range_sums, dim3((rows + 63) / 64, p, std::max(parts, 1)), dim3(256), 0, s,
                           X, ldx, rows, w.ends, to, p);
        if (parts > 1)
            hipLaunchKernelGGL(range_sums_add, dim3((unsigned)((cells + 255) / 256)), dim3(256), 0,
                               s, to, cells, parts, Z);
        MOAO_HIP_TRY(hipGetLastError());
        return MOAO_OK;
    };

    // --- 3. Woodbury terms
    std::vector<double> Sinv;
    if (p) {
        hipLaunchKernelGGL(cvt_f32_f64, grid2(p, N), dim3(256), 0, s, w.X32 + m, xr, w.W, p, p, N);
        MOAO_HIP_TRY(hipGetLastError());
        if (int rc = times_u(w.W, p, p, w.WU, w.E, sizeof(double) * m * n)) return rc;
        std::vector<double> S((size_t)p * p);
        MOAO_HIP_TRY(hipMemcpyAsync(S.data(), w.WU, sizeof(double) * p * p, hipMemcpyDeviceToHost,
                                    s));
        MOAO_HIP_TRY(hipStreamSynchronize(s));
        for (int q = 0; q < p; ++q) S[q + q * p] += 1.0 / rg.cst;
        if (!small_inverse(S, p, Sinv)) {
            set_error("reconstructor_mixed: Woodbury capacitance matrix is singular");
            return MOAO_ERR_NOCONV;
        }
        if (debug) {
            double tr = 0, trs = 0;
            for (int q = 0; q < p; ++q) tr += S[q + q * p], trs += Sinv[q + q * p];
            std::fprintf(stderr, "[mixed] p=%d trace(S)=%.6e trace(S^-1)=%.6e\n", p, tr, trs);
        }
        MOAO_HIP_TRY(hipMemcpyAsync(w.Sinv, Sinv.data(), sizeof(double) * p * p,
                                    hipMemcpyHostToDevice, s));
    }
    // Y (FP64) -> X; X -= (X U) S^{-1} W; the FP32 right-hand sides, of which Y is the copy, are free
    auto woodbury = [&](double* X, long ldx) -> int {
        if (!p) return MOAO_OK;
        if (int rc = times_u(X, ldx, M, w.Z, w.X32, sizeof(float) * xr * n)) return rc;
        auto g = gemm_args<double>(M, p, p, 1.0, w.Z, m, w.Sinv, p, 0, 0.0, w.Z2, m);
        if (int rc = gemm_f64(g, s)) return rc;
        g = gemm_args<double>(M, N, p, -1.0, w.Z2, m, w.W, p, 0, 1.0, X, ldx);
        return gemm_f64(g, s);
    };
    hipLaunchKernelGGL(cvt_f32_f64, grid2(M, N), dim3(256), 0, s, w.X32, xr, Ctm, ldCtm, M, N);
    MOAO_HIP_TRY(hipGetLastError());
    if (debug) {
        double a = 0, b2 = 0;
        norm(Ctm, ldCtm, M, N, &a);
        if (p) norm(w.W, p, p, N, &b2);
        std::fprintf(stderr, "[mixed] |Ctm|=%.6e |Y|=%.6e |W|=%.6e\n", ctm_norm, a, b2);
    }
    if (int rc = woodbury(Ctm, ldCtm)) return rc;  // Ctm now holds R_0
    if (debug && p) {
        double a = 0, b2 = 0, c2 = 0;
        norm(w.Z, m, M, p, &a);
        norm(w.Z2, m, M, p, &b2);
        norm(Ctm, ldCtm, M, N, &c2);
        std::fprintf(stderr, "[mixed] |Z|=%.6e |Z2|=%.6e |R0|=%.6e\n", a, b2, c2);
    }

    // --- 4. refinement (the residual's symmetric operand Cmm written out in full where the
    // workspace has room)
    SymWork sym;
    sym_place(sym, m, n, b + offs.back(), ws_bytes - offs.back());
    double rel = 0;
    int it = 0;
    int status = MOAO_OK;
    for (;; ++it) {
        MOAO_HIP_TRY(hipMemcpyAsync(w.E, w.Ctm0, sizeof(double) * m * n, hipMemcpyDeviceToDevice,
                                    s));
        auto g = gemm_args<double>(M, N, N, -1.0, Ctm, ldCtm, Cmm, ldCmm, 2, 1.0, w.E, m);
        if (int rc = gemm_sym(g, sym, s)) { status = rc; break; }
        double en = 0;
        if (int rc = norm(w.E, m, M, N, &en)) { status = rc; break; }
        rel = ctm_norm > 0 ? en / ctm_norm : en;
        if (debug) std::fprintf(stderr, "[mixed] step %d relative residual %.3e\n", it, rel);
        if (rel <= tol) break;
        if (it >= max_iter) { status = MOAO_ERR_NOCONV; break; }
        // D = E C0^{-1} (FP32 solves), Woodbury-corrected in FP64, R += D
        hipLaunchKernelGGL(cvt_f64_f32, grid2(M, N), dim3(256), 0, s, w.E, m, w.X32, xr, M, N);
        std::vector<RowGroup<float>> rhs{{w.X32, xr, M}};
        if (int rc = trsm_right_lower_trans<float>(n, w.C0, n, w.invL, rhs, s, nullptr, swp)) {
            status = rc;
            break;
        }
        if (int rc = trsm_right_lower_notrans<float>(n, w.C0, n, w.invL, rhs, s, nullptr, swp)) {
            status = rc;
            break;
        }
        hipLaunchKernelGGL(cvt_f32_f64, grid2(M, N), dim3(256), 0, s, w.X32, xr, w.E, m, M, N);
        if (int rc = woodbury(w.E, m)) { status = rc; break; }
        hipLaunchKernelGGL(add_f64, grid2(M, N), dim3(256), 0, s, w.E, m, Ctm, ldCtm, M, N);
        MOAO_HIP_TRY(hipGetLastError());
    }
    MOAO_HIP_TRY(hipStreamSynchronize(s));
    if (resid_out) *resid_out = rel;
    if (iters_out) *iters_out = it;
    if (status == MOAO_ERR_NOCONV)
        set_error("reconstructor_mixed: refinement stopped at relative residual " +
                  std::to_string(rel));
    return status;
}

}  // namespace moao

extern "C" {

int moao_hip_reconstructor_mixed_dev(long nmeas, long nmeasts, const double* dCmm, long ldCmm,
                                     double* dCtm, long ldCtm, const moao_tomo_view* lowrank,
                                     int mode, double tol, int max_iter, double* resid,
                                     int* iters, void* stream) {
    if (int rc = moao::ensure_init()) return rc;
    if (mode != MOAO_MIXED_FP32 && mode != MOAO_MIXED_BF16) {
        moao::set_error("reconstructor_mixed: unsupported mode");
        return MOAO_ERR_ARG;
    }
    if (nmeas < 1 || nmeasts < 1 || nmeas >= (1L << 31) || nmeasts >= (1L << 31)) {
        moao::set_error("reconstructor_mixed: invalid arguments");
        return MOAO_ERR_ARG;
    }
    // workspace of this call only, from the stream-ordered pool; the least where more is not to be had
    hipStream_t s = moao::pick_stream(stream);
    const size_t least = moao::mixed_workspace_bytes(nmeas, nmeasts, lowrank, mode);
    size_t bytes = least + moao::mixed_spare_bytes(nmeas, nmeasts);
    void* ws = nullptr;
    while (hipMallocAsync(&ws, bytes, s) != hipSuccess) {
        (void)hipGetLastError();
        if (bytes == least) {
            moao::set_error("reconstructor_mixed: workspace allocation of " +
                            std::to_string(bytes) + " B failed");
            return MOAO_ERR_NOMEM;
        }
        bytes = least;
    }
    int rc = moao::reconstructor_mixed_dev(nmeas, nmeasts, dCmm, ldCmm, dCtm, ldCtm, lowrank, mode,
                                           tol, max_iter, resid, iters, ws, bytes, s);
    (void)hipFreeAsync(ws, s);
    if (hipStreamSynchronize(s) != hipSuccess && rc == MOAO_OK) {
        moao::set_error("reconstructor_mixed: stream synchronisation failed");
        rc = MOAO_ERR_HIP;
    }
    return rc;
}

}  // extern "C"
