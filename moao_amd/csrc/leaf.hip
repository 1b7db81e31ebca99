// Diagonal-leaf kernels of the reconstructor: FP64 Cholesky of one nb x nb (nb <= 128) block
// held entirely in LDS, followed by the in-place inverse of its triangular factor.
//
// LAPACK semantics of dpotrf('L') for the block: the lower triangle is overwritten by L, the
// strictly-upper part is not touched; a non-positive (or NaN) pivot at local column j stops
// the factorization and records info = j_global + 1 (first failure wins; later leaves see the
// flag and return at once); the leaf's 16-column blocks before the failing pivot's block are
// stored, the rest of the block keeps its input.  The inverse L^{-1} (lower, zero above the diagonal) goes to a
// separate kLeaf x kLeaf buffer and turns every panel triangular solve into an MFMA GEMM.
//
// One workgroup (8 waves) per leaf; the block is zero-padded to kLeaf x kLeaf in LDS and
// processed by 16-column blocks:
//   load:   every element of the lower triangle in flight before the LDS stores;
//   factor: [wave 0] 16x16 diagonal block and its inverse together, in registers: unnormalised
//           elimination of [A | I] (pivots' reciprocals only; one 1/sqrt per lane at the end
//           scales L and D), columns passed between the lanes of a 16-lane row by DPP broadcasts;
//           [all] rows below as A * D^T on f64 MFMA; the rank-16 update of the trailing lower
//           triangle (f64 MFMA) runs one block late, beside the next diagonal factor: wave 0
//           updates that diagonal block first, the other waves the rest;
//   invert: by doubling: from the inverses of the 16x16 diagonal blocks to 32, 64 and 128:
//           inv(L)21 = -inv(L)22 (L21 inv(L)11), both products on f64 MFMA over all waves, the
//           inner one parked in the unused block above the diagonal;
//   store:  L before the inversion overwrites it, inv(L) at the end.
// The time is the serial chain of one workgroup, 128 pivots long.  What it was spent on before
// (70 us): readlane broadcasts under a branch per column, 97 of 166 thousand cycles; an inversion
// by block columns, 45 thousand.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "common.hpp"
#include "leaf.hpp"
#include "profile.hpp"

namespace moao {
namespace {

constexpr int NTL = 512;       // lanes per leaf workgroup
constexpr int NWL = NTL / 64;
constexpr int LD = kLeaf + 1;  // odd stride: a row across columns hits distinct banks
constexpr int kB = 16;         // inner block
constexpr int kNB = kLeaf / kB;

#define S_(r, c) S[(c) * LD + (r)]

typedef double f64x4 __attribute__((ext_vector_type(4)));

// f(0), f(1), ..., f(N - 1) with the index as a compile-time constant
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (N > 0) {
        static_for<N - 1>(f);
        f(std::integral_constant<int, N - 1>{});
    }
}

// Value of v in lane L of the caller's 16-lane row.
template <int L>
__device__ __forceinline__ double row_value(double v) {
    const long long b = __double_as_longlong(v);
    return __longlong_as_double(__builtin_amdgcn_update_dpp(b, b, 0x150 + L, 0xf, 0xf, true));
}

// 1/sqrt(d) for d > 0: hardware estimate refined by two Newton steps.
__device__ __forceinline__ double rsqrt_nr(double d) {
    double r = __builtin_amdgcn_rsq(d);
    r = r * (1.5 - 0.5 * d * r * r);
    r = r * (1.5 - 0.5 * d * r * r);
    return r;
}

// 1/d: hardware estimate refined by two Newton steps (no division on the pivots' chain).
__device__ __forceinline__ double rcp_nr(double d) {
    double r = __builtin_amdgcn_rcp(d);
    r = fma(fma(-d, r, 1.0), r, r);
    return fma(fma(-d, r, 1.0), r, r);
}

// A 16 x 16 block A = L L^T and D = inv(L) in one wave: lane i of every 16-lane row holds row i
// (the four rows work alike).  Elimination of [A | I] with multipliers m_j = a_j / d_j: a[j] keeps
// m_j d_j, x becomes the inverse of the unit factor; then L_ij = a[j] / sqrt(d_j) and
// D_ij = x[j] / sqrt(d_i).  Returns the number of positive pivots before the first that is not.
__device__ __forceinline__ int diag_factor(double (&a)[kB], double (&x)[kB], int li) {
    double dv = 1.0;  // this lane's own pivot
    int good = 0;
    bool all = true;
    static_for<kB>([&](auto J) {
        constexpr int j = decltype(J)::value;
        const double d = row_value<j>(a[j]);
        all = all && d > 0.0;
        good += all ? 1 : 0;
        const double m = li > j ? a[j] * rcp_nr(d) : 0.0;
        dv = li == j ? a[j] : dv;
        // the next pivot's column first
        static_for<kB - 1 - j>([&](auto Q) {
            constexpr int k = j + 1 + decltype(Q)::value;
            a[k] = fma(-m, row_value<k>(a[j]), a[k]);
        });
        static_for<j>([&](auto C) {
            constexpr int c = decltype(C)::value;
            x[c] = fma(-m, row_value<j>(x[c]), x[c]);
        });
        x[j] = li == j ? 1.0 : -m;
    });
    const double rs = rsqrt_nr(dv);
    static_for<kB>([&](auto J) {
        constexpr int j = decltype(J)::value;
        a[j] *= row_value<j>(rs);
        x[j] = li >= j ? x[j] * rs : 0.0;
    });
    return good;
}

// 16 x 16 block product on MFMA: acc += X[r0:r0+16, k0:k0+16*nc] * Y[k0:k0+16*nc, c0:c0+16]
// (nc <= MAXC chunks of 16) with X element (r, k) at X[r + k*ldx] and Y element (k, c) at
// Y[yk*k + yc*c] (LDS).  Lane l supplies X[r0 + l%16][k] and Y[k][c0 + l%16] for
// k = k0 + 4s + l/16; accumulator item t of lane l is row l/16 + 4t, column l%16.  The loop is
// unrolled and the loads of chunk q+1 are issued before the four MFMAs of chunk q, so the LDS
// latency is paid once per call rather than per MFMA; the accumulation order is k ascending.
template <int MAXC>
__device__ __forceinline__ f64x4 mfma_block(const double* X, int ldx, int r0, const double* Y,
                                             int yk, int yc, int c0, int k0, int nc, f64x4 acc,
                                             int lane) {
    const int li = lane & 15, lk = lane >> 4;
    const double* xp = X + (r0 + li) + (k0 + lk) * ldx;  // element (r0 + li, k0 + lk)
    const double* yp = Y + yk * (k0 + lk) + yc * (c0 + li);
    double a[2][4], b[2][4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        a[0][s] = xp[4 * s * ldx];
        b[0][s] = yp[4 * s * yk];
    }
#pragma unroll
    for (int q = 0; q < MAXC; ++q) {
        if (q >= nc) break;
        const int cur = q & 1;
        if (q + 1 < nc) {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                a[cur ^ 1][s] = xp[(16 * (q + 1) + 4 * s) * ldx];
                b[cur ^ 1][s] = yp[(16 * (q + 1) + 4 * s) * yk];
            }
        }
#pragma unroll
        for (int s = 0; s < 4; ++s)
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[cur][s], b[cur][s], acc, 0, 0, 0);
    }
    return acc;
}

template <typename TS>
__global__ void __launch_bounds__(NTL) leaf_potrf_inv(TS* A, long lda, int nb, TS* inv,
                                                      int* info, int j0) {
    __shared__ double S[kLeaf * LD];
    __shared__ double D[kNB][kB * kB];  // inverses of the diagonal blocks, element (r, c) at r*kB+c
    __shared__ int fail;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: scalar branches
    const int li = lane & 15, lq = lane >> 4;
    // Load the lower triangle, zero-padded to kLeaf x kLeaf: wave w takes columns w, w + 8, ...,
    // every load issued before any LDS store (rows and columns clamped into the block, the
    // rows above a column's 64-row half not read, values outside the triangle replaced by 0).
    {
        constexpr int CW = kLeaf / NWL;
        const int rA = min(lane, nb - 1), rB = min(lane + 64, nb - 1);
        double v0[CW / 2], v1[CW];
#pragma unroll
        for (int q = 0; q < CW; ++q) {
            const long cc = min(wave + NWL * q, nb - 1);
            if (q < CW / 2) v0[q] = (double)A[rA + cc * lda];
            v1[q] = (double)A[rB + cc * lda];
        }
        if (*(volatile int*)info != 0) return;  // an earlier leaf failed: R is not computed
#pragma unroll
        for (int q = 0; q < CW; ++q) {
            const int c = wave + NWL * q;
            if (q < CW / 2) S_(lane, c) = (c < nb && lane < nb && lane >= c) ? v0[q] : 0.0;
            S_(lane + 64, c) = (c < nb && lane + 64 < nb && lane + 64 >= c) ? v1[q] : 0.0;
        }
    }
    if (tid == 0) fail = 0;
    __syncthreads();

    // Columns [0, ncol) of L back to global (lower part only), 16 LDS reads per lane in flight
    // before the stores.
    auto store_L = [&](int ncol) {
        for (int cb = wave; cb < ncol; cb += 8 * NWL) {
            double v0[8], v1[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int c = min(cb + NWL * q, kLeaf - 1);
                v0[q] = S_(lane, c);
                v1[q] = S_(lane + 64, c);
            }
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int c = cb + NWL * q;
                if (c >= ncol) break;
                if (lane >= c && lane < nb) A[lane + (long)c * lda] = (TS)v0[q];
                if (lane + 64 >= c && lane + 64 < nb) A[lane + 64 + (long)c * lda] = (TS)v1[q];
            }
        }
    };

    // ------------------------------------------------------------------ factorization
    // Trailing update of block kp's trailing lower triangle, tile t (16 x 16, ti >= tj, tiles
    // numbered row by row), K = 16 on MFMA: S -= P * P^T with P[r][k] = S_(r, kp + k).
    auto trail_tile = [&](int kp, int t) {
        const int base = kp + kB;
        int ti = 0, acc0 = 0;
        while (acc0 + ti + 1 <= t) acc0 += ++ti;
        const int tj = t - acc0;
        f64x4 acc = {0, 0, 0, 0};
        // B operand is P^T: element (k, c) = S_(c, kp + k)
        acc = mfma_block<1>(&S_(0, kp), LD, base + 16 * ti, &S_(0, kp), LD, 1, base + 16 * tj, 0,
                            1, acc, lane);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int r = base + 16 * ti + lq + 4 * e;
            const int c = base + 16 * tj + li;
            if (r < nb && c < nb && r >= c) S_(r, c) -= acc[e];
        }
    };
    for (int kb = 0; kb < nb; kb += kB) {
        const int bs = min(kB, nb - kb);
        double* Db = D[kb / kB];
        // Look-ahead: the previous block's trailing update runs here, beside this block's
        // diagonal factor.  Wave 0 takes tile 0 (this block's diagonal block) and then factors
        // it; the other waves take the other tiles, which this factor neither reads nor writes.
        if (kb > 0) {
            const int ht = (nb - kb + 15) / 16, ntile = ht * (ht + 1) / 2;
            if (wave == 0) trail_tile(kb - kB, 0);
            else
                for (int t = wave; t < ntile; t += NWL - 1) trail_tile(kb - kB, t);
        }
        if (wave == 0) {
            // rows and columns past nb enter as the identity
            double a[kB], x[kB];
#pragma unroll
            for (int k = 0; k < kB; ++k) {
                const double v = S_(kb + li, kb + k);
                a[k] = li < bs && k < bs ? v : (li == k ? 1.0 : 0.0);
                x[k] = 0.0;
            }
            const int good = diag_factor(a, x, li);
            if (good < kB) {
                if (lane == 0) {
                    fail = 1;
                    atomicCAS(info, 0, j0 + kb + good + 1);
                }
            } else if (lq == 0) {
#pragma unroll
                for (int k = 0; k < kB; ++k) {
                    if (li < bs && k <= li) S_(kb + li, kb + k) = a[k];
                    Db[li * kB + k] = li < bs ? x[k] : 0.0;
                }
            }
        }
        __syncthreads();
        if (fail) {
            // the 16-column blocks before the failing one are final: store them (their rows
            // below included), leave the failing block and the rest as they were
            store_L(kb);
            return;
        }
        // rows below the diagonal block: L[r, kb:kb+16] = A[r, kb:kb+16] * D^T on MFMA, a
        // 16-row tile per wave, in place (bs is 16 whenever rows remain below the block)
        const int ht = (nb - kb - bs + 15) / 16;
        for (int i = wave; i < ht; i += NWL) {
            const int r0 = kb + kB + 16 * i;
            f64x4 acc = {0, 0, 0, 0};
            // Y element (k, c) = D^T(k, c) = D(c, k)
            acc = mfma_block<1>(&S_(0, kb), LD, r0, Db, 1, kB, 0, 0, 1, acc, lane);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int r = r0 + lq + 4 * e;
                if (r < nb) S_(r, kb + li) = acc[e];
            }
        }
        __syncthreads();
    }
    store_L(nb);
    __syncthreads();

    // ------------------------------------------------------------------ inverse
    // The diagonal blocks' inverses in their place (zero past nb: rows and columns of zeros, as
    // the padding of S), then doubling.  Level h joins pairs of h x h inverses: T = L21 inv11
    // into the block above the diagonal, then inv21 = -inv22 T.  inv11 and inv22 are lower
    // triangular: 16-wide chunks outside them are skipped.
    for (int t = tid; t < kNB * kB * kB; t += NTL) {
        const int b = t / (kB * kB), r = t / kB % kB, c = t % kB;
        if (b * kB < nb) S_(b * kB + r, b * kB + c) = D[b][r * kB + c];
    }
    __syncthreads();
    auto level = [&](auto H) {
        constexpr int h = decltype(H)::value, nt = h / 16, tiles = kLeaf / 2 / h * nt * nt;
        // tile (i, j) of pair q; the column index of one half of the waves' tiles runs backwards,
        // which evens out the triangles' shorter and longer products
        auto tile = [&](int t, int& q, int& i, int& j) {
            q = t / (nt * nt);
            i = t / nt % nt;
            j = (t / NWL) & 1 ? nt - 1 - t % nt : t % nt;
        };
        for (int t = wave; t < tiles; t += NWL) {
            int q, i, j;
            tile(t, q, i, j);
            const int o = 2 * h * q;
            f64x4 acc = {0, 0, 0, 0};
            acc = mfma_block<nt>(&S_(0, o), LD, o + h + 16 * i, &S_(o, o), 1, LD, 16 * j, 16 * j,
                                 nt - j, acc, lane);
#pragma unroll
            for (int e = 0; e < 4; ++e) S_(o + 16 * i + lq + 4 * e, o + h + 16 * j + li) = acc[e];
        }
        __syncthreads();
        for (int t = wave; t < tiles; t += NWL) {
            int q, j, i;
            tile(t, q, j, i);
            const int o = 2 * h * q;
            f64x4 acc = {0, 0, 0, 0};
            acc = mfma_block<nt>(&S_(0, o + h), LD, o + h + 16 * i, &S_(o, o + h), 1, LD, 16 * j,
                                 0, i + 1, acc, lane);
#pragma unroll
            for (int e = 0; e < 4; ++e) S_(o + h + 16 * i + lq + 4 * e, o + 16 * j + li) = -acc[e];
        }
        __syncthreads();
    };
    if (nb > 16) level(std::integral_constant<int, 16>{});
    if (nb > 32) level(std::integral_constant<int, 32>{});
    if (nb > 64) level(std::integral_constant<int, 64>{});
    for (int cb = wave; cb < kLeaf; cb += 8 * NWL) {
        double v0[8], v1[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            v0[q] = S_(lane, cb + NWL * q);
            v1[q] = S_(lane + 64, cb + NWL * q);
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int c = cb + NWL * q;
            inv[lane + (long)c * kLeaf] = (TS)((lane < nb && c < nb && lane >= c) ? v0[q] : 0.0);
            inv[lane + 64 + (long)c * kLeaf] =
                (TS)((lane + 64 < nb && c < nb && lane + 64 >= c) ? v1[q] : 0.0);
        }
    }
}

#undef S_

}  // namespace

template <typename T>
int leaf_potrf_inv_launch(T* A, long lda, int nb, T* inv, int* info, int j0, hipStream_t stream) {
    if (nb < 1 || nb > kLeaf) {
        set_error("leaf_potrf: bad block size");
        return MOAO_ERR_ARG;
    }
    ProfScope ps(kProfLeaf, (double)nb * nb * nb / 3.0, stream);
    hipLaunchKernelGGL(leaf_potrf_inv<T>, dim3(1), dim3(NTL), 0, stream, A, lda, nb, inv, info,
                       j0);
    MOAO_HIP_TRY(hipGetLastError());
    return MOAO_OK;
}

template int leaf_potrf_inv_launch<double>(double*, long, int, double*, int*, int, hipStream_t);
template int leaf_potrf_inv_launch<float>(float*, long, int, float*, int*, int, hipStream_t);

}  // namespace moao
