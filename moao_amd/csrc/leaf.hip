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
//   factor: [wave 0] 16x16 diagonal block and its inverse together, in registers (diag_factor);
//           [all] rows below as A * D^T on f64 MFMA; beside the next diagonal factor, waves 1-7
//           apply the rank-16 update to the trailing lower triangle (f64 MFMA), store the
//           finished columns of L and put D in the diagonal block's place;
//   invert: by doubling: from the inverses of the 16x16 diagonal blocks to 32, 64 and 128:
//           inv(L)21 = -inv(L)22 (L21 inv(L)11), both products on f64 MFMA over all waves, the
//           inner one parked in the unused block above the diagonal; the last level's result
//           goes from the accumulators to memory.
// The time is the serial chain of one workgroup, 128 pivots long; what a pivot costs is the
// dependent instructions of its 16x16 factor (about 170 cycles) and a block's two barriers and
// LDS round trips.  In cycles of 2.4 GHz for nb = 128: load 6 thousand, eight blocks 51, inverse 17
// (of which 8 the last level, near its MFMA bound of 5).  The first design, readlane broadcasts
// under a branch per column, an inverse by block columns and stores at the end, took 166
// thousand.  70 -> 31 us a leaf.
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

// Workgroup barrier that waits for this wave's LDS accesses only: the stores to global memory,
// which no wave of the workgroup reads back, drain behind it (__syncthreads would wait for them).
__device__ __forceinline__ void lds_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0), vmcnt and expcnt at their maxima
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// 1/sqrt(d) for d > 0: hardware estimate refined by two Newton steps.
__device__ __forceinline__ double rsqrt_nr(double d) {
    double r = __builtin_amdgcn_rsq(d);
    r = r * (1.5 - 0.5 * d * r * r);
    r = r * (1.5 - 0.5 * d * r * r);
    return r;
}

// 1/d: hardware estimate (good to about 2^-23) refined by one step of third order, r (1 + e + e^2)
// with e = 1 - d r (no division on the pivots' chain).
__device__ __forceinline__ double rcp_nr(double d) {
    const double r = __builtin_amdgcn_rcp(d);
    const double e = fma(-d, r, 1.0);
    return fma(r, fma(e, e, e), r);
}

// v of every 16-lane row in all rows: r[q] = v of row q (gfx950 row swaps).
__device__ __forceinline__ void gather_rows(double v, double (&r)[4]) {
    unsigned w[2], o[4][2];
    __builtin_memcpy(w, &v, 8);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const auto p = __builtin_amdgcn_permlane16_swap(w[h], w[h], false, false);  // 0022, 1133
        const auto e = __builtin_amdgcn_permlane32_swap(p[0], p[0], false, false);
        const auto f = __builtin_amdgcn_permlane32_swap(p[1], p[1], false, false);
        o[0][h] = e[0];
        o[1][h] = f[0];
        o[2][h] = e[1];
        o[3][h] = f[1];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) __builtin_memcpy(&r[q], o[q], 8);
}

// Whether the unnormalised elimination below takes pivot d as it is, 2^-1000 <= d < 2^1000: it needs
// reciprocals (they overflow below 2^-1023) where the reciprocal square root has the whole range.
// One unsigned comparison of the high words, which negative numbers, infinities and NaN fail.
__device__ __forceinline__ bool easy_pivot(double d) {
    constexpr unsigned lo = (1023u - 1000) << 20, hi = (1023u + 1000) << 20;
    return (unsigned)__double2hiint(d) - lo < hi - lo;
}

// Exponent e that brings diagonal element li of a block (accumulator layout, see diag_factor) to
// 2^(2 e) A[li][li] in [1/2, 2); 0 where the element is not a positive number.
__device__ __forceinline__ int diag_exponent(f64x4 a, int li, int lq) {
    const int t = li >> 2;
    const double own = t & 2 ? (t & 1 ? a[3] : a[2]) : (t & 1 ? a[1] : a[0]);
    const double d = __shfl(own, li + 16 * (li & 3));  // lane row li % 4 holds column li in a[t]
    return d > 0.0 && d < __builtin_inf() ? -(__builtin_amdgcn_frexp_exp(d) >> 1) : 0;
}

// A 16 x 16 block A = L L^T and D = inv(L) in one wave.  c in MFMA accumulator layout: lane
// (li, lq) = (l % 16, l / 16) holds A[li][lq + 4t] in c[t] (lower triangle used).  Unnormalised
// elimination of [A | I], four columns at a time: columns 4t .. 4t+3 are register t of the four
// lane rows, gathered into every lane; their elimination needs six updates and their pivots'
// reciprocals; the rest of A takes them as one rank-4 MFMA, whose operands are again "column 4t +
// lq in lane row lq", and so does the inverse, with the product of the four eliminations,
// I - sum_q w_q e_q^T.  Out: lo[t] = m d (L[li][4t + lq] times the square root of its pivot, for
// li >= 4t + lq), x[t] = row 4t + lq, column li of the inverse of the unit factor, piv[t] = pivot
// 4t + lq.
__device__ __forceinline__ void diag_factor(f64x4 c, int li, int lq, double (&lo)[4],
                                            double (&piv)[4], f64x4& x) {
#pragma unroll
    for (int t = 0; t < 4; ++t) x[t] = lq + 4 * t == li ? 1.0 : 0.0;
    auto own = [&](const double (&v)[4]) {  // v[lq]
        const double a = lq & 1 ? v[1] : v[0], b = lq & 1 ? v[3] : v[2];
        return lq & 2 ? b : a;
    };
    static_for<4>([&](auto T) {
        constexpr int t = decltype(T)::value;
        double p[4], d[4], m[4], w[4];  // m, w: negated multipliers
        gather_rows(c[t], p);
        static_for<4>([&](auto Q) {
            constexpr int q = decltype(Q)::value, j = 4 * t + q;
            d[q] = row_value<j>(p[q]);
            const double r = rcp_nr(d[q]);
            m[q] = li > j ? -p[q] * r : 0.0;
            static_for<3 - q>([&](auto K) {
                constexpr int k = q + 1 + decltype(K)::value;
                p[k] = fma(m[q], row_value<4 * t + k>(p[q]), p[k]);
            });
        });
        lo[t] = own(p);
        piv[t] = own(d);
        c = __builtin_amdgcn_mfma_f64_16x16x4f64(lo[t], own(m), c, 0, 0, 0);
        static_for<4>([&](auto Q) {
            constexpr int q = 3 - decltype(Q)::value;
            w[q] = m[q];
            static_for<3 - q>([&](auto K) {
                constexpr int k = 3 - decltype(K)::value;
                w[q] = fma(w[k], row_value<4 * t + k>(m[q]), w[q]);
            });
        });
        x = __builtin_amdgcn_mfma_f64_16x16x4f64(own(w), x[t], x, 0, 0, 0);
    });
}

// L of the block to S (leading dimension LD) and its inverse to Db, both up to order bs.
__device__ __forceinline__ void store_block(const double (&lo)[4], const double (&piv)[4], f64x4 x,
                                            int li, int lq, double* S, double* Db, int bs) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const double rs = rsqrt_nr(piv[t]);
        const int col = lq + 4 * t;
        if (li < bs && col <= li) S[li + col * LD] = lo[t] * rs;
        Db[col * kB + li] = col < bs && li <= col ? x[t] * rs : 0.0;
    }
}

// A block with pivots that are not easy: once more with its diagonal scaled to about 1, c row and
// column li by 2^ex, so L's row li by 2^ex and inv(L)'s column li by 2^-ex.  The first pivot that is
// not positive (NaN included), then nothing is stored; else kB.
__device__ __noinline__ int hard_block(f64x4 c, int li, int lq, double* S, double* Db, int bs) {
    const int ex = diag_exponent(c, li, lq);
#pragma unroll
    for (int t = 0; t < 4; ++t) c[t] = ldexp(c[t], ex + __shfl(ex, lq + 4 * t));
    double lo[4], piv[4];
    f64x4 x;
    diag_factor(c, li, lq, lo, piv, x);
    int first = kB;
#pragma unroll
    for (int t = 3; t >= 0; --t)
        for (int q = 3; q >= 0; --q)
            if (__ballot(lq == q && !(piv[t] > 0.0))) first = 4 * t + q;
    if (first < kB) return first;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        lo[t] = ldexp(lo[t], -ex);
        x[t] = ldexp(x[t], ex);
    }
    store_block(lo, piv, x, li, lq, S, Db, bs);
    return kB;
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
    __shared__ double D[2][kB * kB];  // inverses of two successive diagonal blocks, (r, c) at r*kB+c
    __shared__ int fail;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: scalar branches
    const int li = lane & 15, lq = lane >> 4;
    // Load the lower triangle, zero-padded to kLeaf x kLeaf, every load issued before any LDS
    // store (rows and columns clamped into the block, the rows above a column's 64-row half not
    // read, values outside the triangle replaced by 0).  Waves 1-7 take the columns in turn; wave 0
    // reads the first diagonal block alone, into the registers it factors it in, meanwhile.
    f64x4 c = {0, 0, 0, 0};
    if (wave == 0) {
#pragma unroll
        for (int t = 0; t < 4; ++t)
            c[t] = (double)A[min(li, nb - 1) + (long)min(lq + 4 * t, nb - 1) * lda];
        if (*(volatile int*)info != 0) return;  // an earlier leaf failed: R is not computed
        if (lane == 0) fail = 0;
    } else {
        constexpr int NL = NWL - 1, CW = (kLeaf + NL - 1) / NL, CA = (kLeaf / 2 + NL - 1) / NL;
        const int rA = min(lane, nb - 1), rB = min(lane + 64, nb - 1);
        double v0[CA], v1[CW];
#pragma unroll
        for (int q = 0; q < CW; ++q) {
            const long cc = min(wave - 1 + NL * q, nb - 1);
            if (q < CA) v0[q] = (double)A[rA + cc * lda];
            v1[q] = (double)A[rB + cc * lda];
        }
        const int failed = *(volatile int*)info;
        // all in flight before the branch (the compiler would sink each load to its use)
#pragma unroll
        for (int q = 0; q < CW; ++q) {
            if (q < CA) asm volatile("" : "+v"(v0[q]));
            asm volatile("" : "+v"(v1[q]));
        }
        if (failed != 0) return;
#pragma unroll
        for (int q = 0; q < CW; ++q) {
            const int k = wave - 1 + NL * q;
            if (k >= kLeaf) break;
            const bool in = k < nb;
            if (k >= kB || lane >= kB)  // the first diagonal block is wave 0's
                S_(lane, k) = q < CA && in && lane < nb && lane >= k ? v0[q < CA ? q : 0] : 0.0;
            S_(lane + 64, k) = in && lane + 64 < nb && lane + 64 >= k ? v1[q] : 0.0;
        }
    }

    // ------------------------------------------------------------------ factorization
    // Trailing update of block kp's trailing lower triangle, tile t (16 x 16, ti >= tj, tiles
    // numbered row by row), K = 16 on MFMA: S -= P * P^T with P[r][k] = S_(r, kp + k).
    auto trail_tile = [&](int kp, int t) {
        const int base = kp + kB;
        int ti = 0, acc0 = 0;
        while (acc0 + ti + 1 <= t) acc0 += ++ti;
        const int tj = t - acc0;
        // in the accumulators from the start; rows and columns past nb hold zeros on both sides,
        // and what a diagonal tile gets above its diagonal is not read
        f64x4 acc;
        double pa[4], pb[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            acc[e] = S_(base + 16 * ti + lq + 4 * e, base + 16 * tj + li);
            pa[e] = S_(base + 16 * ti + li, kp + 4 * e + lq);
            pb[e] = S_(base + 16 * tj + li, kp + 4 * e + lq);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-pa[e], pb[e], acc, 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) S_(base + 16 * ti + lq + 4 * e, base + 16 * tj + li) = acc[e];
    };
    // Block column kp of L back to global (lower part), its diagonal block replaced by D: columns
    // f, f + stride, ... of it
    auto finish_block = [&](int kp, int f, auto stride) {
        constexpr int st = decltype(stride)::value, n = (kB + st - 1) / st;
        const double* Db = D[kp / kB & 1];
        double v0[n], v1[n], d[n];
#pragma unroll
        for (int q = 0; q < n; ++q) {
            const int k = min(f + st * q, kB - 1);
            v0[q] = S_(lane, kp + k);
            v1[q] = S_(lane + 64, kp + k);
            d[q] = Db[li * kB + k];
        }
#pragma unroll
        for (int q = 0; q < n; ++q) {
            const int k = f + st * q, c = kp + k;
            if (k >= kB || c >= nb) break;
            if (lane >= c && lane < nb) A[lane + (long)c * lda] = (TS)v0[q];
            if (lane + 64 >= c && lane + 64 < nb) A[lane + 64 + (long)c * lda] = (TS)v1[q];
            if (lane < kB) S_(kp + lane, c) = d[q];
        }
    };
    // What lies above the diagonal of the inverse (and its columns past nb): zeros in columns
    // [c0, c1)
    auto clear_inv = [&](int c0, int c1, int f, int stride) {
        for (int c = c0 + f; c < c1; c += stride) {
            if (lane < c || c >= nb) inv[lane + (long)c * kLeaf] = TS(0);
            if (lane + 64 < c || c >= nb) inv[lane + 64 + (long)c * kLeaf] = TS(0);
        }
    };
    for (int kb = 0; kb < nb; kb += kB) {
        const int bs = min(kB, nb - kb);
        double* Db = D[kb / kB & 1];
        // Look-ahead: waves 1-7 apply the previous block's trailing update (all tiles but the
        // first, this block's diagonal block, which wave 0 updates in registers) and finish that
        // block; neither touches what the factor reads or writes.  They also clear what lies above
        // the diagonal in this block's columns of the inverse: more stores where tiles are few.
        if (wave != 0) {
            if (kb > 0) {
                const int ht = (nb - kb + 15) / 16, ntile = ht * (ht + 1) / 2;
                for (int t = wave; t < ntile; t += NWL - 1) trail_tile(kb - kB, t);
                finish_block(kb - kB, wave - 1, std::integral_constant<int, NWL - 1>{});
            }
            clear_inv(kb, kb + kB, wave - 1, NWL - 1);
        } else {
            if (kb > 0) {
                double pr[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    c[t] = S_(kb + li, kb + lq + 4 * t);
                    pr[t] = S_(kb + li, kb - kB + lq + 4 * t);
                }
                // two chains: an MFMA waits 64 cycles for the one whose result it adds to
                f64x4 c2 = {0, 0, 0, 0};
#pragma unroll
                for (int t = 0; t < 4; t += 2) {
                    c = __builtin_amdgcn_mfma_f64_16x16x4f64(pr[t], -pr[t], c, 0, 0, 0);
                    c2 = __builtin_amdgcn_mfma_f64_16x16x4f64(pr[t + 1], -pr[t + 1], c2, 0, 0, 0);
                }
                c += c2;
            }
            // rows and columns past nb enter as the identity
#pragma unroll
            for (int t = 0; t < 4; ++t)
                if (li >= bs || lq + 4 * t >= bs) c[t] = li == lq + 4 * t ? 1.0 : 0.0;
            double lo[4], piv[4];
            f64x4 x;
            diag_factor(c, li, lq, lo, piv, x);
            const bool easy = easy_pivot(piv[0]) && easy_pivot(piv[1]) && easy_pivot(piv[2]) &&
                              easy_pivot(piv[3]);
            if (__ballot(!easy)) {
                const int first = hard_block(c, li, lq, &S_(kb, kb), Db, bs);
                if (first < kB && lane == 0) {
                    fail = 1;
                    atomicCAS(info, 0, j0 + kb + first + 1);
                }
            } else {
                store_block(lo, piv, x, li, lq, &S_(kb, kb), Db, bs);
            }
        }
        lds_barrier();
        const int failed = fail;
        // rows below the diagonal block: L[r, kb:kb+16] = A[r, kb:kb+16] * D^T on MFMA, a
        // 16-row tile per wave, in place (bs is 16 whenever rows remain below the block)
        const int ht = (nb - kb - bs + 15) / 16;
        for (int i = wave; i < ht; i += NWL) {
            const int r0 = kb + kB + 16 * i;
            double pa[4], pb[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                pa[e] = S_(r0 + li, kb + 4 * e + lq);
                pb[e] = Db[li * kB + 4 * e + lq];
            }
            f64x4 acc = {0, 0, 0, 0}, acc2 = {0, 0, 0, 0};
#pragma unroll
            for (int e = 0; e < 4; e += 2) {
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(pa[e], pb[e], acc, 0, 0, 0);
                acc2 = __builtin_amdgcn_mfma_f64_16x16x4f64(pa[e + 1], pb[e + 1], acc2, 0, 0, 0);
            }
            acc += acc2;
            if (failed) break;
#pragma unroll
            for (int e = 0; e < 4; ++e) S_(r0 + lq + 4 * e, kb + li) = acc[e];
        }
        // a failing pivot: the 16-column blocks before this one are final and stored (their rows
        // below included); this block and the rest stay as they were
        if (failed) return;
        lds_barrier();
    }
    finish_block((nb - 1) / kB * kB, wave, std::integral_constant<int, NWL>{});
    clear_inv((nb + kB - 1) / kB * kB, kLeaf, wave, NWL);
    lds_barrier();

    // ------------------------------------------------------------------ inverse
    // The diagonal blocks' inverses are in their place (zero past nb: rows and columns of zeros,
    // as the padding of S).  Doubling: level h joins pairs of h x h inverses: T = L21 inv11 into
    // the block above the diagonal, then inv21 = -inv22 T.  inv11 and inv22 are lower triangular:
    // 16-wide chunks outside them are skipped.
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
        lds_barrier();
        for (int t = wave; t < tiles; t += NWL) {
            int q, j, i;
            tile(t, q, j, i);
            const int o = 2 * h * q;
            f64x4 acc = {0, 0, 0, 0};
            acc = mfma_block<nt>(&S_(0, o + h), LD, o + h + 16 * i, &S_(o, o + h), 1, LD, 16 * j,
                                 0, i + 1, acc, lane);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int r = o + h + 16 * i + lq + 4 * e, c = o + 16 * j + li;
                if (h < kLeaf / 2) S_(r, c) = -acc[e];
                else inv[r + (long)c * kLeaf] = (TS)-acc[e];
            }
        }
        if (h < kLeaf / 2) lds_barrier();
    };
    if (nb > 16) level(std::integral_constant<int, 16>{});
    if (nb > 32) level(std::integral_constant<int, 32>{});
    // the two 64 x 64 diagonal blocks of the inverse are done
    for (int c = wave; c < nb; c += NWL) {
        const int r = (c & 64) + lane;
        const double v = S_(r, c);
        if (r >= c) inv[r + (long)c * kLeaf] = (TS)(r < nb ? v : 0.0);
    }
    if (nb > 64) {
        level(std::integral_constant<int, 64>{});
    } else {
        for (int c = wave; c < nb; c += NWL) inv[lane + 64 + (long)c * kLeaf] = TS(0);
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
