// Intersample PSF (common/tomo_struct/intersample.cpp:72-171) on gfx950, batched over
// directions, FP32 (or FP64) FFTs, two directions per complex grid (real and imaginary parts).
//
// Reference steps, per direction:
//   Map[idx[i]-1] += Cvv[i]; Map /= div; embed Map in the N x N grid at stride dactupix
//   r2c FFT; *= abs2fi[j*N+i] (real part); c2r
//   dphi = exp(-0.5 (norm - dphi/fact2*fact)); _eclat
//   tmp = otf_tel[j*N+i]*dphi[j*N+i]; c2r; _eclat -> PSF
// with the reference's constants: lambda = 1.65e-6, fact = 2 (2*3.14159/lambda)^2,
// fact2 = N^2 dactupix^2, dactupix = N/(3(np-1)) + 1 (integer division), norm at
// (N/2, N/2).  N defaults to the reference's max(512, 8*2^floor(ln(np)+0.5))
// (intersample.cpp:192) and may be set explicitly (a 2048 grid is not reachable by that rule).
//
// Everything after the map is even.  The real part of a real map's spectrum is the spectrum of
// the map's even part (z(x) + z(-x)) / 2, and the half-spectrum product that a c2r transform
// extends by its Hermitian mirror is real and even, so D, dphi, the second spectrum and the PSF
// all satisfy f(-x, -y) = f(x, y).  The map is made even first; then every 2-D array needs its
// lines 0 .. N/2 only, the others being mirrors, and each transform runs half its rows:
//   gather_runs  Cvv -> partial sums of the map bins
//   map_rows     partial sums -> even map; transform of its 2 np - 1 rows (the grid's other rows
//                are zero) -> A
//   map_cols     per column j <= N/2: transform along x, times abs2fi, back along x -> H
//   dphi_rows    per row: along y -> D; dphi, times the OTF; along the shifted row -> H2
//   psf_rows     per row: along the last axis -> PSF, and its mirror row
// Between passes H(x, j) and H(-x, j) are stored for x = N/2 .. N and j = 0 .. N/2, in tiles of
// kRows x kRows that the writing workgroup fills and the reading workgroup takes whole.
// N = 2048, 8 directions, FP32, nact = 4,724: 6 launches, 0.54 ms (gather 0.37, then 0.01, 0.01,
// 0.04, 0.06, 0.06); as full transforms (radix-4 rows, transpose, rows) with pointwise passes and a
// gather by entries between them 15 launches, 2.2 ms, of which the gather 1.17.  N = 512, one
// direction, FP64: 49 -> 18 us.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <deque>
#include <vector>

#include "common.hpp"
#include "fft.hpp"
#include "profile.hpp"

struct moao_isample {
    long N = 0, np = 0, nidx = 0, ncov = 0, nmap = 0;
    double lambda = 1.65e-06, dactupix = 0;
    int prec = 0;  // 0 FP32, 1 FP64
    int batch_cap = 0;
    // Cvv as runs of consecutive entries in consecutive map bins (see gather_runs), or as a list of
    // entries per bin (gather_entries): run_of then holds the bins' offsets, item_of the entries
    bool entries = false;
    int order = 0, width = 0, nslab = 0, ngroup = 0, nitem = 0;
    long slab = 0;
    void* runs = nullptr;
    void* items = nullptr;
    int* run_of = nullptr;
    int* item_of = nullptr;
    double* div = nullptr;     // [nmap] hit counts
    void* a2f = nullptr;       // [N*N] abs2fi (R), reference flat layout
    void* otf = nullptr;       // [N*N] otf_tel (R)
    void* tw = nullptr;        // twiddles
    void* work = nullptr;      // workspace of batch_cap directions, in it:
    double* part = nullptr;    // partial sums of the map bins, one set per slab
    double* sums = nullptr;    // their sums
    void* A = nullptr;         // transformed map rows
    void* X = nullptr;         // H after abs2fi and after the OTF
    void* Y = nullptr;
    void* mid = nullptr;       // H(N/2, j)
    double* dCvv = nullptr;    // host-entry staging
    double* dPsf = nullptr;
};

namespace moao {
namespace {

// Cvv as runs.  The map bins are taken in the order along which consecutive Cvv entries most often
// fall (kOrder*: along a map row or column, up or down), W * 64 of them to a group.  A run is a
// stretch of at most 64 consecutive Cvv entries that fall in consecutive bins of one group: one
// load of neighbouring doubles, bin number mod 64 on each lane, described by 8 bytes (where it
// starts, its first bin, its length) instead of an index per entry.  A pair list of actuators on
// a grid gives whole DM rows, ~50 entries at 80 actuators across; any other index is served too,
// by shorter runs.  Cvv is cut into slabs of equal length; an item is one group in one slab.
struct Run {
    int key;           // first entry, from the slab's start
    unsigned bin_len;  // first bin in the group, length << 16
};
struct Item {
    int slab, group;
};
constexpr int kGatherWaves = 8;  // waves per item
constexpr int kRunsAhead = 8;    // runs that a wave loads at a time
constexpr int kMaxSlabs = 32;
// Entries per run from which runs are used (gather_entries below).  8 directions, nact = 4,724:
// runs take 0.38 ms at 35 entries each and 6.9 ms at one; entry by entry 1.2 ms where neighbouring
// bins read neighbouring entries and 3.3 ms in random order.
constexpr long kRunFrom = 4;
constexpr long kSlabMax = 1L << 26;  // doubles: byte offsets in a slab stay below 2^31
// Bins per group, in blocks of 64: wide groups read a DM row with one wave, so its cache lines are
// fetched once; narrower ones spread the work of a small map or a single direction.  nact = 4,724,
// whole call at N = 512, us by 2, 3, 5, 8 blocks: 8 directions 406, 398, 398, 403; one 62, 72, 99,
// 159.
constexpr int kWide = 3, kWideFrom = 128 * 64;

enum { kOrderRowUp = 0, kOrderRowDown, kOrderColUp, kOrderColDown };
__host__ __device__ inline int bin_place(int order, int ti, int tj, int ncov) {
    const int c = order < kOrderColUp ? ti * ncov + tj : tj * ncov + ti;
    return order & 1 ? ncov * ncov - 1 - c : c;
}

// Partial sums of one item for ND directions; the waves take 8 runs each in turn.  Bound by HBM:
// 1.43 GB of Cvv (nact = 4,724, 8 directions) in 370 us; with groups of 64 bins, where rows are cut
// at every group, 400 us and 1.4 times the cache lines.  Lanes outside a run and directions outside
// the batch read past the buffer resource's end, which the hardware answers with zero and no
// traffic, so the loads stand without branches.  A run lies in blocks k and k + 1 of the group's W
// blocks of 64 bins, k uniform. XCD c takes the c-th eighth of the items. part[((item W + k) batch
// + direction) 64 + lane].
template <int W, int ND>
__global__ __launch_bounds__(kGatherWaves * 64) void gather_runs(
    const double* __restrict__ cvv, long nidx, long slab, const Item* __restrict__ items,
    const int* __restrict__ run_of, const Run* __restrict__ runs, double* __restrict__ part,
    int batch) {
    __shared__ double red[kGatherWaves][ND][64];
    const int n = gridDim.x, per = n / 8, L = blockIdx.x;
    const int it = L < per * 8 ? (L % 8) * per + L / 8 : L;
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r0 = run_of[it], r1 = run_of[it + 1];
    const long i0 = items[it].slab * slab, len = nidx - i0 < slab ? nidx - i0 : slab;
    __amdgpu_buffer_rsrc_t src[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) {
        const int b = blockIdx.y * ND + d;
        src[d] = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(cvv + (size_t)(b < batch ? b : 0) * nidx + i0), 0,
            b < batch ? (int)(len * 8) : 0, 0x00020000);
    }
    double acc[W][ND] = {};
    for (int r = r0 + w * kRunsAhead; r < r1; r += kGatherWaves * kRunsAhead) {
        double v[kRunsAhead][ND];
        int at[kRunsAhead];
#pragma unroll
        for (int a = 0; a < kRunsAhead; ++a) {
            const Run q = runs[r + a < r1 ? r + a : r1 - 1];
            const int m = r + a < r1 ? (int)(q.bin_len >> 16) : 0;
            at[a] = q.bin_len & 0xffff;
            const int o = (lane - at[a]) & 63;
            const unsigned off = o < m ? (unsigned)(q.key + o) * 8u : 0xfffffff8u;
#pragma unroll
            for (int d = 0; d < ND; ++d)
                v[a][d] = __builtin_bit_cast(
                    double, __builtin_amdgcn_raw_buffer_load_b64(src[d], off, 0, 0));
        }
#pragma unroll
        for (int a = 0; a < kRunsAhead; ++a) {
            const bool lo = lane >= (at[a] & 63);
            const int ka = at[a] >> 6;
#pragma unroll
            for (int k = 0; k < W; ++k)
                if (ka == k) {
#pragma unroll
                    for (int d = 0; d < ND; ++d) {
                        acc[k][d] += lo ? v[a][d] : 0.0;
                        if (k + 1 < W) acc[k + 1][d] += lo ? 0.0 : v[a][d];
                    }
                }
        }
    }
#pragma unroll
    for (int k = 0; k < W; ++k) {
        __syncthreads();
#pragma unroll
        for (int d = 0; d < ND; ++d) red[w][d][lane] = acc[k][d];
        __syncthreads();
        const int b = blockIdx.y * ND + w;
        if (w < ND && b < batch) {
            double s = 0;
#pragma unroll
            for (int h = 0; h < kGatherWaves; ++h) s += red[h][w][lane];
            part[((size_t)(it * W + k) * batch + b) * 64 + lane] = s;
        }
    }
}

// The same sums where consecutive entries seldom fall in consecutive bins: one wave per bin over
// the list of its entries.  Sums as map_sums leaves them.
__global__ __launch_bounds__(256) void gather_entries(const double* __restrict__ cvv, long nidx,
                                                      const int* __restrict__ off,
                                                      const int* __restrict__ ent, int nmap,
                                                      double* __restrict__ sums) {
    const int bin = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (bin >= nmap) return;
    const double* c = cvv + (size_t)blockIdx.y * nidx;
    double acc = 0.0;
    for (int e = off[bin] + lane; e < off[bin + 1]; e += 64) acc += c[ent[e]];
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o, 64);
    if (lane == 0) sums[((size_t)(bin >> 6) * gridDim.y + blockIdx.y) * 64 + (bin & 63)] = acc;
}

// Sums over the slabs: one workgroup per 64 bins and direction, each wave every fourth slab, 8
// at a time.  sums[(bins/64 batch + direction) 64 + lane], the layout part has with one slab.
__global__ __launch_bounds__(256) void map_sums(const double* __restrict__ part,
                                                const int* __restrict__ item_of, int nslab,
                                                int ngroup, int W, double* __restrict__ sums) {
    __shared__ double red[4][64];
    const int g = blockIdx.x, b = blockIdx.y, batch = gridDim.y;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    double acc = 0;
    for (int q0 = w; q0 < nslab; q0 += 32) {
        double v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int q = q0 + 4 * k;
            const int it = item_of[(q < nslab ? q : q0) * ngroup + g / W];
            v[k] = part[((size_t)((it < 0 ? 0 : it) * W + g % W) * batch + b) * 64 + lane];
            if (it < 0 || q >= nslab) v[k] = 0;
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) acc += v[k];
    }
    red[w][lane] = acc;
    __syncthreads();
    if (w == 0)
        sums[((size_t)g * batch + b) * 64 + lane] =
            (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]);
}

// What the row passes share.
template <typename R>
struct Grid {
    using C = typename Cplx<R>::type;
    int ncov, first, step;
    const C* tw;
};

// Tile line and pair of directions of a workgroup.  Tile line N/2 / K holds line N/2 alone: those
// go first, so that the launch does not end on them.
template <typename F>
__device__ __forceinline__ int2 tile_line() {
    constexpr int NB = F::N / 2 / F::kRows;
    const int pairs = gridDim.x / (NB + 1), L = (int)blockIdx.x - pairs;
    return L < 0 ? int2{NB, (int)blockIdx.x} : int2{L % NB, L / NB};
}

// Index of column (or row) x of the grid in the map, -1 off the map.
__device__ __forceinline__ int map_index(int x, int first, int step, int ncov) {
    const int d = x - first;
    const int q = (int)(((float)d + 0.5f) * (1.0f / (float)step));  // exact below 2^12
    return d >= 0 && q * step == d && q < ncov ? q : -1;
}

// H of one line j (or r) for all x, to the tiles: x = N/2 + r goes to P(r, j) = H(N/2 + r, j),
// x = N/2 - r to M(r, j) = H(-(N/2 + r), j); r = 0 and N/2 are both.  Tile (r/K, j/K) holds its
// P then its M values, j slow.
template <typename F>
__device__ __forceinline__ size_t tile_at(int r, int j, int m) {
    constexpr int K = F::kRows, NB = F::N / 2 / K + 1;
    return ((((size_t)(r / K) * NB + j / K) * 2 + m) * K + j % K) * K + r % K;
}
template <typename F>
__device__ __forceinline__ size_t grid_size() {
    constexpr int K = F::kRows, NB = F::N / 2 / K + 1;
    return (size_t)NB * NB * 2 * K * K;
}
template <typename F>
__device__ __forceinline__ void store_line(const typename F::C (&v)[F::E], typename F::C* H,
                                           int t, int j) {
    constexpr int N = F::N;
    if (j > N / 2) return;
#pragma unroll
    for (int e = 0; e < F::E; ++e) {
        const int x = t + F::T * e;
        if (e >= F::E / 2)
            H[tile_at<F>(x - N / 2, j, 0)] = v[e];
        else
            H[tile_at<F>(N / 2 - x, j, 1)] = v[e];
        if (e == 0 && t == 0) H[tile_at<F>(N / 2, j, 0)] = v[e];
        if (e == F::E / 2 && t == 0) H[tile_at<F>(0, j, 1)] = v[e];
    }
}
// Line r back, over all j: H(N/2 + r, j) = P(r, j) up to N/2 and M(r, N - j) past it.  Lines
// past N/2 (the last tile's) hold nothing and are not used.
template <typename F>
__device__ __forceinline__ void load_line(typename F::C (&v)[F::E], const typename F::C* H,
                                          int t, int r) {
    constexpr int N = F::N;
#pragma unroll
    for (int e = 0; e < F::E; ++e) {
        const int j = t + F::T * e;
        const bool m = j > N / 2;
        v[e] = H[tile_at<F>(r, m ? N - j : j, m)];
    }
}
// Line j <= N/2 of a weight.  Lines 0 and N/2 hold both k and -k: the weight is averaged over
// the pair, so the product stays even whatever the weights (a c2r transform keeps only that
// even part).
template <typename R, typename F>
__device__ __forceinline__ void load_weight(R (&w)[F::E], const R* __restrict__ W, int t, int j) {
    constexpr int N = F::N;
    const R* row = W + (size_t)(j <= N / 2 ? j : N / 2) * N;
#pragma unroll
    for (int e = 0; e < F::E; ++e) w[e] = row[t + F::T * e];
    if (j == 0 || j == N / 2) {
#pragma unroll
        for (int e = 0; e < F::E; ++e)
            w[e] = (R)0.5 * (w[e] + row[(N - t - F::T * e) & (N - 1)]);
    }
}

// Even map of two directions and its rows' transforms: A(ti, j) at ((j/K) ncov + ti) K + j%K,
// j <= N/2.  A bin's sum is divided by its hit count; the mirror bin of (ti, tj) is
// (ncov-1-ti, ncov-1-tj).
template <typename R, int LOG>
__global__ __launch_bounds__((RowFft<R, LOG>::kThreads), (RowFft<R, LOG>::kWaves)) void map_rows(
    Grid<R> g, const double* __restrict__ sums, int order, const double* __restrict__ div,
    int batch,
    typename Cplx<R>::type* __restrict__ A) {
    using F = RowFft<R, LOG>;
    using C = typename F::C;
    constexpr int N = F::N, K = F::kRows;
    __shared__ C lds[F::kLds];
    const int t = threadIdx.x / K, row = threadIdx.x % K, p = blockIdx.y;
    for (int u = threadIdx.x; u < K * g.ncov; u += F::kThreads) {
        const int ti = blockIdx.x * K + u / g.ncov, tj = u % g.ncov;
        double z[2] = {0, 0};
        if (ti < g.ncov) {
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                const int yi = m ? g.ncov - 1 - ti : ti, yj = m ? g.ncov - 1 - tj : tj;
                const int at = bin_place(order, yi, yj, g.ncov), d1 = 2 * p + 1 < batch;
                const double* v = sums + ((size_t)(at >> 6) * batch + 2 * p) * 64 + (at & 63);
                const double sa = v[0], sb = v[d1 * 64];
                const double h = div[yi * g.ncov + yj];  // no hits: the sum is 0
                z[0] += h > 0 ? 0.5 * (sa / h) : 0.0;
                z[1] += h > 0 && d1 ? 0.5 * (sb / h) : 0.0;
            }
        }
        lds[u] = C{(R)z[0], (R)z[1]};
    }
    __syncthreads();
    C v[F::E];
    const auto tw = F::template twiddles<false>(g.tw, t);
#pragma unroll
    for (int e = 0; e < F::E; ++e) {
        const int tj = map_index(t + F::T * e, g.first, g.step, g.ncov);
        const C c = lds[row * g.ncov + (tj < 0 ? 0 : tj)];
        v[e] = tj < 0 ? C{0, 0} : c;
    }
    F::template run<-1>(v, lds, t, row, tw);
    const int ti = blockIdx.x * K + row;
    if (ti >= g.ncov) return;
    A += (size_t)p * (N / 2 / K + 1) * K * g.ncov;
#pragma unroll
    for (int e = 0; e <= F::E / 2; ++e) {
        const int j = t + F::T * e;
        if (j <= N / 2) A[((size_t)(j / K) * g.ncov + ti) * K + j % K] = v[e];
    }
}

// Whether the middle runs (map_cols, the first of dphi_rows) take their twiddles from the table.  The
// kept ones take registers beside the row's: N = 1024, FP32, 8 directions, kept -> table 16.5 ->
// 14.3 us in map_cols; N = 2048, where a run's loads are more, 40 -> 44.
template <typename F>
constexpr bool middle_from_table = F::N <= 1024;

// Bound by its writes (67 MB at N = 2048 and 4 pairs, 40 us): columns j <= N/2, transform along x,
// product with abs2fi, transform back.  mid[j] = H(N/2, j).
template <typename R, int LOG>
__global__ __launch_bounds__((RowFft<R, LOG>::kThreads), (RowFft<R, LOG>::kWaves)) void map_cols(
    Grid<R> g, const typename Cplx<R>::type* __restrict__ A, const R* __restrict__ w,
    typename Cplx<R>::type* __restrict__ H, typename Cplx<R>::type* __restrict__ mid) {
    using F = RowFft<R, LOG>;
    using C = typename F::C;
    constexpr int N = F::N, K = F::kRows, NB = N / 2 / K + 1;
    __shared__ C lds[F::kLds];
    const int t = threadIdx.x / K, row = threadIdx.x % K;
    const int2 b = tile_line<F>();
    const int j = b.x * K + row, p = b.y;
    A += ((size_t)p * NB + b.x) * K * g.ncov + row;
    C v[F::E];
    const auto tw = F::template twiddles<middle_from_table<F>>(g.tw, t);
    R wt[F::E];
#pragma unroll
    for (int e = 0; e < F::E; ++e) {
        const int ti = map_index(t + F::T * e, g.first, g.step, g.ncov);
        const C c = A[(size_t)(ti < 0 ? 0 : ti) * K];
        v[e] = ti < 0 ? C{0, 0} : c;
    }
    load_weight<R, F>(wt, w, t, j);
    F::template run<-1>(v, lds, t, row, tw);
#pragma unroll
    for (int e = 0; e < F::E; ++e) v[e] = C{v[e].x * wt[e], v[e].y * wt[e]};
    F::template run<1>(v, lds, t, row, tw);
    store_line<F>(v, H + p * grid_size<F>(), t, j);
    if (t == 0 && j <= N / 2) mid[(size_t)p * (N / 2 + 1) + j] = v[F::E / 2];
}

// exp(x).  FP32 transforms: x = n ln 2 + f, |f| <= ln 2 / 2, Taylor's series of e^f to f^11 in FP64
// (remainder below 7e-15), rounded to FP32 by the caller: with the FP64 library function dphi_rows
// takes 80 us, not 57.  The clamp keeps n in range; a NaN passes it.
template <typename R>
__device__ __forceinline__ double phase_exp(double x) {
    if constexpr (sizeof(R) == 8) {
        return exp(x);
    } else {
        x = x > 800.0 ? 800.0 : x;
        x = x < -800.0 ? -800.0 : x;
        const double n = __builtin_rint(x * 1.4426950408889634074);
        const double f = __builtin_fma(n, -0.69314718055994530942, x);
        double y = 1.0 / 39916800;
        y = __builtin_fma(y, f, 1.0 / 3628800);
        y = __builtin_fma(y, f, 1.0 / 362880);
        y = __builtin_fma(y, f, 1.0 / 40320);
        y = __builtin_fma(y, f, 1.0 / 5040);
        y = __builtin_fma(y, f, 1.0 / 720);
        y = __builtin_fma(y, f, 1.0 / 120);
        y = __builtin_fma(y, f, 1.0 / 24);
        y = __builtin_fma(y, f, 1.0 / 6);
        y = __builtin_fma(y, f, 0.5);
        y = __builtin_fma(y, f, 1.0);
        y = __builtin_fma(y, f, 1.0);
        return __builtin_ldexp(y, (int)n);
    }
}

// Bound half by memory (67 MB in, 67 MB out), half by arithmetic; 57 us at N = 2048, 4 pairs.
// Rows N/2 + r, r <= N/2: D along y, dphi = exp(-0.5 (norm - D) scale), scale = fact / fact2,
// shifted by half a row (its row r, column y + N/2), times the OTF's row r, transform along the
// row. norm = D(N/2, N/2) = the alternating sum of H(N/2, j) over all j, taken in FP64.
template <typename R, int LOG>
__global__ __launch_bounds__((RowFft<R, LOG>::kThreads), (RowFft<R, LOG>::kWaves)) void dphi_rows(
    Grid<R> g, const typename Cplx<R>::type* __restrict__ H,
    const typename Cplx<R>::type* __restrict__ mid, const R* __restrict__ otf, double scale,
    typename Cplx<R>::type* __restrict__ H2) {
    using F = RowFft<R, LOG>;
    using C = typename F::C;
    constexpr int N = F::N, K = F::kRows, E = F::E;
    constexpr int kWave = F::kThreads < 64 ? F::kThreads : 64;
    __shared__ C lds[F::kLds];
    __shared__ double red[2][F::kThreads / kWave];
    const int t = threadIdx.x / K, row = threadIdx.x % K;
    const int2 b = tile_line<F>();
    const int r = b.x * K + row, p = b.y;
    C v[E];
    const auto tw = F::template twiddles<middle_from_table<F>>(g.tw, t);
    load_line<F>(v, H + p * grid_size<F>(), t, r);
    mid += (size_t)p * (N / 2 + 1);
    double na = 0, nb = 0;
    for (int j = threadIdx.x; j <= N / 2; j += F::kThreads) {
        const C c = mid[j];
        const double s = (j & 1 ? -1.0 : 1.0) * (j == 0 || j == N / 2 ? 1.0 : 2.0);
        na += s * (double)c.x;
        nb += s * (double)c.y;
    }
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
        na += __shfl_xor(na, o, 64);
        nb += __shfl_xor(nb, o, 64);
    }
    if (threadIdx.x % kWave == 0) {
        red[0][threadIdx.x / kWave] = na;
        red[1][threadIdx.x / kWave] = nb;
    }
    F::template run<1>(v, lds, t, row, tw);  // its barriers order red as well
    R wt[E];
    load_weight<R, F>(wt, otf, t, r);
    na = nb = 0;
#pragma unroll
    for (int q = 0; q < F::kThreads / kWave; ++q) {
        na += red[0][q];
        nb += red[1][q];
    }
    na *= scale;
    nb *= scale;
    C x[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int i = (e + E / 2) % E;  // column y + N/2
        x[i] = C{wt[i] * (R)phase_exp<R>(-0.5 * (na - (double)v[e].x * scale)),
                 wt[i] * (R)phase_exp<R>(-0.5 * (nb - (double)v[e].y * scale))};
    }
    // read again, not kept across the exponentials: the registers decide the occupancy
    int again = t;
    asm volatile("" : "+v"(again));
    F::template run<1>(x, lds, t, row, F::template twiddles<true>(g.tw, again));
    store_line<F>(x, H2 + p * grid_size<F>(), t, r);
}

// Bound by its writes (268 MB of FP64 images in 61 us; 95 us when stored in lane order).
// PSF rows r <= N/2 (grid row N/2 + r before the shift) and their mirrors N - r.
template <typename R, int LOG>
__global__ __launch_bounds__((RowFft<R, LOG>::kThreads), (RowFft<R, LOG>::kWaves)) void psf_rows(
    Grid<R> g, const typename Cplx<R>::type* __restrict__ H2, double* __restrict__ psf,
    int batch) {
    using F = RowFft<R, LOG>;
    using C = typename F::C;
    constexpr int N = F::N, K = F::kRows, E = F::E;
    __shared__ C lds[F::kLds];
    const int t = threadIdx.x / K, row = threadIdx.x % K;
    const int2 b = tile_line<F>();
    const int r = b.x * K + row, p = b.y;
    C v[E];
    const auto tw = F::template twiddles<true>(g.tw, t);
    load_line<F>(v, H2 + p * grid_size<F>(), t, r);
    F::template run<1>(v, lds, t, row, tw);
    // Through LDS by rows, so that every store is a contiguous kilobyte of one image row; lane
    // order would give 128-byte pieces of 4 rows, off the line boundaries in the mirror rows.
    constexpr int kPad = F::T < 16 ? F::T : 16;  // rows a half turn of the banks apart
    static_assert(K * (N + kPad) <= F::kLds);
    __syncthreads();
#pragma unroll
    for (int e = 0; e < E; ++e) lds[row * (N + kPad) + t + F::T * ((e + E / 2) % E)] = v[e];
    __syncthreads();
    const bool two = 2 * p + 1 < batch;
    double* out = psf + (size_t)(2 * p) * N * N;
#pragma unroll
    for (int q = 0; q < E / 2; ++q) {
        const int u = threadIdx.x + q * F::kThreads, c = 2 * (u % (N / 2)), rr = b.x * K + u / (N / 2);
        const C* l = lds + u / (N / 2) * (N + kPad);
        if (rr > N / 2) break;
        const C a0 = l[c], a1 = l[c + 1];
        double* o = out + (size_t)rr * N + c;
        *(double2*)o = double2{(double)a0.x, (double)a1.x};
        if (two) *(double2*)(o + (size_t)N * N) = double2{(double)a0.y, (double)a1.y};
        if (rr == 0 || rr == N / 2) continue;
        const C m0 = l[(N - c) & (N - 1)], m1 = l[N - c - 1];
        o = out + (size_t)(N - rr) * N + c;
        *(double2*)o = double2{(double)m0.x, (double)m1.x};
        if (two) *(double2*)(o + (size_t)N * N) = double2{(double)m0.y, (double)m1.y};
    }
}

// Long-exposure sum: sum[i] += psf[i] (one FP64 addition per element and step, so the sum
// equals a host loop that adds the steps' PSFs in the same order).
__global__ void psf_accumulate(const double* __restrict__ psf, long count,
                               double* __restrict__ sum) {
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i < count) sum[i] += psf[i];
}

template <typename R, int LOG>
int passes(moao_isample* S, int batch, double* dPsf, hipStream_t s) {
    using F = RowFft<R, LOG>;
    using C = typename F::C;
    constexpr int N = F::N, K = F::kRows, NB = N / 2 / K + 1;
    const int ncov = (int)S->ncov, pairs = (batch + 1) / 2;
    const double half = (double)NB * K * N * sizeof(C) * pairs;  // bytes of one H
    Grid<R> g{ncov, (int)(N / 2 - (ncov - 1) / 2 * S->dactupix), (int)S->dactupix,
              (const C*)S->tw};
    const double fact = 2 * std::pow(2 * 3.14159 / S->lambda, 2);
    const double fact2 = (double)N * N * S->dactupix * S->dactupix;
    ProfScope ps(kProfFft, 4 * half + 8.0 * N * N * batch, s);
    const dim3 grid(NB * pairs), block(F::kThreads);
    hipLaunchKernelGGL((map_rows<R, LOG>), dim3((ncov + K - 1) / K, pairs), block, 0, s, g,
                       S->entries || S->nslab > 1 ? S->sums : S->part, S->order, S->div, batch, (C*)S->A);
    hipLaunchKernelGGL((map_cols<R, LOG>), grid, block, 0, s, g, (const C*)S->A,
                       (const R*)S->a2f, (C*)S->X, (C*)S->mid);
    hipLaunchKernelGGL((dphi_rows<R, LOG>), grid, block, 0, s, g, (const C*)S->X,
                       (const C*)S->mid, (const R*)S->otf, fact / fact2, (C*)S->Y);
    hipLaunchKernelGGL((psf_rows<R, LOG>), grid, block, 0, s, g, (const C*)S->Y, dPsf, batch);
    MOAO_HIP_TRY(hipGetLastError());
    return MOAO_OK;
}

// Complex values of H, A and mid per pair of directions (K rows per workgroup, NB tiles)
struct Sizes {
    size_t h, a, mid;
};
Sizes sizes(const moao_isample* S) {
    const size_t K = S->prec == 1 && S->N == 4096 ? 2 : 4, NB = S->N / 2 / K + 1;
    return {NB * NB * 2 * K * K, NB * K * S->ncov, (size_t)S->N / 2 + 1};
}

template <typename R>
int process(moao_isample* S, const double* dCvv, int batch, double* dPsf, hipStream_t s) {
    using C = typename Cplx<R>::type;
    const size_t pairs = (batch + 1) / 2;
    if (batch > S->batch_cap) {
        const Sizes z = sizes(S);
        void** const buf[] = {&S->X, &S->Y, &S->A, &S->mid, (void**)&S->part, (void**)&S->sums};
        const size_t bytes[] = {sizeof(C) * z.h * pairs, sizeof(C) * z.h * pairs,
                                sizeof(C) * z.a * pairs, sizeof(C) * z.mid * pairs,
                                sizeof(double) * 64 * S->width * S->nitem * batch,
                                sizeof(double) * 64 * S->width * S->ngroup * batch};
        size_t at[7] = {};
        for (int k = 0; k < 6; ++k) at[k + 1] = at[k] + (bytes[k] + 255) / 256 * 256;
        S->batch_cap = 0;
        if (S->work) (void)hipFree(S->work);
        S->work = nullptr;
        MOAO_HIP_TRY(hipMalloc(&S->work, at[6]));
        for (int k = 0; k < 6; ++k) *buf[k] = (char*)S->work + at[k];
        S->batch_cap = batch;
    }
    {
        ProfScope ps(kProfOther, 8.0 * S->nidx * batch, s);
        if (S->entries) {
            hipLaunchKernelGGL(gather_entries, dim3((S->nmap + 3) / 4, batch), dim3(256), 0, s, dCvv,
                               S->nidx, S->run_of, S->item_of, (int)S->nmap, S->sums);
        } else {
            const int nd = batch > 1 ? 2 : 1;  // directions per reading of the runs
            const dim3 grid(S->nitem, (batch + nd - 1) / nd);
            auto* k = S->width == kWide ? (nd == 2 ? gather_runs<kWide, 2> : gather_runs<kWide, 1>)
                                        : (nd == 2 ? gather_runs<1, 2> : gather_runs<1, 1>);
            hipLaunchKernelGGL(k, grid, dim3(kGatherWaves * 64), 0, s, dCvv, S->nidx, S->slab,
                               (const Item*)S->items, S->run_of, (const Run*)S->runs, S->part, batch);
            if (S->nslab > 1)
                hipLaunchKernelGGL(map_sums, dim3((S->nmap + 63) / 64, batch), dim3(256), 0, s, S->part,
                                   S->item_of, S->nslab, S->ngroup, S->width, S->sums);
        }
        MOAO_HIP_TRY(hipGetLastError());
    }
    switch (S->N) {
        case 32: return passes<R, 5>(S, batch, dPsf, s);
        case 64: return passes<R, 6>(S, batch, dPsf, s);
        case 128: return passes<R, 7>(S, batch, dPsf, s);
        case 256: return passes<R, 8>(S, batch, dPsf, s);
        case 512: return passes<R, 9>(S, batch, dPsf, s);
        case 1024: return passes<R, 10>(S, batch, dPsf, s);
        case 2048: return passes<R, 11>(S, batch, dPsf, s);
        default: return passes<R, 12>(S, batch, dPsf, s);
    }
}

// The runs of every item, from idx.
struct Plan {
    bool entries = false;  // by entries: run_of has the bins' offsets, item_of the entries
    int order = 0, width = 1, nslab = 1, ngroup = 0;
    long slab = 0;
    std::vector<Run> runs;
    std::vector<Item> items;
    std::vector<double> div;   // hits per map bin
    std::vector<int> run_of;   // [items + 1]
    std::vector<int> item_of;  // [nslab][ngroup], -1 where a group has nothing in a slab
};
// False if an index lies off the map.
bool make_plan(const long* idx, long nidx, int ncov, Plan* plan) {
    Plan& P = *plan;
    const long nmap = (long)ncov * ncov;
    long votes[4] = {};
    for (long i = 0; i + 1 < nidx; i += nidx >> 20 | 1) {  // a million pairs tell
        const long d = idx[i + 1] - idx[i];
        votes[0] += d == 1;
        votes[1] += d == -1;
        votes[2] += d == ncov;
        votes[3] += d == -ncov;
    }
    for (int o = 1; o < 4; ++o)
        if (votes[o] > votes[P.order]) P.order = o;
    std::vector<int> place(nmap);
    for (int b = 0; b < nmap; ++b) place[b] = bin_place(P.order, b / ncov, b % ncov, ncov);
    P.width = nmap >= kWideFrom ? kWide : 1;
    const int bins = P.width * 64;
    P.ngroup = (int)((nmap + bins - 1) / bins);
    P.div.assign(nmap, 0.0);
    const long kEntryMax = 0x7fffffff;  // entries are listed by 32-bit numbers
    struct Flat {
        long i;
        int place, len;
    };
    // by entries as soon as the runs are too many; the list grows in pieces, not by doubling
    const long most = nidx <= kEntryMax ? nidx / kRunFrom : nidx;
    std::deque<Flat> flat;
    for (long i = 0, next = -1; i < nidx && !P.entries; ++i) {
        const long b = idx[i] - 1;
        if (b < 0 || b >= nmap) return false;
        P.div[b] += 1;
        const int p = place[b];
        if (p == next && flat.back().len < 64 && p % bins)
            ++flat.back().len;
        else if ((long)flat.size() < most)
            flat.push_back({i, p, 1});
        else
            P.entries = true;
        next = p + 1;
    }
    if (P.entries) {
        flat.clear();
        std::vector<int> at(nmap, 0);  // entries of a bin, then where its next one goes
        for (long i = 0; i < nidx; ++i) {
            const long b = idx[i] - 1;
            if (b < 0 || b >= nmap) return false;
            ++at[b];
        }
        P.run_of.assign(nmap + 1, 0);
        for (long b = 0; b < nmap; ++b) P.div[b] = P.run_of[place[b] + 1] = at[b];
        for (long b = 0; b < nmap; ++b) P.run_of[b + 1] += P.run_of[b];
        for (long b = 0; b < nmap; ++b) at[b] = P.run_of[place[b]];
        P.item_of.resize(nidx);
        for (long i = 0; i < nidx; ++i) P.item_of[at[idx[i] - 1]++] = (int)i;
        return true;
    }
    // slabs: at least two rounds of loads per wave; runs are cut where slabs meet
    const long per_slab = (long)P.ngroup * kGatherWaves * kRunsAhead * 2;
    const long want = std::min<long>(kMaxSlabs, std::max<long>(1, (long)flat.size() / per_slab));
    P.slab = std::min(kSlabMax, (nidx + want - 1) / want);
    P.nslab = (int)((nidx + P.slab - 1) / P.slab);
    // f(group of the slab, run) for every run
    auto walk = [&](auto&& f) {
        for (Flat r : flat)
            while (r.len > 0) {
                const long q = r.i / P.slab, at = r.i - q * P.slab;
                const int n = (int)std::min<long>(r.len, P.slab - at);
                f((size_t)q * P.ngroup + r.place / bins,
                  Run{(int)at, (unsigned)(r.place % bins) | (unsigned)n << 16});
                r.i += n;
                r.place += n;
                r.len -= n;
            }
    };
    std::vector<int> count((size_t)P.nslab * P.ngroup, 0), at(count.size());
    walk([&](size_t k, Run) { ++count[k]; });
    P.item_of.assign(count.size(), -1);
    P.run_of.push_back(0);
    for (size_t k = 0; k < count.size(); ++k) {
        if (P.nslab > 1 && count[k] == 0) continue;
        P.item_of[k] = (int)P.items.size();
        P.items.push_back({(int)(k / P.ngroup), (int)(k % P.ngroup)});
        at[k] = P.run_of.back();
        P.run_of.push_back(at[k] + count[k]);
    }
    P.runs.resize(P.run_of.back());
    walk([&](size_t k, Run r) { P.runs[at[k]++] = r; });
    return true;
}

}  // namespace
}  // namespace moao

using moao::ctx;
using moao::set_error;

extern "C" {

long moao_intersample_default_n(long np) {
    // intersample.cpp:192: MAX(512, 8*pow(2, (long)(log(np)+0.5)))  (natural log)
    const double v = 8 * std::pow(2.0, (double)(long)(std::log((double)np) + 0.5));
    return (long)std::max(512.0, v);
}

int moao_hip_intersample_create(long nidx, long np, long N, const long* idx, const double* abs2fi,
                                const double* otf_tel, int precision, moao_isample** out) {
    if (int rc = moao::ensure_init()) return rc;
    if (!out || !idx || !abs2fi || !otf_tel || nidx < 1 || np < 2 || precision < 0 ||
        precision > 1) {
        set_error("intersample_create: invalid arguments");
        return MOAO_ERR_ARG;
    }
    if (N <= 0) N = moao_intersample_default_n(np);
    if (N < 32 || N > 4096 || (N & (N - 1))) {
        set_error("intersample_create: N must be a power of two in [32, 4096]");
        return MOAO_ERR_ARG;
    }
    auto* S = new moao_isample;
    S->N = N;
    S->np = np;
    S->nidx = nidx;
    S->ncov = 2 * np - 1;
    S->nmap = S->ncov * S->ncov;
    S->prec = precision;
    S->dactupix = (double)(N / (3 * (np - 1)) + 1);  // intersample.cpp:199 (integer division)
    const long nelem = (S->ncov - 1) / 2, ncmap = N / 2 + 1;
    const long first = (long)(ncmap - nelem * S->dactupix - 1);
    const long last = (long)(first + (S->ncov - 1) * S->dactupix);
    if (first < 0 || last >= N) {
        delete S;
        set_error("intersample_create: the covariance map does not fit the N x N grid");
        return MOAO_ERR_ARG;
    }
    moao::Plan plan;
    if (!moao::make_plan(idx, nidx, (int)S->ncov, &plan)) {
        delete S;
        set_error("intersample_create: idx entry out of range");
        return MOAO_ERR_ARG;
    }
    S->entries = plan.entries;
    S->order = plan.order;
    S->nslab = plan.nslab;
    S->width = plan.width;
    S->ngroup = plan.ngroup;
    S->slab = plan.slab;
    S->nitem = (int)plan.items.size();
    hipStream_t s = ctx().stream;
    auto fail = [&](int rc) {
        moao_hip_intersample_destroy(S);
        return rc;
    };
    auto H2D = [&](void** d, const void* h, size_t bytes) -> int {
        if (bytes == 0) return MOAO_OK;
        if (hipMalloc(d, bytes) != hipSuccess) return MOAO_ERR_NOMEM;
        if (hipMemcpyAsync(*d, h, bytes, hipMemcpyHostToDevice, s) != hipSuccess) return MOAO_ERR_HIP;
        return MOAO_OK;
    };
    if (int rc = H2D(&S->runs, plan.runs.data(), sizeof(moao::Run) * plan.runs.size()))
        return fail(rc);
    if (int rc = H2D(&S->items, plan.items.data(), sizeof(moao::Item) * plan.items.size()))
        return fail(rc);
    if (int rc = H2D((void**)&S->run_of, plan.run_of.data(), sizeof(int) * plan.run_of.size()))
        return fail(rc);
    if (int rc = H2D((void**)&S->item_of, plan.item_of.data(), sizeof(int) * plan.item_of.size()))
        return fail(rc);
    if (int rc = H2D((void**)&S->div, plan.div.data(), sizeof(double) * S->nmap)) return fail(rc);
    const size_t nn = (size_t)N * N;
    if (precision == 0) {
        std::vector<float> a(nn), o(nn);
        for (size_t k = 0; k < nn; ++k) a[k] = (float)abs2fi[k], o[k] = (float)otf_tel[k];
        if (int rc = H2D(&S->a2f, a.data(), sizeof(float) * nn)) return fail(rc);
        if (int rc = H2D(&S->otf, o.data(), sizeof(float) * nn)) return fail(rc);
        if (hipStreamSynchronize(s) != hipSuccess) return fail(MOAO_ERR_HIP);
        if (int rc = moao::fft_twiddles<float>((int)N, (float2**)&S->tw, s)) return fail(rc);
    } else {
        if (int rc = H2D(&S->a2f, abs2fi, sizeof(double) * nn)) return fail(rc);
        if (int rc = H2D(&S->otf, otf_tel, sizeof(double) * nn)) return fail(rc);
        if (int rc = moao::fft_twiddles<double>((int)N, (double2**)&S->tw, s)) return fail(rc);
    }
    if (hipStreamSynchronize(s) != hipSuccess) return fail(MOAO_ERR_HIP);
    *out = S;
    return MOAO_OK;
}

long moao_hip_intersample_n(const moao_isample* S) { return S ? S->N : MOAO_ERR_ARG; }

int moao_hip_psf_accumulate_dev(const double* dPsf, long count, double* dSum, void* stream) {
    if (int rc = moao::ensure_init()) return rc;
    if (count < 0 || (count > 0 && (!dPsf || !dSum))) {
        set_error("psf_accumulate: invalid arguments");
        return MOAO_ERR_ARG;
    }
    if (count == 0) return MOAO_OK;
    hipStream_t s = moao::pick_stream(stream);
    hipLaunchKernelGGL(moao::psf_accumulate, dim3((unsigned)((count + 255) / 256)), dim3(256), 0,
                       s, dPsf, count, dSum);
    MOAO_HIP_TRY(hipGetLastError());
    return MOAO_OK;
}

int moao_hip_intersample_process_dev(moao_isample* S, const double* dCvv, int batch,
                                     double* dPsf, void* stream) {
    if (int rc = moao::ensure_init()) return rc;
    if (!S || !dCvv || !dPsf || batch < 1) {
        set_error("intersample_process: invalid arguments");
        return MOAO_ERR_ARG;
    }
    hipStream_t s = moao::pick_stream(stream);
    return S->prec == 0 ? moao::process<float>(S, dCvv, batch, dPsf, s)
                        : moao::process<double>(S, dCvv, batch, dPsf, s);
}

// Host drop-in of intersample_process (intersample.cpp:72-171): Cvv is the flat nact x nact
// covariance (nidx doubles), psf receives the N x N PSF in the reference's layout.
int moao_hip_intersample_process(moao_isample* S, const double* Cvv, double* psf) {
    if (int rc = moao::ensure_init()) return rc;
    if (!S || !Cvv || !psf) return MOAO_ERR_ARG;
    hipStream_t s = ctx().stream;
    if (!S->dCvv) MOAO_HIP_TRY(hipMalloc((void**)&S->dCvv, sizeof(double) * S->nidx));
    if (!S->dPsf) MOAO_HIP_TRY(hipMalloc((void**)&S->dPsf, sizeof(double) * S->N * S->N));
    MOAO_HIP_TRY(hipMemcpyAsync(S->dCvv, Cvv, sizeof(double) * S->nidx, hipMemcpyHostToDevice, s));
    if (int rc = moao_hip_intersample_process_dev(S, S->dCvv, 1, S->dPsf, s)) return rc;
    MOAO_HIP_TRY(hipMemcpyAsync(psf, S->dPsf, sizeof(double) * S->N * S->N, hipMemcpyDeviceToHost,
                                s));
    MOAO_HIP_TRY(hipStreamSynchronize(s));
    return MOAO_OK;
}

void moao_hip_intersample_destroy(moao_isample* S) {
    if (!S) return;
    void* ptrs[] = {S->runs, S->items, S->run_of, S->item_of, S->div, S->a2f, S->otf, S->tw,
                    S->work, S->dCvv, S->dPsf};
    (void)hipDeviceSynchronize();
    for (void* p : ptrs)
        if (p) (void)hipFree(p);
    delete S;
}

}  // extern "C"
