// The deepest levels of the backward solve Y L = X in one launch.
//
// The recursion over columns ends in segments of up to four 128-column leaves: four products with the
// leaves' inverses and the updates between them, each of a few hundred rows and each a launch of 8
// to 12 us, of which the products themselves are 1 to 2.  The rows are independent, so a workgroup
// takes 16 of them through the whole segment: eight waves, wave w holding columns 16 w .. 16 w + 15 of
// every leaf in MFMA accumulator registers; finished values pass to the other waves through LDS,
// where [k][row] is both what an accumulator's lanes write and what the MFMA takes as its A operand.
// L and the inverses come from memory (L2) in MFMA order, the next product's while the current one
// runs.  The order of the products and of k within each sum is that of the launches it replaces,
// so the bits are the same.
// Bound by the operands' way from L2 to the CU (1.4 MB per 16 rows and segment of four leaves: 44 us
// in FP64; the seven launches 63 and more), beside a chain of 8 x 128 k of dependent MFMAs (7 us).
#include <hip/hip_runtime.h>

#include "common.hpp"
#include "leaf.hpp"
#include "mfma.hpp"
#include "profile.hpp"
#include "segment.hpp"

namespace moao {
namespace {

// Barrier for LDS alone: __syncthreads would also wait for the operands still on their way from
// memory (60 us a launch).
__device__ __forceinline__ void lds_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0), vmcnt and expcnt at their maxima
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <typename T>
struct SegArgs {
    SegRows<T> g[kSegGroups];
    const T* L;    // (first column, first column) of the segment
    long lda;
    const T* inv;  // inverses of its leaves, kLeaf x kLeaf each
    const int* skip_if;
};

template <typename T, int NL>
__global__ void __launch_bounds__(512) trsm_segment_kernel(SegArgs<T> a) {
    using M = Mfma<T>;
    using acc_t = typename M::acc_t;
    __shared__ T sh[5][kLeaf * 16];  // X of the leaf being solved, Y of the four leaves
    const SegRows<T> g = a.g[blockIdx.y];
    const int m0 = blockIdx.x * 16;
    if (m0 >= g.rows) return;
    const int skip = a.skip_if ? *(volatile const int*)a.skip_if : 0;
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 15, lq = lane >> 4;
    const int row = min(m0 + li, g.rows - 1);

    // the wave's 16 columns of a leaf, element (row li, column M::row(lane, t))
    T x0[4], x1[4], x2[4], x3[4];
    auto load = [&](T (&x)[4], int leaf) __attribute__((always_inline)) {
        const T* X = g.X + row + (long)leaf * kLeaf * g.ld;
#pragma unroll
        for (int t = 0; t < 4; ++t) x[t] = X[(long)(16 * w + M::row(lane, t)) * g.ld];
    };
    auto store = [&](const T (&x)[4], int leaf) __attribute__((always_inline)) {
        if (skip || m0 + li >= g.rows) return;
        T* X = g.X + row + (long)leaf * kLeaf * g.ld;
#pragma unroll
        for (int t = 0; t < 4; ++t) X[(long)(16 * w + M::row(lane, t)) * g.ld] = x[t];
        if constexpr (sizeof(T) == 4)  // a lane's 4 columns are 4 consecutive k of a plane row
            if (g.cp)
                write_planes(x, g.cp + (long)row * g.cpld, g.cpps, leaf * kLeaf + 16 * w + 4 * lq,
                             (leaf + 1) * kLeaf);
    };

    // 128 k of op(B) for the wave's columns: lane (column li, k = 16 c + 4 lq ..) of column-major B;
    // one product's operands are under way during another's MFMAs
    T p[8][4], q[8][4];
    auto fetch = [&](T (&b)[8][4], const T* B, long ld) __attribute__((always_inline)) {
        const T* s = B + (long)(16 * w + li) * ld + 4 * lq;
#pragma unroll
        for (int c = 0; c < 8; ++c) __builtin_memcpy(b[c], s + 16 * c, sizeof(b[c]));
    };
    auto fetch_inv = [&](T (&b)[8][4], int leaf) __attribute__((always_inline)) {
        fetch(b, a.inv + (long)leaf * kLeaf * kLeaf, kLeaf);
    };
    auto fetch_l = [&](T (&b)[8][4], int rows_of, int cols_of) __attribute__((always_inline)) {
        fetch(b, a.L + (long)rows_of * kLeaf + (long)cols_of * kLeaf * a.lda, a.lda);
    };
    auto share = [&](const T (&v)[4], T* to) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < 4; ++t) to[(16 * w + M::row(lane, t)) * 16 + li] = v[t];
        lds_barrier();
    };
    auto mma = [&](acc_t& acc, T (&b)[8][4], const T* A) __attribute__((always_inline)) {
        T av[32];  // read in one go: one by one each MFMA would wait for its own
#pragma unroll
        for (int k = 0; k < 32; ++k) av[k] = A[(4 * k + lq) * 16 + li];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            lane_rows_transpose(b[c][0], b[c][1], b[c][2], b[c][3]);
#pragma unroll
            for (int t = 0; t < 4; ++t) acc = M::mac(b[c][t], av[4 * c + t], acc);
        }
    };
    const acc_t zero{0, 0, 0, 0};
    // Y_leaf = X_leaf inv; b holds the inverse
    auto solve = [&](int leaf, T (&xl)[4], T (&b)[8][4]) __attribute__((always_inline)) {
        share(xl, sh[4]);
        acc_t acc = zero;
        mma(acc, b, sh[4]);
#pragma unroll
        for (int t = 0; t < 4; ++t) xl[t] = acc[t];
        share(xl, sh[leaf]);
        store(xl, leaf);
    };
    auto minus = [&](T (&xl)[4], const acc_t& acc) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < 4; ++t) xl[t] = xl[t] - acc[t];
    };
    acc_t u = zero, v = zero;
    if constexpr (NL == 4) {
        fetch_inv(p, 3);
        load(x3, 3);
        fetch_l(q, 3, 2);
        load(x2, 2);
        solve(3, x3, p);
        fetch_inv(p, 2);
        mma(u, q, sh[3]);
        minus(x2, u);
        fetch_l(q, 2, 1);
        solve(2, x2, p);
        fetch_l(p, 2, 0);
        u = zero;
        mma(u, q, sh[2]);
        fetch_l(q, 3, 1);
        mma(v, p, sh[2]);
        fetch_l(p, 3, 0);
        load(x1, 1);
        mma(u, q, sh[3]);
        fetch_inv(q, 1);
        load(x0, 0);
        mma(v, p, sh[3]);
    } else if constexpr (NL == 3) {
        fetch_inv(p, 2);
        load(x2, 2);
        fetch_l(q, 2, 1);
        solve(2, x2, p);
        fetch_l(p, 2, 0);
        load(x1, 1);
        mma(u, q, sh[2]);
        fetch_inv(q, 1);
        load(x0, 0);
        mma(v, p, sh[2]);
    } else {
        fetch_inv(q, 1);
        load(x1, 1);
        load(x0, 0);
    }
    if constexpr (NL > 2) {
        minus(x1, u);
        minus(x0, v);
    }
    fetch_l(p, 1, 0);
    solve(1, x1, q);
    fetch_inv(q, 0);
    u = zero;
    mma(u, p, sh[1]);
    minus(x0, u);
    solve(0, x0, q);
}

}  // namespace

template <typename T>
int trsm_segment(const SegRows<T>* rows, int ngroups, const T* L, long lda, const T* inv, int nn,
                 const int* skip_if, hipStream_t s) {
    SegArgs<T> a{};
    a.L = L;
    a.lda = lda;
    a.inv = inv;
    const int nl = nn / kLeaf;
    a.skip_if = skip_if;
    if (nn % kLeaf || nl < 2 || nl > 4 || ngroups < 1 || ngroups > kSegGroups) {
        set_error("trsm_segment: invalid arguments");
        return MOAO_ERR_ARG;
    }
    int most = 0;
    double work = 0;
    for (int i = 0; i < ngroups; ++i) {
        a.g[i] = rows[i];
        most = rows[i].rows > most ? rows[i].rows : most;
        work += (double)rows[i].rows * nn * (nn + 1.0);
    }
    if (most == 0) return MOAO_OK;
    ProfScope ps(sizeof(T) == 8 ? kProfGemmF64 : kProfGemmF32, work, s);
    auto* k = nl == 4   ? trsm_segment_kernel<T, 4>
              : nl == 3 ? trsm_segment_kernel<T, 3>
                        : trsm_segment_kernel<T, 2>;
    hipLaunchKernelGGL(k, dim3((most + 15) / 16, ngroups), dim3(512), 0, s, a);
    MOAO_HIP_TRY(hipGetLastError());
    return MOAO_OK;
}

template int trsm_segment<double>(const SegRows<double>*, int, const double*, long, const double*,
                                  int, const int*, hipStream_t);
template int trsm_segment<float>(const SegRows<float>*, int, const float*, long, const float*, int,
                                 const int*, hipStream_t);

}  // namespace moao
