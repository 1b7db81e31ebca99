// Row FFTs of the PSF stage (power-of-two N, 32 <= N <= 4096), held in registers.
//
// One row of N complex values is spread over N/E lanes, E values each; a Stockham stage of
// radix E is a butterfly of the lane's own registers, and between stages the row crosses LDS
// once (N = 2048: radices 16, 16, 8, two crossings; six radix-4/2 stages through LDS before).
// Lane t holds the elements t + (N/E) e of the input and, since the transform sorts itself, of
// the output too: a product with a weight or a second transform follows in the same registers
// with no exchange, and a half rotation (fftshift) is a renaming of them.
// A workgroup carries kRows rows interleaved over its lanes (lane = t * kRows + row), so global
// accesses at one e cover kRows rows x 64/kRows consecutive elements: whole 128-byte lines of
// arrays stored in kRows x kRows tiles, which is how the passes hand over a transposed grid
// without a transpose pass.  LDS index i is padded to i + i/E: the first stage's stride-E
// writes then fall into different banks.
#pragma once

#include <hip/hip_runtime.h>

namespace moao {

template <typename R>
struct Cplx;
template <>
struct Cplx<float> { using type = float2; };
template <>
struct Cplx<double> { using type = double2; };

// Twiddle table W_N^e = exp(-2 pi i e / N), e < N, built on the host in FP64 and rounded once.
template <typename R>
int fft_twiddles(int N, typename Cplx<R>::type** d_table, hipStream_t s);

template <typename R, int LOG>
struct RowFft {
    using C = typename Cplx<R>::type;
    static constexpr int N = 1 << LOG;
    // 8 values per lane where the radices come out even (8.4, 8.8, 8.8.8), else 16
    static constexpr int E = LOG == 5 || LOG == 6 || LOG == 9 ? 8 : 16;
    static constexpr int T = N / E;
    // 4 rows per workgroup; 2 where 4 would not fit the 160 KB of LDS
    static constexpr int kRows = sizeof(R) == 8 && LOG == 12 ? 2 : 4;
    static constexpr int kThreads = T * kRows;
    static constexpr int kWaves = sizeof(R) == 4 ? 4 : 2;  // per SIMD: two workgroups of 512 in FP32
    static constexpr int kLds = (N + N / E) * kRows;  // complex values

    static __device__ __forceinline__ C mul(C a, C b) {
        return C{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
    }
    static __device__ __forceinline__ C add(C a, C b) { return C{a.x + b.x, a.y + b.y}; }
    static __device__ __forceinline__ C sub(C a, C b) { return C{a.x - b.x, a.y - b.y}; }
    template <int DIR>
    static __device__ __forceinline__ C mul_i(C a) {  // a * (DIR * i)
        return DIR > 0 ? C{-a.y, a.x} : C{a.y, -a.x};
    }
    template <int DIR>
    static __device__ __forceinline__ void dft4(C& a, C& b, C& c, C& d) {
        const C s = add(a, c), u = sub(a, c), v = add(b, d), w = mul_i<DIR>(sub(b, d));
        a = add(s, v);
        b = add(u, w);
        c = sub(s, v);
        d = sub(u, w);
    }
    // X[k] = sum_m x[m] exp(DIR 2 pi i m k / P), in place, natural order
    template <int P, int DIR>
    static __device__ __forceinline__ void dft(C (&x)[P]) {
        if constexpr (P == 2) {
            const C a = x[0], b = x[1];
            x[0] = add(a, b);
            x[1] = sub(a, b);
        } else if constexpr (P == 4) {
            dft4<DIR>(x[0], x[1], x[2], x[3]);
        } else {  // P = A * 4: A four-point transforms, twiddles W_P^(a b), 4 of A points
            constexpr int A = P / 4;
            constexpr R c1 = (R)0.92387953251128675613, s1 = (R)0.38268343236508977173,
                        h = (R)0.70710678118654752440;
#pragma unroll
            for (int a = 0; a < A; ++a) dft4<DIR>(x[a], x[a + A], x[a + 2 * A], x[a + 3 * A]);
            constexpr R co[10] = {1, c1, h, s1, 0, -s1, -h, -c1, -1, -c1};
            constexpr R si[10] = {0, s1, h, c1, 1, c1, h, s1, 0, -s1};
#pragma unroll
            for (int a = 1; a < A; ++a)
#pragma unroll
                for (int b = 1; b < 4; ++b) {
                    const int f = a * b * (16 / P);
                    C& v = x[a + A * b];
                    v = f == 4 ? mul_i<DIR>(v) : mul(v, C{co[f], DIR * si[f]});
                }
            C y[P];
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                if constexpr (A == 4) {
                    dft4<DIR>(x[4 * b], x[4 * b + 1], x[4 * b + 2], x[4 * b + 3]);
                    for (int c = 0; c < 4; ++c) y[b + 4 * c] = x[4 * b + c];
                } else {
                    y[b] = add(x[2 * b], x[2 * b + 1]);
                    y[b + 4] = sub(x[2 * b], x[2 * b + 1]);
                }
            }
#pragma unroll
            for (int k = 0; k < P; ++k) x[k] = y[k];
        }
    }

    // Twiddles of one stage: W^(m k), m < P, from the entries m = 1, 2, 3 and the multiples of 4
    static constexpr int radix(int ns) { return E < N / ns ? E : N / ns; }
    static constexpr int entries(int p) { return p == 16 ? 6 : p == 8 ? 4 : p - 1; }
    static constexpr int tw_count(int ns) {
        return ns >= N ? 0
                       : (ns > 1 ? E / radix(ns) * entries(radix(ns)) : 0) + tw_count(ns * radix(ns));
    }
    static constexpr int kTw = tw_count(1);
    template <int NS = 1, int AT = 0>
    static __device__ __forceinline__ void load_twiddles(C (&w)[kTw], int t,
                                                         const C* __restrict__ tw) {
        if constexpr (NS < N) {
            constexpr int P = radix(NS), Q = E / P, M = NS > 1 ? entries(P) : 0;
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const int k = ((t + q * T) & (NS - 1)) * (N / (NS * P));
#pragma unroll
                for (int m = 0; m < M; ++m) w[AT + q * M + m] = tw[(m < 3 ? m + 1 : 4 * m - 8) * k];
            }
            load_twiddles<NS * P, AT + Q * M>(w, t, tw);
        }
    }

    // Stage over sub-transforms of length NS, then the later ones.  Butterfly j = t + q T takes
    // elements j + m N/P, m < P.
    template <int DIR, int NS, int AT>
    static __device__ __forceinline__ void stage(C (&v)[E], C* lds, int t, int row,
                                                 const C (&tw)[kTw]) {
        if constexpr (NS < N) {
            constexpr int P = radix(NS), Q = E / P, M = NS > 1 ? entries(P) : 0;
            if constexpr (NS * P < N) __syncthreads();  // the last reads of lds are done
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const int j = t + q * T;
                C x[P];
#pragma unroll
                for (int m = 0; m < P; ++m) x[m] = v[q + m * Q];
                if constexpr (NS > 1) {
                    C w[P];
#pragma unroll
                    for (int m = 0; m < M; ++m) {
                        C& c = w[m < 3 ? m + 1 : 4 * m - 8];
                        c = tw[AT + q * M + m];
                        if (DIR > 0) c.y = -c.y;
                    }
#pragma unroll
                    for (int m = 5; m < P; ++m)
                        if (m % 4) w[m] = mul(w[m & ~3], w[m & 3]);
#pragma unroll
                    for (int m = 1; m < P; ++m) x[m] = mul(x[m], w[m]);
                }
                dft<P, DIR>(x);
                if constexpr (NS * P < N) {
                    const int o = (j / NS) * NS * P + (j & (NS - 1));
#pragma unroll
                    for (int m = 0; m < P; ++m) {
                        const int i = o + m * NS;
                        lds[(i + i / E) * kRows + row] = x[m];
                    }
                } else {
#pragma unroll
                    for (int m = 0; m < P; ++m) v[q + m * Q] = x[m];
                }
            }
            if constexpr (NS * P < N) {
                __syncthreads();
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    const int i = t + T * e;
                    v[e] = lds[(i + i / E) * kRows + row];
                }
                stage<DIR, NS * P, AT + Q * M>(v, lds, t, row, tw);
            }
        }
    }
    // v[e] = element t + T e of the row, before and after; unnormalised; every thread of the
    // workgroup calls it.
    template <int DIR>
    static __device__ __forceinline__ void run(C (&v)[E], C* lds, int t, int row,
                                               const C (&tw)[kTw]) {
        stage<DIR, 1, 0>(v, lds, t, row, tw);
    }
};

}  // namespace moao
