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

#include <type_traits>

namespace moao {

template <typename R>
struct Cplx;
template <>
struct Cplx<float> { using type = float2; };
template <>
struct Cplx<double> { using type = double2; };

// Values per lane of a transform of 2^log: 8 where the radices come out even (8.4, 8.8, 8.8.8), else
// 16; and the radix of its stage over sub-transforms of length ns.
constexpr int fft_values(int log) { return log == 5 || log == 6 || log == 9 ? 8 : 16; }
constexpr int fft_radix(int log, int ns) {
    return fft_values(log) < (1 << log) / ns ? fft_values(log) : (1 << log) / ns;
}

// Twiddles of a transform of N values, stage by stage: exp(-2 pi i m k / (ns P)) for m = 1 .. P - 1 and
// k < ns (k fast: neighbouring lanes read neighbouring entries), computed on the host in FP64 and
// rounded once.
template <typename R>
int fft_twiddles(int N, typename Cplx<R>::type** d_table, hipStream_t s);

template <typename R, int LOG>
struct RowFft {
    using C = typename Cplx<R>::type;
    static constexpr int N = 1 << LOG;
    static constexpr int E = fft_values(LOG);
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
    static __device__ __forceinline__ C conj_if(C a) {  // a's conjugate for the backward direction
        return DIR > 0 ? C{a.x, -a.y} : a;
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

    static constexpr int radix(int ns) { return fft_radix(LOG, ns); }
    // A run takes its twiddles from the table, a stage's while the row crosses LDS on the way to it, or
    // from registers filled before the run.  There a lane keeps, of a stage's factors m = 1 .. P - 1,
    // those with m = 1, 2, 3 and the multiples of 4 and multiplies out the others: at N = 2048 14
    // loads and not 29, but with the roundings of the products.  With those in every run the FP32
    // PSF is 8, 2 and 3% (N = 512, 1024, 2048) further from the exact one than by radix-4 stages
    // with table entries alone; with the table in its last two runs 0.4 +- 0.6% further, 0.6 and 0.4%
    // nearer.
    struct Table {
        const C* w;
    };
    static constexpr int entries(int p) { return p == 16 ? 6 : p == 8 ? 4 : p - 1; }
    static constexpr int factor(int k) { return k < 3 ? k + 1 : 4 * k - 8; }
    static constexpr int tw_count(int ns) {
        return ns >= N ? 0
                       : (ns > 1 ? E / radix(ns) * entries(radix(ns)) : 0) + tw_count(ns * radix(ns));
    }
    struct Kept {
        C w[tw_count(1)];
    };
    // AT, FROM: where the stage's entries start in Kept and in the table
    template <int NS = 1, int AT = 0, int FROM = 0>
    static __device__ __forceinline__ void keep(Kept& kept, const Table& tw, int t) {
        if constexpr (NS < N) {
            constexpr int P = radix(NS), Q = E / P, M = NS > 1 ? entries(P) : 0;
#pragma unroll
            for (int q = 0; q < Q; ++q)
#pragma unroll
                for (int k = 0; k < M; ++k)
                    kept.w[AT + q * M + k] =
                        tw.w[FROM + (factor(k) - 1) * NS + ((t + q * T) & (NS - 1))];
            keep<NS * P, AT + Q * M, FROM + (NS > 1 ? (P - 1) * NS : 0)>(kept, tw, t);
        }
    }
    // A run's twiddles: the table's own, or kept ones.  FP64 keeps them always (its PSF is nearer to
    // the exact one than by radix-4 stages all the same, and 8 directions at N = 1024 take 98 us
    // with the table, 93 without).
    template <bool TABLE>
    static __device__ __forceinline__ auto twiddles(const C* tw, int t) {
        if constexpr (TABLE && sizeof(R) == 4) {
            return Table{tw};
        } else {
            Kept kept;
            keep(kept, Table{tw}, t);
            return kept;
        }
    }

    // Stage over sub-transforms of length NS, then the later ones.  Butterfly j = t + q T takes
    // elements j + m N/P times factor m, m < P; from the table f holds factor m at q (P - 1) + m - 1.
    template <int DIR, int NS, int AT, int FROM, typename W, int L>
    static __device__ __forceinline__ void stage(C (&v)[E], C* lds, int t, int row, const W& tw,
                                                 const C (&f)[L]) {
        constexpr bool kTable = std::is_same<W, Table>::value;
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
                if constexpr (kTable) {
#pragma unroll
                    for (int m = 1; m < P; ++m) w[m] = conj_if<DIR>(f[q * (P - 1) + m - 1]);
                } else {
#pragma unroll
                    for (int k = 0; k < M; ++k) w[factor(k)] = conj_if<DIR>(tw.w[AT + q * M + k]);
#pragma unroll
                    for (int m = 5; m < P; ++m)
                        if (m % 4) w[m] = mul(w[m & ~3], w[m & 3]);
                }
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
            constexpr int NS2 = NS * P, P2 = radix(NS2), Q2 = E / P2;
            C f2[kTable ? Q2 * (P2 - 1) : 1];
            if constexpr (kTable) {
                // at an address that the compiler takes for another run to run: what it kept from one
                // run for the next would fill the registers of the work between them
                int k = t;
                asm volatile("" : "+v"(k));
#pragma unroll
                for (int q = 0; q < Q2; ++q)
#pragma unroll
                    for (int m = 1; m < P2; ++m)
                        f2[q * (P2 - 1) + m - 1] =
                            tw.w[FROM + (m - 1) * NS2 + ((k + q * T) & (NS2 - 1))];
            }
            __syncthreads();
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int i = t + T * e;
                v[e] = lds[(i + i / E) * kRows + row];
            }
            stage<DIR, NS2, AT + Q * M, FROM + (P2 - 1) * NS2>(v, lds, t, row, tw, f2);
        }
    }
    // v[e] = element t + T e of the row, before and after; unnormalised; every thread of the
    // workgroup calls it.  tw: a Table or a Kept.
    template <int DIR, typename W>
    static __device__ __forceinline__ void run(C (&v)[E], C* lds, int t, int row, const W& tw) {
        const C none[1] = {};
        stage<DIR, 1, 0, 0>(v, lds, t, row, tw, none);
    }
};

}  // namespace moao
