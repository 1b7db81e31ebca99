// 16x16x4 MFMA steps, the lane exchange that feeds them from memory order, and the split-BF16 planes
// of what they leave (gfx950).
#pragma once

#include <hip/hip_runtime.h>

namespace moao {
namespace {

template <typename T>
struct Mfma;

template <>
struct Mfma<double> {
    typedef double acc_t __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ acc_t mac(double a, double b, acc_t c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    // accumulator item t of lane l holds row (l/16) + 4t of the 16x16 block
    static __device__ __forceinline__ int row(int lane, int t) { return (lane >> 4) + 4 * t; }
};

template <>
struct Mfma<float> {
    typedef float acc_t __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ acc_t mac(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    // accumulator item t of lane l holds row 4*(l/16) + t of the 16x16 block
    static __device__ __forceinline__ int row(int lane, int t) { return 4 * (lane >> 4) + t; }
};

// 4x4 transpose between four registers and the four 16-lane rows of a wave: lane row q's
// register t becomes lane row t's register q (gfx950 row swaps; no LDS).
__device__ __forceinline__ void swap_rows(unsigned (&x)[4]) {
    auto p = __builtin_amdgcn_permlane32_swap(x[0], x[2], false, false);
    auto q = __builtin_amdgcn_permlane32_swap(x[1], x[3], false, false);
    auto r = __builtin_amdgcn_permlane16_swap(p[0], q[0], false, false);
    auto s = __builtin_amdgcn_permlane16_swap(p[1], q[1], false, false);
    x[0] = r[0];
    x[1] = r[1];
    x[2] = s[0];
    x[3] = s[1];
}
template <typename T>
__device__ __forceinline__ void lane_rows_transpose(T& a, T& b, T& c, T& d) {
    constexpr int W = sizeof(T) / 4;
    unsigned v[4][W], x[4];
    __builtin_memcpy(v[0], &a, sizeof(T));
    __builtin_memcpy(v[1], &b, sizeof(T));
    __builtin_memcpy(v[2], &c, sizeof(T));
    __builtin_memcpy(v[3], &d, sizeof(T));
#pragma unroll
    for (int w = 0; w < W; ++w) {
        for (int t = 0; t < 4; ++t) x[t] = v[t][w];
        swap_rows(x);
        for (int t = 0; t < 4; ++t) v[t][w] = x[t];
    }
    __builtin_memcpy(&a, v[0], sizeof(T));
    __builtin_memcpy(&b, v[1], sizeof(T));
    __builtin_memcpy(&c, v[2], sizeof(T));
    __builtin_memcpy(&d, v[3], sizeof(T));
}

// hi and lo planes of four consecutive k of one row, those below N (see Planes).
__device__ __forceinline__ void write_planes(const float (&v)[4], unsigned short* hi, long ps,
                                             int k, int N) {
    typedef unsigned short us4 __attribute__((ext_vector_type(4)));
    us4 h, l;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const __bf16 a = (__bf16)v[t];
        h[t] = __builtin_bit_cast(unsigned short, a);
        l[t] = __builtin_bit_cast(unsigned short, (__bf16)(v[t] - (float)a));
    }
    if (k + 4 <= N) {
        *(us4*)(hi + k) = h;
        *(us4*)(hi + ps + k) = l;
        return;
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
        if (k + t < N) {
            hi[k + t] = h[t];
            hi[ps + k + t] = l[t];
        }
}
__device__ __forceinline__ void write_planes(const double (&)[4], unsigned short*, long, int, int) {}

}  // namespace
}  // namespace moao
