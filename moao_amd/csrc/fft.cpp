// Twiddle tables of the PSF stage's transforms.
#include "fft.hpp"

#include <cmath>
#include <vector>

#include "common.hpp"

namespace moao {

template <typename R>
int fft_twiddles(int N, typename Cplx<R>::type** d_table, hipStream_t s) {
    using C = typename Cplx<R>::type;
    std::vector<C> h(N);
    const double pi = 3.14159265358979323846;
    for (int e = 0; e < N; ++e) {
        const double a = -2.0 * pi * (double)e / (double)N;
        h[e] = C{(R)std::cos(a), (R)std::sin(a)};
    }
    MOAO_HIP_TRY(hipMalloc((void**)d_table, sizeof(C) * N));
    MOAO_HIP_TRY(hipMemcpyAsync(*d_table, h.data(), sizeof(C) * N, hipMemcpyHostToDevice, s));
    MOAO_HIP_TRY(hipStreamSynchronize(s));
    return MOAO_OK;
}

template int fft_twiddles<float>(int, float2**, hipStream_t);
template int fft_twiddles<double>(int, double2**, hipStream_t);

}  // namespace moao
