// Twiddle tables of the PSF stage's transforms.
#include "fft.hpp"

#include <cmath>
#include <vector>

#include "common.hpp"

namespace moao {

template <typename R>
int fft_twiddles(int N, typename Cplx<R>::type** d_table, hipStream_t s) {
    using C = typename Cplx<R>::type;
    int log = 0;
    while (1 << log < N) ++log;
    std::vector<C> h;  // N - (first radix) values
    const double pi = 3.14159265358979323846;
    for (int ns = fft_radix(log, 1); ns < N; ns *= fft_radix(log, ns))
        for (int m = 1; m < fft_radix(log, ns); ++m)
            for (int k = 0; k < ns; ++k) {
                const double a = -2.0 * pi * m * k / ((double)ns * fft_radix(log, ns));
                h.push_back(C{(R)std::cos(a), (R)std::sin(a)});
            }
    MOAO_HIP_TRY(hipMalloc((void**)d_table, sizeof(C) * h.size()));
    MOAO_HIP_TRY(hipMemcpyAsync(*d_table, h.data(), sizeof(C) * h.size(), hipMemcpyHostToDevice, s));
    MOAO_HIP_TRY(hipStreamSynchronize(s));
    return MOAO_OK;
}

template int fft_twiddles<float>(int, float2**, hipStream_t);
template int fft_twiddles<double>(int, double2**, hipStream_t);

}  // namespace moao
