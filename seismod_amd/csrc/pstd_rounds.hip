// pstd_rounds.hip -- the spectral derivatives' kernels for lines whose passes
// take several rounds of a workgroup (FftPlan::loop).
#define PSTD_ROUNDS
#include "pstd_fft.hpp"

namespace sm {
namespace pstd {

template <typename T>
const void *rounds_kernel()
{
    return (const void *)rounds::pstd_dfft<T, 1, true>;
}

template <typename T>
void rounds_launch(unsigned grid, unsigned nt, size_t lds, hipStream_t st, const DfftArgs<T> &ax, const DfftArgs<T> &az)
{
    rounds::pstd_dfft<T, 1, true><<<grid, nt, lds, st>>>(ax, az);
}

template const void *rounds_kernel<float>();
template const void *rounds_kernel<double>();
template void rounds_launch<float>(unsigned, unsigned, size_t, hipStream_t, const DfftArgs<float> &,
                                   const DfftArgs<float> &);
template void rounds_launch<double>(unsigned, unsigned, size_t, hipStream_t, const DfftArgs<double> &,
                                    const DfftArgs<double> &);

}  // namespace pstd
}  // namespace sm
