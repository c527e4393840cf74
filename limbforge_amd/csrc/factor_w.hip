// One width of the Cholesky / triangular-solve kernels: compiled once per LF_WORDS in [2, 32].
#include "factor_kernels.hpp"
#include "factor_launch.hpp"

#include <algorithm>

#ifndef LF_WORDS
#error "compile with -DLF_WORDS=<2..32>"
#endif

namespace lf {

template <int N> hipError_t launch_chol_diag(const FactorArgs& f, hipStream_t s)
{
    if (f.k1 <= f.k0) return hipSuccess;
    uint32_t resume = 0;
    if constexpr (wd_fits<N>())
        if (f.k1 - f.k0 <= WD_ROWS) { // what it leaves, usually nothing, is the general kernel's
            hipLaunchKernelGGL((chol_diag_wave_kernel<N>), dim3(1), dim3(DIAG_WAVES * WAVE), 0, s, f);
            if (hipError_t e = hipGetLastError()) return e;
            resume = 1;
        }
    hipLaunchKernelGGL((chol_diag_kernel<N>), dim3(1), dim3(diag_waves<N>() * WAVE), 0, s, f, resume);
    return hipGetLastError();
}

template <int N> hipError_t launch_tri_block(const TriArgs& g, hipStream_t s)
{
    if (!g.count || !g.rows) return hipSuccess;
    if constexpr (wd_fits<N>())
        if (g.rows <= WD_ROWS) {
            hipLaunchKernelGGL((tri_block_kernel<N>), dim3((g.count + TRI_WAVES - 1) / TRI_WAVES), dim3(64 * TRI_WAVES), 0, s, g);
            return hipGetLastError();
        }
    hipLaunchKernelGGL((tri_general_kernel<N>), dim3(g.count), dim3(64), 0, s, g);
    return hipGetLastError();
}

template <int N> hipError_t launch_update(const UpdateArgs& g, uint32_t waves, hipStream_t s)
{
    if (!g.rows || !g.cols || !waves) return hipSuccess;
    if constexpr (wd_fits<N>())
        if (g.K <= WD_ROWS && waves >= UPD_WAVES) {
            const uint32_t tc = upd_cols(g.cols), tr = upd_rows(tc);
            const uint64_t tiles = (uint64_t)((g.rows + tr - 1) / tr) * ((g.cols + tc - 1) / tc);
            hipLaunchKernelGGL((update_wave_kernel<N>), dim3((unsigned)std::min<uint64_t>(tiles, waves / UPD_WAVES)), dim3(64 * UPD_WAVES), 0, s, g);
            return hipGetLastError();
        }
    hipLaunchKernelGGL((update_kernel<N>), dim3((unsigned)std::min<uint64_t>((uint64_t)g.rows * g.cols, waves)), dim3(WAVE), 0, s, g);
    return hipGetLastError();
}

template <int N> hipError_t launch_chol_invalid(uint32_t* w, uint64_t pitch, uint32_t n, uint32_t p, hipStream_t s)
{
    const uint64_t m = n - p;
    if (!m) return hipSuccess;
    hipLaunchKernelGGL((chol_invalid_kernel<N>), dim3((unsigned)((m * m + 255u) / 256u)), dim3(256), 0, s, w, pitch, n, p);
    return hipGetLastError();
}

template <int N> hipError_t launch_zero_upper(uint32_t* w, uint64_t pitch, uint32_t n, hipStream_t s)
{
    const uint64_t total = (uint64_t)n * n;
    if (!total) return hipSuccess;
    hipLaunchKernelGGL((zero_upper_kernel<N>), dim3((unsigned)((total + 255u) / 256u)), dim3(256), 0, s, w, pitch, n);
    return hipGetLastError();
}

template <int N> hipError_t launch_reciprocals(const uint32_t* w, uint64_t pitch, uint32_t n, uint32_t* recip, uint64_t rpitch, hipStream_t s)
{
    if (!n) return hipSuccess;
    hipLaunchKernelGGL((reciprocals_kernel<N>), dim3((n + 63) / 64), dim3(64), 0, s, w, pitch, n, recip, rpitch);
    return hipGetLastError();
}

template <int N>
hipError_t launch_factor_steps(const uint32_t* v, uint64_t pitch, uint32_t* scratch, uint64_t swords, int32_t* err, int reps, uint64_t* out,
                               uint32_t* sink, hipStream_t s)
{
    hipLaunchKernelGGL((factor_steps_kernel<N, 0>), dim3(1), dim3(WAVE), 0, s, v, pitch, scratch, swords, err, reps, out, sink);
    hipLaunchKernelGGL((factor_steps_kernel<N, 1>), dim3(1), dim3(WAVE), 0, s, v, pitch, scratch, swords, err, reps, out, sink);
    hipLaunchKernelGGL((factor_steps_kernel<N, 2>), dim3(1), dim3(WAVE), 0, s, v, pitch, scratch, swords, err, reps, out, sink);
    hipLaunchKernelGGL((factor_steps_kernel<N, 3>), dim3(1), dim3(WAVE), 0, s, v, pitch, scratch, swords, err, reps, out, sink);
    hipLaunchKernelGGL((factor_steps_kernel<N, 4>), dim3(1), dim3(WAVE), 0, s, v, pitch, scratch, swords, err, reps, out, sink);
    return hipGetLastError();
}

template hipError_t launch_chol_diag<LF_WORDS>(const FactorArgs&, hipStream_t);
template hipError_t launch_factor_steps<LF_WORDS>(const uint32_t*, uint64_t, uint32_t*, uint64_t, int32_t*, int, uint64_t*, uint32_t*, hipStream_t);
template hipError_t launch_tri_block<LF_WORDS>(const TriArgs&, hipStream_t);
template hipError_t launch_update<LF_WORDS>(const UpdateArgs&, uint32_t, hipStream_t);
template hipError_t launch_chol_invalid<LF_WORDS>(uint32_t*, uint64_t, uint32_t, uint32_t, hipStream_t);
template hipError_t launch_zero_upper<LF_WORDS>(uint32_t*, uint64_t, uint32_t, hipStream_t);
template hipError_t launch_reciprocals<LF_WORDS>(const uint32_t*, uint64_t, uint32_t, uint32_t*, uint64_t, hipStream_t);

} // namespace lf
