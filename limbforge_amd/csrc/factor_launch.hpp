// factor_launch.hpp — launch entry points of the Cholesky / triangular-solve kernels (instantiated per
// width in factor_w.hip) and the argument records they share with the host driver (factor.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace lf {

struct FactorInfo {
    int32_t pivot;   // first failing column, -1 while none
    int32_t sign;    // sign of the failing s_pp (0 for zero or a status)
    uint32_t status; // its status
    int32_t resume;  // columns of the block that the wave-parallel diagonal kernel decided
};

struct FactorArgs {
    uint32_t* w;   // work matrix planes, element (i, j) at i*n + j
    uint64_t pitch;
    uint32_t n, k0, k1;
    FactorInfo* info;
    FactorInfo* host;  // a failed pivot's record in pinned host memory (read only after the block's event)
    int32_t* error;    // cluster scratch overflow (never expected)
    uint32_t* scratch; // per thread: 2 * swords words
    uint64_t swords;
    uint32_t* recip;   // reciprocals of the pivots l_jj (up to N+3 planes, entry j), written by the diagonal kernel
    uint64_t rpitch;
};

// A triangular block T x = b for many right-hand sides, in place: element (r, k), k <= r, of the block at plane
// element fbase + r*fr + k*fk, element r of right-hand side c at xbase + r*xr + c*xc, the reciprocal of diagonal
// entry r at rbase + r*rstep.  Forward and backward solves and the rows below a Cholesky block are this one
// recurrence with other strides.
struct TriArgs {
    const uint32_t* f;
    uint64_t fpitch;
    int64_t fbase, fr, fk;
    uint32_t* x;
    uint64_t xpitch;
    int64_t xbase, xr, xc;
    const uint32_t* recip;
    uint64_t rpitch;
    int64_t rbase, rstep;
    uint32_t rows, count;  // block rows, right-hand sides
    uint32_t* scratch;     // per right-hand side: 2 * swords words
    uint64_t swords;
    int32_t* error;
    const FactorInfo* info; // not null: only the rows before a failed pivot (row 0 is column k0)
    uint32_t k0;
};

// Off-block update out_ic = D(out_ic; x_i, y_c; K) of rows x cols entries in place: element k of line x_i at
// xbase + i*xr + k*xk, of line y_c at ybase + c*yc + k*yk, entry (i, c) at obase + i*orow + c*ocol; with `lower` the
// entries c <= i alone.
struct UpdateArgs {
    const uint32_t* x;
    uint64_t xpitch;
    int64_t xbase, xr, xk;
    const uint32_t* y;
    uint64_t ypitch;
    int64_t ybase, yc, yk;
    uint32_t* out;
    uint64_t opitch;
    int64_t obase, orow, ocol;
    uint32_t rows, cols, K, lower;
    uint32_t* scratch; // 2 * swords words per wavefront
    uint64_t swords;
    int32_t* error;
};

// Window words of the register path of the exact dot: 2N product words plus 24 words (768 bits) of
// exponent spread; wider spreads take the cluster path.
constexpr int factor_window(int N) { return 2 * N + 24; }

// Scratch words per accumulator of the cluster path for dots of up to K terms (plus the addend): a
// cluster spans at most 64N bits plus (K+1) * (64N + gap) bits, gap = 32N + ceil(log2(K+1)) + 4.
inline uint64_t factor_scratch_words(int N, uint64_t K)
{
    int logk = 0;
    while ((uint64_t(1) << logk) < K + 1) ++logk;
    const uint64_t bits = 64ull * N + (K + 1) * (64ull * N + 32ull * N + logk + 4);
    return bits / 32 + 4;
}

template <int N> hipError_t launch_chol_diag(const FactorArgs& f, hipStream_t s);
// one wavefront timing the per-row steps (factor_steps_kernel)
template <int N>
hipError_t launch_factor_steps(const uint32_t* v, uint64_t pitch, uint32_t* scratch, uint64_t swords, int32_t* err, int reps, uint64_t* out,
                               uint32_t* sink, hipStream_t s);
// T x = b of one block for every right-hand side
template <int N> hipError_t launch_tri_block(const TriArgs& g, hipStream_t s);
// at most `waves` wavefronts (scratch slots)
template <int N> hipError_t launch_update(const UpdateArgs& g, uint32_t waves, hipStream_t s);
template <int N> hipError_t launch_chol_invalid(uint32_t* w, uint64_t pitch, uint32_t n, uint32_t p, hipStream_t s);
template <int N> hipError_t launch_zero_upper(uint32_t* w, uint64_t pitch, uint32_t n, hipStream_t s);
// recip entry i = reciprocal of the mantissa of the diagonal element (i, i) of the n x n planes, i < n (up to
// N+3 planes)
template <int N> hipError_t launch_reciprocals(const uint32_t* w, uint64_t pitch, uint32_t n, uint32_t* recip, uint64_t rpitch, hipStream_t s);

} // namespace lf
