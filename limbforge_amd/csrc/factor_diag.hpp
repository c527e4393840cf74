// factor_diag.hpp — the diagonal block of a Cholesky panel with a digit per lane (factor_wave.hpp).
#pragma once
#include "factor_wave.hpp"

namespace lf {

// ------------------------------------------------------------------ fixed point: F fraction digits
// Fraction digits of the square root's Newton iteration: those of a stored reciprocal (32N + 65 bits).
template <int N> constexpr int wd_frac() { return wd_recip<N>(); }

// a * b truncated to F fraction digits, a's digits below FROM left out (a, b: lanes 0 .. F, an integer digit
// in lane F).
template <int F, int FROM> __device__ __forceinline__ u32 wd_mul_fixed(u32 a, u32 b, u32 lane)
{
    u64 S = 0;
    u32 bs = b;
    if constexpr (FROM > 0) {
        bs = (u32)__shfl((int)b, (int)((lane - (u32)FROM) & 63u));
        bs = lane >= (u32)FROM ? bs : 0u;
    }
#pragma unroll
    for (int i = FROM; i <= F; ++i) {
        S += (u64)wd_read(a, i) * bs;
        bs = wave_from_previous_lane(bs);
    }
    const u32 d = wd_resolve((i64)S, lane);
    const u32 r = (u32)__shfl((int)d, (int)((lane + (u32)F) & 63u));
    return lane + (u32)F < 64u ? r : 0u;
}

// m << s (s uniform, >= 0)
__device__ __forceinline__ u32 wd_shift_left(u32 m, int s, u32 lane)
{
    const int q = s / WD_BITS, b = s - WD_BITS * q;
    u32 y = (u32)__shfl((int)m, (int)((lane - (u32)q) & 63u));
    y = lane >= (u32)q ? y : 0u;
    return ((y << b) | (wave_from_previous_lane(y) >> (WD_BITS - b))) & WD_MASK;
}

// 2^61 / sqrt(x), x = top / 2^64 in [1/4, 1), to about 57 bits: the FP32 reciprocal square root and two Newton
// steps in 64-bit fixed point (limb_core.hpp rsqrt_seed takes five from a constant).
__device__ __forceinline__ u64 wd_rsqrt_seed(u64 top)
{
    const float x = (float)(u32)(top >> 40) * 0x1p-24f;
    u64 z = (u64)(u32)(__builtin_amdgcn_rsqf(x) * 0x1p30f) << 31;
#pragma unroll
    for (int it = 0; it < 2; ++it) {
        const u64 t = ((u64)3 << 61) - mul_hi64(top, mul_hi64(z, z) << 3);
        z = mul_hi64(z, t) << 2;
    }
    return z;
}

// y <- y (3 - u y^2) / 2 with uh = u / 2, the result good to twice y's bits; FROM as in wd_mul_fixed
template <int F, int FROM> __device__ __forceinline__ u32 wd_rsqrt_step(u32 y, u32 uh, u32 lane)
{
    const u32 t = wd_mul_fixed<F, FROM>(wd_mul_fixed<F, FROM>(y, y, lane), uh, lane);
    const i64 c = (int)lane == F ? 1 : (int)lane == F - 1 ? (i64)1 << (WD_BITS - 1) : 0; // 3/2
    return wd_mul_fixed<F, FROM>(y, wd_resolve(c - (i64)t, lane), lane);
}
template <int N, int BITS> __device__ __forceinline__ u32 wd_rsqrt(u32 y, u32 uh, u32 lane)
{
    constexpr int F = wd_frac<N>();
    if constexpr (BITS >= 32 * N + 40) return y;
    else {
        constexpr int keep = (2 * BITS) / WD_BITS + 2;
        return wd_rsqrt<N, 2 * BITS - 1>(wd_rsqrt_step<F, (keep < F ? F - keep : 0)>(y, uh, lane), uh, lane);
    }
}

// l = RN(sqrt(s)) for s > 0, and R = the reciprocal of l's mantissa, 2^(64N + 64) / L to within 2^30 units.
// With M = m 2^odd / 2^(32N-1) in [1, 4) and y = 2 / sqrt(M): sqrt(M) = M y / 2, and one step from y/2 gives
// 1 / l.  A root is never halfway between two mantissas; false when the 24 bits below the last one do not
// tell which side of halfway it lies on (about one root in 2^23), or when R's last words are too close to
// a carry for its leading words to be those of the exact quotient.
template <int N> __device__ __forceinline__ bool wd_sqrt(const WaveNum& s, u32 lane, WaveNum& l, u32& R)
{
    constexpr int D = wd_mant<N>(), F = wd_frac<N>();
    const int e = (int)(s.e >> 1), odd = (int)s.e - 2 * e;
    // M / 8 on the fixed-point grid
    const u32 uh = wd_shift_left(s.m, WD_BITS * F - 32 * N - 2 + odd, lane);
    u64 top = 0; // the leading 64 bits of m (digits from 32N - 64 up)
    {
        constexpr int p = 32 * N - 64, q = p / WD_BITS, b = p - WD_BITS * q;
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (q + k < D) {
                const u64 d = wd_read(s.m, q + k);
                const int at = WD_BITS * k - b;
                if (at < 0) top |= d >> -at;
                else if (at < 64) top |= d << at;
            }
    }
    const u64 z = wd_rsqrt_seed(odd ? top : top >> 1);
    const int sh = 61 - WD_BITS * (F - (int)lane);
    u32 y = 0;
    if (sh >= 0 && sh < 64) y = (u32)(z >> sh) & WD_MASK;
    else if (sh < 0 && sh > -WD_BITS) y = (u32)(z << -sh) & WD_MASK;
    y = wd_rsqrt<N, 56>(y, uh, lane);
    const u32 p = wd_mul_fixed<F, 0>(uh, y, lane); // sqrt(M) / 4
    constexpr int sigma = WD_BITS * F - 32 * N - 1;
    l.m = wd_shift_right(p, sigma, lane);
    l.e = e;
    l.s = 1;
    const u32 g = wd_below(p, sigma);
    if (g == 0x7fffffu || g == 0x800000u) return false;
    if (g >> 23) l.m = wd_increment<N>(l.m, l.e, lane);
    if (l.e != e) return false; // rounded up to the next power of two
    const u32 r = wd_shift_left(l.m, WD_BITS * F - (32 * N - 1), lane);
    const u32 t = wd_mul_fixed<F, 0>(r, y, lane); // near 2
    const u32 c = wd_resolve(((int)lane == F ? (i64)4 : 0) - (i64)t, lane);
    R = wd_shift_right(wd_mul_fixed<F, 0>(y, c, lane), WD_BITS * F - 32 * N - 63, lane);
    const u32 low = (u32)((((u64)wd_read(R, 2) << (2 * WD_BITS)) | ((u64)wd_read(R, 1) << WD_BITS)) >> 32);
    return low != 0u && low != 0xffffffffu;
}

// Stores words 0 .. N + 2 of the reciprocal digits R at entry i of the reciprocal planes.
template <int N> __device__ __forceinline__ void wd_store_recip(u32* recip, u64 rpitch, u32 i, u32 R, u32 lane)
{
    const u32 bit = 32u * (lane < (u32)N + 3 ? lane : 0u), k = bit / WD_BITS, s = bit - WD_BITS * k;
    const u32 a = (u32)__shfl((int)R, (int)k), b = (u32)__shfl((int)R, (int)k + 1), c = (u32)__shfl((int)R, (int)k + 2);
    const u64 v = (u64)a | ((u64)b << WD_BITS) | ((u64)c << (2 * WD_BITS));
    if (lane < (u32)N + 3) recip[(u64)lane * rpitch + i] = (u32)(v >> s);
}

// ------------------------------------------------------------------ the block
// The block [k0, k1) of up to 32 columns in one workgroup of DIAG_WAVES wavefronts, column by column.  LDS
// holds the lower triangle as signed grid digits (entries of columns not yet done: a_ij; done: l_ij), one
// accumulator for each row of the column at work, and two for pivots.  Column j:
//   A  wave 0 takes the last term off the pivot's accumulator and forms l_jj = sqrt(s_jj) and its reciprocal;
//      meanwhile the other waves add the terms k < j to the accumulators of the rows below, and those of the
//      next pivot, two lanes a term (half of the digits each);
//   B  one wave a row rounds its accumulator and divides by l_jj, replaces a_ij by l_ij in LDS and starts the
//      accumulator of the row's next column.
// A column's entries go to global memory only when all of it is decided; info->resume is the number of
// columns done, and chol_diag_kernel does the rest (a failed pivot, a status, spreads past the columns).
// What bounds it is wave 0's instruction count in A (about 1,000, two thirds of them the Newton products)
// and one row's in B.  A 32-column block at 256 bits took 512 us with an exact dot a wavefront per entry and
// one-lane roots and divisions; with this the factorization of n = 512 went from 10.9 to 5.9 ms.
constexpr int DIAG_WAVES = 16;
template <int N> struct DiagLds {
    i64 acc[WD_ROWS][WD_COLS + 1];
    i64 pacc[2][WD_COLS + 1];
    int digit[wd_grid<N>()][WD_TRI];
    int origin[WD_TRI];
    int ddigit[wd_grid<N>()][WD_ROWS];
    int dorigin[WD_ROWS];
    u32 recip[wd_mant<N>() - 1 + WD_COLS];
    int pe;      // exponent of the pivot
    int slow[3]; // something this kernel does not decide, seen in A, in B, or on loading (each read only after a
                 // barrier that its next write follows by another)
};

// Origin of the accumulator of entry (i, j) from those of a_ii and a_jj: |a_ij| and every |l_ik l_jk| are at most
// sqrt(a_ii a_jj), so that magnitude goes near the top column and the room below is for small terms.
template <int N> __device__ __forceinline__ int diag_alpha(int oi, int oj) { return ((oi + oj) >> 1) + wd_grid<N>() - 1 - (WD_TOP - 4); }

__device__ __forceinline__ u32 wd_at(u32 i, u32 k) { return wd_col_start(k) + (i - k - 1); }

template <int N> __global__ void __launch_bounds__(DIAG_WAVES * 64) chol_diag_wave_kernel(FactorArgs f)
{
    constexpr int D = wd_mant<N>(), GD = wd_grid<N>(), RD = wd_recip<N>(), H = (GD + 1) / 2;
    __shared__ __attribute__((aligned(16))) unsigned char lds[sizeof(DiagLds<N>)];
    DiagLds<N>& L = *reinterpret_cast<DiagLds<N>*>(lds);
    const u32 t = threadIdx.x, wave = t / 64u, lane = t % 64u, B = f.k1 - f.k0;
    if (t < 3) L.slow[t] = 0;
    if (t < sizeof(L.recip) / 4) L.recip[t] = 0;
    __syncthreads();
    {   // the block's lower triangle
        const u32 i = t / WD_ROWS, k = t % WD_ROWS;
        if (i < B && k <= i) {
            const Num<N> a = load_out<N>(f.w, f.pitch, (u64)(f.k0 + i) * f.n + f.k0 + k);
            if (a.st || (i == k && !a.s)) L.slow[2] = 1;
            int d[GD], o;
            lane_to_grid<N>(a, d, o);
            if (i == k) {
#pragma unroll
                for (int j = 0; j < GD; ++j) L.ddigit[j][i] = a.s < 0 ? -d[j] : d[j];
                L.dorigin[i] = a.s ? o : WD_ZERO;
            } else {
                const u32 at = wd_at(i, k);
#pragma unroll
                for (int j = 0; j < GD; ++j) L.digit[j][at] = a.s < 0 ? -d[j] : d[j];
                L.origin[at] = a.s ? o : WD_ZERO;
            }
        }
    }
    __syncthreads();
    // start an accumulator from an entry's digits (one wave); false when they do not fit its columns
    auto start = [&](i64* acc, int o, int alpha, const int* digit, u32 pitch) -> bool {
        const int off = o == WD_ZERO ? 0 : o - alpha, dj = (int)lane - off;
        acc[lane] = dj >= 0 && dj < GD ? digit[(u32)(dj >= 0 && dj < GD ? dj : 0) * pitch] : 0;
        return off >= 0 && off + GD - 1 <= WD_TOP;
    };
    auto start_row = [&](u32 i, u32 k) -> bool {
        const u32 at = wd_at(i, k);
        return start(L.acc[i], L.origin[at], diag_alpha<N>(L.dorigin[i], L.dorigin[k]), &L.digit[0][at], WD_TRI);
    };
    auto start_pivot = [&](u32 j) -> bool {
        return start(L.pacc[j & 1u], L.dorigin[j], diag_alpha<N>(L.dorigin[j], L.dorigin[j]), &L.ddigit[0][j], WD_ROWS);
    };
    {
        bool fits = true;
        for (u32 i = 1 + wave; i < B; i += DIAG_WAVES) fits = start_row(i, 0) && fits;
        if (wave < 2 && wave < B) fits = start_pivot(wave) && fits;
        if (!fits) L.slow[2] = 1;
    }
    __syncthreads();
    if (L.slow[2]) {
        if (t == 0) f.info->resume = 0;
        return;
    }
    WaveNum piv{0, 0, 0}, x[2];
    u32 R = 0, j = 0;
    for (; j < B; ++j) {
        // ---- A
        if (wave == 0) {
            i64 S = L.pacc[j & 1u][lane];
            const int pa = diag_alpha<N>(L.dorigin[j], L.dorigin[j]);
            bool ok = true;
            if (j) {
                const u32 at = wd_at(j, j - 1);
                const int lo = L.origin[at];
                if (lo != WD_ZERO) {
                    const int o = 2 * lo - pa;
                    ok = o >= 0 && o + 2 * GD - 1 <= WD_TOP;
                    if (ok) {
                        const int g = (int)lane < GD ? L.digit[lane < (u32)GD ? lane : 0][at] : 0;
                        const u32 m = (u32)(g < 0 ? -g : g); // all of one sign
                        u64 q = 0;
                        u32 ms = m;
#pragma unroll
                        for (int i = 0; i < GD; ++i) {
                            q += (u64)wd_read(m, i) * ms;
                            ms = wave_from_previous_lane(ms);
                        }
                        const int from = (int)lane - o;
                        const u32 qa = (u32)__shfl((int)(u32)q, from & 63), qb = (u32)__shfl((int)(u32)(q >> 32), from & 63);
                        S -= from >= 0 ? (i64)(((u64)qb << 32) | qa) : 0;
                    }
                }
            }
            WaveNum s;
            ok = ok && wd_round<N>(S, pa, lane, s);
            ok = ok && s.s > 0 && wd_sqrt<N>(s, lane, piv, R);
            if (ok) {
                if ((int)lane < RD) L.recip[D - 1 + (int)lane] = R;
                if (lane == 0) L.pe = (int)piv.e;
            } else if (lane == 0)
                L.slow[0] = 1;
        } else if (j && j + 1 < B) {
            // slots: rows j + 1 .. B - 1 of column j, then the pivot of column j + 1; lanes next to each other take
            // different rows, so that their adds go to different accumulators
            const u32 slots = B - j, u = t - 64u, half = u & 1u, rest = u >> 1;
            const u32 k = rest / slots, slot = rest - k * slots;
            if (k < j) {
                const bool pivot = slot == slots - 1;
                const u32 i = pivot ? j + 1 : j + 1 + slot;
                const u32 ax = wd_at(i, k), al = pivot ? ax : wd_at(j, k);
                const int ox = L.origin[ax], ol = L.origin[al];
                if (ox != WD_ZERO && ol != WD_ZERO) {
                    const int o = ox + ol - diag_alpha<N>(L.dorigin[i], L.dorigin[pivot ? i : j]);
                    if (o < 0 || o + 2 * GD - 1 > WD_TOP) L.slow[0] = 1;
                    else {
                        int xd[H], ld[GD];
#pragma unroll
                        for (int q = 0; q < H; ++q) {
                            const int d = q + H * (int)half;
                            xd[q] = d < GD ? -L.digit[d < GD ? d : 0][ax] : 0;
                        }
#pragma unroll
                        for (int q = 0; q < GD; ++q) ld[q] = L.digit[q][al];
                        wd_accumulate<GD, H>((pivot ? &L.pacc[i & 1u][0] : &L.acc[i][0]) + o + H * (int)half, xd, ld);
                    }
                }
            }
        }
        __syncthreads();
        if (L.slow[0]) break;
        // ---- B
        {
            u32 Rs[D];
#pragma unroll
            for (int k = 0; k < D; ++k) Rs[k] = L.recip[D - 1 + (int)lane - k];
            const i64 pe = L.pe;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const u32 i = j + 1 + wave + (u32)q * DIAG_WAVES;
                if (i >= B) break;
                WaveNum v;
                if (!wd_round<N>(L.acc[i][lane], diag_alpha<N>(L.dorigin[i], L.dorigin[j]), lane, v) || !wd_divide<N>(v, Rs, pe, 1, lane, x[q])) {
                    if (lane == 0) L.slow[1] = 1;
                    break;
                }
                int o;
                const int gd = (int)wd_to_grid<N>(x[q], o);
                const u32 at = wd_at(i, j);
                if ((int)lane < GD) L.digit[lane][at] = x[q].s < 0 ? -gd : gd;
                if (lane == 0) L.origin[at] = x[q].s ? o : WD_ZERO;
                bool fits = true;
                if (i > j + 1) fits = start_row(i, j + 1);
                if (i == j + 2) fits = start_pivot(i) && fits;
                if (!fits) L.slow[1] = 1;
            }
        }
        __syncthreads();
        if (L.slow[1]) break;
        // ---- the column is decided
        if (wave == 0) {
            wd_store<N>(f.w, f.pitch, (u64)(f.k0 + j) * f.n + f.k0 + j, piv, lane);
            wd_store_recip<N>(f.recip, f.rpitch, f.k0 + j, R, lane);
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const u32 i = j + 1 + wave + (u32)q * DIAG_WAVES;
            if (i < B) wd_store<N>(f.w, f.pitch, (u64)(f.k0 + i) * f.n + f.k0 + j, x[q], lane);
        }
    }
    if (t == 0) f.info->resume = (int32_t)j;
}

} // namespace lf
