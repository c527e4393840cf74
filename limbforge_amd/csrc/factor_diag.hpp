// factor_diag.hpp — the diagonal block of a Cholesky panel with a digit per lane (factor_wave.hpp).
#pragma once
#include "factor_wave.hpp"

namespace lf {

// ------------------------------------------------------------------ fixed point: F fraction digits
// Fraction digits of the square root's Newton iteration: those of a stored reciprocal (32N + 65 bits).
template <int N> constexpr int wd_frac() { return wd_recip<N>(); }

// Columns of a * b for a's digits FROM .. F, held in lanes A0 + FROM .. A0 + F, and b aligned (digit i in lane i, an
// integer digit in lane F).  The columns of a product of two aligned numbers are "raised": F more fraction digits,
// the integer digit in lane 2F; their digits from lane F up serve as the next a with A0 = F, with no shift.
template <int F, int FROM, int A0> __device__ __forceinline__ i64 wd_columns(u32 a, u32 b, u32 lane)
{
    i64 S = 0;
    u32 bs = b;
    if constexpr (FROM > 0) {
        bs = (u32)__shfl((int)b, (int)((lane - (u32)FROM) & 63u));
        bs = lane >= (u32)FROM ? bs : 0u;
    }
#pragma unroll
    for (int i = FROM; i <= F; ++i) {
        S += (i64)(int)wd_read(a, A0 + i) * (int)bs;
        bs = wave_from_previous_lane(bs);
    }
    return S;
}
// Columns split into their three balanced digits and added up, no carries after that: signed digits below 2^26.1 in
// magnitude, which serve as factors where a result's exact digits are not needed.  Balanced, a small column of either
// sign stays in its lane, so the digits of a raised number end at lane 2F.
__device__ __forceinline__ u32 wd_loose(i64 S)
{
    const i64 T = S + ((i64)1 << (WD_BITS - 1)) + ((i64)1 << (2 * WD_BITS - 1));
    const u32 lo = (u32)T & WD_MASK, mid = (u32)(T >> WD_BITS) & WD_MASK, hi = (u32)(int)(T >> (2 * WD_BITS));
    return lo + wave_from_previous_lane(mid + wave_from_previous_lane(hi)) - (1u << WD_BITS);
}
// raised <-> aligned digits
template <int F> __device__ __forceinline__ u32 wd_align(u32 d, u32 lane)
{
    const u32 r = (u32)__shfl((int)d, (int)((lane + (u32)F) & 63u));
    return lane + (u32)F < 64u ? r : 0u;
}
template <int F> __device__ __forceinline__ u32 wd_raise(u32 d, u32 lane)
{
    const u32 r = (u32)__shfl((int)d, (int)((lane - (u32)F) & 63u));
    return lane >= (u32)F ? r : 0u;
}

// m << s (s uniform, >= 0)
__device__ __forceinline__ u32 wd_shift_left(u32 m, int s, u32 lane)
{
    const int q = s / WD_BITS, b = s - WD_BITS * q;
    u32 y = (u32)__shfl((int)m, (int)((lane - (u32)q) & 63u));
    y = lane >= (u32)q ? y : 0u;
    return ((y << b) | (wave_from_previous_lane(y) >> (WD_BITS - b))) & WD_MASK;
}

// 2^61 / sqrt(x), x = top / 2^64 in [1/4, 1), from below, to about 56 bits: the FP32 reciprocal square root and one
// third-order step z (1 + g/2 + 3 g^2 / 8), g = 1 - x z^2, in 64-bit fixed point (g is below 2^-20, so g^2 takes 32
// bits).
__device__ __forceinline__ u64 wd_rsqrt_seed(u64 top)
{
    const float x = (float)(u32)(top >> 40) * 0x1p-24f;
    const u64 z = ((u64)(u32)(__builtin_amdgcn_rsqf(x) * 0x1p30f) - 1024u) << 31; // below 2^61 / sqrt(x) by 2^-21 to 2^-18
    const u64 g = ((u64)1 << 61) - mul_hi64(top, mul_hi64(z, z) << 3);           // g * 2^61, positive
    const u32 gs = (u32)(g >> 16);                                               // g * 2^45
    const u64 q = (g >> 1) + (((u64)gs * gs * 3u) >> 32);                        // (g/2 + 3 g^2 / 8) * 2^61
    return z + (mul_hi64(z, q) << 3) - 32u;
}

// y <- y (3 - u y^2) / 2 with uh = u / 2: twice y's bits; a's digits below FROM left out of the products
template <int F, int FROM> __device__ __forceinline__ u32 wd_rsqrt_step(u32 y, u32 uh, u32 lane)
{
    const u32 p = wd_resolve(wd_columns<F, FROM, 0>(y, y, lane), lane);
    const i64 c = (int)lane == 2 * F ? 1 : (int)lane == 2 * F - 1 ? (i64)1 << (WD_BITS - 1) : 0; // 3/2
    const u32 e = wd_resolve(c - wd_columns<F, FROM, F>(p, uh, lane), lane);
    return wd_align<F>(wd_resolve(wd_columns<F, FROM, F>(e, y, lane), lane), lane);
}
// The same from the 56-bit seed to three times its bits: with k = 1/2 - uh y^2 >= 0 (y is from below),
// 2 y' = 2 y + y k (2 + 3 k).
template <int F> __device__ __forceinline__ u32 wd_rsqrt_first(u32 y, u32 uh, u32 lane)
{
    constexpr int A = F > 3 ? F - 3 : 0, B = F > 6 ? F - 6 : 0, C = F > 8 ? F - 8 : 0;
    const u32 p = wd_resolve(wd_columns<F, A, 0>(y, y, lane), lane);
    const u32 k = wd_resolve(((int)lane == 2 * F - 1 ? (i64)1 << (WD_BITS - 1) : 0) - wd_columns<F, B, F>(p, uh, lane), lane);
    const u32 k23 = 3u * wd_align<F>(k, lane) + ((int)lane == F ? 2u : 0u);
    const u32 q = wd_resolve(wd_columns<F, C, F>(k, k23, lane), lane);
    const u32 y2 = wd_resolve(wd_columns<F, C, F>(q, y, lane) + 2 * (i64)wd_raise<F>(y, lane), lane);
    return wd_shift_right(y2, WD_BITS * F + 1, lane);
}
// Steps until y has half the bits that the root and the reciprocal need (each doubles them once more).
template <int N, int BITS> __device__ __forceinline__ u32 wd_rsqrt(u32 y, u32 uh, u32 lane)
{
    constexpr int F = wd_frac<N>();
    if constexpr (2 * BITS - 4 >= 32 * N + 40) return y;
    else {
        constexpr int keep = (2 * BITS) / WD_BITS + 2;
        return wd_rsqrt<N, 2 * BITS - 2>(wd_rsqrt_step<F, (keep < F ? F - keep : 0)>(y, uh, lane), uh, lane);
    }
}

// l = RN(sqrt(s)) for s > 0, and R = the reciprocal of l's mantissa, 2^(64N + 64) / L to within 2^30 units.
// With M = m 2^odd / 2^(32N-1) in [1, 4), uh = M / 8 and y = 2 / sqrt(M) to half of the bits: r0 = uh y is sqrt(M) / 4
// from below, 2 r0 + (uh - 2 r0^2) y is sqrt(M) / 2 to all of them, and y (4 - l y) / 4 is 1 / l.  A root is never
// halfway between two mantissas; false when the 24 bits below the last one do not tell which side of halfway it
// lies on (about one root in 2^23), or when R's last words are too close to a carry for its leading words to be
// those of the exact quotient (about one in 2^31 of the others).  That would be every root that is a power of two
// (2^(64N + 64) / L is one itself), and such roots are common: a unit diagonal's, an identity's, those of scaled integers.
// Their reciprocal, ones in all its bits, is known.
template <int N> __device__ __forceinline__ bool wd_sqrt(const WaveNum& s, u32 lane, WaveNum& l, u32& R)
{
    constexpr int D = wd_mant<N>(), F = wd_frac<N>();
    static_assert(2 * F + 2 <= 64, "raised digits fit the wavefront");
    const int e = (int)(s.e >> 1), odd = (int)s.e - 2 * e;
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
    const u32 uhr = wd_raise<F>(uh, lane);
    u32 p, g, r, c;
    auto power_of_two = [&]() -> bool {
        constexpr int ones = 32 * N + 65; // bits of 2^(32N + 65) - 1
        if (wd_read(l.m, D - 1) != 1u << (32 * N - 1 - WD_BITS * (D - 1)) || __ballot(l.m != 0) != (u64)1 << (D - 1)) return false;
        const int left = ones - WD_BITS * (int)lane;
        R = left >= WD_BITS ? WD_MASK : left > 0 ? (1u << left) - 1u : 0u;
        return true;
    };
    auto root = [&](int sigma) -> bool {
        l.m = wd_shift_right(p, sigma, lane);
        l.e = e;
        l.s = 1;
        g = wd_below(p, sigma);
        if (g == 0x7fffffu || g == 0x800000u) return false;
        if (g >> 23) l.m = wd_increment<N>(l.m, l.e, lane);
        if (l.e != e) return false; // rounded up to the next power of two
        r = wd_shift_left(l.m, WD_BITS * F - (32 * N - 1), lane);
        return true;
    };
    if constexpr (2 * 164 - 4 >= 32 * N + 40) {
        // the first step's 164 bits are half enough: on loose digits, with Y = 8 y (k = 1/2 - uh y^2, Y = 8 y +
        // y k (8 + 12 k)), q0 = uh Y = 2 sqrt(M), 128 sqrt(M) = 64 q0 + (32 uh - q0^2) Y, and Y (32 - l Y) / 256 = 1 / l
        constexpr int A = F > 3 ? F - 3 : 0, B = F > 6 ? F - 6 : 0, C = F > 8 ? F - 8 : 0;
        const u32 y2 = wd_loose(wd_columns<F, A, 0>(y, y, lane));
        const u32 k = wd_loose(((int)lane == 2 * F - 1 ? (i64)1 << (WD_BITS - 1) : 0) - wd_columns<F, B, F>(y2, uh, lane));
        const u32 k12 = 12u * wd_align<F>(k, lane) + ((int)lane == F ? 8u : 0u);
        const u32 q = wd_loose(wd_columns<F, C, F>(k, k12, lane));
        const u32 Y = wd_align<F>(wd_loose(wd_columns<F, C, F>(q, y, lane) + 8 * (i64)wd_raise<F>(y, lane)), lane);
        const u32 q0 = wd_loose(wd_columns<F, 0, 0>(Y, uh, lane)), qa = wd_align<F>(q0, lane);
        const u32 d = wd_loose(32 * (i64)uhr - wd_columns<F, 0, 0>(qa, qa, lane));
        p = wd_resolve(wd_columns<F, 0, F>(d, Y, lane) + (lane >= (u32)F ? 64 * (i64)(int)q0 : 0), lane);
        if (!root(2 * WD_BITS * F - 32 * N + 8)) return false;
        if (power_of_two()) return true;
        c = wd_loose(((int)lane == 2 * F ? (i64)32 : 0) - wd_columns<F, 0, 0>(Y, r, lane));
        R = wd_shift_right(wd_resolve(wd_columns<F, 0, F>(c, Y, lane), lane), 2 * WD_BITS * F - 32 * N - 57, lane);
    } else {
        y = wd_rsqrt<N, 164>(wd_rsqrt_first<F>(y, uh, lane), uh, lane);
        const u32 p0 = wd_resolve(wd_columns<F, 0, 0>(y, uh, lane), lane), r0 = wd_align<F>(p0, lane);
        const u32 d2 = wd_resolve((i64)uhr - 2 * wd_columns<F, 0, 0>(r0, r0, lane), lane);
        p = wd_resolve(wd_columns<F, 0, F>(d2, y, lane) + (lane >= (u32)F ? 2 * (i64)p0 : 0), lane);
        if (!root(2 * WD_BITS * F - 32 * N)) return false;
        if (power_of_two()) return true;
        c = wd_resolve(((int)lane == 2 * F ? (i64)4 : 0) - wd_columns<F, 0, 0>(y, r, lane), lane);
        R = wd_shift_right(wd_resolve(wd_columns<F, 0, F>(c, y, lane), lane), 2 * WD_BITS * F - 32 * N - 63, lane);
    }
    const u32 low = (u32)((((u64)wd_read(R, 2) << (2 * WD_BITS)) | ((u64)wd_read(R, 1) << WD_BITS)) >> 32);
    return low != 0u && low != 0xffffffffu;
}

// Word `lane` of the N + 3 words of the reciprocal digits R.
template <int N> __device__ __forceinline__ u32 wd_recip_word(u32 R, u32 lane)
{
    const u32 bit = 32u * (lane < (u32)N + 3 ? lane : 0u), k = bit / WD_BITS, s = bit - WD_BITS * k;
    const u32 a = (u32)__shfl((int)R, (int)k), b = (u32)__shfl((int)R, (int)k + 1), c = (u32)__shfl((int)R, (int)k + 2);
    return (u32)(((u64)a | ((u64)b << WD_BITS) | ((u64)c << (2 * WD_BITS))) >> s);
}

// ------------------------------------------------------------------ the block
// The block [k0, k1) of up to 32 columns in one workgroup of DIAG_WAVES wavefronts, column by column.  LDS
// holds the lower triangle as signed grid digits (entries of columns not yet done: a_ij; done: l_ij) and the
// accumulators of three columns.  Column j:
//   A  wave 0 takes the last term off the pivot's accumulator and forms l_jj = sqrt(s_jj) and its reciprocal;
//      meanwhile the others add the terms k < j of column j + 1, two lanes a term (half of the digits each), start
//      column j + 2, take the last term off the accumulators of their rows and round them;
//   B  each row is divided by l_jj and l_ij replaces a_ij in LDS.
// A column's entries go to global memory only when all of it is decided; info->resume is the number of
// columns done, and chol_diag_kernel does the rest (a failed pivot, a status, spreads past the columns).
// What bounds it is the chain of wave 0's wave-parallel products in A: nine for the root and the reciprocal at
// 256 bits.  A 32-column block at 256 bits took 512 us with an exact dot a wavefront per entry and one-lane roots
// and divisions, 194 us with twelve products for the pivot and the rows rounded after it, and 131 us so.
constexpr int DIAG_WAVES = 16;
template <int N> struct DiagLds {
    i64 acc[3][WD_ROWS][WD_COLS + 1]; // column j: acc[j % 3], row i
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
    if (f.info->pivot >= 0) return; // a block before this one failed
    if (t < 3) L.slow[t] = 0;
    if (t < sizeof(L.recip) / 4) L.recip[t] = 0;
    __syncthreads();
    {   // the block's lower triangle
        const u32 i = t / WD_ROWS, k = t % WD_ROWS;
        if (i < B && k <= i) {
            const Num<N> a = load_out<N>(f.w, f.pitch, (u64)(f.k0 + i) * f.n + f.k0 + k);
            if (a.st || (i == k && !a.s)) L.slow[2] = 1;
            int d[GD], o;
            lane_to_grid<N>(a, d, o); // (a record of sign 0 is zero whatever its limbs hold, and its accumulator starts from its digits)
            if (i == k) {
#pragma unroll
                for (int j = 0; j < GD; ++j) L.ddigit[j][i] = a.s < 0 ? -d[j] : a.s ? d[j] : 0;
                L.dorigin[i] = a.s ? o : WD_ZERO;
            } else {
                const u32 at = wd_at(i, k);
#pragma unroll
                for (int j = 0; j < GD; ++j) L.digit[j][at] = a.s < 0 ? -d[j] : a.s ? d[j] : 0;
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
    auto start_entry = [&](u32 i, u32 k) -> bool {
        const u32 at = i == k ? 0u : wd_at(i, k);
        const int alpha = diag_alpha<N>(L.dorigin[i], L.dorigin[k]);
        return i == k ? start(L.acc[k % 3u][i], L.dorigin[i], alpha, &L.ddigit[0][i], WD_ROWS)
                      : start(L.acc[k % 3u][i], L.origin[at], alpha, &L.digit[0][at], WD_TRI);
    };
    // S less the last term l_ik l_jk of entry (i, j), both factors' digits spread over the lanes; false when it does
    // not fit the accumulator's columns
    auto last_term = [&](u32 i, u32 j, i64& S, int alpha) -> bool {
        const u32 ax = wd_at(i, j - 1), ay = wd_at(j, j - 1);
        const int ox = L.origin[ax], oy = L.origin[ay];
        if (ox == WD_ZERO || oy == WD_ZERO) return true;
        const int o = ox + oy - alpha;
        if (o < 0 || o + 2 * GD - 1 > WD_TOP) return false;
        const u32 dl = lane < (u32)GD ? lane : 0u;
        const int x = lane < (u32)GD ? L.digit[dl][ax] : 0;
        int y = lane < (u32)GD ? L.digit[dl][ay] : 0;
        i64 q = 0;
#pragma unroll
        for (int k = 0; k < GD; ++k) {
            q += (i64)(int)wd_read((u32)x, k) * y;
            y = (int)wave_from_previous_lane((u32)y);
        }
        const int from = (int)lane - o;
        const u32 lo = (u32)__shfl((int)(u32)q, from & 63), hi = (u32)__shfl((int)(u32)((u64)q >> 32), from & 63);
        S -= from >= 0 ? (i64)(((u64)hi << 32) | lo) : 0;
        return true;
    };
    {
        bool fits = true;
        for (u32 i = wave; i < B; i += DIAG_WAVES) {
            fits = start_entry(i, 0) && fits;
            if (i) fits = start_entry(i, 1) && fits;
        }
        if (!fits) L.slow[2] = 1;
    }
    __syncthreads();
    if (L.slow[2]) {
        if (t == 0) f.info->resume = 0;
        return;
    }
    constexpr int ROWS = (WD_ROWS - 1 + DIAG_WAVES - 2) / (DIAG_WAVES - 1); // rows of a column that one wave takes
    WaveNum piv{0, 0, 0}, x[ROWS];
    u32 R = 0, pivot_word = 0, recip_word = 0, j = 0;
    for (; j < B; ++j) {
        // ---- A
        if (wave == 0) {
            i64 S = L.acc[j % 3u][j][lane];
            const int alpha = diag_alpha<N>(L.dorigin[j], L.dorigin[j]);
            WaveNum s;
            bool ok = true;
            if (j) ok = last_term(j, j, S, alpha);
            ok = ok && wd_round<N>(S, alpha, lane, s) && s.s > 0 && wd_sqrt<N>(s, lane, piv, R);
            if (ok) {
                if ((int)lane < RD) L.recip[D - 1 + (int)lane] = R;
                if (lane == 0) L.pe = (int)piv.e;
            } else if (lane == 0)
                L.slow[0] = 1;
        } else {
            // the terms k < j of column j + 1: lanes next to each other take different rows, so that their adds go to
            // different accumulators
            if (j && j + 1 < B) {
                const u32 rows = B - 1 - j, u = t - 64u, half = u & 1u, rest = u >> 1;
                const u32 k = rest / rows, i = j + 1 + rest - k * rows;
                if (k < j) {
                    const u32 ax = wd_at(i, k), al = wd_at(j + 1, k);
                    const int ox = L.origin[ax], ol = L.origin[al];
                    if (ox != WD_ZERO && ol != WD_ZERO) {
                        const int o = ox + ol - diag_alpha<N>(L.dorigin[i], L.dorigin[j + 1]);
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
                            wd_accumulate<GD, H>(&L.acc[(j + 1) % 3u][i][0] + o + H * (int)half, xd, ld);
                        }
                    }
                }
            }
            // this wave's rows of column j
#pragma unroll
            for (int q = 0; q < ROWS; ++q) {
                const u32 i = j + wave + (u32)q * (DIAG_WAVES - 1);
                if (i >= B) break;
                if (i >= j + 2 && !start_entry(i, j + 2)) L.slow[0] = 1;
                i64 S = L.acc[j % 3u][i][lane];
                const int alpha = diag_alpha<N>(L.dorigin[i], L.dorigin[j]);
                if ((j && !last_term(i, j, S, alpha)) || !wd_round<N>(S, alpha, lane, x[q])) {
                    if (lane == 0) L.slow[0] = 1;
                    break;
                }
            }
        }
        __syncthreads();
        if (L.slow[0]) break;
        // ---- B
        if (wave) {
            u32 Rs[D];
#pragma unroll
            for (int k = 0; k < D; ++k) Rs[k] = L.recip[D - 1 + (int)lane - k];
            const i64 pe = L.pe;
#pragma unroll
            for (int q = 0; q < ROWS; ++q) {
                const u32 i = j + wave + (u32)q * (DIAG_WAVES - 1);
                if (i >= B) break;
                WaveNum l;
                if (!wd_divide<N>(x[q], Rs, pe, 1, lane, l)) {
                    if (lane == 0) L.slow[1] = 1;
                    break;
                }
                x[q] = l;
                int o;
                const int gd = (int)wd_to_grid<N>(l, o);
                const u32 at = wd_at(i, j);
                if ((int)lane < GD) L.digit[lane][at] = l.s < 0 ? -gd : gd;
                if (lane == 0) L.origin[at] = l.s ? o : WD_ZERO;
            }
        } else { // the pivot's and the reciprocal's words, while the rows divide
            pivot_word = wd_record_word<N>(piv, lane);
            recip_word = wd_recip_word<N>(R, lane);
        }
        __syncthreads();
        if (L.slow[1]) break;
        // ---- the column is decided
        if (wave == 0) {
            if (lane < (u32)N + 3) {
                f.w[(u64)lane * f.pitch + (u64)(f.k0 + j) * f.n + f.k0 + j] = pivot_word;
                f.recip[(u64)lane * f.rpitch + f.k0 + j] = recip_word;
            }
        } else {
#pragma unroll
            for (int q = 0; q < ROWS; ++q) {
                const u32 i = j + wave + (u32)q * (DIAG_WAVES - 1);
                if (i < B) wd_store<N>(f.w, f.pitch, (u64)(f.k0 + i) * f.n + f.k0 + j, x[q], lane);
            }
        }
    }
    if (t == 0) f.info->resume = (int32_t)j;
}

} // namespace lf
