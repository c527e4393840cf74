// factor_wave.hpp — wave-parallel exact sums, roundings and divisions of the factorization and the solves.
//
// A number is spread over the 64 lanes of a wavefront as 26-bit digits on one absolute grid: lane j of a
// grid number with origin a holds the digit of weight 2^(26(j + a)).  Digit products are below 2^52, so a
// 64-bit column takes the products of 32 terms of up to 26 digits each without a carry
// (32 * 26 * 2^52 < 2^62), and because every operand sits on the same grid, a product's columns meet an
// accumulator's columns with no shift: adding x_k * l_rk to row r's accumulator is a run of 64-bit LDS adds.
//
// What bounds the in-block recurrences is the instruction count of one wavefront (a step follows the one
// before, and few wavefronts are in flight), and the old step ran the exact dot of the row's terms, its
// rounding and a one-lane division one after another: about 12k cycles at 256 bits.  Here a row's terms are
// added as soon as their x is known, all rows of the block at once (one row on two lanes, half of x's digits
// each), so what remains on the chain is the rounding of one accumulator and one division, both with a digit
// per lane.
#pragma once
#include "factor_launch.hpp"
#include "gemm_kernels.hpp"

namespace lf {

constexpr int WD_BITS = 26;
constexpr u32 WD_MASK = (1u << WD_BITS) - 1;
constexpr int WD_COLS = 64; // accumulator columns: one per lane
// Digits of a 32N-bit mantissa; of a grid number (a mantissa shifted by up to 25 bits); of a reciprocal of
// N + 2 words and a bit.
template <int N> constexpr int wd_mant() { return (32 * N + WD_BITS - 1) / WD_BITS; }
template <int N> constexpr int wd_grid() { return (32 * N + 25 + WD_BITS - 1) / WD_BITS; }
template <int N> constexpr int wd_recip() { return (32 * N + 65 + WD_BITS - 1) / WD_BITS; }
// Widths whose products leave spare columns for the spread of a row's terms (20 limbs: 52 of 64 columns).
template <int N> constexpr bool wd_fits() { return N <= 20; }
// The addend's top digit goes to this column of its accumulator, in the middle of the room a product leaves;
// terms reach at most column WD_TOP (two columns and more hold the sum's growth and sign).
template <int N> constexpr int wd_center() { return wd_grid<N>() + 30; }
constexpr int WD_TOP = 61;

// Words of a stored reciprocal: floor((2^(64N) - 1) / B) with two more words of fraction where the
// wave-parallel division reads them.
template <int N> constexpr int recip_words() { return wd_fits<N>() ? N + 3 : N + 1; }

// The value of lane l + 1 in lane l (0 in lane 63): DPP wave_shl:1.  Every lane must be active.
__device__ __forceinline__ u32 wave_from_next_lane(u32 v) { return (u32)__builtin_amdgcn_update_dpp(0, (int)v, 0x130, 0xF, 0xF, true); }

__device__ __forceinline__ u32 wd_read(u32 v, int lane) { return (u32)__builtin_amdgcn_readlane((int)v, lane); }

// Digits of the two's-complement sum of signed columns (lane w: column w), modulo 2^(26 * 64).  Each column
// splits into three digits for this lane and the two above; a constant 2^26 - 1 added in every lane (-1 in
// all, taken back as the carry into lane 0) keeps the digit sums non-negative, so one add of carries leaves
// single-bit carries for the ballots.
__device__ __forceinline__ u32 wd_resolve(i64 S, u32 lane)
{
    const u32 lo = (u32)S & WD_MASK, mid = (u32)(S >> WD_BITS) & WD_MASK, hi = (u32)(int)(S >> (2 * WD_BITS));
    const u32 v = lo + wave_from_previous_lane(mid + wave_from_previous_lane(hi)) + WD_MASK;
    const u32 w = (v & WD_MASK) + wave_from_previous_lane(v >> WD_BITS);
    u64 cin = 1;
    const u32 c = wave_carry_in(w > WD_MASK, w == WD_MASK, lane, cin);
    return (w + c) & WD_MASK;
}

// Digits of -d modulo 2^(26 * 64).
__device__ __forceinline__ u32 wd_negate(u32 d, u32 lane)
{
    const u32 v = WD_MASK - d;
    u64 cin = 1;
    const u32 c = wave_carry_in(false, v == WD_MASK, lane, cin);
    return (v + c) & WD_MASK;
}

// d >> sigma (sigma uniform, 0 <= sigma < 26 * 64).
__device__ __forceinline__ u32 wd_shift_right(u32 d, int sigma, u32 lane)
{
    const int q = sigma / WD_BITS, b = sigma - WD_BITS * q;
    u32 y = (u32)__shfl((int)d, (int)((lane + (u32)q) & 63u));
    y = lane + (u32)q < 64u ? y : 0u;
    return ((y >> b) | (wave_from_next_lane(y) << (WD_BITS - b))) & WD_MASK;
}

// The 24 bits of d right below bit sigma (sigma uniform, >= 24).
__device__ __forceinline__ u32 wd_below(u32 d, int sigma)
{
    const int p = sigma - 24, q = p / WD_BITS, b = p - WD_BITS * q;
    const u64 two = (u64)wd_read(d, q) | ((u64)wd_read(d, (q + 1) & 63) << WD_BITS);
    return (u32)(two >> b) & 0xffffffu;
}

// A + 1 for a 32N-bit mantissa; e + 1 and the mantissa 2^(32N-1) when it leaves 32N bits.
template <int N> __device__ __forceinline__ u32 wd_increment(u32 A, i64& e, u32 lane)
{
    constexpr int D = wd_mant<N>(), TB = 32 * N - WD_BITS * (D - 1);
    if (wd_read(A, 0) != WD_MASK) return A + (lane == 0 ? 1u : 0u);
    const u64 ones = __ballot(A == WD_MASK);
    const int k = (int)__builtin_ctzll(~ones); // lanes from D on hold 0
    if (k >= D - 1 && wd_read(A, D - 1) == (1u << TB) - 1u) {
        ++e;
        return (int)lane == D - 1 ? 1u << (TB - 1) : 0u;
    }
    return (int)lane < k ? 0u : A + ((int)lane == k ? 1u : 0u);
}

// A number of the wave: 32N-bit mantissa (a digit per lane), exponent, sign (0: zero); no status.
struct WaveNum {
    u32 m;
    i64 e;
    int s;
};

// RN of the sum in the columns S of weight 2^(26(w + alpha)); false when a general routine has to decide
// (the sum reaches below the columns, or the exponent leaves the number range).
template <int N> __device__ __forceinline__ bool wd_round(i64 S, i64 alpha, u32 lane, WaveNum& r)
{
    u32 d = wd_resolve(S, lane);
    r.s = 1;
    if (wd_read(d, 63) >> (WD_BITS - 1)) {
        r.s = -1;
        d = wd_negate(d, lane);
    }
    const u64 nz = __ballot(d != 0);
    if (!nz) {
        r.m = 0;
        r.e = 0;
        r.s = 0;
        return true;
    }
    const int t = 63 - (int)__builtin_clzll(nz);
    const int top = WD_BITS * t + 31 - __builtin_clz(wd_read(d, t));
    const int sigma = top - (32 * N - 1);
    if (sigma < 24) return false;
    r.m = wd_shift_right(d, sigma, lane);
    r.e = (i64)WD_BITS * alpha + top;
    const u32 g = wd_below(d, sigma);
    const int p = sigma - 24, q = p / WD_BITS, b = p - WD_BITS * q;
    const bool sticky = (g & 0x7fffffu) != 0 || (wd_read(d, q) & ((1u << b) - 1u)) != 0 || (nz & (((u64)1 << q) - 1u)) != 0;
    if ((g >> 23) && (sticky || (wd_read(r.m, 0) & 1u))) r.m = wd_increment<N>(r.m, r.e, lane);
    return r.e <= EMAX && r.e >= -(i64)EMAX;
}

// RN(a / b) from the reciprocal R of b's mantissa, 2^P / B to within 2^30 units, P = 64N + 64, given as Rs[i] =
// digit lane - i of R (0 outside it); be, bs: b's exponent and sign.  V = A R is 2^P A / B to within 2^(32N + 30),
// and the quotient's last place is 2^(32N + 64) or more: the rounding bit tells, unless it and the 23 bits below it
// are 0111...1 or 1000...0 (about one division in 2^23 takes the general routine).  A quotient of two 32N-bit
// mantissas is never halfway between two others, so a set rounding bit rounds up.
template <int N>
__device__ __forceinline__ bool wd_divide(const WaveNum& a, const u32 (&Rs)[wd_mant<N>()], i64 be, int bs, u32 lane, WaveNum& q)
{
    q = WaveNum{0, 0, 0};
    if (!a.s) return true;
    constexpr int P = 64 * N + 64;
    u64 S = 0;
#pragma unroll
    for (int i = 0; i < wd_mant<N>(); ++i) S += (u64)wd_read(a.m, i) * Rs[i];
    const u32 V = wd_resolve((i64)S, lane);
    const bool ge = (wd_read(V, P / WD_BITS) >> (P % WD_BITS)) & 1u;
    const int sigma = P - 32 * N + (ge ? 1 : 0);
    q.m = wd_shift_right(V, sigma, lane);
    q.e = a.e - be - (ge ? 0 : 1);
    q.s = a.s * bs;
    const u32 g = wd_below(V, sigma);
    if (g == 0x7fffffu || g == 0x800000u) return false;
    if (g >> 23) q.m = wd_increment<N>(q.m, q.e, lane);
    return q.e <= EMAX && q.e >= -(i64)EMAX;
}

// floor(x / 26) for |x| < 2^31
__device__ __forceinline__ int wd_floor_div(int x)
{
    const int q = x / WD_BITS;
    return q - (x - WD_BITS * q < 0 ? 1 : 0);
}

// Grid digits (lane j: digit j) and origin of a wave number.
template <int N> __device__ __forceinline__ u32 wd_to_grid(const WaveNum& x, int& origin)
{
    const int low = (int)x.e - (32 * N - 1);
    origin = wd_floor_div(low);
    const int b = low - WD_BITS * origin;
    return ((x.m << b) | (wave_from_previous_lane(x.m) >> (WD_BITS - b))) & WD_MASK;
}

// Word `lane` of the mantissa (lanes below N).
template <int N> __device__ __forceinline__ u32 wd_word(u32 m, u32 lane)
{
    const u32 bit = 32u * (lane < (u32)N ? lane : 0u), k = bit / WD_BITS, s = bit - WD_BITS * k;
    const u32 a = (u32)__shfl((int)m, (int)k), b = (u32)__shfl((int)m, (int)k + 1), c = (u32)__shfl((int)m, (int)k + 2);
    const u64 v = (u64)a | ((u64)b << WD_BITS) | ((u64)c << (2 * WD_BITS));
    return (u32)(v >> s);
}

// Plane `lane` of a wave number's record (lanes below N + 3), and the record stored at plane element `at`.
template <int N> __device__ __forceinline__ u32 wd_record_word(const WaveNum& x, u32 lane)
{
    const u32 v = wd_word<N>(x.m, lane);
    return lane == (u32)N ? (u32)(int)x.e : lane == (u32)N + 1 ? (u32)x.s : lane == (u32)N + 2 ? 0u : v;
}
template <int N> __device__ __forceinline__ void wd_store(u32* planes, u64 pitch, u64 at, const WaveNum& x, u32 lane)
{
    const u32 v = wd_record_word<N>(x, lane);
    if (lane < (u32)N + 3) planes[(u64)lane * pitch + at] = v;
}

// Per-lane grid digits of a number (a digit array in one lane), with its origin.
template <int N> __device__ __forceinline__ void lane_to_grid(const Num<N>& x, int (&d)[wd_grid<N>()], int& origin)
{
    const int low = x.e - (32 * N - 1);
    origin = wd_floor_div(low);
    const u32 b = (u32)(low - WD_BITS * origin), r = (32u - b) & 31u;
    u32 w[N + 1];
#pragma unroll
    for (int i = 0; i <= N; ++i) {
        const u32 hi = i < N ? x.w[i] : 0u, lo = i ? x.w[i - 1] : 0u;
        w[i] = b ? __builtin_amdgcn_alignbit(hi, lo, r) : hi;
    }
#pragma unroll
    for (int j = 0; j < wd_grid<N>(); ++j) {
        const int bit = WD_BITS * j, wi = bit / 32, s = bit % 32;
        u32 v = wi <= N ? w[wi] >> s : 0u;
        if (s > 32 - WD_BITS && wi + 1 <= N) v |= w[wi + 1] << (32 - s);
        d[j] = (int)(v & WD_MASK);
    }
}

// floor((2^(64N) - 1) / B), followed below by the next words of (2^(64N) - 1/2^(32 K)) / B (K = M - N - 1 of them):
// Knuth's division of an all-ones dividend (limb_core.hpp reciprocal) run K steps further.
template <int N, int M> __device__ __forceinline__ void reciprocal_words(const u32 (&b)[N], u32 (&v)[M])
{
    u32 R[N + 1];
#pragma unroll
    for (int i = 0; i < N; ++i) R[i] = ~b[i];
    R[N] = 0;
    v[M - 1] = 1;
    const u32 inv = (u32)(~(u64)0 / b[N - 1] - ((u64)1 << 32));
#pragma unroll
    for (int j = M - 2; j >= 0; --j) v[j] = knuth_step<N>(R, b, 0xffffffffu, inv);
}

// The reciprocal of the pivot or diagonal entry i: its leading N+1 words (limb_core.hpp reciprocal) are the last
// planes stored.
template <int N> __device__ __forceinline__ void load_recip(const u32* r, u64 rpitch, u64 i, u32 (&v)[N + 1])
{
#pragma unroll
    for (int k = 0; k <= N; ++k) v[k] = r[(u64)(k + recip_words<N>() - (N + 1)) * rpitch + i];
}
// A wave number from a record in LDS (its status apart).
template <int N> __device__ __forceinline__ WaveNum wd_from_record(const u32* rec, u32 lane)
{
    const u32 wi = WD_BITS * lane / 32u, s = WD_BITS * lane % 32u;
    const u32 lo = wi < (u32)N ? rec[wi] : 0u, hi = wi + 1 < (u32)N ? rec[wi + 1] : 0u;
    return {(u32)((((u64)hi << 32) | lo) >> s) & WD_MASK, (i64)__builtin_amdgcn_readfirstlane((int)rec[N]),
            __builtin_amdgcn_readfirstlane((int)rec[N + 1])};
}

// ------------------------------------------------------------------ triangular blocks
// LDS of a block: the signed grid digits of the strict lower triangle packed by columns with their origins (zero
// entries: WD_ZERO), the reciprocals of the diagonal between zeros, so that lane c reads digit c - i without a
// bound, and for each wavefront, which runs one right-hand side, its rows' accumulators (an odd number of 64-bit
// columns a row, so that lanes adding at the same column of their rows hit distinct banks).
constexpr u32 WD_ROWS = 32;
constexpr int WD_TRI = WD_ROWS * (WD_ROWS - 1) / 2;
constexpr int WD_ZERO = 0x7fffffff;
constexpr u32 TRI_WAVES = 4;
template <int N> struct alignas(16) TriLds {
    i64 acc[TRI_WAVES][WD_ROWS][WD_COLS + 1];
    int digit[wd_grid<N>()][WD_TRI];
    int origin[WD_TRI];
    u32 recip[WD_ROWS][wd_mant<N>() - 1 + WD_COLS];
    u32 odd; // rows with a status in the block
};

// first index of column k of the strict lower triangle: rows k + 1 .. WD_ROWS - 1
__device__ __forceinline__ u32 wd_col_start(u32 k) { return k * (2 * WD_ROWS - 1 - k) / 2; }

// Workgroup scope: the diagonal block's and the updates' accumulators take the terms of several wavefronts between
// two barriers (the triangular blocks' belong to one; the instruction is the same).
__device__ __forceinline__ void lds_add(i64* p, i64 v)
{
    __hip_atomic_fetch_add((u64*)p, (u64)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Adds x * l to columns from `at` on, for one lane: H digits of x and GD digits of l.
template <int GD, int H> __device__ __forceinline__ void wd_accumulate(i64* at, const int (&x)[H], const int (&l)[GD])
{
#pragma unroll
    for (int c = 0; c < GD + H - 1; ++c) {
        i64 s = 0;
#pragma unroll
        for (int j = 0; j < H; ++j)
            if (c - j >= 0 && c - j < GD) s += (i64)x[j] * l[c - j];
        lds_add(at + c, s);
    }
}

// Row i's exact dot and its one-lane division, for rows that the wave-parallel forms do not decide: the dot's record
// goes to `rec`, the division replaces it by the quotient's and stores x_i.  `rec` is also the dot's LDS, of rows
// 0 .. i + 1.  Both read the kernel's arguments again, through a pointer that the compiler cannot follow, so that neither
// they nor what is formed from them takes scalar registers of the recurrence's loop (52.8 and 51.9 us a block at 256 bits
// without and with it).
__device__ __forceinline__ TriArgs tri_args_again()
{
    typedef const __attribute__((address_space(4))) TriArgs* args_ptr; // the kernel's one argument
    args_ptr p = (args_ptr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const TriArgs*)p;
}
template <int N> __device__ __forceinline__ void tri_exact_dot(u32 c, u32 i, u32 lane, u32* rec)
{
    const TriArgs g = tri_args_again();
    const i64 xb = g.xbase + (i64)c * g.xc;
    wave_sync();
    const Num<N> d = wave_dot_sub<N>(load_out<N>(g.x, g.xpitch, (u64)(xb + (i64)i * g.xr)), VecView{g.f, g.fpitch, g.fbase + (i64)i * g.fr, g.fk},
                                     VecView{g.x, g.xpitch, xb, g.xr}, i, lane,
                                     DotRows<N>{reinterpret_cast<u32(*)[dot_row_stride<N>()]>(rec), (int)i},
                                     DotScratch{g.scratch + (u64)c * 2 * g.swords, g.swords, g.error});
    if (lane == 0) store_out<N>(rec, 1, 0, 0, 0, false, d);
    wave_sync();
}
template <int N> __device__ __forceinline__ void tri_exact_divide(u32 c, u32 i, u32 lane, u32* rec)
{
    const TriArgs g = tri_args_again();
    if (lane == 0) {
        u32 rv[N + 1];
        load_recip<N>(g.recip, g.rpitch, (u64)(g.rbase + (i64)i * g.rstep), rv);
        const Num<N> l = load_out<N>(g.f, g.fpitch, (u64)(g.fbase + (i64)i * (g.fr + g.fk)));
        const Num<N> q = div_by_reciprocal<N>(load_out<N>(rec, 1, 0), l, rv);
        store_out<N>(g.x, g.xpitch, 0, 0, (u32)(g.xbase + (i64)c * g.xc + (i64)i * g.xr), false, q);
        store_out<N>(rec, 1, 0, 0, 0, false, q);
    }
    wave_sync();
}

// The recurrence x_r = (b_r - sum_{k<r} l_rk x_k) / l_rr over the rows of a block of up to 32 rows, one
// rounding of the exact sum and one of the quotient per row, for right-hand side c on one wavefront of the
// workgroup.  A row whose terms spread past its columns takes the exact dot of them instead (in the LDS of the
// accumulators up to its own, which no later row needs), a quotient too close to a rounding boundary the one-lane
// division, and the recurrence goes on from their result: where most rows of a block need the exact dot, the division
// and the sums that stay in their columns still pay for the digits (terms spread over 700 bits, 256-bit values: 164 us a
// block, 640 bits: 330 us; with the exact dot and the one-lane division for every row 169 and 400 us, and 259 and 680 us
// where the digits gave up the rest of a block at its first such row).  After the first row that ends in a status every row
// is a zero with the statuses of its terms, which are all that it reads.
// The block is staged by the whole workgroup: its loads' latency, 16 rounds of them for one wavefront, was about
// a quarter of the kernel.
template <int N> __device__ __forceinline__ void tri_block(const TriArgs& g, u32 c, u32 B, u32 wave, u32 lane, TriLds<N>& L)
{
    constexpr int D = wd_mant<N>(), GD = wd_grid<N>(), RD = wd_recip<N>(), H = (GD + 1) / 2;
    const u32 t = 64u * wave + lane, row = lane & 31u, half = lane >> 5;
    const bool mine = c < g.count;
    const u64 xb = (u64)(g.xbase + (i64)c * g.xc);
    {
        int4* z = reinterpret_cast<int4*>(&L.acc[0][0][0]);
        static_assert(sizeof(L.acc) % 16 == 0, "whole 16-byte chunks");
        for (u32 k = t; k < sizeof(L.acc) / 16; k += 64u * TRI_WAVES) z[k] = make_int4(0, 0, 0, 0);
        u32* r = &L.recip[0][0];
        for (u32 k = t; k < sizeof(L.recip) / 4; k += 64u * TRI_WAVES) r[k] = 0u;
        if (t == 0) L.odd = 0;
    }
    __syncthreads();
    for (u32 k = t >> 5; k < B; k += 2u * TRI_WAVES)
        if (row > k && row < B) {
            const Num<N> l = load_out<N>(g.f, g.fpitch, (u64)(g.fbase + (i64)row * g.fr + (i64)k * g.fk));
            if (l.st) atomicOr(&L.odd, 1u << row);
            int d[GD], o;
            lane_to_grid<N>(l, d, o);
            const u32 at = wd_col_start(k) + (row - k - 1);
#pragma unroll
            for (int j = 0; j < GD; ++j) L.digit[j][at] = l.s < 0 ? -d[j] : d[j];
            L.origin[at] = l.s ? o : WD_ZERO;
        }
    int le = 0, ls = 0, alpha = 0;
    bool placed = false; // alpha is set: the row has an addend or a term
    bool odd = false;
    if (lane < B) {
        const u64 at = (u64)(g.fbase + (i64)lane * (g.fr + g.fk));
        le = (int)g.f[(u64)N * g.fpitch + at];
        ls = (int)g.f[(u64)(N + 1) * g.fpitch + at];
        odd = g.f[(u64)(N + 2) * g.fpitch + at] != 0 || ls == 0;
        if (wave == TRI_WAVES - 1) {
            u32 v[N + 3];
#pragma unroll
            for (int k = 0; k < N + 3; ++k) v[k] = g.recip[(u64)k * g.rpitch + (u64)(g.rbase + (i64)lane * g.rstep)];
#pragma unroll
            for (int j = 0; j < RD; ++j) {
                const int bit = WD_BITS * j, wi = bit / 32, s = bit % 32;
                u32 e = wi < N + 3 ? v[wi] >> s : 0u;
                if (s > 32 - WD_BITS && wi + 1 < N + 3) e |= v[wi + 1] << (32 - s);
                L.recip[lane][D - 1 + j] = e & WD_MASK;
            }
        }
        if (mine) {
            const Num<N> b = load_out<N>(g.x, g.xpitch, xb + (u64)((i64)lane * g.xr));
            odd = odd || b.st != 0;
            if (b.s) {
                int d[GD], o;
                lane_to_grid<N>(b, d, o);
                alpha = o + GD - 1 - wd_center<N>();
                placed = true;
#pragma unroll
                for (int j = 0; j < GD; ++j) L.acc[wave][lane][wd_center<N>() - (GD - 1) + j] = b.s < 0 ? -(i64)d[j] : (i64)d[j];
            }
        }
    }
    __syncthreads();
    if (!mine) return;
    // the first row with a status or a zero divisor: it and all rows after it end in a status
    const u32 odds = L.odd | (u32)__ballot(odd), first = odds ? (u32)__builtin_ctz(odds) : WD_ROWS;
    // both lanes of a row carry its origin
    alpha = __shfl(alpha, (int)row);
    placed = __shfl((int)placed, (int)row) != 0;
    i64(&acc)[WD_ROWS][WD_COLS + 1] = L.acc[wave];
    static_assert(2 * dot_row_stride<N>() * 4 <= (WD_COLS + 1) * 8, "the rows of an exact dot of i terms fit the accumulators of rows 0 .. i");
    u32* rec = reinterpret_cast<u32*>(&acc[0][0]);
    u32 outside = 0; // rows with a term outside their columns
    WaveNum v, x{0, 0, 0};
    for (u32 i = 0;; ++i) {
        // rows as far as the digits decide them; what they do not decide stays out of this loop, whose registers it would
        // spill (57 instead of 52 us a block)
        bool summed = false;
        for (; i < B; ++i) {
            if (x.s) { // the terms of row k = i - 1
                const u32 k = i - 1;
                int xo;
                const int gx = (int)wd_to_grid<N>(x, xo);
                const int sx = x.s > 0 ? -gx : gx; // the term is subtracted
                int xd[H];
#pragma unroll
                for (int j = 0; j < H; ++j) xd[j] = __shfl(sx, j + H * (int)half);
                const bool live = row > k && row < B;
                const u32 at = wd_col_start(k) + (live ? row - k - 1 : 0u);
                const int lo = live ? L.origin[at] : WD_ZERO;
                bool bad = false;
                if (lo != WD_ZERO) {
                    if (!placed) {
                        alpha = lo + xo + 2 * GD - 1 - wd_center<N>();
                        placed = true;
                    }
                    const int o = lo + xo - alpha;
                    bad = o < 0 || o + 2 * GD - 1 > WD_TOP;
                    if (!bad) {
                        int ld[GD];
#pragma unroll
                        for (int j = 0; j < GD; ++j) ld[j] = L.digit[j][at];
                        wd_accumulate<GD, H>(&acc[row][o + H * (int)half], xd, ld);
                    }
                }
                const u64 bads = __ballot(bad); // either lane of a row
                outside |= (u32)bads | (u32)(bads >> 32);
                wave_sync();
            }
            summed = false;
            if (i >= first || ((outside >> i) & 1u)) break;
            u32 Rs[D];
#pragma unroll
            for (int k = 0; k < D; ++k) Rs[k] = L.recip[i][D - 1 + (int)lane - k];
            const i64 S = acc[i][lane];
            if (!wd_round<N>(S, (i64)(int)wd_read((u32)alpha, (int)i), lane, v)) break;
            summed = true;
            if (!wd_divide<N>(v, Rs, (i64)(int)wd_read((u32)le, (int)i), (int)wd_read((u32)ls, (int)i), lane, x)) break;
            wd_store<N>(g.x, g.xpitch, xb + (u64)((i64)i * g.xr), x, lane);
        }
        if (i >= B) return;
        // row i by the exact dot, the one-lane division, or both
        bool divided = false;
        if (!summed) {
            tri_exact_dot<N>(c, i, lane, rec);
            v = wd_from_record<N>(rec, lane);
            if (i < first && !__builtin_amdgcn_readfirstlane((int)rec[N + 2])) {
                u32 Rs[D];
#pragma unroll
                for (int k = 0; k < D; ++k) Rs[k] = L.recip[i][D - 1 + (int)lane - k];
                divided = wd_divide<N>(v, Rs, (i64)(int)wd_read((u32)le, (int)i), (int)wd_read((u32)ls, (int)i), lane, x);
            }
        } else {
            wave_sync();
            const u32 w = wd_record_word<N>(v, lane);
            if (lane < (u32)N + 3) rec[lane] = w;
            wave_sync();
        }
        if (divided) {
            wd_store<N>(g.x, g.xpitch, xb + (u64)((i64)i * g.xr), x, lane);
            continue;
        }
        tri_exact_divide<N>(c, i, lane, rec);
        x = wd_from_record<N>(rec, lane);
        if (!__builtin_amdgcn_readfirstlane((int)rec[N + 2])) continue;
        // the rows after one that ended in a status
        for (++i; i < B; ++i) {
            const u64 fat = (u64)(g.fbase + (i64)i * g.fr + (i64)lane * g.fk), xat = xb + (u64)((i64)lane * g.xr);
            wave_sync();
            u32 st = 0;
            if (lane <= i) st = g.f[(u64)(N + 2) * g.fpitch + fat] | g.x[(u64)(N + 2) * g.xpitch + xat];
            st = (u32)wave_or((int)st);
            if (lane < (u32)N + 3) g.x[(u64)lane * g.xpitch + xb + (u64)((i64)i * g.xr)] = lane == (u32)N + 2 ? st : 0u;
        }
        return;
    }
}

} // namespace lf
