// div_core.hpp — division by a signed-digit recurrence whose partial remainder is kept in 64-bit columns.
//
// With 26-bit digits (D of them), the remainder's columns R_j take the products -q b_j of every step with one
// v_mad_i64_i32 each and no carries (41 steps of products below 2^54.4 stay below 2^60).  A step shifts the
// columns up by one, which is a choice of registers, estimates the quotient digit from the top three columns
// and a 30-bit reciprocal of the divisor's top bits (within 5 units, which the signed digits absorb), and adds
// the products.  Columns too low to reach the digits still to come are left out, half of them over all steps, so
// that the quotient comes out with 30 bits or more below its last place, right to a few units there: enough for the
// rounding unless it lies within 8 units of 2^-28 of halfway (about one quotient in 2^24), which the caller
// gives to Knuth's division (limb_core.hpp div).  Knuth's steps take a multiply-add, a subtract pair and a digit
// correction for every word (11,700 static instructions at 1024 bits, about 2,300 here).
#pragma once
#include "limb_core.hpp"

namespace lf {

constexpr int CD_BITS = 26;
constexpr u32 CD_MASK = (1u << CD_BITS) - 1;
template <int N> constexpr int cd_digits() { return (32 * N + CD_BITS - 1) / CD_BITS; }
template <int N> constexpr int cd_fraction() { return (32 * N + 30 + CD_BITS - 1) / CD_BITS; }

// Digits of a normalized mantissa shifted up so that its top bit is the top digit's.
template <int N> __device__ __forceinline__ void cd_align(const u32 (&w)[N], int (&d)[cd_digits<N>()])
{
    constexpr int D = cd_digits<N>(), S = CD_BITS * D - 32 * N;
#pragma unroll
    for (int j = 0; j < D; ++j) {
        const int bit = CD_BITS * j - S; // of digit j in w; negative in digit 0 alone
        if (bit < 0) d[j] = (int)((w[0] << -bit) & CD_MASK);
        else {
            const int wi = bit / 32, s = bit % 32;
            u32 v = w[wi] >> s;
            if (s > 32 - CD_BITS && wi + 1 < N) v |= w[wi + 1] << (32 - s);
            d[j] = (int)(v & CD_MASK);
        }
    }
}

// A divisor: its digits and floor(2^60 / its top 31 bits), to a few units.
template <int N> struct Divisor {
    int d[cd_digits<N>()];
    int inv;
};
template <int N> __device__ __forceinline__ Divisor<N> cd_divisor(const u32 (&w)[N])
{
    Divisor<N> v;
    cd_align<N>(w, v.d);
    const u32 top = (w[N - 1] >> 1) | 0x40000000u; // (a zero divisor's quotient is discarded)
    const u32 r = (u32)((1.0f / (float)top) * 0x1.fffff8p59f); // below 2^60 / top by up to 2^-21
    const u64 e = ((u64)1 << 60) - (u64)r * top;
    v.inv = (int)(r + (u32)(((u64)r * (u32)(e >> 30)) >> 30));
    return v;
}

__device__ __forceinline__ int cd_mul_hi(int a, int b) { return (int)(((i64)a * b) >> 32); }

// z = RN(a / b) (the contract of div), v = cd_divisor of b's mantissa; false when z is not decided.
template <int N> __device__ __forceinline__ bool cd_div(const Num<N>& a, const Num<N>& b, const Divisor<N>& v, Num<N>& z)
{
    constexpr int D = cd_digits<N>(), F = cd_fraction<N>();
    static_assert(D >= 3 && F <= 42, "columns of the top estimate, and the bound on their growth");
    u32 st = a.st | b.st;
    if (!st && !b.s) st = ST_DIV0;
    const bool kill = st || !a.s;
    i64 R[D];
    int q[F + 1]; // q[k]: digit of weight 2^(26 (k - F))
    {
        int ad[D];
        cd_align<N>(a.w, ad);
        q[F] = ad[D - 1] >= v.d[D - 1] ? 1 : 0;
#pragma unroll
        for (int j = 0; j < D; ++j) R[j] = (i64)ad[j] - (q[F] ? v.d[j] : 0);
    }
#pragma unroll
    for (int s = 1; s <= F; ++s) {
        const int J = D - (F - s) - 3 > 0 ? D - (F - s) - 3 : 0; // lowest column that the digits to come can see
        const i64 top = (i64)((u64)R[D - 1] << CD_BITS);
#pragma unroll
        for (int j = D - 1; j > 0; --j) R[j] = R[j - 1];
        R[0] = 0;
        R[D - 1] += top;
        const i64 T = R[D - 1] + (R[D - 2] >> CD_BITS);
        const int e = (int)((u32)cd_mul_hi((int)(T >> 24), v.inv) << 1);
        q[F - s] = e;
#pragma unroll
        for (int j = 0; j < D; ++j)
            if (j >= J) R[j] += (i64)(-e) * v.d[j];
    }
    // non-negative digits of the quotient, 2^(26 F) times: the integer digit 0 or 1
    u32 g[F + 1];
    int c = 0;
#pragma unroll
    for (int k = 0; k <= F; ++k) {
        const int t = q[k] + c;
        g[k] = (u32)t & CD_MASK;
        c = t >> CD_BITS;
    }
    const bool ge = g[F] != 0;
    constexpr int P = CD_BITS * F - 32 * N; // bit of the last place of a quotient below 1
    auto bits = [&](int p) -> u32 {         // bits p .. p + 31
        const int k = p / CD_BITS, s = p % CD_BITS;
        u32 t = g[k] >> s;
        if (k + 1 <= F) t |= g[k + 1] << (CD_BITS - s);
        if (k + 2 <= F && 2 * CD_BITS - s < 32) t |= g[k + 2] << (2 * CD_BITS - s);
        return t;
    };
    u32 w[N + 1];
#pragma unroll
    for (int i = 0; i <= N; ++i) w[i] = 32 * i + P <= CD_BITS * F + CD_BITS - 1 ? bits(32 * i + P) : 0u;
    const u32 E = bits(P - 29) & 0x3fffffffu, half = ge ? 1u << 29 : 1u << 28, tail = ge ? E : E & 0x1fffffffu;
#pragma unroll
    for (int i = 0; i < N; ++i) z.w[i] = ge ? __builtin_amdgcn_alignbit(w[i + 1], w[i], 1u) : w[i];
    const u32 carry = increment_mantissa<N>(z.w, tail >= half);
    z.w[N - 1] |= carry << 31;
    finish_rounded<N>(z, (i64)a.e - b.e - (ge ? 0 : 1) + carry, a.s * b.s, st, kill);
    return kill || tail + 8u - half > 16u;
}

} // namespace lf
