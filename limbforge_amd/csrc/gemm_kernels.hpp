// gemm_kernels.hpp — kernels of the exact dense products C = RN(op(A) B) and RN(C - op(A) B).
//
// Residue path (the reference's algorithm, src/linalg.metal:24-152, rebuilt for CDNA4):
//   digits_kernel   each entry's exact band integer X = m * 2^(e-lo) reduced modulo every prime (its bytes times
//                   2^(8h) mod m on v_mfma_i32_32x32x32_i8), balanced residue v in [-m/2, m/2], split into
//                   int8 digits v = 256 d1 + d0 (linalg.metal:24-39)
//   product_kernel  per modulus and 128x128 tile: G11 = D1 D1', G00 = D0 D0', Gmid = D1 D0' + D0 D1' on
//                   v_mfma_i32_32x32x32_i8 with int32 accumulation from LDS-staged tiles, then
//                   y = (65536 G11 + 256 Gmid + G00) (M/m)^-1 mod m written as uint16 (linalg.metal:66-96
//                   writes the residue itself; the CRT factor rides on the digit weights here)
//   crt_round_kernel  one band per line: one lane per output, CRT and rounding
//   crt_pairs_kernel, rebuild_kernel  several bands, and updates; one lane per output: for each band pair, the exact integer by direct
//                   CRT X' = sum_q y_q (M/m_q) 2^t (independent 64-bit column sums, no carry chains),
//                   reduced mod M' and mapped to the symmetric range,
//                   then one rounding, or exact accumulation over the band pairs then one rounding
//                   (the reference's Garner `reconstruct` + `finish`, linalg.metal:109-152; the same integer)
// Exact dot kernels (plain limb GEMM and the lines the residue path does not take, linalg.hpp:268-318):
//   dot_window_kernel   every exact 2N-word product added into one two's-complement window
//   dot_cluster_kernel  exponent clusters with a sticky sign for outputs whose terms spread further
#pragma once
#include "gemm_common.hpp"
#include "gemm_launch.hpp"
#include "limb_core.hpp"
#include "residue_reduce.hpp"

namespace lf {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

// Residue digits of both operands.  An entry's exact integer X = mantissa << (exponent - band lo) is a string
// of bytes x_h, and X mod m = sum_h x_h (2^(8h) mod m): a matrix product of entries by moduli with at most 256
// terms.  It runs on v_mfma_i32_32x32x32_i8: the bytes less 128 as int8 (the 128s come back as one constant a
// modulus), the powers as two int8 digits, so that two int32 sums give T = 256 s1 + s0 + offset, |T| < 2^30, and
// one FP32 quotient estimate reduces T to the balanced residue.  A workgroup takes 256 entries (tk consecutive
// k of 256 / tk lines; where lines are adjacent in memory consecutive threads take consecutive lines, so that
// loads coalesce), places their shifted bytes in LDS, and for 32 moduli at a time leaves the digit bytes in
// LDS and writes every band row of its lines as 16-byte chunks, zero where the entry is not a member of that
// band (or is zero, carries a status, or lies past K).  Rows past the last line are left as they are: no
// kernel reads the residues they give.
// What bounds it is the reduction of each residue (about 17 instructions) and the LDS that limits the workgroups in
// flight: each wavefront keeps its entries' bytes in registers over the moduli, so that the digit bytes' stage takes
// the place of the mantissas.  On the operands of a 512-bit 512^3 product joined to one band (123 moduli) two
// launches of 16-bit chunks by powers, reduced twice, took 260 us, this form 107 us with both in LDS and 102 us so.
constexpr u32 DIG_QB = 32;                      // moduli per LDS batch
constexpr u32 DIG_STAGE_ROW = 2 * 256 + 16;     // bytes of a modulus's stage row: both digits of 256 entries
// a shifted mantissa's LDS row: an odd number of 16-byte chunks, so that the 16 lanes of a fragment read hit
// distinct banks
__host__ __device__ constexpr u32 digits_row_bytes(u32 bytes) { return bytes + 16; }
__host__ __device__ constexpr u32 digits_area(u32 bytes) // the mantissas, then the stage
{
    return 256 * digits_row_bytes(bytes) > DIG_QB * DIG_STAGE_ROW ? 256 * digits_row_bytes(bytes) : DIG_QB * DIG_STAGE_ROW;
}
__host__ __device__ constexpr u64 digits_lds_bytes(u32 bytes) { return digits_area(bytes) + 256 + 64; }

__device__ __forceinline__ u32 byte_eq_mask(u32 x, u32 b4)
{
    // 0xff in each byte of x equal to the byte of b4, 0 elsewhere (the exact zero-byte test)
    const u32 t = x ^ b4;
    const u32 z = ~(((t & 0x7f7f7f7fu) + 0x7f7f7f7fu) | t | 0x7f7f7f7fu); // 0x80 where t's byte is zero
    return (z >> 7) * 0xffu;
}

template <int N> __global__ void __launch_bounds__(256, 2) digits_kernel(DigitsArgs g)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const u32 rowb = digits_row_bytes(g.bytes);
    unsigned char* stage = lds;
    unsigned char* bandof = lds + digits_area(g.bytes);
    u32* signs = reinterpret_cast<u32*>(bandof + 256); // bit e % 32 of word e / 32: entry e is negative
    const bool second = blockIdx.x >= g.side[0].blocks;
    const DigitsSide S = second ? g.side[1] : g.side[0];
    const u32 blk = blockIdx.x - (second ? g.side[0].blocks : 0u);
    const u32 tk = S.tk, tl = 256u / tk, kblocks = (g.Kp + tk - 1) / tk;
    const u32 line0 = (blk / kblocks) * tl, k0 = (blk % kblocks) * tk;
    const u32 t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    for (u32 i = t; i < 256u * rowb / 16u; i += 256u) reinterpret_cast<uint4*>(lds)[i] = make_uint4(0x80808080u, 0x80808080u, 0x80808080u, 0x80808080u);
    if (t < 8) signs[t] = 0;
    __syncthreads();
    {
        const u32 tline = S.by_line ? t % tl : t / tk, tkk = S.by_line ? t / tl : t % tk, e = tline * tk + tkk;
        const u32 line = line0 + tline, k = k0 + tkk;
        u32 band = 0xffu;
        if (line < S.nlines && k < g.K && S.lines[line].cls == 0) {
            const GemmLine* L = S.lines + line;
            const u64 idx = (u64)line * S.v.ls + (u64)k * S.v.ks;
            const u32* P = S.v.planes;
            const u64 pitch = S.v.pitch;
            const u32 st = P[(u64)(N + 2) * pitch + idx];
            const int s = (int)P[(u64)(N + 1) * pitch + idx];
            if (!st && s) {
                const int ex = (int)P[(u64)N * pitch + idx];
                u32 shift = 0;
                if (g.joined) {
                    band = 0;
                    shift = (u32)(ex - L->low);
                } else
                    for (int b = 0; b < L->nb; ++b)
                        if (ex >= L->lo[b] && ex <= L->hi[b]) {
                            band = (u32)b;
                            shift = (u32)(ex - L->lo[b]);
                        }
                // the band's width bounds the shift, and the planner sized the row for the widest band
                if (band != 0xffu && shift / 8u + 4u * N + 4u <= rowb) {
                    const u32 ws = shift >> 5, b = shift & 31u;
                    u32* row = reinterpret_cast<u32*>(lds + e * rowb) + ws;
                    u32 lo = 0;
#pragma unroll
                    for (int w = 0; w < N; ++w) {
                        const u32 x = P[(u64)w * pitch + idx];
                        row[w] = (b ? __builtin_amdgcn_alignbit(x, lo, 32u - b) : x) ^ 0x80808080u;
                        lo = x;
                    }
                    if (b) row[N] = (lo >> (32u - b)) ^ 0x80808080u;
                    if (s < 0) atomicOr(&signs[e >> 5], 1u << (e & 31u));
                }
            }
        }
        bandof[e] = (unsigned char)band;
    }
    __syncthreads();
    // waves 0-3: entries 64 wave + 32 h + (lane % 32); bytes 32 step + 16 (lane / 32) of each
    const u32 steps = g.bytes / 32u, r = lane & 31u, kh = lane >> 5;
    const u32 sg[2] = {signs[2u * wave], signs[2u * wave + 1u]};
    constexpr u32 STEPS = digit_bytes_max(N) / 32;
    v4i a[STEPS][2];
#pragma unroll
    for (u32 st = 0; st < STEPS; ++st)
#pragma unroll
        for (int h = 0; h < 2; ++h)
            if (st < steps) a[st][h] = *(const v4i*)(lds + (64u * wave + 32u * h + r) * rowb + 32u * st + 16u * kh);
    __syncthreads(); // the mantissas' LDS becomes the stage
    for (u32 qb = 0; qb < g.L; qb += DIG_QB) {
        const u32 q = qb + r < g.L ? qb + r : g.L - 1; // lanes past the last modulus repeat it
        const int8_t* tab = g.table + (u64)q * 2 * DIGIT_TABLE_BYTES + 16u * kh;
        v16i s1[2] = {}, s0[2] = {};
#pragma unroll
        for (u32 st = 0; st < STEPS; ++st)
            if (st < steps) {
                const v4i b1 = *(const v4i*)(tab + 32u * st), b0 = *(const v4i*)(tab + DIGIT_TABLE_BYTES + 32u * st);
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    s1[h] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[st][h], b1, s1[h], 0, 0, 0);
                    s0[h] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[st][h], b0, s0[h], 0, 0, 0);
                }
            }
        const int m = (int)g.moduli[q], half = m >> 1, off = g.offset[q];
        const float inv = g.inverse[q];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4) {
                // accumulator element 4 i4 + i: entry row 8 i4 + 4 (lane / 32) + i, modulus column lane % 32
                const u32 e = 8u * i4 + 4u * kh;
                u32 v[4], v1[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int T = (int)((u32)s1[h][4 * i4 + i] << 8) + s0[h][4 * i4 + i] + off;
                    // T - q m + half lies in (-m, 2m): one unsigned minimum takes a negative value up by m, one a value
                    // from m on down by m
                    u32 u = (u32)(T + half - residue_mul24((int)__builtin_rintf((float)T * inv), m));
                    u = min(u, u + (u32)m);
                    u = min(u, u - (u32)m);
                    const int neg = -(int)((sg[h] >> (e + i)) & 1u);
                    v[i] = (u32)(((int)u - half) ^ neg) - (u32)neg;
                    v1[i] = v[i] + 128u; // its second byte is the high digit, v's first the low one
                }
                const u32 w0 = __builtin_amdgcn_perm(__builtin_amdgcn_perm(v[3], v[2], 0x0c0c0400u), __builtin_amdgcn_perm(v[1], v[0], 0x0c0c0400u), 0x05040100u);
                const u32 w1 = __builtin_amdgcn_perm(__builtin_amdgcn_perm(v1[3], v1[2], 0x0c0c0501u), __builtin_amdgcn_perm(v1[1], v1[0], 0x0c0c0501u), 0x05040100u);
                unsigned char* at = stage + r * DIG_STAGE_ROW + 64u * wave + 32u * h + e;
                *reinterpret_cast<u32*>(at) = w1;
                *reinterpret_cast<u32*>(at + 256) = w0;
            }
        __syncthreads();
        const u32 nq = g.L - qb < DIG_QB ? g.L - qb : DIG_QB;
        // chunk j: 16 entries (c16) of digit plane pl of modulus qb + qi, written to every band row of their line
        for (u32 j = t; j < nq * 32u; j += 256u) {
            const u32 c16 = j & 15u, pl = (j >> 4) & 1u, qi = j >> 5;
            const u32 line = line0 + 16u * c16 / tk, kk = k0 + 16u * c16 % tk;
            if (line >= S.nlines || kk >= g.Kp || S.lines[line].cls != 0) continue;
            const GemmLine* L = S.lines + line;
            const uint4 dv = *reinterpret_cast<const uint4*>(stage + qi * DIG_STAGE_ROW + 256u * pl + 16u * c16);
            int8_t* plane = (pl ? S.d0 : S.d1) + (u64)(qb + qi) * S.rows_p * g.Kp + kk;
            if (g.joined || L->nb == 1) {
                *reinterpret_cast<uint4*>(plane + (u64)L->member[0] * g.Kp) = dv;
                continue;
            }
            const uint4 bv = *reinterpret_cast<const uint4*>(bandof + 16u * c16);
            for (int b = 0; b < L->nb; ++b) {
                const u32 b4 = (u32)b * 0x01010101u;
                *reinterpret_cast<uint4*>(plane + (u64)L->member[b] * g.Kp) =
                    make_uint4(dv.x & byte_eq_mask(bv.x, b4), dv.y & byte_eq_mask(bv.y, b4), dv.z & byte_eq_mask(bv.z, b4),
                               dv.w & byte_eq_mask(bv.w, b4));
            }
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------- CRT rebuild
// The symmetric representative of X' = sum y_q (M/m_q) 2^t < L M' (Mb: M', then floor(M'/2)): X becomes its magnitude;
// returns its sign (+1/-1).
template <int WX> __device__ __forceinline__ int crt_reduce(const u32* Mb, u32 (&X)[WX])
{
    // X' < L M' with M' normalised to bit 32(WX-1)-1: estimate q = floor(X'/M') from the top words
    const u64 xt = ((u64)X[WX - 1] << 32) | X[WX - 2];
    u64 qe = xt / ((u64)Mb[WX - 2] + 1u);
    // X' -= qe * M'
    u64 bw = 0;
#pragma unroll
    for (int w = 0; w < WX; ++w) {
        const u64 p = qe * Mb[w] + bw;
        const u32 lo = (u32)p, old = X[w];
        X[w] = old - lo;
        bw = (p >> 32) + (old < lo ? 1u : 0u);
    }
    for (int rep = 0; rep < 3; ++rep) {
        int cmp = 0;
#pragma unroll
        for (int w = WX - 1; w >= 0; --w)
            if (cmp == 0 && X[w] != Mb[w]) cmp = X[w] > Mb[w] ? 1 : -1;
        if (cmp < 0) break;
        u32 b2 = 0;
#pragma unroll
        for (int w = 0; w < WX; ++w) {
            const u64 v = (u64)X[w] - Mb[w] - b2;
            X[w] = (u32)v;
            b2 = (u32)(v >> 63);
        }
    }
    // symmetric range: X' > floor(M'/2) means the negative value X' - M'
    const u32* H = Mb + WX;
    int cmp = 0;
#pragma unroll
    for (int w = WX - 1; w >= 0; --w)
        if (cmp == 0 && X[w] != H[w]) cmp = X[w] > H[w] ? 1 : -1;
    if (cmp <= 0) return 1;
    u32 b3 = 0;
#pragma unroll
    for (int w = 0; w < WX; ++w) {
        const u64 v = (u64)Mb[w] - X[w] - b3;
        X[w] = (u32)v;
        b3 = (u32)(v >> 63);
    }
    return -1;
}

// X' = |sum| * 2^t from the L values y_q = r_q (M/m_q)^-1 mod m_q at (row, col) (the product kernel writes
// the residues already multiplied by that factor); returns the sign (+1/-1) of the symmetric value.  The
// CRT words come from LDS (staged by the kernel, rows padded to whole 16-byte groups, read 16 bytes at a
// time) for wide integers, from scalar loads otherwise.  Measured on the 512-bit 512^3 products (with the
// factor still applied here): 67-word rows 300 us scalar against 173 us staged; 39-word rows 500 us scalar
// against 531 us staged.
constexpr int CRT_LDS_MIN_WX = 48;
template <int WX>
__device__ __forceinline__ int crt_rebuild(const RebuildArgs& g, const u32* tab, u32 row, u32 col, u32 (&X)[WX])
{
    // tab (LDS, when WX >= CRT_LDS_MIN_WX): the L rows of WX CRT words
    constexpr bool STAGED = WX >= CRT_LDS_MIN_WX;
    constexpr int WXP = (WX + 3) & ~3;
    u64 colsum[WX];
#pragma unroll
    for (int w = 0; w < WX; ++w) colsum[w] = 0;
    const u64 plane = (u64)g.Mp * g.Np, at = (u64)row * g.Np + col;
    // residues in batches of 8 moduli, the next batch's loads in flight while this one accumulates
    constexpr u32 RB = 8;
    u32 rr[RB], rn[RB];
#pragma unroll
    for (u32 u = 0; u < RB; ++u) rr[u] = u < g.L ? (u32)g.res[(u64)u * plane + at] : 0u;
    for (u32 q0 = 0; q0 < g.L; q0 += RB) {
#pragma unroll
        for (u32 u = 0; u < RB; ++u) rn[u] = q0 + RB + u < g.L ? (u32)g.res[(u64)(q0 + RB + u) * plane + at] : 0u;
#pragma unroll
        for (u32 u = 0; u < RB; ++u) {
            const u32 q = q0 + u;
            if (q >= g.L) break;
            u32 y = rr[u];
            // y < 2^16 is known to the compiler from the 16-bit load; knowing it, the compiler splits the
            // 64-bit column sums over unaligned register pairs and copies every one around its
            // multiply-add (one extra move per v_mad_u64_u32).  The empty asm hides the range.
            asm("" : "+v"(y));
            if constexpr (STAGED) {
                const uint4* C4 = reinterpret_cast<const uint4*>(tab + q * WXP);
#pragma unroll
                for (int w4 = 0; w4 < WXP / 4; ++w4) {
                    const uint4 c = C4[w4];
                    const u32 cw[4] = {c.x, c.y, c.z, c.w};
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (4 * w4 + k < WX) colsum[4 * w4 + k] += (u64)y * cw[k];
                }
            } else {
                const u32* C = g.crt + q * WX;
#pragma unroll
                for (int w = 0; w < WX; ++w) colsum[w] += (u64)y * C[w];
            }
        }
#pragma unroll
        for (u32 u = 0; u < RB; ++u) rr[u] = rn[u];
    }
    u64 carry = 0;
#pragma unroll
    for (int w = 0; w < WX; ++w) {
        const u64 v = colsum[w] + carry;
        X[w] = (u32)v;
        carry = v >> 32;
    }
    return crt_reduce<WX>(g.bound, X);
}

template <int N> __device__ __forceinline__ void store_out(u32* base, u64 pitch, u64 stride, u32 i, u32 j, bool mirror, const Num<N>& r)
{
    const u64 at = (u64)i * stride + j;
#pragma unroll
    for (int k = 0; k < N; ++k) base[k * pitch + at] = r.w[k];
    base[N * pitch + at] = (u32)r.e;
    base[(N + 1) * pitch + at] = (u32)r.s;
    base[(N + 2) * pitch + at] = r.st;
    if (mirror && i != j) {
        const u64 bt = (u64)j * stride + i;
#pragma unroll
        for (int k = 0; k < N; ++k) base[k * pitch + bt] = r.w[k];
        base[N * pitch + bt] = (u32)r.e;
        base[(N + 1) * pitch + bt] = (u32)r.s;
        base[(N + 2) * pitch + bt] = r.st;
    }
}

template <int N> __device__ __forceinline__ Num<N> load_out(const u32* base, u64 pitch, u64 at)
{
    Num<N> r;
#pragma unroll
    for (int k = 0; k < N; ++k) r.w[k] = base[k * pitch + at];
    r.e = (int)base[N * pitch + at];
    r.s = (int)base[(N + 1) * pitch + at];
    r.st = base[(N + 2) * pitch + at];
    return r;
}

// Stage 1 of the rebuild: one lane per (band pair, output) of rows [row0, row0 + rows) reconstructs the
// pair's exact integer by CRT, reduced to the symmetric range, into the stage (WX words and a sign word).
// Only this stage touches the residues; the register budget holds the column sums and nothing else.
// Wide CRT integers stage their words in LDS once per workgroup (dynamic shared memory of
// crt_table_bytes(L, WX)).
constexpr u64 crt_table_bytes(u32 L, int WX) { return WX >= CRT_LDS_MIN_WX ? (u64)L * ((WX + 3) & ~3) * 4 : 0; }
template <int WX> __global__ void __launch_bounds__(256) crt_pairs_kernel(RebuildArgs g)
{
    constexpr int WXP = (WX + 3) & ~3;
    extern __shared__ __attribute__((aligned(16))) u32 tab[];
    if constexpr (WX >= CRT_LDS_MIN_WX) {
        for (u32 k = threadIdx.x; k < g.L * WXP; k += 256u) {
            const u32 q = k / WXP, w = k % WXP;
            tab[k] = w < (u32)WX ? g.crt[q * WX + w] : 0u;
        }
        __syncthreads();
    }
    const u64 span = (u64)g.rows * g.n;
    const u64 idx = (u64)blockIdx.x * 256u + threadIdx.x;
    if (idx >= span) return;
    const u32 i = g.row0 + (u32)(idx / g.n), j = (u32)(idx % g.n);
    if (g.syrk && j > i) return;
    const GemmLine* Li = g.left + i;
    const GemmLine* Lj = g.right + j;
    if (Li->cls != 0 || Lj->cls != 0) return;
    const u32 p = blockIdx.y, b = p / g.pj, c = p % g.pj;
    if ((int)b >= Li->nb || (int)c >= Lj->nb) return;
    u32 rr = (u32)Li->member[b], rc = (u32)Lj->member[c];
    if (g.syrk && rc > rr) { // the extended SYRK product is symmetric: read its lower triangle
        const u32 t0 = rr;
        rr = rc;
        rc = t0;
    }
    u32 X[WX];
    const int sg = crt_rebuild<WX>(g, tab, rr, rc, X);
    u32* dst = g.stage + (u64)p * span + idx;
    const u64 wstride = (u64)g.pairs * span;
#pragma unroll
    for (int w = 0; w < WX; ++w) dst[w * wstride] = X[w];
    dst[WX * wstride] = (u32)sg;
}

template <int WX> __device__ __forceinline__ int read_stage(const RebuildArgs& g, u32 b, u32 c, u32 i, u32 j, u32 (&X)[WX])
{
    const u64 span = (u64)g.rows * g.n;
    const u32* src = g.stage + (u64)(b * g.pj + c) * span + (u64)(i - g.row0) * g.n + j;
    const u64 wstride = (u64)g.pairs * span;
#pragma unroll
    for (int w = 0; w < WX; ++w) X[w] = src[w * wstride];
    return (int)src[WX * wstride];
}

// The value of lane `SRC` of this lane's quad, and of the lane one or two places away in it.
template <int CTRL> __device__ __forceinline__ u32 quad_read(u32 v) { return (u32)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, 0xF, 0xF, false); }

// One pass from the residues to the rounded output where every line is one band: nothing is staged between the
// CRT and the rounding.  Four consecutive outputs form a quad of lanes, and each lane forms one quarter
// of the CRT words of all four, then the quad exchanges quarters: a lane's multiply-adds are as many as for one
// output of its own, and it reads a quarter of the table from LDS.  What bounds it is those multiply-adds; with the
// whole table read by every lane (17 16-byte reads a modulus at 67 words against 5) it was LDS bound: 158 us on
// the 512-bit 512^3 product joined to one band, 145 us so; 34 and 27 us on the 256-bit SYRK of 2048 x 512.
constexpr u32 ROUND_BLOCK = 256;
constexpr int quarter_words(int wx) { return (wx + 3) / 4; }
constexpr int quarter_pitch(int wx) { return (quarter_words(wx) + 3) & ~3; }
constexpr u64 round_table_bytes(u32 L, int wx) { return (u64)L * 4 * quarter_pitch(wx) * 4; }
template <int N, int WX> __global__ void __launch_bounds__(ROUND_BLOCK) crt_round_kernel(RoundArgs g)
{
    constexpr int QW = quarter_words(WX), QP = quarter_pitch(WX);
    extern __shared__ __attribute__((aligned(16))) u32 tab[];
    // outputs in row order, whatever the rows' length: a workgroup takes consecutive ones (of one wavefront instead of
    // four it was no faster from 4,096 outputs to 200,000: 87.6 and 86.4 us the 256-bit 96 x 75 x 130 product)
    constexpr u32 block = ROUND_BLOCK;
    const u32 total = g.m * g.n, first = blockIdx.x * block, idx = first + threadIdx.x, quarter = threadIdx.x & 3u;
    if (g.syrk) { // nothing to do where the whole workgroup lies above the diagonal, in one row
        const u32 i0 = first / g.n, i1 = min(first + block, total) - 1u;
        if (first - i0 * g.n > i0 && i1 / g.n == i0) return;
    }
    for (u32 k = threadIdx.x; k < g.L * 4 * QP; k += block) {
        const u32 q = k / (4 * QP), p = (k / QP) % 4u, w = p * QW + k % QP;
        tab[k] = k % QP < (u32)QW && w < (u32)WX ? g.crt[q * WX + w] : 0u;
    }
    __syncthreads();
    const u32 i = idx < total ? idx / g.n : 0u, j = idx < total ? idx - i * g.n : 0u;
    const bool inside = idx < total && !(g.syrk && j > i);
    if (!__ballot(inside)) return;
    const GemmLine* Li = g.left + i;
    const GemmLine* Lj = g.right + j;
    const bool live = inside && Li->cls == 0 && Lj->cls == 0;
    u64 sum[4][QW];
#pragma unroll
    for (int o = 0; o < 4; ++o)
#pragma unroll
        for (int w = 0; w < QW; ++w) sum[o][w] = 0;
    // a SYRK's members are in line order, so the row's is the larger: the product's lower triangle
    const u64 plane = (u64)g.Mp * g.Np, at = live ? (u64)(u32)Li->member[0] * g.Np + (u32)Lj->member[0] : 0;
    // residues in batches of 8 moduli, the next batch's loads in flight while this one accumulates
    constexpr u32 RB = 8;
    u32 rr[RB], rn[RB];
#pragma unroll
    for (u32 u = 0; u < RB; ++u) rr[u] = live && u < g.L ? (u32)g.res[(u64)u * plane + at] : 0u;
    for (u32 q0 = 0; q0 < g.L; q0 += RB) {
#pragma unroll
        for (u32 u = 0; u < RB; ++u) rn[u] = live && q0 + RB + u < g.L ? (u32)g.res[(u64)(q0 + RB + u) * plane + at] : 0u;
#pragma unroll
        for (u32 u = 0; u < RB; ++u) {
            const u32 q = q0 + u;
            if (q >= g.L) break;
            u32 y[4] = {quad_read<0x00>(rr[u]), quad_read<0x55>(rr[u]), quad_read<0xAA>(rr[u]), quad_read<0xFF>(rr[u])};
            const uint4* C4 = reinterpret_cast<const uint4*>(tab + (q * 4 + quarter) * QP);
#pragma unroll
            for (int w4 = 0; w4 < QP / 4; ++w4) {
                const uint4 c = C4[w4];
                const u32 cw[4] = {c.x, c.y, c.z, c.w};
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (4 * w4 + k < QW)
#pragma unroll
                        for (int o = 0; o < 4; ++o) sum[o][4 * w4 + k] += (u64)y[o] * cw[k];
            }
        }
#pragma unroll
        for (u32 u = 0; u < RB; ++u) rr[u] = rn[u];
    }
    // each quarter's words and the carry out of it; then lane k of the quad takes the quarters of output k
    u32 x[4][QW + 1];
#pragma unroll
    for (int o = 0; o < 4; ++o) {
        u64 carry = 0;
#pragma unroll
        for (int w = 0; w < QW; ++w) {
            const u64 v = sum[o][w] + carry;
            x[o][w] = (u32)v;
            carry = v >> 32;
        }
        x[o][QW] = (u32)carry; // below L 2^16
    }
    const bool odd = quarter & 1u, high = quarter & 2u;
#pragma unroll
    for (int w = 0; w <= QW; ++w) {
#pragma unroll
        for (int o = 0; o < 4; o += 2) { // neighbours exchange (o, o + 1)
            const u32 r = quad_read<0xB1>(odd ? x[o][w] : x[o + 1][w]);
            x[o][w] = odd ? r : x[o][w];
            x[o + 1][w] = odd ? x[o + 1][w] : r;
        }
#pragma unroll
        for (int o = 0; o < 2; ++o) { // pairs exchange (o, o + 2)
            const u32 r = quad_read<0x4E>(high ? x[o][w] : x[o + 2][w]);
            x[o][w] = high ? r : x[o][w];
            x[o + 2][w] = high ? x[o + 2][w] : r;
        }
    }
    if (!inside) return;
    const bool mirror = g.syrk && !g.lower_only;
    if (Li->cls == 1 || Lj->cls == 1) { // zero or status line
        store_out<N>(g.out, g.out_pitch, g.out_stride, i, j, mirror, zero<N>(Li->status | Lj->status));
        return;
    }
    if (!live) return; // exact dot kernels
    u32 X[WX];
    u32 from = 0, cy = 0;
#pragma unroll
    for (int w = 0; w < WX; ++w) {
        const int p = w / QW, k = w % QW;
        if (k == 0) from = p ? x[p - 1][QW] : 0u;
        X[w] = add_carry(x[p][k], k == 0 ? from : 0u, cy);
    }
    const int sg = crt_reduce<WX>(g.bound, X);
    const i64 scale = (i64)Li->low + Lj->low - 2 * (32 * N - 1) - g.t;
    store_out<N>(g.out, g.out_pitch, g.out_stride, i, j, mirror, pack<N, WX>(X, scale, sg, ST_OK));
}

// WX: CRT integer words (M' normalised to bit 32(WX-1)-1); ACC: multi-band accumulator words (kept in LDS,
// one row of ACC+1 words per lane; 1 = no multi-band outputs in this instantiation).
constexpr u32 REBUILD_BLOCK = 128;
template <int N, int WX, int ACC> __global__ void __launch_bounds__(REBUILD_BLOCK) rebuild_kernel(RebuildArgs g)
{
    __shared__ u32 rebuild_acc[ACC > 1 ? REBUILD_BLOCK * (ACC + 1) : 1];
    const u32 nblocks = (g.n + REBUILD_BLOCK - 1) / REBUILD_BLOCK;
    const u32 i = g.row0 + blockIdx.x / nblocks;
    const u32 j = (blockIdx.x % nblocks) * REBUILD_BLOCK + threadIdx.x;
    if (i >= g.row0 + g.rows || i >= g.m || j >= g.n) return;
    if (g.syrk && j > i) return; // SYRK computes the lower triangle (mirrored when full)
    const bool mirror = g.syrk && !g.lower_only;
    const GemmLine* Li = g.left + i;
    const GemmLine* Lj = g.right + j;
    const u64 at = (u64)i * g.out_stride + j;
    Num<N> old = zero<N>(ST_OK);
    if (g.subtract) old = load_out<N>(g.out, g.out_pitch, at);
    if (Li->cls == 1 || Lj->cls == 1) {
        // zero or status line: zero with the statuses; a zero line leaves an update unchanged
        u32 st = Li->status | Lj->status | (g.subtract ? old.st : 0u);
        if (!g.subtract || st) store_out<N>(g.out, g.out_pitch, g.out_stride, i, j, mirror, zero<N>(st));
        return;
    }
    if (Li->cls != 0 || Lj->cls != 0) return; // exact dot kernels
    if (g.subtract && old.st) {
        store_out<N>(g.out, g.out_pitch, g.out_stride, i, j, mirror, zero<N>(old.st));
        return;
    }
    const int nbi = Li->nb, nbj = Lj->nb;
    const i64 base = (i64)Li->low + Lj->low - 2 * (32 * N - 1);
    const i64 old_scale = (i64)old.e - (32 * N - 1);
    Num<N> result;
    if (nbi == 1 && nbj == 1) {
        u32 X[WX];
        const int sg = read_stage<WX>(g, 0, 0, i, j, X);
        if (!g.subtract) result = pack<N, WX>(X, base - g.t, sg, ST_OK);
        else result = round_sum2<N, WX, N>(X, base - g.t, -sg, old.w, old_scale, old.s);
    } else if constexpr (ACC <= WX) {
        result = zero<N>(ST_INVALID); // not reached: the planner sends multi-band lines of this class elsewhere
    } else {
        // exact sum over the band pairs in this lane's LDS accumulator (two's complement, ACC words): each
        // pair's integer is added at its word offset with a runtime address, so no register barrel shifter
        const int tb = (g.t + 31) & ~31;
        u32* acc = rebuild_acc + threadIdx.x * (ACC + 1);
        for (int w = 0; w < ACC; ++w) acc[w] = 0;
        for (int b = 0; b < nbi; ++b)
            for (int c = 0; c < nbj; ++c) {
                u32 X[WX];
                const int sg = read_stage<WX>(g, (u32)b, (u32)c, i, j, X);
                const i64 shift = (i64)(Li->lo[b] - Li->low) + (Lj->lo[c] - Lj->low) + tb - g.t;
                const int o = (int)(shift >> 5);
                const u32 bs = (u32)(shift & 31);
                if (sg > 0) {
                    u32 cy = 0;
#pragma unroll
                    for (int t = 0; t <= WX; ++t) {
                        const u32 hi = t < WX ? X[t] : 0u, lo = t ? X[t - 1] : 0u;
                        const u32 v = bs ? __builtin_amdgcn_alignbit(hi, lo, 32u - bs) : hi;
                        const u64 z = (u64)acc[o + t] + v + cy;
                        acc[o + t] = (u32)z;
                        cy = (u32)(z >> 32);
                    }
                    for (int w = o + WX + 1; cy && w < ACC; ++w) {
                        const u64 z = (u64)acc[w] + cy;
                        acc[w] = (u32)z;
                        cy = (u32)(z >> 32);
                    }
                } else {
                    u32 bw = 0;
#pragma unroll
                    for (int t = 0; t <= WX; ++t) {
                        const u32 hi = t < WX ? X[t] : 0u, lo = t ? X[t - 1] : 0u;
                        const u32 v = bs ? __builtin_amdgcn_alignbit(hi, lo, 32u - bs) : hi;
                        const u64 z = (u64)acc[o + t] - v - bw;
                        acc[o + t] = (u32)z;
                        bw = (u32)(z >> 63);
                    }
                    for (int w = o + WX + 1; bw && w < ACC; ++w) {
                        const u64 z = (u64)acc[w] - bw;
                        acc[w] = (u32)z;
                        bw = (u32)(z >> 63);
                    }
                }
            }
        u32 A[ACC];
#pragma unroll
        for (int w = 0; w < ACC; ++w) A[w] = acc[w];
        int sign = 1;
        if (A[ACC - 1] >> 31) {
            sign = -1;
            u32 cy = 1;
#pragma unroll
            for (int w = 0; w < ACC; ++w) {
                const u64 v = (u64)(u32)~A[w] + cy;
                A[w] = (u32)v;
                cy = (u32)(v >> 32);
            }
        }
        if (!g.subtract) result = pack<N, ACC>(A, base - tb, sign, ST_OK);
        else result = round_sum2<N, ACC, N>(A, base - tb, -sign, old.w, old_scale, old.s);
    }
    store_out<N>(g.out, g.out_pitch, g.out_stride, i, j, mirror, result);
}

// ---------------------------------------------------------------- exact dot products
__device__ __forceinline__ void output_of(const DotArgs& g, u32 idx, u32& i, u32& j)
{
    if (g.list) {
        i = g.list[2 * idx];
        j = g.list[2 * idx + 1];
    } else {
        i = idx / g.n;
        j = idx - i * g.n;
    }
}

template <int N> __device__ __forceinline__ Num<N> load_view(const MatView& v, u32 line, u32 k)
{
    return load_out<N>(v.planes, v.pitch, (u64)line * v.ls + (u64)k * v.ks);
}

// The plain exact limb GEMM: every term a_k b_k is formed exactly (2N words) and added into one W-word
// two's-complement window whose lsb is the smallest possible term exponent of the output; one rounding.
template <int N, int W> __global__ void __launch_bounds__(256) dot_window_kernel(DotArgs g)
{
    const u32 idx = blockIdx.x * 256u + threadIdx.x;
    if (idx >= g.count) return;
    u32 i, j;
    output_of(g, idx, i, j);
    if (g.syrk && j > i) return;
    const GemmLine* Li = g.lrows + i;
    const GemmLine* Lj = g.rcols + j;
    const u64 at = (u64)i * g.out_stride + j;
    const bool mirror = g.mirror != 0;
    Num<N> old = zero<N>(ST_OK);
    if (g.subtract) old = load_out<N>(g.out, g.out_pitch, at);
    if (Li->cls == 1 || Lj->cls == 1) {
        u32 st = Li->status | Lj->status | (g.subtract ? old.st : 0u);
        if (!g.subtract || st) store_out<N>(g.out, g.out_pitch, g.out_stride, i, j, mirror, zero<N>(st));
        return;
    }
    if (g.subtract && old.st) {
        store_out<N>(g.out, g.out_pitch, g.out_stride, i, j, mirror, zero<N>(old.st));
        return;
    }
    const i64 lo = (i64)Li->bottom + Lj->bottom;
    u32 acc[W];
#pragma unroll
    for (int w = 0; w < W; ++w) acc[w] = 0;
    for (u32 k = 0; k < g.K; ++k) {
        const Num<N> a = load_view<N>(g.left, i, k);
        const Num<N> b = load_view<N>(g.right, j, k);
        if (!a.s || !b.s) continue;
        u32 p[2 * N], w[W];
        mantissa_product<N>(a.w, b.w, p);
        place<W, 2 * N>(w, p, (i64)a.e + b.e - lo);
        accumulate_signed<W>(acc, w, a.s * b.s);
    }
    int sign = 1;
    if (acc[W - 1] >> 31) {
        sign = -1;
        u32 cy = 1;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const u64 v = (u64)(u32)~acc[w] + cy;
            acc[w] = (u32)v;
            cy = (u32)(v >> 32);
        }
    }
    const i64 scale = lo - 2 * (32 * N - 1);
    Num<N> r;
    if (!g.subtract) r = pack<N, W>(acc, scale, sign, ST_OK);
    else r = round_sum2<N, W, N>(acc, scale, -sign, old.w, (i64)old.e - (32 * N - 1), old.s);
    store_out<N>(g.out, g.out_pitch, g.out_stride, i, j, mirror, r);
}

// Exact dot product for terms spread beyond any fixed window: the cluster algorithm of
// linalg.hpp:298-317.  Terms in descending exponent order form clusters (a term joins while its top bit
// lies within gap = 32N + ceil(log2(K+1)) + 4 bits of the cluster's lowest bit); the first nonzero cluster
// sum S is exact and only the sign of the next nonzero cluster matters, so the result is
// RN(S * 2^D +/- 1) * 2^-D with D = 32N + 64.  Clusters are found by repeated passes over the term
// exponents (no sort).  cluster_size_kernel measures the widest cluster of every listed output;
// cluster_sum_kernel then sums each cluster exactly in that output's own global scratch (separate
// positive and negative accumulators, so carries stay short) and keeps only the top N+3 words of S and a
// sticky unit for the rounding.  The update's old value is one more term.
struct ClusterTerms {
    const DotArgs& g;
    u32 i, j;
    Num<1> cinfo; // sign and exponent of the old value (limbs not used)
    bool has_c;
    __device__ i64 scale_of(u32 k, int& sg, int N) const
    {
        if (k == g.K) {
            sg = cinfo.s;
            return (i64)cinfo.e - (32 * N - 1);
        }
        const u64 ia = (u64)i * g.left.ls + (u64)k * g.left.ks, ib = (u64)j * g.right.ls + (u64)k * g.right.ks;
        const int sa = (int)g.left.planes[(u64)(N + 1) * g.left.pitch + ia];
        const int sb = (int)g.right.planes[(u64)(N + 1) * g.right.pitch + ib];
        sg = g.subtract ? -sa * sb : sa * sb;
        if (!sg) return -((i64)1 << 62);
        const int ea = (int)g.left.planes[(u64)N * g.left.pitch + ia];
        const int eb = (int)g.right.planes[(u64)N * g.right.pitch + ib];
        return (i64)ea + eb - 2 * (32 * N - 1);
    }
    __device__ u32 terms() const { return g.K + (has_c ? 1u : 0u); }
    // next cluster below `cutoff`: its highest and lowest term exponents; false when none is left
    __device__ bool next(i64 cutoff, i64& hi, i64& low, int N) const
    {
        const i64 width = 64 * N, gap = 32 * N + (i64)g.logk + 4, NONE = -((i64)1 << 62);
        hi = NONE;
        for (u32 k = 0; k < terms(); ++k) {
            int sg;
            const i64 sc = scale_of(k, sg, N);
            if (sg && sc < cutoff && sc > hi) hi = sc;
        }
        if (hi == NONE) return false;
        low = hi;
        for (bool changed = true; changed;) {
            changed = false;
            for (u32 k = 0; k < terms(); ++k) {
                int sg;
                const i64 sc = scale_of(k, sg, N);
                if (sg && sc < low && sc + width - 1 + gap >= low) {
                    low = sc;
                    changed = true;
                }
            }
        }
        return true;
    }
};

// Trivial outputs and updates of status entries; true when the output is finished.
template <int N> __device__ __forceinline__ bool dot_prologue(const DotArgs& g, u32 i, u32 j, Num<N>& old)
{
    const GemmLine* Li = g.lrows + i;
    const GemmLine* Lj = g.rcols + j;
    const bool mirror = g.mirror != 0;
    old = zero<N>(ST_OK);
    if (g.subtract) old = load_out<N>(g.out, g.out_pitch, (u64)i * g.out_stride + j);
    if (Li->cls == 1 || Lj->cls == 1) {
        u32 st = Li->status | Lj->status | (g.subtract ? old.st : 0u);
        if (!g.subtract || st) store_out<N>(g.out, g.out_pitch, g.out_stride, i, j, mirror, zero<N>(st));
        return true;
    }
    if (g.subtract && old.st) {
        store_out<N>(g.out, g.out_pitch, g.out_stride, i, j, mirror, zero<N>(old.st));
        return true;
    }
    return false;
}

// words[idx] = accumulator words of the widest cluster of listed output idx (0 if trivial)
template <int N> __global__ void __launch_bounds__(256) cluster_size_kernel(DotArgs g, u32* words)
{
    const u32 idx = blockIdx.x * 256u + threadIdx.x;
    if (idx >= g.count) return;
    u32 i, j;
    output_of(g, idx, i, j);
    words[idx] = 0;
    if (g.syrk && j > i) return;
    const GemmLine* Li = g.lrows + i;
    const GemmLine* Lj = g.rcols + j;
    if (Li->cls == 1 || Lj->cls == 1) return;
    Num<1> c = zero<1>(ST_OK);
    bool has_c = false;
    if (g.subtract) {
        const u64 at = (u64)i * g.out_stride + j;
        c.e = (int)g.out[(u64)N * g.out_pitch + at];
        c.s = (int)g.out[(u64)(N + 1) * g.out_pitch + at];
        has_c = c.s != 0;
    }
    const ClusterTerms T{g, i, j, c, has_c};
    i64 cutoff = ((i64)1 << 62), hi, low;
    i64 widest = 0;
    while (T.next(cutoff, hi, low, N)) {
        const i64 w = (hi + 64 * N - low) / 32 + 3;
        widest = w > widest ? w : widest;
        cutoff = low;
    }
    words[idx] = (u32)(widest < 0xffffffffll ? widest : 0xffffffffll);
}

// acc[0..W) += x (S words) * 2^off, off >= 0, in global memory; carries propagate as far as needed
__device__ __forceinline__ void global_add(u32* acc, u64 W, const u32* x, int S, i64 off)
{
    const u64 ws = (u64)(off >> 5);
    const u32 bs = (u32)(off & 31);
    u64 carry = 0;
    for (int t = 0; t <= S; ++t) {
        const u32 hi = t < S ? x[t] : 0u, lo = t ? x[t - 1] : 0u;
        const u32 v = bs ? __builtin_amdgcn_alignbit(hi, lo, 32u - bs) : hi;
        const u64 at = ws + (u64)t;
        if (at >= W) break;
        const u64 s = (u64)acc[at] + v + carry;
        acc[at] = (u32)s;
        carry = s >> 32;
    }
    for (u64 at = ws + (u64)S + 1; carry && at < W; ++at) {
        const u64 s = (u64)acc[at] + carry;
        acc[at] = (u32)s;
        carry = s >> 32;
    }
}

template <int N> __global__ void __launch_bounds__(256) cluster_sum_kernel(DotArgs g, const u32* words, const u64* offsets, u32* scratch)
{
    const u32 idx = blockIdx.x * 256u + threadIdx.x;
    if (idx >= g.count) return;
    u32 i, j;
    output_of(g, idx, i, j);
    if (g.syrk && j > i) return;
    Num<N> old;
    if (dot_prologue<N>(g, i, j, old)) return;
    Num<1> c = zero<1>(ST_OK);
    c.e = old.e;
    c.s = old.s;
    const ClusterTerms T{g, i, j, c, g.subtract && old.s != 0};
    const u64 W = words[idx];
    u32* pos = scratch + offsets[idx];
    u32* neg = pos + W;
    constexpr int KW = N + 4; // kept words of S: a sticky word, then the top N+3 words
    u32 S[KW];
#pragma unroll
    for (int w = 0; w < KW; ++w) S[w] = 0;
    i64 scale1 = 0, cutoff = ((i64)1 << 62), hi, low;
    int nsums = 0, sign1 = 0, sign2 = 0;
    while (nsums < 2 && T.next(cutoff, hi, low, N)) {
        for (u64 w = 0; w < 2 * W; ++w) pos[w] = 0;
        for (u32 k = 0; k < T.terms(); ++k) {
            int sg;
            const i64 sc = T.scale_of(k, sg, N);
            if (!sg || sc < low || sc >= cutoff) continue;
            u32* dst = sg > 0 ? pos : neg;
            if (k == g.K) global_add(dst, W, old.w, N, sc - low);
            else {
                const Num<N> a = load_view<N>(g.left, i, k);
                const Num<N> b = load_view<N>(g.right, j, k);
                u32 p[2 * N];
                mantissa_product<N>(a.w, b.w, p);
                global_add(dst, W, p, 2 * N, sc - low);
            }
        }
        // sign and magnitude of pos - neg
        int cmp = 0;
        for (u64 w = W; w-- > 0;)
            if (pos[w] != neg[w]) {
                cmp = pos[w] > neg[w] ? 1 : -1;
                break;
            }
        if (cmp) {
            if (!nsums) {
                u32* big = cmp > 0 ? pos : neg;
                const u32* small = cmp > 0 ? neg : pos;
                u32 bw = 0;
                u64 top = 0;
                for (u64 w = 0; w < W; ++w) {
                    const u64 v = (u64)big[w] - small[w] - bw;
                    big[w] = (u32)v;
                    bw = (u32)(v >> 63);
                    if (big[w]) top = w;
                }
                // keep words [top-(N+2), top] and a sticky word for everything below
                const i64 first = (i64)top - (N + 2);
                bool sticky = false;
                for (i64 w = 0; w < first; ++w) sticky = sticky || big[w] != 0;
                S[0] = sticky ? 1u : 0u;
#pragma unroll
                for (int t = 0; t < N + 3; ++t) {
                    const i64 w = first + t;
                    S[t + 1] = (w >= 0 && w < (i64)W) ? big[w] : 0u;
                }
                scale1 = low + 32 * (first - 1);
                sign1 = cmp;
            } else
                sign2 = cmp;
            ++nsums;
        }
        cutoff = low;
    }
    Num<N> r;
    if (!nsums) r = zero<N>(ST_OK);
    else if (nsums == 1) r = pack<N, KW>(S, scale1, sign1, ST_OK);
    else {
        // S * 2^D -/+ 1 puts the sticky unit below the rounding position of S
        constexpr int DW = N + 2, EW = KW + DW;
        u32 ext[EW];
#pragma unroll
        for (int w = 0; w < EW; ++w) ext[w] = w >= DW ? S[w - DW] : 0u;
        if (sign2 == sign1) ext[0] = 1;
        else {
            u32 bw = 1;
#pragma unroll
            for (int w = 0; w < EW; ++w) {
                const u64 v = (u64)ext[w] - bw;
                ext[w] = (u32)v;
                bw = (u32)(v >> 63);
            }
        }
        r = pack<N, EW>(ext, scale1 - 32 * DW, sign1, ST_OK);
    }
    store_out<N>(g.out, g.out_pitch, g.out_stride, i, j, g.mirror != 0, r);
}

} // namespace lf
