// gemm.hip — exact dense products on MI355X: the int8-MFMA residue product kernel and the host planner
// behind lf_gemm_host / lf_syrk_host / lf_gemm_planes (the reference's Linalg::gemm / syrk and
// Linalg::Impl::run, src/linalg.mm:295-407).
//
// Per call: band analysis of every line on the device (linalg.mm:82-111, same classes and bands; only the
// line table comes back to the host), modulus count from the widest band (linalg.mm:341-345), CRT constants
// in exact integer arithmetic, then on one
// stream: digits of both extended operands, the residue GEMM per modulus on int8 MFMA, one output-centric
// CRT rebuild pass that also writes the trivial outputs, and the exact-dot kernels for the outputs of lines
// outside the residue path.  Nothing is computed on the host besides the plan.
#include "limbforge_hip.h"
#include "gemm_kernels.hpp"
#include "gemm_launch.hpp"
#include "gemm_plan.hpp"
#include "host_copy.hpp"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <climits>
#include <cmath>
#include <cstring>
#include <limits>
#include <map>
#include <string>
#include <thread>
#include <vector>

namespace lf {

// ------------------------------------------------------------------ int8 MFMA residue product
constexpr int PT = 128;       // output tile per workgroup (rows and columns)
constexpr int PK = 32;        // K per MFMA step
constexpr u32 XCDS = 8;       // MI355X: 8 XCDs, workgroups dealt to them round-robin by linear id

// One 32x32 block of residues times the CRT factor y = (M/m)^-1 mod m: (65536 G11 + 256 Gmid + G00) y mod m,
// written as uint16, in 32-bit integer and FP32 arithmetic (residue_fold; the factor rides on the digit
// weights, so the CRT kernel reads y_q itself).
struct FoldWeights {
    int k11, kmid, k00;
};
__device__ __forceinline__ void store_block(uint16_t* out, u32 Np, u32 row, u32 col, u32 lane, const v16i& c11, const v16i& c00,
                                            const v16i& cmid, const FoldWeights& k, int m, float inv, int c32)
{
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        // 32x32 accumulator layout: lane l, element i -> row 8(i/4) + 4(l/32) + i%4, column l%32
        const u32 rr = row + 8u * (u32)(i / 4) + 4u * (lane >> 5) + (u32)(i % 4);
        const u32 cc = col + (lane & 31u);
        out[(u64)rr * Np + cc] = (uint16_t)residue_fold(c11[i], cmid[i], c00[i], k.k11, k.kmid, k.k00, m, inv, c32);
    }
}

// One 128x128 output tile of one modulus: four waves, each a 64x64 sub-tile of 2x2 MFMA blocks with three
// int32 accumulators each (G11, G00, Gmid).  The digit tiles of a 32-deep K step (both planes of 128 A
// rows and 128 B columns, 16 KB) travel from global memory straight into LDS (global_load_lds_dwordx4: lane
// i's 16 bytes land at 16 i of the instruction's LDS base) through a ring of four stages, so three steps
// are in flight while one is computed: each wave issues four loads per step, waits for its own loads of
// the step it is about to use (vmcnt), and one barrier per step both publishes them and frees the oldest
// stage for refilling.  In a stage, row r's two 16-byte halves sit at chunks 2r + (h xor bit 3 of r), so
// the 16 lanes of an MFMA operand read hit distinct banks.  Each wave then reads 8 fragments and issues
// 16 v_mfma_i32_32x32x32_i8.  The 1-D grid is dealt to the XCDs so that all tiles of a modulus run on
// one XCD (modulus q on XCD q mod 8): a modulus's digit planes are fetched into one L2 instead of eight.
constexpr u32 STAGES = 4;
__device__ __forceinline__ u32 chunk_of(u32 r, u32 h) { return 2u * r + (h ^ ((r >> 3) & 1u)); }

template <u32 V> __device__ __forceinline__ void wait_vmcnt()
{
    static_assert(V < 64, "vmcnt field");
    __builtin_amdgcn_s_waitcnt((int)((V & 15u) | (7u << 4) | (15u << 8) | ((V >> 4) << 14)));
}

__global__ void __launch_bounds__(256, 2) product_kernel(ProductArgs g)
{
    const u32 tiles_x = g.Np / PT, tiles = tiles_x * (g.Mp / PT);
    const u32 xcd = blockIdx.x % XCDS, slot = blockIdx.x / XCDS;
    const u32 q = xcd + XCDS * (slot / tiles), tile = slot % tiles;
    if (q >= g.L) return;
    const u32 row0 = (tile / tiles_x) * PT, col0 = (tile % tiles_x) * PT;
    if (g.lower && col0 > row0 + PT - 1) return; // tile strictly above the diagonal
    __shared__ __attribute__((aligned(16))) int8_t ring[STAGES][4][PT * PK]; // [stage][a1, a0, b1, b0][chunks]
    const u64 aplane = (u64)g.Mp * g.Kp, bplane = (u64)g.Np * g.Kp;
    const u32 t = threadIdx.x;
    const u32 lane = t & 63u, wave = t >> 6;
    const u32 wr = (wave >> 1) * 64u, wc = (wave & 1u) * 64u;
    // loads: this wave fills chunks [64 wave, 64 wave + 64) of each of the four regions; lane i takes the
    // chunk at position 64 wave + i, i.e. row p/2, half (p & 1) xor bit 3 of the row
    const u32 p = 64u * wave + lane, pr = p >> 1, ph = (p & 1u) ^ ((pr >> 3) & 1u);
    const int8_t* src[4] = {g.a1 + q * aplane + (u64)(row0 + pr) * g.Kp + 16u * ph, g.a0 + q * aplane + (u64)(row0 + pr) * g.Kp + 16u * ph,
                            g.b1 + q * bplane + (u64)(col0 + pr) * g.Kp + 16u * ph, g.b0 + q * bplane + (u64)(col0 + pr) * g.Kp + 16u * ph};
    auto issue = [&](u32 st) {
        const u32 buf = st % STAGES, k0 = st * PK;
#pragma unroll
        for (int rg = 0; rg < 4; ++rg)
            __builtin_amdgcn_global_load_lds((const void*)(src[rg] + k0), (__attribute__((address_space(3))) void*)&ring[buf][rg][1024u * wave], 16, 0,
                                             0);
    };
    v16i c11[2][2] = {}, c00[2][2] = {}, cmid[2][2] = {};
    const u32 r = lane & 31u, kh = lane >> 5;
    const u32 steps = g.Kp / PK;
#pragma unroll
    for (u32 st = 0; st + 1 < STAGES; ++st)
        if (st < steps) issue(st);
    for (u32 s = 0; s < steps; ++s) {
        const u32 ahead = steps - 1 - s; // stages issued after s, capped at STAGES - 2
        if (ahead >= STAGES - 2) wait_vmcnt<4 * (STAGES - 2)>();
        else if (ahead == 1) wait_vmcnt<4>();
        else wait_vmcnt<0>();
        // a bare barrier: __syncthreads' fence would wait for every load in flight (vmcnt 0); the loads
        // this step reads were waited for above, and the reads of the stage refilled next have completed
        // (their values fed the previous step's MFMAs)
        __builtin_amdgcn_s_barrier();
        if (s + STAGES - 1 < steps) issue(s + STAGES - 1);
        const u32 cur = s % STAGES;
        v4i a1[2], a0[2], b1[2], b0[2];
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
            const u32 ca = 16u * chunk_of(wr + 32u * hh + r, kh), cb = 16u * chunk_of(wc + 32u * hh + r, kh);
            a1[hh] = *(const v4i*)(&ring[cur][0][ca]);
            a0[hh] = *(const v4i*)(&ring[cur][1][ca]);
            b1[hh] = *(const v4i*)(&ring[cur][2][cb]);
            b0[hh] = *(const v4i*)(&ring[cur][3][cb]);
        }
#pragma unroll
        for (int mi = 0; mi < 2; ++mi)
#pragma unroll
            for (int ni = 0; ni < 2; ++ni) {
                c11[mi][ni] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a1[mi], b1[ni], c11[mi][ni], 0, 0, 0);
                c00[mi][ni] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a0[mi], b0[ni], c00[mi][ni], 0, 0, 0);
                cmid[mi][ni] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a1[mi], b0[ni], cmid[mi][ni], 0, 0, 0);
                cmid[mi][ni] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a0[mi], b1[ni], cmid[mi][ni], 0, 0, 0);
            }
    }
    const int m = (int)g.moduli[q];
    const float inv = 1.0f / (float)m;
    const int c32u = (int)(((u64)1 << 32) % (u64)m), c32 = c32u > m / 2 ? c32u - m : c32u; // balanced 2^32 mod m
    const FoldWeights k{g.fold[3 * q], g.fold[3 * q + 1], g.fold[3 * q + 2]};
    uint16_t* out = g.res + (u64)q * g.Mp * g.Np;
    // one block at a time (the scheduling barriers keep the accumulators in AGPRs until their turn)
    store_block(out, g.Np, row0 + wr, col0 + wc, lane, c11[0][0], c00[0][0], cmid[0][0], k, m, inv, c32);
    __builtin_amdgcn_sched_barrier(0);
    store_block(out, g.Np, row0 + wr, col0 + wc + 32u, lane, c11[0][1], c00[0][1], cmid[0][1], k, m, inv, c32);
    __builtin_amdgcn_sched_barrier(0);
    store_block(out, g.Np, row0 + wr + 32u, col0 + wc, lane, c11[1][0], c00[1][0], cmid[1][0], k, m, inv, c32);
    __builtin_amdgcn_sched_barrier(0);
    store_block(out, g.Np, row0 + wr + 32u, col0 + wc + 32u, lane, c11[1][1], c00[1][1], cmid[1][1], k, m, inv, c32);
}

hipError_t launch_product(const ProductArgs& g, hipStream_t s)
{
    if (!g.L || !g.Mp || !g.Np) return hipSuccess;
    const u32 tiles = (g.Np / PT) * (g.Mp / PT);
    const u32 per_xcd = (g.L + XCDS - 1) / XCDS; // moduli per XCD (the last ones may idle)
    hipLaunchKernelGGL(product_kernel, dim3(XCDS * tiles * per_xcd), dim3(256), 0, s, g);
    return hipGetLastError();
}

} // namespace lf

// the C ABI's per-thread error message (capi.hip)
void lf_set_last_error(const std::string& message);

namespace {
using lf::GemmLine;
using lf::GEMM_MAX_BANDS;
typedef unsigned __int128 u128;

constexpr std::size_t MAX_K = 65472; // 2 Kp 2^14 < 2^31 keeps every int8 product sum exact in int32

int fail(int code, const std::string& m)
{
    lf_set_last_error(m);
    return code;
}

// ---- exact multiword helpers (host) ----
struct Big {
    std::vector<uint32_t> w; // little endian
    void trim()
    {
        while (!w.empty() && !w.back()) w.pop_back();
    }
    int bits() const
    {
        for (int i = int(w.size()) - 1; i >= 0; --i)
            if (w[i]) return 32 * i + 32 - __builtin_clz(w[i]);
        return 0;
    }
};
Big big_from(uint64_t v)
{
    Big b;
    b.w = {uint32_t(v), uint32_t(v >> 32)};
    b.trim();
    return b;
}
void big_mul_small(Big& b, uint32_t m)
{
    uint64_t c = 0;
    for (auto& x : b.w) {
        uint64_t t = uint64_t(x) * m + c;
        x = uint32_t(t);
        c = t >> 32;
    }
    if (c) b.w.push_back(uint32_t(c));
}
// b / m exactly (m divides b)
Big big_div_small(const Big& b, uint32_t m)
{
    Big q;
    q.w.assign(b.w.size(), 0);
    uint64_t r = 0;
    for (int i = int(b.w.size()) - 1; i >= 0; --i) {
        uint64_t cur = (r << 32) | b.w[i];
        q.w[i] = uint32_t(cur / m);
        r = cur % m;
    }
    q.trim();
    return q;
}
uint32_t big_mod_small(const Big& b, uint32_t m)
{
    uint64_t r = 0;
    for (int i = int(b.w.size()) - 1; i >= 0; --i) r = ((r << 32) | b.w[i]) % m;
    return uint32_t(r);
}
// b << s into exactly `words` words (must fit)
std::vector<uint32_t> big_shifted(const Big& b, int s, int words)
{
    std::vector<uint32_t> out(words, 0);
    const int ws = s / 32, bs = s % 32;
    for (std::size_t i = 0; i < b.w.size(); ++i) {
        uint64_t v = uint64_t(b.w[i]) << bs;
        if (i + ws < std::size_t(words)) out[i + ws] |= uint32_t(v);
        if (i + ws + 1 < std::size_t(words)) out[i + ws + 1] |= uint32_t(v >> 32);
    }
    return out;
}
uint32_t inverse_mod(uint64_t a, uint64_t m) // a^-1 mod m (gcd 1)
{
    int64_t t = 0, nt = 1, r = int64_t(m), nr = int64_t(a % m);
    while (nr) {
        int64_t q = r / nr, x = t - q * nt;
        t = nt;
        nt = x;
        x = r - q * nr;
        r = nr;
        nr = x;
    }
    return uint32_t(t < 0 ? t + int64_t(m) : t);
}

// ------------------------------------------------------------------ band analysis on the device
// The reference's per-line analysis (linalg.mm:82-111) from the lines' exponent, sign and status planes: status OR, largest and smallest exponent of a nonzero status-free entry, the class
// (0 bands, 1 zero or status line, 2 exact fallback) and the greedy bands [hi - G, hi] taken from the largest
// exponent down (lo: the smallest exponent inside), one pass over the line per band.  Lines with more than
// max_bands bands or a spread above max_spread are class 2; the first GEMM_MAX_BANDS bands are stored and nb
// counts them all (up to max_bands + 1).
using lf::GemmLine;
using lf::MatView;
using lf::u32;
using lf::u64;
using lf::GEMM_MAX_BANDS;
using lf::DIGIT_TABLE_BYTES;
using lf::PT;

struct AnalyzeSide {
    MatView v;
    uint32_t nlines, blocks;
    uint32_t by_line; // lines adjacent in memory: a workgroup takes 16 lines, else one wavefront a line
    GemmLine* out;
    GemmLine* host; // the same table in pinned host memory
};
struct AnalyzeArgs {
    AnalyzeSide side[2];
    uint32_t field_plane; // N: exponent plane (sign N + 1, status N + 2)
    uint32_t K;
    int32_t G, max_bands, max_spread;
    uint32_t force;
};

constexpr u32 ANALYZE_THREADS = 1024, ANALYZE_LINES = 16;

// Reductions over the threads of one line: the 64 lanes of its wavefront, or lanes l, l + 16, l + 32, l + 48 of
// every wavefront of the workgroup (through red, 16 values a wavefront), with every thread getting the result.
template <bool BY_LINE, class F> __device__ __forceinline__ int line_reduce(int x, int (*red)[ANALYZE_LINES], F pick)
{
    const u32 lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
#pragma unroll
    for (int o = 32; o >= (BY_LINE ? 16 : 1); o >>= 1) x = pick(x, __shfl_xor(x, o));
    if constexpr (BY_LINE) {
        if (lane < ANALYZE_LINES) red[wave][lane] = x;
        __syncthreads();
        x = red[0][lane % ANALYZE_LINES];
#pragma unroll
        for (u32 w = 1; w < ANALYZE_THREADS / 64u; ++w) x = pick(x, red[w][lane % ANALYZE_LINES]);
        __syncthreads();
    }
    return x;
}

// One line's record, its threads striding over the line's K entries: first status and exponent range, then one
// pass per band.  BY_LINE: the workgroup's 16 lines go through the same passes together.
template <bool BY_LINE> __device__ __forceinline__ void analyze_line(const AnalyzeArgs& a, const AnalyzeSide& S, u32 line, bool live, u32 first,
                                                                     u32 step, bool leader, GemmLine& L, int (*red)[ANALYZE_LINES])
{
    const u32* ep = S.v.planes + (u64)a.field_plane * S.v.pitch;
    const u32* sp = ep + S.v.pitch;
    const u32* tp = sp + S.v.pitch;
    const u64 base = (u64)line * S.v.ls;
    const u32 K = live ? a.K : 0u;
    const auto mx = [](int x, int y) { return max(x, y); };
    const auto mn = [](int x, int y) { return min(x, y); };
    u32 status = 0;
    int top = INT_MIN, bottom = INT_MAX;
    // a thread's exponents stay in registers for the band passes (INT_MIN: zero, status or past K) where they fit, in 32
    // registers for lines of up to 2,048 entries; all their loads are then in flight together.  Longer lines are read
    // again by each pass: 64 lines of 2,048 and of 2,112 entries take 27 and 43 us with adjacent entries (one band), 30
    // and 57 with adjacent lines (three bands).
    constexpr u32 KEPT = 32;
    const bool kept = a.K <= KEPT * step;
    int own[KEPT];
    if (kept) {
#pragma unroll
        for (u32 n = 0; n < KEPT; ++n) {
            const u32 k = first + n * step;
            own[n] = INT_MIN;
            if (k < K) {
                const u64 i = base + (u64)k * S.v.ks;
                const int e = (int)ep[i], sg = (int)sp[i];
                const u32 st = tp[i];
                status |= st;
                own[n] = !st && sg ? e : INT_MIN;
            }
        }
#pragma unroll
        for (u32 n = 0; n < KEPT; ++n) {
            top = max(top, own[n]);
            bottom = own[n] == INT_MIN ? bottom : min(bottom, own[n]);
        }
    } else
#pragma unroll 4
        for (u32 k = first; k < K; k += step) {
            const u64 i = base + (u64)k * S.v.ks;
            const int e = (int)ep[i], sg = (int)sp[i];
            const u32 st = tp[i];
            status |= st;
            if (!st && sg) {
                top = max(top, e);
                bottom = min(bottom, e);
            }
        }
    status = (u32)line_reduce<BY_LINE>((int)status, red, [](int x, int y) { return x | y; });
    top = line_reduce<BY_LINE>(top, red, mx);
    bottom = line_reduce<BY_LINE>(bottom, red, mn);
    const bool any = top != INT_MIN;
    int cls = 1, nb = 0, low = 0, hi = top;
    bool more = false;
    if (leader)
#pragma unroll
        for (int b = 0; b < GEMM_MAX_BANDS; ++b) L.member[b] = L.lo[b] = L.hi[b] = 0;
    if (live && !status && any) {
        if (a.force) cls = 2;
        else if (a.max_bands >= 1 && (long)top - bottom <= a.G) {
            cls = 0;
            nb = 1;
            low = bottom;
            if (leader) {
                L.lo[0] = bottom;
                L.hi[0] = top;
            }
        } else if ((long)top - bottom > a.max_spread) cls = 2;
        else more = true;
    }
    while (BY_LINE ? __syncthreads_or(more) != 0 : more) {
        int lo = hi, next = INT_MIN;
        if (more && kept) {
#pragma unroll
            for (u32 n = 0; n < KEPT; ++n) {
                const int e = own[n];
                if (e == INT_MIN || e > hi) continue;
                if ((long)e >= (long)hi - a.G) lo = min(lo, e);
                else next = max(next, e);
            }
        } else if (more)
#pragma unroll 4
            for (u32 k = first; k < K; k += step) {
                const u64 i = base + (u64)k * S.v.ks;
                const int e = (int)ep[i], sg = (int)sp[i];
                const u32 st = tp[i];
                if (st || !sg || e > hi) continue;
                if ((long)e >= (long)hi - a.G) lo = min(lo, e);
                else next = max(next, e);
            }
        lo = line_reduce<BY_LINE>(lo, red, mn);
        next = line_reduce<BY_LINE>(next, red, mx);
        if (!more) continue;
        if (leader && nb < GEMM_MAX_BANDS) {
            L.lo[nb] = lo;
            L.hi[nb] = hi;
        }
        ++nb;
        low = lo;
        if (nb > a.max_bands) {
            cls = 2;
            nb = 0;
            more = false;
        } else if (next == INT_MIN) {
            cls = 0;
            more = false;
        } else
            hi = next;
    }
    if (leader) {
        L.cls = cls;
        L.nb = nb;
        L.low = low;
        L.status = status;
        L.top = any ? top : 0;
        L.bottom = any ? bottom : 0;
        L.member[0] = (int)line; // its extended row while every line is one band
    }
}

// Both sides of a product in one launch; the records go to the device table and to the host's.  What bounds it is
// the latency of its loads: 16 lines and 64 rows of them at a time where lines are adjacent (a wavefront per
// line there read one word per 64 bytes: 56 us for 512 columns of 2048 entries).
__global__ void __launch_bounds__(ANALYZE_THREADS) analyze_kernel(AnalyzeArgs a)
{
    __shared__ int red[ANALYZE_THREADS / 64][ANALYZE_LINES];
    __shared__ GemmLine rec[ANALYZE_LINES];
    const bool second = blockIdx.x >= a.side[0].blocks;
    const AnalyzeSide S = second ? a.side[1] : a.side[0];
    const u32 line0 = (blockIdx.x - (second ? a.side[0].blocks : 0u)) * ANALYZE_LINES;
    const u32 t = threadIdx.x;
    if (S.by_line) {
        const u32 l = t % ANALYZE_LINES;
        analyze_line<true>(a, S, line0 + l, line0 + l < S.nlines, t / ANALYZE_LINES, ANALYZE_THREADS / ANALYZE_LINES, t < ANALYZE_LINES, rec[l], red);
    } else {
        const u32 l = t / 64u;
        analyze_line<false>(a, S, line0 + l, line0 + l < S.nlines, t % 64u, 64u, t % 64u == 0, rec[l], red);
    }
    __syncthreads();
    const u32 lines = min(ANALYZE_LINES, S.nlines - line0), words = sizeof(GemmLine) / 4;
    for (u32 w = t; w < lines * words; w += ANALYZE_THREADS) {
        const u32 v = reinterpret_cast<const u32*>(rec)[w];
        reinterpret_cast<u32*>(S.out + line0)[w] = v;
        reinterpret_cast<u32*>(S.host + line0)[w] = v;
    }
}

// Primes <= 65279, descending: balanced residues then split into two int8 digits (linalg.mm:38-40).
const std::vector<uint32_t>& primes()
{
    static const std::vector<uint32_t> p = [] {
        std::vector<uint32_t> r;
        for (uint32_t q = 65279; r.size() < 1200; --q) {
            bool prime = true;
            for (uint32_t d = 2; d * d <= q; ++d)
                if (q % d == 0) {
                    prime = false;
                    break;
                }
            if (prime) r.push_back(q);
        }
        return r;
    }();
    return p;
}

using lf::Product;

// One side of a product: its line table (in pinned host memory) and what the report says of it.
struct Side {
    GemmLine* lines = nullptr;
    std::size_t count = 0;
    std::vector<uint64_t> histogram;
    uint64_t fallback = 0;
};

void read_side(Side& s, int max_bands)
{
    s.histogram.assign(std::size_t(std::max(max_bands, 0)) + 1, 0);
    for (std::size_t i = 0; i < s.count; ++i) {
        const GemmLine& L = s.lines[i];
        if (L.cls == 2) ++s.fallback;
        else ++s.histogram[L.cls == 1 ? 0 : L.nb];
    }
}

// GPU-path capacity: lines whose bands this build's rebuild kernels cannot hold take the exact-dot path
// (same results; the report counts them as fallback lines).
void route_capacity(Side& s, int wx_class)
{
    for (std::size_t i = 0; i < s.count; ++i) {
        GemmLine& L = s.lines[i];
        if (L.cls != 0) continue;
        const bool too_many = L.nb > GEMM_MAX_BANDS;
        const bool too_wide = L.nb > 1 && (wx_class != 0 || long(L.hi[0]) - L.low > 512);
        if (too_many || too_wide) {
            L.cls = 2;
            ++s.fallback;
            --s.histogram[L.nb];
        }
    }
}

// What a thread keeps for a device is found by the device's own number (a node in a partitioned mode shows more devices
// than GPUs) in a std::map, whose entries stay where they are when another device's is added.

// Five timing events per host thread and device, created once and reused by every product.
hipError_t stage_events(hipEvent_t** out)
{
    struct Set {
        hipEvent_t e[5] = {};
        ~Set()
        {
            for (auto x : e)
                if (x) (void)hipEventDestroy(x);
        }
    };
    thread_local std::map<int, Set> sets;
    int device = 0;
    if (hipError_t err = hipGetDevice(&device)) return err;
    Set& s = sets[device];
    for (auto& x : s.e)
        if (!x)
            if (hipError_t err = hipEventCreate(&x)) return err;
    *out = s.e;
    return hipSuccess;
}

int ceil_log2(std::size_t x)
{
    int l = 0;
    while ((std::size_t(1) << l) < x) ++l;
    return l;
}

struct DeviceBuf {
    void* p = nullptr;
    ~DeviceBuf()
    {
        if (p) (void)hipFree(p);
    }
    hipError_t alloc(std::size_t bytes)
    {
        if (p) (void)hipFree(p);
        p = nullptr;
        return hipMalloc(&p, std::max<std::size_t>(bytes, 16));
    }
};

// Device work buffers of the planner, kept per host thread and device and grown on demand, so that a
// sequence of products (the updates of a factorization) does not allocate and free on every call.  A
// product synchronizes its stream before returning, so the next call on the thread may reuse them.
struct Workspace {
    std::vector<std::pair<void*, std::size_t>> slots;
    ~Workspace()
    {
        for (auto& s : slots)
            if (s.first) (void)hipFree(s.first);
    }
};
struct PoolBuf {
    int slot;
    void* p = nullptr;
    hipError_t alloc(std::size_t bytes)
    {
        std::pair<void*, std::size_t>* s = nullptr;
        if (hipError_t e = find(&s)) return e;
        bytes = std::max<std::size_t>(bytes, 16);
        if (s->second < bytes) {
            if (hipError_t e = release()) return e;
            void* q = nullptr;
            if (hipError_t e = hipMalloc(&q, bytes)) return e;
            *s = {q, bytes};
        }
        p = s->first;
        return hipSuccess;
    }
    // the slot's memory back to the device
    hipError_t release()
    {
        std::pair<void*, std::size_t>* s = nullptr;
        if (hipError_t e = find(&s)) return e;
        if (s->first) (void)hipFree(s->first);
        *s = {nullptr, 0};
        p = nullptr;
        return hipSuccess;
    }

private:
    hipError_t find(std::pair<void*, std::size_t>** s) const
    {
        thread_local std::map<int, Workspace> pools;
        int dev = 0;
        if (hipError_t e = hipGetDevice(&dev)) return e;
        Workspace& ws = pools[dev];
        if (ws.slots.size() <= std::size_t(slot)) ws.slots.resize(slot + 1, {nullptr, 0});
        *s = &ws.slots[slot];
        return hipSuccess;
    }
};

// The line tables' pinned host memory, kept per host thread and device and grown on demand (a product waits for
// its stream before it returns, so the next one may overwrite it).
struct PinnedTable {
    GemmLine* p = nullptr;
    std::size_t lines = 0;
    ~PinnedTable()
    {
        if (p) (void)hipHostFree(p);
    }
};
hipError_t pinned_table(std::size_t lines, GemmLine** out)
{
    thread_local std::map<int, PinnedTable> tables;
    int dev = 0;
    if (hipError_t e = hipGetDevice(&dev)) return e;
    PinnedTable& t = tables[dev];
    if (t.lines < lines) {
        if (t.p) (void)hipHostFree(t.p);
        t.p = nullptr;
        t.lines = 0;
        if (hipError_t e = hipHostMalloc((void**)&t.p, lines * sizeof(GemmLine), hipHostMallocDefault)) return e;
        t.lines = lines;
    }
    *out = t.p;
    return hipSuccess;
}

// ------------------------------------------------------------------ constants of the residue path
// Modulus counts up to the widest CRT class: bits and double log2 sums of the products of the first L primes.
constexpr unsigned MAX_L = 208;
struct ModulusSums {
    double have[MAX_L + 1];
    int bits[MAX_L + 1];
    ModulusSums()
    {
        Big M = big_from(1);
        have[0] = 0;
        bits[0] = M.bits();
        for (unsigned q = 0; q < MAX_L; ++q) {
            have[q + 1] = have[q] + std::log2(double(primes()[q]));
            big_mul_small(M, primes()[q]);
            bits[q + 1] = M.bits();
        }
    }
};
// The fewest moduli for an integer of `need` bits: the reference's double sum, then the same bound exactly (M is
// odd and `need` an integer, so M > 2^need means more than `need` bits), which only guards against the sum's
// rounding.  0: more than MAX_L.
unsigned modulus_count(double need, int* bits)
{
    static const ModulusSums sums;
    unsigned L = 0;
    while (L <= MAX_L && sums.have[L] <= need) ++L;
    while (L <= MAX_L && sums.bits[L] <= int(need)) ++L;
    if (L > MAX_L) return 0;
    *bits = sums.bits[L];
    return L;
}

// Device tables kept per host thread and device: the digit table of all moduli (once), and the CRT constants of
// the (moduli, words) sizes used last, at most CRT_SETS of them (each below 100 KB).
struct DigitTable {
    const int8_t* table;
    const int32_t* offset[DIGIT_TABLE_BYTES / 32 + 1]; // by byte length / 32
    const uint32_t* moduli;
    const float* inverse;
};
struct CrtSet {
    unsigned L = 0;
    int WX = 0;
    int shift = 0;
    const int32_t* fold;
    const uint32_t* crt;
    const uint32_t* bound;
};
constexpr std::size_t CRT_SETS = 16;
struct ConstantCache {
    void* digits_mem = nullptr;
    DigitTable digits{};
    struct Entry {
        CrtSet set;
        void* mem = nullptr;
        uint64_t used = 0;
    };
    std::vector<Entry> sets;
    uint64_t clock = 0;
    ~ConstantCache()
    {
        if (digits_mem) (void)hipFree(digits_mem);
        for (auto& e : sets)
            if (e.mem) (void)hipFree(e.mem);
    }
};
ConstantCache& constant_cache(int dev)
{
    thread_local std::map<int, ConstantCache> caches;
    return caches[dev];
}

// Uploads `words` into new device memory, complete on return.
hipError_t upload_words(const std::vector<uint32_t>& words, void** mem)
{
    if (hipError_t e = hipMalloc(mem, words.size() * 4)) return e;
    if (hipError_t e = hipMemcpy(*mem, words.data(), words.size() * 4, hipMemcpyHostToDevice)) {
        (void)hipFree(*mem);
        *mem = nullptr;
        return e;
    }
    return hipSuccess;
}

hipError_t digit_table(const DigitTable** out)
{
    int dev = 0;
    if (hipError_t e = hipGetDevice(&dev)) return e;
    ConstantCache& c = constant_cache(dev);
    if (!c.digits_mem) {
        constexpr unsigned W = DIGIT_TABLE_BYTES, S = W / 32 + 1;
        std::vector<uint32_t> w(MAX_L * 2 * W / 4 + S * MAX_L + 2 * MAX_L, 0);
        int8_t* tab = reinterpret_cast<int8_t*>(w.data());
        uint32_t *off = w.data() + MAX_L * 2 * W / 4, *mod = off + S * MAX_L, *inv = mod + MAX_L;
        for (unsigned q = 0; q < MAX_L; ++q) {
            const uint32_t m = primes()[q];
            uint64_t p = 1, sum = 0;
            for (unsigned h = 0; h < W; ++h) {
                if (h % 32 == 0) off[h / 32 * MAX_L + q] = uint32_t(128 * sum % m);
                const int v = p > m / 2 ? int(p) - int(m) : int(p), d0 = ((v + 128) & 255) - 128;
                tab[(q * 2) * W + h] = int8_t((v - d0) / 256);
                tab[(q * 2 + 1) * W + h] = int8_t(d0);
                sum += p;
                p = (p << 8) % m;
            }
            off[(S - 1) * MAX_L + q] = uint32_t(128 * sum % m);
            mod[q] = m;
            const float f = 1.0f / float(m);
            std::memcpy(&inv[q], &f, 4);
        }
        if (hipError_t e = upload_words(w, &c.digits_mem)) return e;
        const uint32_t* d = (const uint32_t*)c.digits_mem;
        c.digits.table = (const int8_t*)d;
        for (unsigned k = 0; k < S; ++k) c.digits.offset[k] = (const int32_t*)(d + MAX_L * 2 * W / 4 + k * MAX_L);
        c.digits.moduli = d + MAX_L * 2 * W / 4 + S * MAX_L;
        c.digits.inverse = (const float*)(c.digits.moduli + MAX_L);
    }
    *out = &c.digits;
    return hipSuccess;
}

// fold[L][3] | crt[L][WX] | bound[2][WX] for the first L primes and WX CRT words
hipError_t crt_constants(unsigned L, int WX, CrtSet* out)
{
    int dev = 0;
    if (hipError_t e = hipGetDevice(&dev)) return e;
    ConstantCache& c = constant_cache(dev);
    for (auto& e : c.sets)
        if (e.set.L == L && e.set.WX == WX) {
            e.used = ++c.clock;
            *out = e.set;
            return hipSuccess;
        }
    Big M = big_from(1);
    for (unsigned q = 0; q < L; ++q) big_mul_small(M, primes()[q]);
    CrtSet set;
    set.L = L;
    set.WX = WX;
    set.shift = 32 * (WX - 1) - M.bits();
    std::vector<uint32_t> w, crt;
    for (unsigned q = 0; q < L; ++q) {
        const uint32_t m = primes()[q];
        const Big Mq = big_div_small(M, m);
        // the product kernel's digit weights 65536 y, 256 y, y (mod m, balanced), y = (M/m)^-1 mod m
        const uint64_t y = inverse_mod(big_mod_small(Mq, m), m);
        for (uint64_t d : {uint64_t(65536), uint64_t(256), uint64_t(1)}) {
            const int64_t k = int64_t(d * y % m);
            w.push_back(uint32_t(int32_t(k > int64_t(m / 2) ? k - int64_t(m) : k)));
        }
        const std::vector<uint32_t> words = big_shifted(Mq, set.shift, WX);
        crt.insert(crt.end(), words.begin(), words.end());
    }
    const std::size_t o_crt = w.size(), o_bound = o_crt + crt.size();
    w.insert(w.end(), crt.begin(), crt.end());
    const std::vector<uint32_t> Ms = big_shifted(M, set.shift, WX);
    w.insert(w.end(), Ms.begin(), Ms.end());
    for (int i = 0; i < WX; ++i) w.push_back((Ms[i] >> 1) | (i + 1 < WX ? Ms[i + 1] << 31 : 0u));
    ConstantCache::Entry* slot = nullptr;
    if (c.sets.size() < CRT_SETS) {
        c.sets.emplace_back();
        slot = &c.sets.back();
    } else {
        slot = &*std::min_element(c.sets.begin(), c.sets.end(), [](const auto& x, const auto& y) { return x.used < y.used; });
        (void)hipFree(slot->mem); // the products that used it have finished
        *slot = {};
    }
    if (hipError_t e = upload_words(w, &slot->mem)) return e;
    const uint32_t* d = (const uint32_t*)slot->mem;
    set.fold = (const int32_t*)d;
    set.crt = d + o_crt;
    set.bound = d + o_bound;
    slot->set = set;
    slot->used = ++c.clock;
    *out = set;
    return hipSuccess;
}

// ------------------------------------------------------------------ the plan of a residue product
// How the class 0 lines run: by their bands, or joined, every line one band from its lowest exponent.  Joined lines
// need more moduli and CRT words, and save the extra rows and band pairs: on the 512-bit 512^3 product with three
// bands a line (73 moduli, nine pairs an output, against 123 moduli) 1.62 ms by bands, 0.43 ms joined.
struct Plan {
    bool joined = false;
    unsigned L = 0;
    int wx_class = 0, width = 0; // widest band: bits an entry is shifted by
    double cost = 0;
};
// Bits an exact product of band integers needs, and the CRT class that holds M (2: none compiled).
bool plan_moduli(Plan& p, int bits, int logk)
{
    int mbits = 0;
    p.L = modulus_count(2.0 * bits + 2 * p.width + logk + 2, &mbits);
    const int N = bits / 32;
    p.wx_class = !p.L ? 2 : mbits + 1 <= 32 * (lf::rebuild_words(N, 0) - 1) ? 0 : mbits + 1 <= 32 * (lf::rebuild_words(N, 1) - 1) ? 1 : 2;
    return p.wx_class < 2;
}
std::size_t digit_bytes(int N, int width) { return (std::size_t(4 * N) + (width + 7) / 8 + 31) / 32 * 32; }
// Nanoseconds of the three large stages, from their measured rates on an MI355X: 2.8 for a 32-deep step of a 128 x 128
// product tile of one modulus; 6.2e-5 for each modulus and CRT word of an output (16 multiply-adds a picosecond) and
// 0.06 for each band pair of an output that passes through the stage; 7e-4 for a residue's digits.  It only has to rank two plans of one product, which differ by their moduli and rows; memory is not
// part of it (a joined plan that does not fit gives way when its buffers are reserved).
double plan_cost(const Plan& p, int N, std::size_t rows, std::size_t cols, std::size_t lines, std::size_t K, double pairs, bool syrk)
{
    const double tr = double((rows + PT - 1) / PT), tc = double((cols + PT - 1) / PT), tiles = syrk ? tr * (tr + 1) / 2 : tr * tc;
    const double steps = double((K + 63) / 64 * 2), WX = lf::rebuild_words(N, p.wx_class);
    return 2.8 * tiles * steps * p.L + pairs * (6.2e-5 * p.L * WX + (p.joined ? 0.0 : 0.06)) + 7e-4 * double(lines) * double(K) * p.L;
}

#define GEMM_HIP(call, where)                                                                                          \
    do {                                                                                                               \
        hipError_t e_ = (call);                                                                                        \
        if (e_ != hipSuccess) return fail(LF_RUNTIME_ERROR, std::string(where) + ": " + hipGetErrorString(e_));         \
    } while (0)

typedef hipError_t (*digits_fn)(const lf::DigitsArgs&, hipStream_t);
typedef hipError_t (*round_fn)(int, const lf::RoundArgs&, hipStream_t);
typedef hipError_t (*rebuild_fn)(int, const lf::RebuildArgs&, hipStream_t);
typedef hipError_t (*dot_fn)(int, const lf::DotArgs&, hipStream_t);
typedef hipError_t (*csize_fn)(const lf::DotArgs&, uint32_t*, hipStream_t);
typedef hipError_t (*csum_fn)(const lf::DotArgs&, const uint32_t*, const uint64_t*, uint32_t*, hipStream_t);
struct GemmTables;
template <int N> void fill_gemm(GemmTables& t);
struct GemmTables {
    digits_fn digits[33] = {};
    round_fn round[33] = {};
    rebuild_fn rebuild[33] = {};
    dot_fn dot[33] = {};
    csize_fn cluster_size[33] = {};
    csum_fn cluster_sum[33] = {};
    GemmTables() { fill_gemm<2>(*this); }
};
template <int N> void fill_gemm(GemmTables& t)
{
    t.digits[N] = lf::launch_digits<N>;
    t.round[N] = lf::launch_round<N>;
    t.rebuild[N] = lf::launch_rebuild<N>;
    t.dot[N] = lf::launch_dot<N>;
    t.cluster_size[N] = lf::launch_cluster_size<N>;
    t.cluster_sum[N] = lf::launch_cluster_sum<N>;
    if constexpr (N < 32) fill_gemm<N + 1>(t);
}
const GemmTables& gemm_tables()
{
    static const GemmTables t;
    return t;
}

} // namespace

int lf::run_product(const Product& P, lf_linalg_report* rep, float* device_ms)
{
    using Clock = std::chrono::steady_clock;
    const auto since = [](Clock::time_point t) { return std::chrono::duration<double>(Clock::now() - t).count(); };
    const int N = P.bits / 32;
    if (rep) {
        std::memset(rep, 0, sizeof *rep);
        rep->m = P.m;
        rep->n = P.n;
        rep->k = P.K;
    }
    auto t0 = Clock::now();
    const bool force = P.opt.force_fallback || P.K > MAX_K || P.opt.method == 1;
    // line tables: written by the analysis on the device and into pinned host memory in one launch, completed with
    // the member lists on the host where lines are not their own extended rows
    const std::size_t nlines = P.m + (P.syrk ? 0 : P.n);
    PoolBuf dtab{0};
    GEMM_HIP(dtab.alloc(sizeof(GemmLine) * std::max<std::size_t>(nlines, 1)), "hipMalloc (lines)");
    GemmLine* htab = nullptr;
    GEMM_HIP(pinned_table(std::max<std::size_t>(nlines, 1), &htab), "hipHostMalloc (lines)");
    const GemmLine* dleft = (const GemmLine*)dtab.p;
    const GemmLine* dright = P.syrk ? dleft : dleft + P.m;
    {
        AnalyzeArgs a{};
        a.field_plane = uint32_t(N);
        a.K = uint32_t(P.K);
        a.G = P.opt.band_bits;
        a.max_bands = P.opt.max_bands;
        a.max_spread = P.opt.max_spread;
        a.force = force ? 1u : 0u;
        uint32_t blocks = 0;
        for (int k = 0; k < (P.syrk ? 1 : 2); ++k) {
            AnalyzeSide& S = a.side[k];
            S.v = k ? P.right : P.left;
            S.nlines = uint32_t(k ? P.n : P.m);
            S.blocks = (S.nlines + ANALYZE_LINES - 1) / ANALYZE_LINES;
            S.by_line = S.v.ls == 1 && S.v.ks != 1;
            S.out = (GemmLine*)dtab.p + (k ? P.m : 0);
            S.host = htab + (k ? P.m : 0);
            blocks += S.blocks;
        }
        if (blocks) {
            hipLaunchKernelGGL(analyze_kernel, dim3(blocks), dim3(ANALYZE_THREADS), 0, P.stream, a);
            GEMM_HIP(hipGetLastError(), "analysis launch");
            GEMM_HIP(hipStreamSynchronize(P.stream), "device execution (analysis)");
        }
    }
    Side ls, rs_own;
    ls.lines = htab;
    ls.count = P.m;
    read_side(ls, P.opt.max_bands);
    if (!P.syrk) {
        rs_own.lines = htab + P.m;
        rs_own.count = P.n;
        read_side(rs_own, P.opt.max_bands);
    }
    Side& rs = P.syrk ? ls : rs_own;
    const int logk = ceil_log2(P.K);
    // the band plan: modulus count from the widest band of both sides (linalg.mm:341-345)
    Plan bands;
    for (const Side* s : {&ls, &rs})
        for (std::size_t i = 0; i < s->count; ++i)
            if (s->lines[i].cls == 0)
                for (int b = 0; b < s->lines[i].nb && b < GEMM_MAX_BANDS; ++b) bands.width = std::max(bands.width, s->lines[i].hi[b] - s->lines[i].lo[b]);
    if (!plan_moduli(bands, P.bits, logk)) { // beyond the compiled CRT classes: every band line takes the exact-dot path
        for (Side* s : {&ls, &rs})
            for (std::size_t i = 0; i < s->count; ++i) {
                GemmLine& Ln = s->lines[i];
                if (Ln.cls == 0) {
                    --s->histogram[Ln.nb];
                    Ln.cls = 2;
                    ++s->fallback;
                }
            }
        bands.wx_class = 0;
    }
    route_capacity(ls, bands.wx_class);
    if (!P.syrk) route_capacity(rs, bands.wx_class);
    // lines by class and bands: extended rows, and what the outputs are
    struct Count {
        std::size_t rows = 0, lines0 = 0, single = 0, trivial = 0, dots = 0;
        int widest = 0, most = 0; // widest line, most bands
    };
    auto count_side = [](const Side& s) {
        Count c;
        for (std::size_t i = 0; i < s.count; ++i) {
            const GemmLine& Ln = s.lines[i];
            if (Ln.cls == 0) {
                ++c.lines0;
                c.rows += std::size_t(Ln.nb);
                c.single += Ln.nb == 1;
                c.widest = std::max(c.widest, Ln.top - Ln.bottom);
                c.most = std::max(c.most, Ln.nb);
            } else if (Ln.cls == 1) ++c.trivial;
            else ++c.dots;
        }
        return c;
    };
    const Count cl = count_side(ls), cr = P.syrk ? cl : count_side(rs);
    const bool any_pair = cl.lines0 && cr.lines0;
    const std::size_t rep_rows = cl.rows, rep_cols = cr.rows;
    // the plan that runs
    Plan plan = bands;
    bool single = cl.single == cl.lines0 && cr.single == cr.lines0; // every line is one band
    if (any_pair && !single) {
        Plan join;
        join.joined = true;
        join.width = std::max(cl.widest, cr.widest);
        if (plan_moduli(join, P.bits, logk) && digit_bytes(N, join.width) <= DIGIT_TABLE_BYTES) {
            const double share = P.syrk ? 0.5 : 1.0; // outputs of the lower triangle
            const double out = share * double(cl.lines0) * double(cr.lines0);
            bands.cost = plan_cost(bands, N, cl.rows, cr.rows, nlines, P.K, share * double(cl.rows) * double(cr.rows), P.syrk);
            join.cost = plan_cost(join, N, cl.lines0, cr.lines0, nlines, P.K, out, P.syrk);
            if (join.cost < bands.cost) {
                plan = join;
                single = true;
            }
        }
    }
    // extended operands: band-major member lists (linalg.mm:326-330); a side whose lines are all one band in the
    // device's table is its own list
    bool upload = false;
    auto assign_members = [&](Side& s, const Count& c) {
        if (c.lines0 == s.count && single && !(plan.joined && P.subtract)) return;
        upload = upload || s.count;
        std::size_t next = 0;
        if (plan.joined)
            for (std::size_t i = 0; i < s.count; ++i)
                if (s.lines[i].cls == 0) {
                    GemmLine& Ln = s.lines[i];
                    Ln.nb = 1;
                    Ln.lo[0] = Ln.low = Ln.bottom;
                    Ln.hi[0] = Ln.top;
                }
        for (int b = 0; b < GEMM_MAX_BANDS; ++b)
            for (std::size_t i = 0; i < s.count; ++i)
                if (s.lines[i].cls == 0 && s.lines[i].nb > b) s.lines[i].member[b] = int(next++);
    };
    if (rep) {
        rep->band_slots = uint32_t(std::min<std::size_t>(ls.histogram.size(), 65));
        for (std::size_t b = 0; b < ls.histogram.size() && b < 65; ++b) rep->left_bands[b] = ls.histogram[b];
        for (std::size_t b = 0; b < rs.histogram.size() && b < 65; ++b) rep->right_bands[b] = rs.histogram[b];
        rep->left_fallback = ls.fallback;
        rep->right_fallback = rs.fallback;
        uint32_t np = 0;
        if (any_pair)
            for (int b = 0; b < cl.most; ++b)
                for (int c = 0; c < (P.syrk ? b + 1 : cr.most) && np < 64; ++c) {
                    uint32_t rows = 0, cols = 0;
                    for (std::size_t i = 0; i < ls.count; ++i) rows += ls.lines[i].cls == 0 && ls.lines[i].nb > b;
                    for (std::size_t i = 0; i < rs.count; ++i) cols += rs.lines[i].cls == 0 && rs.lines[i].nb > c;
                    rep->pairs[np++] = {uint32_t(b), uint32_t(c), rows, cols, bands.L};
                }
        rep->npairs = np;
        rep->analysis_seconds = since(t0);
    }
    // outputs for the exact-dot kernels, by window class; the others are counted from the lines
    std::vector<uint32_t> lists[3];
    uint64_t trivial = 0, gpu_out = 0, multi = 0;
    if (cl.dots || cr.dots) {
        for (std::size_t i = 0; i < P.m; ++i)
            for (std::size_t j = 0; j < (P.syrk ? i + 1 : P.n); ++j) {
                const GemmLine &a = ls.lines[i], &b = rs.lines[j];
                if (a.cls == 1 || b.cls == 1) {
                    ++trivial;
                    continue;
                }
                if (a.cls == 0 && b.cls == 0) {
                    ++gpu_out;
                    multi += a.nb > 1 || b.nb > 1;
                    continue;
                }
                const long span = (long(a.top) + b.top) - (long(a.bottom) + b.bottom) + 64L * N + logk + 3;
                const int cls = span <= 32L * lf::dot_window_words(0) ? 0 : span <= 32L * lf::dot_window_words(1) ? 1 : 2;
                lists[cls].push_back(uint32_t(i));
                lists[cls].push_back(uint32_t(j));
            }
    } else {
        const auto pairs_of = [&](uint64_t a, uint64_t b) { return P.syrk ? a * (a + 1) / 2 : a * b; };
        gpu_out = pairs_of(cl.lines0, cr.lines0);
        multi = gpu_out - pairs_of(cl.single, cr.single);
        trivial = pairs_of(P.m, P.n) - gpu_out;
    }
    const uint64_t fallback_outputs = (lists[0].size() + lists[1].size() + lists[2].size()) / 2;
    // digits and residues of the plan that runs.  A joined plan needs more of them than the bands where few lines have
    // several; one that does not fit the device's free memory gives way to the bands.
    const std::size_t Kp = std::max<std::size_t>((std::max<std::size_t>(P.K, 1) + 63) / 64 * 64, 64);
    std::size_t Mp = 0, Np = 0; // extended rows and columns in whole product tiles
    PoolBuf dig_l1{3}, dig_l0{4}, dig_r1{5}, dig_r0{6}, dres{7}, dlist[3] = {{8}, {9}, {10}};
    const auto reserve = [&]() -> hipError_t {
        const auto tiles = [&](const Count& c) { return ((plan.joined ? c.lines0 : c.rows) + PT - 1) / PT * PT; };
        Mp = tiles(cl);
        Np = tiles(cr);
        if (!any_pair) return hipSuccess;
        if (hipError_t e = dig_l1.alloc(plan.L * Mp * Kp)) return e;
        if (hipError_t e = dig_l0.alloc(plan.L * Mp * Kp)) return e;
        if (!P.syrk) {
            if (hipError_t e = dig_r1.alloc(plan.L * Np * Kp)) return e;
            if (hipError_t e = dig_r0.alloc(plan.L * Np * Kp)) return e;
        }
        return dres.alloc(plan.L * Mp * Np * 2);
    };
    t0 = Clock::now();
    hipError_t reserved = reserve();
    if (reserved == hipErrorOutOfMemory && plan.joined) {
        (void)hipGetLastError(); // taken care of here
        for (PoolBuf* b : {&dig_l1, &dig_l0, &dig_r1, &dig_r0, &dres}) GEMM_HIP(b->release(), "hipFree (digits, residues)");
        plan = bands;
        single = false;
        reserved = reserve();
    }
    GEMM_HIP(reserved, "hipMalloc (digits, residues)");
    const unsigned L = plan.L;
    assign_members(ls, cl);
    if (!P.syrk) assign_members(rs, cr);
    if (upload) GEMM_HIP(hipMemcpyAsync(dtab.p, htab, sizeof(GemmLine) * nlines, hipMemcpyHostToDevice, P.stream), "upload lines");
    // events bounding the stages: start, digits done, products done, rebuild done, exact dots done (attached to the
    // kernels' own dispatches instead, they cost the 98 us of a small product 13 us more)
    hipEvent_t* ev = nullptr;
    GEMM_HIP(stage_events(&ev), "hipEventCreate");
    const int WX = lf::rebuild_words(N, plan.wx_class);
    const DigitTable* dt = nullptr;
    CrtSet crt{};
    if (any_pair) {
        GEMM_HIP(digit_table(&dt), "digit table");
        GEMM_HIP(crt_constants(L, WX, &crt), "CRT constants");
    }
    for (int c = 0; c < 3; ++c)
        if (!lists[c].empty()) {
            GEMM_HIP(dlist[c].alloc(lists[c].size() * 4), "hipMalloc (outputs)");
            GEMM_HIP(hipMemcpyAsync(dlist[c].p, lists[c].data(), lists[c].size() * 4, hipMemcpyHostToDevice, P.stream), "upload outputs");
        }
    if (rep) rep->upload_seconds = since(t0);
    t0 = Clock::now();
    GEMM_HIP(hipEventRecord(ev[0], P.stream), "hipEventRecord");
    if (any_pair) {
        // the digits kernel writes every byte of the lines' rows; the padding rows past them only feed residues
        // that nothing reads
        lf::DigitsArgs d{};
        d.L = L;
        d.Kp = uint32_t(Kp);
        d.K = uint32_t(P.K);
        d.joined = plan.joined;
        d.bytes = uint32_t(digit_bytes(N, plan.width));
        d.table = dt->table;
        d.offset = dt->offset[d.bytes / 32];
        d.moduli = dt->moduli;
        d.inverse = dt->inverse;
        for (int k = 0; k < (P.syrk ? 1 : 2); ++k) {
            lf::DigitsSide& S = d.side[k];
            S.v = k ? P.right : P.left;
            S.lines = k ? dright : dleft;
            S.nlines = uint32_t(k ? P.n : P.m);
            S.rows_p = uint32_t(k ? Np : Mp);
            S.d1 = (int8_t*)(k ? dig_r1.p : dig_l1.p);
            S.d0 = (int8_t*)(k ? dig_r0.p : dig_l0.p);
            S.by_line = S.v.ls == 1 && S.v.ks != 1;
            S.tk = S.by_line ? 32u : Kp >= 256 ? 256u : Kp >= 128 ? 128u : 64u;
            const uint64_t blocks = (S.nlines + 256u / S.tk - 1) / (256u / S.tk) * ((Kp + S.tk - 1) / S.tk);
            S.blocks = uint32_t(blocks);
        }
        GEMM_HIP(gemm_tables().digits[N](d, P.stream), "digits launch");
        GEMM_HIP(hipEventRecord(ev[1], P.stream), "hipEventRecord");
        lf::ProductArgs pa{};
        pa.a1 = (const int8_t*)dig_l1.p;
        pa.a0 = (const int8_t*)dig_l0.p;
        pa.b1 = (const int8_t*)(P.syrk ? dig_l1.p : dig_r1.p);
        pa.b0 = (const int8_t*)(P.syrk ? dig_l0.p : dig_r0.p);
        pa.res = (uint16_t*)dres.p;
        pa.Mp = uint32_t(Mp);
        pa.Np = uint32_t(Np);
        pa.Kp = uint32_t(Kp);
        pa.L = L;
        pa.moduli = dt->moduli;
        pa.fold = crt.fold;
        pa.lower = P.syrk;
        GEMM_HIP(lf::launch_product(pa, P.stream), "product launch");
    } else
        GEMM_HIP(hipEventRecord(ev[1], P.stream), "hipEventRecord");
    GEMM_HIP(hipEventRecord(ev[2], P.stream), "hipEventRecord");
    if (single && !P.subtract) {
        lf::RoundArgs r{};
        r.res = (const uint16_t*)dres.p;
        r.Mp = uint32_t(Mp);
        r.Np = uint32_t(Np);
        r.L = any_pair ? L : 0;
        r.crt = crt.crt;
        r.bound = crt.bound;
        r.t = crt.shift;
        r.left = dleft;
        r.right = dright;
        r.m = uint32_t(P.m);
        r.n = uint32_t(P.n);
        r.out = (uint32_t*)P.C.planes;
        r.out_pitch = P.C.pitch;
        r.out_stride = P.out_stride ? P.out_stride : P.n;
        r.syrk = P.syrk;
        r.lower_only = P.lower_only;
        GEMM_HIP(gemm_tables().round[N](plan.wx_class, r, P.stream), "rebuild launch");
    } else {
        lf::RebuildArgs r{};
        r.res = (const uint16_t*)dres.p;
        r.Mp = uint32_t(Mp);
        r.Np = uint32_t(Np);
        r.L = any_pair ? L : 0;
        r.crt = crt.crt;
        r.bound = crt.bound;
        r.t = crt.shift;
        r.left = dleft;
        r.right = dright;
        r.m = uint32_t(P.m);
        r.n = uint32_t(P.n);
        r.out = (uint32_t*)P.C.planes;
        r.out_pitch = P.C.pitch;
        r.out_stride = P.out_stride ? P.out_stride : P.n;
        r.syrk = P.syrk;
        r.lower_only = P.lower_only;
        r.subtract = P.subtract;
        // band pairs per output and the stage of the pair CRTs, in row chunks of at most 1 GiB
        r.pj = single ? 1u : std::max<uint32_t>(uint32_t(cr.most), 1);
        r.pairs = any_pair ? (single ? 1u : uint32_t(cl.most)) * r.pj : 0;
        const uint64_t per_row = uint64_t(r.pairs) * P.n * (WX + 1) * 4;
        const uint64_t chunk = per_row ? std::max<uint64_t>(1, (uint64_t(1) << 30) / per_row) : P.m;
        PoolBuf dstage{12};
        if (r.pairs) GEMM_HIP(dstage.alloc(per_row * std::min<uint64_t>(chunk, P.m)), "hipMalloc (CRT stage)");
        r.stage = (uint32_t*)dstage.p;
        for (uint64_t row0 = 0; row0 < P.m; row0 += chunk) {
            r.row0 = uint32_t(row0);
            r.rows = uint32_t(std::min<uint64_t>(chunk, P.m - row0));
            GEMM_HIP(gemm_tables().rebuild[N](plan.wx_class, r, P.stream), "rebuild launch");
        }
    }
    GEMM_HIP(hipEventRecord(ev[3], P.stream), "hipEventRecord");
    for (int c = 0; c < 3; ++c) {
        if (lists[c].empty()) continue;
        lf::DotArgs x{};
        x.left = P.left;
        x.right = P.right;
        x.lrows = dleft;
        x.rcols = dright;
        x.list = (const uint32_t*)dlist[c].p;
        x.count = uint32_t(lists[c].size() / 2);
        x.m = uint32_t(P.m);
        x.n = uint32_t(P.n);
        x.K = uint32_t(P.K);
        x.logk = uint32_t(ceil_log2(P.K + 1));
        x.out = (uint32_t*)P.C.planes;
        x.out_pitch = P.C.pitch;
        x.out_stride = P.out_stride ? P.out_stride : P.n;
        x.syrk = P.syrk;
        x.lower_only = P.lower_only;
        x.subtract = P.subtract;
        x.mirror = P.syrk && !P.lower_only;
        if (c < 2) {
            GEMM_HIP(gemm_tables().dot[N](c, x, P.stream), "exact dot launch");
            continue;
        }
        // exponent clusters: size every output's widest cluster, then sum in exactly sized scratch
        const std::size_t cnt = x.count;
        DeviceBuf dwords, doffs, dscratch;
        GEMM_HIP(dwords.alloc(cnt * 4), "hipMalloc (cluster sizes)");
        GEMM_HIP(gemm_tables().cluster_size[N](x, (uint32_t*)dwords.p, P.stream), "cluster size launch");
        std::vector<uint32_t> words(cnt);
        GEMM_HIP(hipMemcpyAsync(words.data(), dwords.p, cnt * 4, hipMemcpyDeviceToHost, P.stream), "download cluster sizes");
        GEMM_HIP(hipStreamSynchronize(P.stream), "device execution (cluster sizes)");
        // scratch in chunks of outputs within a budget (two accumulators per output)
        const uint64_t budget = uint64_t(4) << 30; // bytes
        for (std::size_t first = 0; first < cnt;) {
            std::vector<uint64_t> offs;
            uint64_t total = 0;
            std::size_t last = first;
            while (last < cnt && (last == first || (total + 2ull * words[last]) * 4 <= budget)) {
                offs.push_back(total);
                total += 2ull * words[last];
                ++last;
            }
            if (total * 4 > (uint64_t(64) << 30))
                return fail(LF_RUNTIME_ERROR, "exact dot: an exponent cluster needs more than 64 GB of accumulator");
            GEMM_HIP(doffs.alloc(offs.size() * 8), "hipMalloc (cluster offsets)");
            GEMM_HIP(dscratch.alloc(std::max<uint64_t>(total, 1) * 4), "hipMalloc (cluster scratch)");
            GEMM_HIP(hipMemcpyAsync(doffs.p, offs.data(), offs.size() * 8, hipMemcpyHostToDevice, P.stream), "upload offsets");
            lf::DotArgs y = x;
            y.list = x.list + 2 * first;
            y.count = uint32_t(last - first);
            GEMM_HIP(gemm_tables().cluster_sum[N](y, (const uint32_t*)dwords.p + first, (const uint64_t*)doffs.p, (uint32_t*)dscratch.p, P.stream),
                     "cluster sum launch");
            GEMM_HIP(hipStreamSynchronize(P.stream), "device execution (clusters)");
            first = last;
        }
    }
    if (fallback_outputs) GEMM_HIP(hipEventRecord(ev[4], P.stream), "hipEventRecord");
    GEMM_HIP(hipStreamSynchronize(P.stream), "device execution (linalg)");
    float ms = 0, stage_ms[4] = {};
    for (int q = 0; q < (fallback_outputs ? 4 : 3); ++q) {
        GEMM_HIP(hipEventElapsedTime(&stage_ms[q], ev[q], ev[q + 1]), "hipEventElapsedTime");
        ms += stage_ms[q];
    }
    if (device_ms) *device_ms = ms;
    if (rep) {
        rep->gpu_seconds = ms * 1e-3;
        rep->digits_seconds = stage_ms[0] * 1e-3;
        rep->product_seconds = stage_ms[1] * 1e-3;
        rep->rebuild_seconds = stage_ms[2] * 1e-3;
        rep->dot_seconds = stage_ms[3] * 1e-3;
        rep->gemm_rows = rep_rows;
        rep->gemm_cols = rep_cols;
        rep->moduli = any_pair ? bands.L : 0;
        rep->int8_gemms = any_pair ? 3ull * bands.L : 0;
        rep->gpu_outputs = gpu_out;
        rep->multi_band_outputs = multi;
        rep->fallback_outputs = fallback_outputs;
        rep->trivial_outputs = trivial;
        rep->crt_words = any_pair ? uint32_t(lf::rebuild_words(N, bands.wx_class)) : 0;
        rep->assembly_seconds = since(t0);
    }
    return LF_OK;
}

int lf::check_linalg_options(const lf_linalg_options* o)
{
    if (o->band_bits < 0 || o->band_bits > 1024 || o->max_bands < 0 || o->max_spread < 0 || o->max_spread > 8192)
        return fail(LF_INVALID_ARGUMENT, "linalg options: band_bits in [0,1024], max_bands >= 0, max_spread in [0,8192]");
    if (o->method < 0 || o->method > 1) return fail(LF_INVALID_ARGUMENT, "linalg options: method 0 (residue GEMM) or 1 (limb GEMM)");
    return LF_OK;
}

namespace {
using lf::check_linalg_options;

// Staging of the host-array products, kept per host thread and device and grown on demand, so repeated
// calls allocate nothing after the first: a stream and the device AoS / limb-plane buffers (planner pool
// slots); the host arrays pass through host_copy's pinned chunk ring.
struct HostStage {
    int device = -1;
    hipStream_t stream = nullptr;
    ~HostStage()
    {
        if (stream) (void)hipStreamDestroy(stream);
    }
    hipError_t ready()
    {
        if (!stream)
            if (hipError_t e = hipStreamCreateWithFlags(&stream, hipStreamNonBlocking)) return e;
        return hipSuccess;
    }
};
HostStage& host_stage()
{
    thread_local std::map<int, HostStage> stages;
    int device = 0;
    (void)hipGetDevice(&device);
    return stages[device];
}

} // namespace

extern "C" {

void lf_linalg_default_options(lf_linalg_options* o)
{
    if (!o) return;
    std::memset(o, 0, sizeof *o);
    o->band_bits = 64;
    o->max_bands = 4;
    o->max_spread = 512;
    o->resident_bands = 2;
}

int lf_gemm_host(int bits, int transpose_a, const void* A, const void* B, uint64_t m, uint64_t n, uint64_t k, void* C, int subtract,
                 const lf_linalg_options* options, lf_linalg_report* report, double* gpu_seconds, double* wall_seconds)
{
    const auto start = std::chrono::steady_clock::now();
    if (gpu_seconds) *gpu_seconds = 0;
    if (wall_seconds) *wall_seconds = 0;
    lf_linalg_options o;
    if (options) o = *options;
    else lf_linalg_default_options(&o);
    if (int r = check_linalg_options(&o)) return r;
    if (bits < 64 || bits > 1024 || bits % 32) return fail(LF_INVALID_ARGUMENT, "bits must be a multiple of 32 in [64,1024]");
    const uint64_t limit = uint64_t(1) << 31;
    if (m >= limit || n >= limit || k >= limit || m * n >= limit || m * k >= limit || k * n >= limit)
        return fail(LF_INVALID_ARGUMENT, "matrix dimensions exceed 32-bit indexing");
    if (m && n && !C) return fail(LF_INVALID_ARGUMENT, "null output");
    if (m * n && k && (!A || !B)) return fail(LF_INVALID_ARGUMENT, "null input");
    if (report) {
        std::memset(report, 0, sizeof *report);
        report->m = m;
        report->n = n;
        report->k = k;
    }
    if (!m || !n) return LF_OK;
    const int N = bits / 32;
    const std::size_t E = bits / 8 + 12;
    HostStage& st = host_stage();
    GEMM_HIP(st.ready(), "hipStreamCreate");
    const std::size_t na = m * k, nb = k * n, nc = m * n;
    // AoS staging of all three operands on the device (the uploads run back to back), then their planes
    PoolBuf aos{13}, pa{14}, pb{15}, pc{16};
    GEMM_HIP(aos.alloc((na + nb + nc) * E), "hipMalloc (staging)");
    GEMM_HIP(pa.alloc(lf_planes_bytes(bits, 0, std::max<uint64_t>(na, 1))), "hipMalloc (A)");
    GEMM_HIP(pb.alloc(lf_planes_bytes(bits, 0, std::max<uint64_t>(nb, 1))), "hipMalloc (B)");
    GEMM_HIP(pc.alloc(lf_planes_bytes(bits, 0, nc)), "hipMalloc (C)");
    char* daos = static_cast<char*>(aos.p);
    lf_operand OA{pa.p, lf_plane_pitch(std::max<uint64_t>(na, 1))}, OB{pb.p, lf_plane_pitch(std::max<uint64_t>(nb, 1))},
        OC{pc.p, lf_plane_pitch(nc)};
    if (na) {
        GEMM_HIP(lf::copy_to_device(daos, A, na * E, st.stream), "upload A");
        if (int r = lf_aos_to_planes(bits, 0, daos, &OA, na, st.stream)) return r;
    }
    if (nb) {
        GEMM_HIP(lf::copy_to_device(daos + na * E, B, nb * E, st.stream), "upload B");
        if (int r = lf_aos_to_planes(bits, 0, daos + na * E, &OB, nb, st.stream)) return r;
    }
    if (subtract) {
        GEMM_HIP(lf::copy_to_device(daos + (na + nb) * E, C, nc * E, st.stream), "upload C");
        if (int r = lf_aos_to_planes(bits, 0, daos + (na + nb) * E, &OC, nc, st.stream)) return r;
    }
    Product P{};
    P.bits = bits;
    P.syrk = false;
    P.lower_only = false;
    P.subtract = subtract != 0;
    // op(A) row i, entry k: A[i*k + kk] or (transpose) A[kk*m + i]; B column j, entry kk: B[kk*n + j]
    P.left = {(const uint32_t*)OA.planes, OA.pitch, transpose_a ? 1 : k, transpose_a ? m : 1};
    P.right = {(const uint32_t*)OB.planes, OB.pitch, 1, n};
    P.m = m;
    P.n = n;
    P.K = k;
    P.C = OC;
    P.opt = o;
    P.stream = st.stream;
    float ms = 0;
    if (int r = run_product(P, report, &ms)) return r;
    if (int r = lf_planes_to_aos(bits, 0, &OC, daos, nc, st.stream)) return r;
    GEMM_HIP(lf::copy_to_host(C, daos, nc * E, st.stream), "download C");
    if (gpu_seconds) *gpu_seconds = ms * 1e-3;
    if (wall_seconds) *wall_seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - start).count();
    return LF_OK;
}

// ---- products on device operands (resident products) ----
namespace {
int check_product_planes(const lf_operand* o, uint64_t elements, const char* name)
{
    if (!elements) return LF_OK;
    if (!o || !o->planes) return fail(LF_INVALID_ARGUMENT, std::string("null operand ") + name);
    if (o->pitch < elements) return fail(LF_INVALID_ARGUMENT, std::string("operand ") + name + " pitch is smaller than its element count");
    return LF_OK;
}
bool overlaps(int N, const lf_operand& a, const lf_operand& b)
{
    const uintptr_t a0 = (uintptr_t)a.planes, a1 = a0 + (uintptr_t)(N + 3) * a.pitch * 4;
    const uintptr_t b0 = (uintptr_t)b.planes, b1 = b0 + (uintptr_t)(N + 3) * b.pitch * 4;
    return a0 < b1 && b0 < a1;
}
} // namespace

int lf_gemm(int bits, int transpose_a, const lf_operand* A, const lf_operand* B, uint64_t m, uint64_t n, uint64_t k, const lf_operand* C,
            int subtract, const lf_linalg_options* options, lf_linalg_report* report, double* gpu_seconds, void* stream)
{
    if (gpu_seconds) *gpu_seconds = 0;
    lf_linalg_options o;
    if (options) o = *options;
    else lf_linalg_default_options(&o);
    if (int r = check_linalg_options(&o)) return r;
    if (bits < 64 || bits > 1024 || bits % 32) return fail(LF_INVALID_ARGUMENT, "bits must be a multiple of 32 in [64,1024]");
    const uint64_t limit = uint64_t(1) << 31;
    if (m >= limit || n >= limit || k >= limit || m * n >= limit || m * k >= limit || k * n >= limit)
        return fail(LF_INVALID_ARGUMENT, "matrix dimensions exceed 32-bit indexing");
    if (report) {
        std::memset(report, 0, sizeof *report);
        report->m = m;
        report->n = n;
        report->k = k;
    }
    if (!m || !n) return LF_OK;
    if (int r = check_product_planes(C, m * n, "C")) return r;
    if (k) {
        if (int r = check_product_planes(A, m * k, "A")) return r;
        if (int r = check_product_planes(B, k * n, "B")) return r;
        if (overlaps(bits / 32, *C, *A) || overlaps(bits / 32, *C, *B)) return fail(LF_INVALID_ARGUMENT, "gemm: C must not overlap A or B");
    }
    Product P{};
    P.bits = bits;
    P.subtract = subtract != 0;
    const uint32_t* a = k ? (const uint32_t*)A->planes : (const uint32_t*)C->planes;
    const uint32_t* b = k ? (const uint32_t*)B->planes : (const uint32_t*)C->planes;
    P.left = {a, k ? A->pitch : C->pitch, transpose_a ? 1 : k, transpose_a ? m : 1};
    P.right = {b, k ? B->pitch : C->pitch, 1, n};
    P.m = m;
    P.n = n;
    P.K = k;
    P.C = *C;
    P.opt = o;
    P.stream = (hipStream_t)stream;
    float ms = 0;
    if (int r = run_product(P, report, &ms)) return r;
    if (gpu_seconds) *gpu_seconds = ms * 1e-3;
    return LF_OK;
}

int lf_syrk(int bits, const lf_operand* A, uint64_t rows, uint64_t cols, const lf_operand* C, int lower_only, int subtract,
            const lf_linalg_options* options, lf_linalg_report* report, double* gpu_seconds, void* stream)
{
    if (gpu_seconds) *gpu_seconds = 0;
    lf_linalg_options o;
    if (options) o = *options;
    else lf_linalg_default_options(&o);
    if (int r = check_linalg_options(&o)) return r;
    if (bits < 64 || bits > 1024 || bits % 32) return fail(LF_INVALID_ARGUMENT, "bits must be a multiple of 32 in [64,1024]");
    if (subtract && !lower_only) return fail(LF_INVALID_ARGUMENT, "syrk: subtract updates the lower triangle only (lower_only)");
    const uint64_t limit = uint64_t(1) << 31;
    if (rows >= limit || cols >= limit || cols * cols >= limit || rows * cols >= limit)
        return fail(LF_INVALID_ARGUMENT, "matrix dimensions exceed 32-bit indexing");
    if (report) {
        std::memset(report, 0, sizeof *report);
        report->m = cols;
        report->n = cols;
        report->k = rows;
    }
    if (!cols) return LF_OK;
    if (int r = check_product_planes(C, cols * cols, "C")) return r;
    if (rows) {
        if (int r = check_product_planes(A, rows * cols, "A")) return r;
        if (overlaps(bits / 32, *C, *A)) return fail(LF_INVALID_ARGUMENT, "syrk: C must not overlap A");
    }
    Product P{};
    P.bits = bits;
    P.syrk = true;
    P.lower_only = lower_only != 0;
    P.subtract = subtract != 0;
    P.left = {rows ? (const uint32_t*)A->planes : (const uint32_t*)C->planes, rows ? A->pitch : C->pitch, 1, cols};
    P.right = P.left;
    P.m = cols;
    P.n = cols;
    P.K = rows;
    P.C = *C;
    P.opt = o;
    P.stream = (hipStream_t)stream;
    float ms = 0;
    if (int r = run_product(P, report, &ms)) return r;
    if (gpu_seconds) *gpu_seconds = ms * 1e-3;
    return LF_OK;
}

int lf_syrk_host(int bits, const void* A, uint64_t rows, uint64_t cols, void* C, int lower_only, int subtract,
                 const lf_linalg_options* options, lf_linalg_report* report, double* gpu_seconds, double* wall_seconds)
{
    const auto start = std::chrono::steady_clock::now();
    if (gpu_seconds) *gpu_seconds = 0;
    if (wall_seconds) *wall_seconds = 0;
    lf_linalg_options o;
    if (options) o = *options;
    else lf_linalg_default_options(&o);
    if (int r = check_linalg_options(&o)) return r;
    if (bits < 64 || bits > 1024 || bits % 32) return fail(LF_INVALID_ARGUMENT, "bits must be a multiple of 32 in [64,1024]");
    if (subtract && !lower_only) return fail(LF_INVALID_ARGUMENT, "syrk: subtract updates the lower triangle only (lower_only)");
    const uint64_t limit = uint64_t(1) << 31;
    if (rows >= limit || cols >= limit || cols * cols >= limit || rows * cols >= limit)
        return fail(LF_INVALID_ARGUMENT, "matrix dimensions exceed 32-bit indexing");
    if (cols && !C) return fail(LF_INVALID_ARGUMENT, "null output");
    if (cols && rows && !A) return fail(LF_INVALID_ARGUMENT, "null input");
    if (report) {
        std::memset(report, 0, sizeof *report);
        report->m = cols;
        report->n = cols;
        report->k = rows;
    }
    if (!cols) return LF_OK;
    const int N = bits / 32;
    const std::size_t E = bits / 8 + 12;
    HostStage& st = host_stage();
    GEMM_HIP(st.ready(), "hipStreamCreate");
    const std::size_t na = rows * cols, nc = cols * cols;
    PoolBuf aos{13}, pa{14}, pc{16};
    GEMM_HIP(aos.alloc((na + nc) * E), "hipMalloc (staging)");
    GEMM_HIP(pa.alloc(lf_planes_bytes(bits, 0, std::max<uint64_t>(na, 1))), "hipMalloc (A)");
    GEMM_HIP(pc.alloc(lf_planes_bytes(bits, 0, nc)), "hipMalloc (C)");
    char* daos = static_cast<char*>(aos.p);
    lf_operand OA{pa.p, lf_plane_pitch(std::max<uint64_t>(na, 1))}, OC{pc.p, lf_plane_pitch(nc)};
    if (na) {
        GEMM_HIP(lf::copy_to_device(daos, A, na * E, st.stream), "upload A");
        if (int r = lf_aos_to_planes(bits, 0, daos, &OA, na, st.stream)) return r;
    }
    if (subtract || lower_only) { // untouched entries keep their old values
        GEMM_HIP(lf::copy_to_device(daos + na * E, C, nc * E, st.stream), "upload C");
        if (int r = lf_aos_to_planes(bits, 0, daos + na * E, &OC, nc, st.stream)) return r;
    }
    Product P{};
    P.bits = bits;
    P.syrk = true;
    P.lower_only = lower_only != 0;
    P.subtract = subtract != 0;
    // line i = column i of A: element (i, kk) = A[kk*cols + i]
    P.left = {(const uint32_t*)OA.planes, OA.pitch, 1, cols};
    P.right = P.left;
    P.m = cols;
    P.n = cols;
    P.K = rows;
    P.C = OC;
    P.opt = o;
    P.stream = st.stream;
    float ms = 0;
    if (int r = run_product(P, report, &ms)) return r;
    if (int r = lf_planes_to_aos(bits, 0, &OC, daos, nc, st.stream)) return r;
    GEMM_HIP(lf::copy_to_host(C, daos, nc * E, st.stream), "download C");
    if (gpu_seconds) *gpu_seconds = ms * 1e-3;
    if (wall_seconds) *wall_seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - start).count();
    return LF_OK;
}

} // extern "C"
