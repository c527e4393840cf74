// factor_update.hpp — off-block updates c_ic = D(c_ic; x_i, y_c; K) of the factorization and the solves, 64
// entries a workgroup.
#pragma once
#include "factor_wave.hpp"

namespace lf {

// Tiles of rows x columns entries, at most UPD_ENTRIES of them from at most UPD_LINES lines (rows and columns
// together) of at most 32 terms.
constexpr u32 UPD_ENTRIES = 64, UPD_LINES = 17, UPD_WAVES = 8;
template <int N> struct UpdLds {
    i64 acc[UPD_ENTRIES][WD_COLS + 1];
    int digit[wd_grid<N>()][WD_ROWS * UPD_LINES]; // number (line, k) at k * UPD_LINES + line
    int origin[WD_ROWS * UPD_LINES];
    int top[UPD_ENTRIES], low[UPD_ENTRIES]; // largest and smallest origin of an entry's terms
    u32 status[UPD_LINES];                  // statuses of a line's numbers
};

// The tile's columns (up to 8) and rows: what is left of the lines and the entries.
__host__ __device__ __forceinline__ u32 upd_cols(u32 cols) { return cols < 8u ? cols : 8u; }
__host__ __device__ __forceinline__ u32 upd_rows(u32 tc) { return UPD_LINES - tc < UPD_ENTRIES / tc ? UPD_LINES - tc : UPD_ENTRIES / tc; }

// One workgroup of eight wavefronts a tile.  The lines' terms are turned into signed grid digits once; every
// entry's accumulator is placed under its largest term; then each lane adds the products of one entry, two
// wavefronts to a term (half of the row's digits each) and four terms at a time; and the accumulators are
// rounded a digit a lane, eight a wavefront.  A term costs its lane about 150 instructions and an entry's
// rounding 120 instructions of a wavefront, where one wavefront per entry (an exact dot of 32 terms) took
// about 1,500: at 256 bits 62 us for 15,360 entries, 18 us here, and 52 against 24 us for the updates of a solve with
// 64 right-hand sides.  Entries whose terms spread past the columns (seen from their smallest and largest origins,
// before anything is added) take the exact dot; those with a status and those without a term need none.
// The exact dot sets the registers: with four wavefronts a SIMD it spills 46 of 128 at 320 bits and 143 at 512, which
// all entries paid for (22.9 against 20.1 us at 320 bits, 36.5 against 27.6 at 512, 197 against 96 where every entry
// takes the exact dot).  At 256 bits, with 16, four are better than two (23.4 against 26.2 us).
template <int N> __global__ void __launch_bounds__(64 * UPD_WAVES, N <= 8 ? 4 : 2) update_wave_kernel(UpdateArgs g)
{
    constexpr int GD = wd_grid<N>(), H = (GD + 1) / 2;
    constexpr std::size_t bytes = sizeof(UpdLds<N>) > UPD_WAVES * sizeof(WaveLds<N>) ? sizeof(UpdLds<N>) : UPD_WAVES * sizeof(WaveLds<N>);
    __shared__ __attribute__((aligned(16))) unsigned char lds[bytes];
    UpdLds<N>& L = *reinterpret_cast<UpdLds<N>*>(lds);
    const u32 t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t / 64u), lane = t % 64u;
    const u32 tc = upd_cols(g.cols), tr = upd_rows(tc), tiles_c = (g.cols + tc - 1) / tc, tiles = ((g.rows + tr - 1) / tr) * tiles_c;
    const DotScratch sc{g.scratch + (u64)(blockIdx.x * UPD_WAVES + wave) * 2 * g.swords, g.swords, g.error};
    for (u32 tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const u32 r0 = (tile / tiles_c) * tr, c0 = (tile % tiles_c) * tc;
        const u32 rows = min(tr, g.rows - r0), cols = min(tc, g.cols - c0);
        if (g.lower && c0 > r0 + rows - 1) continue;
        __syncthreads(); // the tile before is done with the LDS
        if (t < UPD_LINES) L.status[t] = 0;
        if (t < UPD_ENTRIES) {
            L.top[t] = -WD_ZERO;
            L.low[t] = WD_ZERO;
        }
        for (u32 e = t; e < UPD_ENTRIES * (WD_COLS + 1); e += 64u * UPD_WAVES) (&L.acc[0][0])[e] = 0;
        __syncthreads();
        const u32 lines = rows + cols;
        for (u32 e = t; e < lines * g.K; e += 64u * UPD_WAVES) {
            const u32 line = e / g.K, k = e - line * g.K;
            const bool isrow = line < rows;
            const Num<N> a = isrow ? load_out<N>(g.x, g.xpitch, (u64)(g.xbase + (i64)(r0 + line) * g.xr + (i64)k * g.xk))
                                   : load_out<N>(g.y, g.ypitch, (u64)(g.ybase + (i64)(c0 + line - rows) * g.yc + (i64)k * g.yk));
            if (a.st) atomicOr(&L.status[line], a.st);
            int d[GD], o;
            lane_to_grid<N>(a, d, o);
            const bool neg = (a.s < 0) != isrow; // the products are subtracted
            const u32 at = k * UPD_LINES + line;
#pragma unroll
            for (int j = 0; j < GD; ++j) L.digit[j][at] = neg ? -d[j] : d[j];
            L.origin[at] = a.s ? o : WD_ZERO;
        }
        __syncthreads();
        // lane = entry
        const u32 er = lane / tc, ec = lane - er * tc;
        const bool live = er < rows && ec < cols && !(g.lower && c0 + ec > r0 + er);
        const u32 lr = live ? er : 0u, lc = rows + (live ? ec : 0u);
        {
            int hi = -WD_ZERO, lo = WD_ZERO;
            for (u32 k = wave; k < g.K; k += UPD_WAVES) {
                const int ox = L.origin[k * UPD_LINES + lr], oy = L.origin[k * UPD_LINES + lc];
                if (ox == WD_ZERO || oy == WD_ZERO) continue;
                hi = max(hi, ox + oy);
                lo = min(lo, ox + oy);
            }
            if (live && hi != -WD_ZERO) {
                atomicMax(&L.top[lane], hi);
                atomicMin(&L.low[lane], lo);
            }
        }
        const u64 out = live ? (u64)(g.obase + (i64)(r0 + er) * g.orow + (i64)(c0 + ec) * g.ocol) : 0;
        Num<N> c = zero<N>(ST_OK);
        if (live) c = load_out<N>(g.out, g.opitch, out);
        int cd[GD], co;
        lane_to_grid<N>(c, cd, co);
        __syncthreads();
        // an entry with a status is zero with all of them, one without a nonzero product stays as it is
        const u32 st = live ? L.status[lr] | L.status[lc] | c.st : 0u;
        constexpr u32 OWN = UPD_ENTRIES / UPD_WAVES;
        if (st && lane / OWN == wave) store_out<N>(g.out, g.opitch, 0, 0, (u32)out, false, zero<N>(st));
        const bool sum = live && !st && L.top[lane] != -WD_ZERO;
        int top = L.top[lane] + 2 * GD - 1;
        if (c.s) top = max(top, co + GD - 1);
        const int alpha = top - (WD_TOP - 1);
        const bool fits = sum && L.low[lane] >= alpha && (!c.s || co >= alpha);
        if (fits && c.s && wave == 0)
#pragma unroll
            for (int j = 0; j < GD; ++j) lds_add(&L.acc[lane][co - alpha + j], c.s < 0 ? -(i64)cd[j] : (i64)cd[j]);
        const u32 half = wave & 1u;
        for (u32 k = wave >> 1; k < g.K; k += UPD_WAVES / 2) {
            const u32 ax = k * UPD_LINES + lr, ay = k * UPD_LINES + lc;
            const int ox = L.origin[ax], oy = L.origin[ay];
            if (!fits || ox == WD_ZERO || oy == WD_ZERO) continue;
            const int o = ox + oy - alpha;
            int xd[H], yd[GD];
#pragma unroll
            for (int q = 0; q < H; ++q) {
                const int d = q + H * (int)half;
                xd[q] = d < GD ? L.digit[d < GD ? d : 0][ax] : 0;
            }
#pragma unroll
            for (int q = 0; q < GD; ++q) yd[q] = L.digit[q][ay];
            wd_accumulate<GD, H>(&L.acc[lane][o + H * (int)half], xd, yd);
        }
        __syncthreads();
        const u64 good = __ballot(fits);
        u64 rest = __ballot(sum) & ((((u64)1 << OWN) - 1u) << (OWN * wave)); // this wavefront's entries
        for (u64 todo = rest & good; todo; todo &= todo - 1) {
            const int e = (int)__builtin_ctzll(todo);
            WaveNum v;
            if (!wd_round<N>(L.acc[e][lane], (i64)(int)wd_read((u32)alpha, e), lane, v)) continue;
            const u64 at = (u64)wd_read((u32)out, e) | ((u64)wd_read((u32)(out >> 32), e) << 32);
            wd_store<N>(g.out, g.opitch, at, v, lane);
            rest &= ~((u64)1 << e);
        }
        __syncthreads(); // the accumulators' LDS becomes the exact dot's
        for (; rest; rest &= rest - 1) {
            const u32 e = (u32)__builtin_ctzll(rest), i = r0 + e / tc, j = c0 + e % tc;
            const VecView x{g.x, g.xpitch, g.xbase + (i64)i * g.xr, g.xk}, y{g.y, g.ypitch, g.ybase + (i64)j * g.yc, g.yk};
            const u64 at = (u64)(g.obase + (i64)i * g.orow + (i64)j * g.ocol);
            const Num<N> v = wave_dot_sub<N, true>(load_out<N>(g.out, g.opitch, at), x, y, g.K, lane, reinterpret_cast<WaveLds<N>*>(lds)[wave].rows(), sc);
            if (lane == 0) store_out<N>(g.out, g.opitch, 0, 0, (u32)at, false, v);
        }
    }
}

// The same updates one wavefront per entry (wider values and longer dots), grid-stride; wavefront b uses
// scratch slot b.
template <int N> __global__ void __launch_bounds__(64) update_kernel(UpdateArgs g)
{
    __shared__ WaveLds<N> lds;
    const DotRows<N> L = lds.rows();
    const u32 lane = threadIdx.x;
    const u64 entries = (u64)g.rows * g.cols;
    const DotScratch sc{g.scratch + (u64)blockIdx.x * 2 * g.swords, g.swords, g.error};
    for (u64 e = blockIdx.x; e < entries; e += gridDim.x) {
        const u32 i = (u32)(e / g.cols), j = (u32)(e % g.cols);
        if (g.lower && j > i) continue; // the whole wavefront skips the strict upper part
        const VecView x{g.x, g.xpitch, g.xbase + (i64)i * g.xr, g.xk}, y{g.y, g.ypitch, g.ybase + (i64)j * g.yc, g.yk};
        const u64 at = (u64)(g.obase + (i64)i * g.orow + (i64)j * g.ocol);
        const Num<N> v = wave_dot_sub<N>(load_out<N>(g.out, g.opitch, at), x, y, g.K, lane, L, sc);
        if (lane == 0) store_out<N>(g.out, g.opitch, 0, 0, (u32)at, false, v);
    }
}

} // namespace lf
