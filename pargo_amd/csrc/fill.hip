// fill.hip -- depression filling (pitremove) on the device.
//
// The reference (apps/hydrology/pitremove/pitRemoveOperator.cpp:26-72, run
// by RasterOperator::Work, gpro/rasterOperator.h:170-216) starts from
// W = 10000 on valid cells and NoData elsewhere (the border too, through
// copyLayerInfo) and sweeps the interior in row-major order until a sweep
// assigns nothing.  A valid cell with W > dem looks at its 3x3 window:
//   if dem >= W(n) + 0.0005 or W(n) is NoData for some n:  W = dem
//   otherwise                                              W = min(W, min_n W(n) + 0.0005)
// (the window loop never breaks, and once W = dem no later neighbour
// changes it again).
//
// That update is monotone in the neighbours' values as long as no valid
// cell's W can come within 1e-6 of NoData (W stays in [min(dem, 10000),
// 10000]; pargo_pit_remove checks this and refuses other inputs).  The
// reference's loop then ends at the greatest fixed point below the start,
// and so does any order of the same updates: every update reads values that
// are >= that fixed point, and a state in which no update changes anything
// is a fixed point.  The result is therefore bit-identical to the
// reference's while the order is free.
//
// A NoData or border neighbour sends a cell to its own elevation, and that is
// the least value the cell can take, so the init kernel writes it (at most
// 10000) into W at once.  For every other cell, and with NoData read as
// +infinity, the update is
//   W = min(W, max(dem, min_n W(n) + 0.0005))
// (if dem >= some W(n) + gap it is dem, as above; the rounded addition is
// monotone, so min_n RN(W(n) + gap) = RN(min_n W(n) + gap)); taking the cell
// itself into min_n changes nothing, since W + gap >= W.
//
// Device order: 64 x 32 tiles, one workgroup of four waves each (two for
// large rasters), a wave holding 8 (16) rows in registers, one column per
// lane.  With h(r) the minimum
// of a row's W over each column and its two neighbours (two DPP moves), an
// update of row r is two minima over h(r-1), h(r), h(r+1), one addition, a
// maximum and a compare; h(r) is formed again only when the row changed.
// Only rows whose inputs changed are evaluated: a bit per row (a scalar)
// says so, set by a change of the row itself or of a row next to it.  The
// waves exchange the h of their first and last rows through LDS.  When no
// row of the tile is left, the changed rows are written back (with copies
// of the tile's first and last columns, which the tiles beside it read as
// their halo columns), and the tiles across each changed edge or corner are
// scheduled for the next pass with flags that say which edge (and for side
// edges which waves' rows) changed; only the waves next to such a
// change start with rows to evaluate, and the others load nothing unless
// the change reaches them.  Passes repeat until none is scheduled.  Tiles
// read each other's edges while they change; that only feeds the monotone
// iteration earlier values, never wrong ones, and a change made during a
// pass schedules its neighbours for the next one.
//
// Only scheduled tiles run: a pass's workgroups walk a device worklist with
// a fixed stride, and a tile enters the next pass's list with its first
// flag.  Pass 0's list holds the tiles with a cell in or around them that
// the init kernel opened: with every valid W at 10000, nothing else can
// change.
//
// Measured at 16384^2 on the synthetic DEM: 6.1 ms (19.3 ms with nine-cell
// windows swept over whole tiles, two launches per pass): 0.60 ms init and
// 5.5 ms in 35 to 40 passes, 534,000 visits of which 54 % change an edge,
// 2.5 rounds a visit.  A visit that changes nothing reads 26 KB at 5.1 TB/s
// (0.67 ms for all 131,072 tiles), 2.2 ms of the passes; the rest is the
// evaluations, the rows written (4.8 GB) and the 15-20 us a pass of few tiles
// takes.  Measured with four waves a tile (6.8 to 7.2 ms): occupancy (4 to 6
// waves per SIMD) and a tiled layout of W changed nothing, 16- and 64-row
// tiles lost (11.2 and 8.9 ms), and putting a visit off when a neighbour has
// changed during the pass saved no visits.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "internal.h"

namespace pargo {

namespace {

constexpr int kTW = 64, kTH = 32;  // tile: 64 columns x 32 rows
static_assert(kTW == 64, "a lane is a column of the tile");
// From this many tiles on, a tile is held by two waves of 16 rows instead of
// four of 8 (eight waves of 4 rows took 12.4 ms at 16384^2, four 6.8, two
// 6.1).  As many visits, but a change crosses fewer bands: 2.5 rounds a visit
// instead of 3.4, with them 1.08 G VALU instructions instead of 1.43 and
// 0.75 G scalar ones instead of 1.33, and of the wave cycles (6.7 G instead
// of 12.9) 51 % wait instead of 60.  A wave's chain of rows is longer, though,
// which a raster that does not fill the GPU many times over waits for.  us,
// four waves / two: 1000^2 (512 tiles) 438 / 484, 2048^2 678 / 734,
// 3000 x 4000 (5,922) 1014 / 1057, 5003 x 7001 (17,270) 1785 / 1735,
// 8192^2 2827 / 2610, 16384^2 6989 / 6173.
constexpr int kTallTiles = 16384;
constexpr double kGap = 0.0005;    // pitRemoveOperator.cpp:36
constexpr double kStart = 10000.0; // pitRemoveOperator.cpp:41

// What changed around a tile since it was last settled.
constexpr unsigned kLeft = 1u, kRight = 1u << 4;  // halo column, one bit per wave's band of rows (at most 4)
constexpr unsigned kTop = 1u << 8, kBottom = 1u << 9;
constexpr unsigned kTopLeft = 1u << 10, kTopRight = 1u << 11, kBottomLeft = 1u << 12, kBottomRight = 1u << 13;
constexpr unsigned kAll = 1u << 15;  // never visited: every row is to be evaluated

// A worklist is kSub lists, a tile's by its number modulo kSub, each with a
// counter in a cache line of its own: returning atomics on one address take
// turns (577,000 of them, from a cursor over the list, added 6.4 ms at
// 16384^2, 11 ns each).  With one counter per list the passes took 7.09 ms
// with their init against 6.85, the init 0.89 against 0.62.
constexpr int kSub = 64, kSubStride = 32;  // stride in 4-byte words
constexpr int kSetWords = kSub * kSubStride;

struct FillParams {
    const float *__restrict__ dem;
    double *__restrict__ w;
    unsigned *__restrict__ flags;    // [2][tiles]: what the tile's next visit starts from (even, odd passes)
    unsigned *__restrict__ count;    // [3][kSub]: entries of the worklists (kSubStride apart), pass p's in set p % 3
    unsigned *__restrict__ ran;      // passes that had tiles on their list
    int *__restrict__ list;          // [2][kSub][sub_cap]: tiles of the pass (even, odd)
    double *__restrict__ edge;       // [tiles][2][kTH]: W of each tile's first and last column, NoData as +infinity
    unsigned *__restrict__ range;    // [0] smallest valid elevation (ordered bits), [1] NaN cells
    long long pitch;
    int rows, cols, tiles_x, tiles_y, sub_cap;
    float nd_lo, nd_hi;  // float32 values with fabs((double)v - nodata) <= 1e-6
    int opens;           // a NoData neighbour opens a cell (not with NoData +infinity, which tests unequal to itself)
    double nodata;
};

// The least filled value there can be, min(smallest valid elevation, 10000),
// from the range word; NaN when no cell is valid.
__host__ __device__ inline double lowest_filled(unsigned key)
{
    const unsigned u = (key & 0x80000000u) ? (key & 0x7fffffffu) : ~key;
    float mn;
    __builtin_memcpy(&mn, &u, sizeof(mn));
    return mn < kStart ? (double)mn : (mn != mn ? (double)mn : kStart);
}

// Whether the DEM is refused: NaN cells, or a NoData value that a filled one
// can come within 1e-6 of (every valid W lies in [min(dem, 10000), 10000]).
__host__ __device__ inline bool fill_refused(unsigned key, unsigned nans, double nodata)
{
    const double lo = lowest_filled(key);
    return nans != 0 || (lo == lo && !(nodata < lo - 0.000001 || nodata > kStart + 0.000001));
}

__device__ __forceinline__ bool is_nd(const FillParams &p, float v) { return v >= p.nd_lo && v <= p.nd_hi; }

// FP64 minimum and maximum without the quieting the compiler puts in front
// of fmin/fmax for operands it cannot prove canonical (a DEM that holds NaN
// is refused, so which operand a NaN selects does not matter).
__device__ __forceinline__ double vmin(double a, double b)
{
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ double vmax(double a, double b)
{
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// Lane i gets lane i-1's (from_left) or lane i+1's (from_right) v; the lane
// without a source (0, resp. 63) gets `edge`.  Two 32-bit DPP wave shifts.
__device__ __forceinline__ double dpp_from_left(double v, double edge)
{
    const long long b = __double_as_longlong(v), e = __double_as_longlong(edge);
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp((int)(unsigned)e, (int)(unsigned)b, 0x138, 0xf, 0xf, false);
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp((int)(e >> 32), (int)(b >> 32), 0x138, 0xf, 0xf, false);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ double dpp_from_right(double v, double edge)
{
    const long long b = __double_as_longlong(v), e = __double_as_longlong(edge);
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp((int)(unsigned)e, (int)(unsigned)b, 0x130, 0xf, 0xf, false);
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp((int)(e >> 32), (int)(b >> 32), 0x130, 0xf, 0xf, false);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Each tile's first and last column of W, also kept contiguously per tile:
// a tile's halo columns are its neighbours' edge columns, read as two short
// runs instead of one extra cache line per halo row on each side.
__device__ __forceinline__ long long edge_index(const FillParams &p, int ty, int tx, int right, int row_in_tile)
{
    return (((long long)ty * p.tiles_x + tx) * 2 + right) * kTH + row_in_tile;
}

// Sets flags of tile t for pass `pass`; 0 for the first ones, with which the
// caller appends the tile to that pass's list.
__device__ __forceinline__ unsigned flag_tile(const FillParams &p, int t, unsigned f, int pass)
{
    return atomicOr(&p.flags[(long long)(pass & 1) * p.tiles_x * p.tiles_y + t], f);
}
__device__ __forceinline__ void append_tile(const FillParams &p, int t, int pass)
{
    const int sub = t % kSub;
    const unsigned k = atomicAdd(&p.count[(pass % 3) * kSetWords + sub * kSubStride], 1u);
    p.list[((long long)(pass & 1) * kSub + sub) * p.sub_cap + k] = t;
}

// W before the first sweep (pitRemoveOperator.cpp:39-45 plus copyLayerInfo,
// with the cells next to NoData or the border at their own elevation), pass
// 0's worklist, and the smallest valid elevation and the NaN count for the
// monotonicity check.  One wave per tile, walking its rows: which cells of a
// row are excluded is one 64-bit mask, widened by a column on either side
// (the columns beside the tile are read by lanes 0 and 63) and merged with
// the rows above and below.  At 16384^2 it replaces an init pass of 0.75 ms
// and a range pass of 0.33 ms that read the DEM once more.
constexpr int kInitBatch = 8;  // rows whose loads are in flight together
static_assert(kTH % kInitBatch == 0, "whole batches");

// What the walk over a tile's rows finds.
struct InitSeen {
    unsigned least = 0xffffffffu, nans = 0;            // per lane: smallest elevation (ordered bits), NaN cells
    unsigned long long any = 0, top = 0, bottom = 0;  // opened or excluded cells: all rows, the first and the last row
};

// INNER: every cell of the tile and around it is an interior cell, so no row
// or column is tested (all tiles but the border's; the tests are scalar work
// for every row).  0.62 ms at 16384^2 (3.2 GB moved, 5.2 TB/s).
template <bool INNER>
__device__ __forceinline__ void fill_init_tile(const FillParams &p, int ty, int tx, int lane, double *edge, InitSeen &o)
{
    const int c = tx * kTW + lane, r0 = ty * kTH;
    // lanes 0 and 63: the column beside the tile (the others: their own)
    const int ce = lane == 0 ? c - 1 : (lane == 63 ? c + 1 : c);
    const bool cin = INNER || (c >= 1 && c <= p.cols - 2), ein = INNER || (ce >= 1 && ce <= p.cols - 2);
    const bool opens = p.opens != 0;
    auto rin = [&](int r) { return INNER || (r >= 1 && r <= p.rows - 2); };
    auto load = [&](int r, float &f, float &e) {
        const float *row = p.dem + (long long)r * p.pitch;
        f = rin(r) && cin ? row[c] : 0.0f;
        e = rin(r) && ein ? row[ce] : 0.0f;
    };
    // excluded cells of row r, and the same widened by a column
    auto excluded = [&](int r, float f) -> unsigned long long {
        return __builtin_amdgcn_ballot_w64(!(rin(r) && cin) || is_nd(p, f));
    };
    auto widened = [&](int r, unsigned long long m, float e) -> unsigned long long {
        return m | (m << 1) | (m >> 1) | __builtin_amdgcn_ballot_w64(!(rin(r) && ein) || is_nd(p, e));
    };
    float f, e;
    load(r0 - 1, f, e);
    unsigned long long above = widened(r0 - 1, excluded(r0 - 1, f), e);
    load(r0, f, e);
    float cur = f;
    unsigned long long cur_m = excluded(r0, f), cur_w = widened(r0, cur_m, e);
    for (int b = 0; b < kTH; b += kInitBatch) {
        if (!INNER && r0 + b >= p.rows) break;
        float fn[kInitBatch], en[kInitBatch];  // the rows below each row of the batch
#pragma unroll
        for (int k = 0; k < kInitBatch; k++) load(r0 + b + k + 1, fn[k], en[k]);
#pragma unroll
        for (int k = 0; k < kInitBatch; k++) {
            const int r = r0 + b + k;
            const unsigned long long next_m = excluded(r + 1, fn[k]), next_w = widened(r + 1, next_m, en[k]);
            if (INNER || r < p.rows) {
                const unsigned long long open = above | cur_w | next_w;
                const bool valid = !((cur_m >> lane) & 1ull);
                double w0 = p.nodata;
                if (valid) {
                    w0 = opens && ((open >> lane) & 1ull) ? fmin((double)cur, kStart) : kStart;
                    if (cur != cur) {
                        o.nans++;
                    } else {
                        unsigned u = __float_as_uint(cur);  // order-preserving map of floats to unsigned
                        u = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
                        o.least = u < o.least ? u : o.least;
                    }
                }
                // streamed past the caches: the passes read W back much later
                if (INNER || c < p.cols) __builtin_nontemporal_store(w0, &p.w[(long long)r * p.pitch + c]);
                if (lane == 0 || lane == 63) edge[(lane ? kTH : 0) + b + k] = valid ? w0 : __builtin_huge_val();
                o.any |= open;
                if (b + k == 0) o.top = open;
                if (b + k == kTH - 1) o.bottom = open;
            }
            above = cur_w;
            cur_w = next_w;
            cur_m = next_m;
            cur = fn[k];
        }
    }
}

__global__ __launch_bounds__(256) void fill_init_kernel(FillParams p)
{
    __shared__ double edges[4][2 * kTH];  // each wave's first and last column
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int tx = (int)blockIdx.x * 4 + wave, ty = blockIdx.y;
    if (tx >= p.tiles_x) return;  // the whole wave
    InitSeen o;
    if (ty > 0 && tx > 0 && (ty + 1) * kTH + 1 < p.rows && (tx + 1) * kTW + 1 < p.cols)
        fill_init_tile<true>(p, ty, tx, lane, edges[wave], o);
    else
        fill_init_tile<false>(p, ty, tx, lane, edges[wave], o);
    // lanes 0-31 the first column, lanes 32-63 the last: one run of 512 bytes
    // (rows and columns past the raster are never read)
    p.edge[edge_index(p, ty, tx, 0, 0) + lane] = edges[wave][lane];
    // the tiles with an opened cell in them or around them
    {
        const int dy = lane / 3 - 1, dx = lane % 3 - 1;
        const int nty = ty + dy, ntx = tx + dx;
        const unsigned long long m = dy < 0 ? o.top : (dy > 0 ? o.bottom : o.any);
        const bool need = lane < 9 && (dx < 0 ? (m & 1ull) != 0 : (dx > 0 ? (m >> 63) != 0 : m != 0)) && nty >= 0 &&
                          nty < p.tiles_y && ntx >= 0 && ntx < p.tiles_x;
        const int t = nty * p.tiles_x + ntx;
        if (need && flag_tile(p, t, kAll, 0) == 0) append_tile(p, t, 0);
    }
    unsigned least = o.least, nans = o.nans;
    for (int off = 32; off > 0; off >>= 1) {
        const unsigned u = __shfl_xor(least, off);
        least = u < least ? u : least;
        nans += __shfl_xor(nans, off);
    }
    if (lane == 0) {
        // the plain read skips the atomic unless it would lower the value
        // (or the read is stale): same-address atomics serialise
        if (least < __atomic_load_n(&p.range[0], __ATOMIC_RELAXED)) atomicMin(&p.range[0], least);
        if (nans) atomicAdd(&p.range[1], nans);
    }
}

// Flags cleared, empty worklists, no range and no passes, before the init kernel.
__global__ void fill_reset_kernel(FillParams p, int n)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) p.flags[i] = 0;
    if (i < 3 * kSetWords) p.count[i] = 0;
    if (i == 0) {
        p.range[0] = 0xffffffffu;
        p.range[1] = 0;
        *p.ran = 0;
    }
}

template <int RW>
struct FillShared {
    static constexpr int kWaves = kTH / RW;
    double h[2][kWaves][2][kTW];  // per round parity and wave: h of its first and last row
    unsigned note[2][kWaves];     // per round parity and wave: kSentTop, kSentBottom, kGoing
    unsigned start[2];            // by parity of the visit: its flags (0: none)
    unsigned out[2];              // by parity of the visit: which edges and corners changed
};
constexpr unsigned kSentTop = 1u, kSentBottom = 2u, kGoing = 4u;

// The flags a visit starts from, requested a visit ahead by thread 0 so that
// no wave waits for them (list entry, flags and barrier in turn cost a visit
// about 2 us of its 15).
__device__ __forceinline__ unsigned *visit_flags(const FillParams &p, int tile, int pass)
{
    return &p.flags[(long long)(pass & 1) * p.tiles_x * p.tiles_y + tile];
}

// Tiles flagged at the end of a visit and not on a list yet: wave 0 appends
// them during the next visit, while that visit's loads are on their way.
struct Flagged {
    int tile = 0;
    unsigned old = 1;  // the flags found (0: the lane's tile goes on the list)
};

// One visit of one tile (see the top of the file).
template <int RW>
__device__ __forceinline__ void fill_tile(const FillParams &p, int tile, unsigned start, int parity, int pass,
                                          FillShared<RW> &S, Flagged &flagged)
{
    constexpr int kRW = RW, kWaves = kTH / RW;
    static_assert(kWaves <= 4, "the flags hold one bit per wave and side, four of each");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    auto flush = [&]() {
        if (flagged.old == 0) append_tile(p, flagged.tile, pass + 1);
        flagged.old = 1;
    };
    const int ty = tile / p.tiles_x, tx = tile - ty * p.tiles_x;
    const int r0 = ty * kTH + wave * kRW, c = tx * kTW + lane;  // the wave's first row, the lane's column
    constexpr unsigned kRows = (1u << kRW) - 1u;
    unsigned dirty = 0;  // bit k: row r0 + k is to be evaluated
    if ((start & kAll) || (start & ((kLeft | kRight) << wave))) dirty = kRows;
    if (wave == 0 && (start & (kTop | kTopLeft | kTopRight))) dirty |= 1u;
    if (wave == kWaves - 1 && (start & (kBottom | kBottomLeft | kBottomRight))) dirty |= 1u << (kRW - 1);

    const double inf = __builtin_huge_val();
    double w[kRW], h[kRW], side[kRW];  // side: halo columns, left in lane 0, right in lane 63
    double up = inf, down = inf;       // h of the rows above and below the wave's
    float dem[kRW];
    bool up_sent = false, down_sent = false;
    unsigned touched = 0;                              // bit k: row r0 + k changed
    unsigned long long cols = 0, first = 0, last = 0;  // columns that changed: any row, the first, the last row
    auto row_h = [&](double v, double e) -> double { return vmin(vmin(dpp_from_left(v, e), v), dpp_from_right(v, e)); };
    auto load = [&]() {
        double eu = inf, ed = inf, wu = p.nodata, wd = p.nodata;
        // the edge copies beside the tile: the left tile's last column (which
        // precedes this tile's copies) and the right tile's first
        const bool ein = (lane == 0 && tx > 0) || (lane == 63 && tx + 1 < p.tiles_x);
        const double *edge = p.edge + (edge_index(p, ty, tx, 0, wave * kRW) + (lane == 0 ? -kTH : 2 * kTH));
        const double *row = p.w + ((long long)r0 * p.pitch + tx * kTW);
        const float *drow = p.dem + ((long long)r0 * p.pitch + tx * kTW);
        // every load is issued before the first value is used
        if (ty > 0 && r0 + kRW < p.rows && tx * kTW + kTW <= p.cols) {
            // every row the wave reads lies in the raster, and so do its columns
            const double *rw = row - p.pitch;
            wu = rw[(unsigned)lane];
#pragma unroll
            for (int k = 0; k < kRW; k++) {
                rw += p.pitch;
                w[k] = rw[(unsigned)lane];
                dem[k] = drow[(unsigned)lane];
                drow += p.pitch;
                side[k] = inf;
            }
            rw += p.pitch;
            wd = rw[(unsigned)lane];
            if (ein) {
                // the tile rows above and below hold their own copies
                const long long stride = (long long)p.tiles_x * 2 * kTH;
                eu = wave > 0 ? edge[-1] : edge[kTH - 1 - stride];
                ed = wave < kWaves - 1 ? edge[kRW] : edge[stride - (kTH - kRW)];
#pragma unroll
                for (int k = 0; k < kRW; k++) side[k] = edge[k];
            }
        } else {
            const bool cin = c < p.cols;
            auto get = [&](int r, double &v, double &e) {
                v = p.nodata;
                e = inf;
                if (r >= 0 && r < p.rows) {
                    if (cin) v = p.w[(long long)r * p.pitch + c];
                    if (ein) e = p.edge[edge_index(p, r / kTH, tx, 0, r % kTH) + (lane == 0 ? -kTH : 2 * kTH)];
                }
            };
            get(r0 - 1, wu, eu);
#pragma unroll
            for (int k = 0; k < kRW; k++) {
                get(r0 + k, w[k], side[k]);
                dem[k] = cin && r0 + k < p.rows ? p.dem[(long long)(r0 + k) * p.pitch + c] : 0.0f;
            }
            get(r0 + kRW, wd, ed);
        }
        if (wave == 0) flush();
        // NoData reads as +infinity: never a minimum, never lowered
        auto open = [&](double v) -> double { return v == p.nodata ? inf : v; };
#pragma unroll
        for (int k = 0; k < kRW; k++) {
            w[k] = open(w[k]);
            dem[k] = w[k] == inf ? __builtin_huge_valf() : dem[k];
            h[k] = row_h(w[k], side[k]);
        }
        if (!up_sent) up = row_h(open(wu), eu);
        if (!down_sent) down = row_h(open(wd), ed);
    };
    // One evaluation of row r0 + k by every lane.
    auto evaluate = [&](int k) {
        dirty &= ~(1u << k);
        const double above = k == 0 ? up : h[k > 0 ? k - 1 : 0], below = k == kRW - 1 ? down : h[k < kRW - 1 ? k + 1 : 0];
        // t = max(dem, min(h(r-1), h(r), h(r+1)) + gap), as one block: the
        // DEM value is widened where it is used (kept widened, the rows would
        // take 16 more registers)
        double t, d;
        asm volatile("v_min_f64 %0, %2, %3\n\tv_cvt_f64_f32 %1, %5\n\tv_min_f64 %0, %0, %4\n\t"
                     "v_add_f64 %0, %0, %6\n\tv_max_f64 %0, %1, %0"
                     : "=&v"(t), "=&v"(d)
                     : "v"(above), "v"(h[k]), "v"(below), "v"(dem[k]), "s"(kGap));
        const unsigned long long ch = __builtin_amdgcn_ballot_w64(t < w[k]);
        if (ch != 0) {
            w[k] = vmin(w[k], t);
            h[k] = row_h(w[k], side[k]);
            dirty |= (7u << k >> 1) & kRows;
            touched |= 1u << k;
            cols |= ch;
            if (k == 0) first |= ch;
            if (k == kRW - 1) last |= ch;
        }
    };
    // Ends a round: tells the other waves what this one sent and takes what
    // they sent; true when no wave has anything left.  One barrier per round:
    // what a round sends is read before the next barrier and written over
    // only after it.
    int round = 0;
    auto exchange = [&](unsigned note) -> bool {
        if (lane == 0) S.note[round][wave] = note;
        __syncthreads();
        unsigned notes = 0;
#pragma unroll
        for (int v = 0; v < kWaves; v++) {
            const unsigned n = (unsigned)__builtin_amdgcn_readfirstlane((int)S.note[round][v]);
            notes |= n;
            if (v == wave - 1 && (n & kSentBottom)) {
                up = S.h[round][v][1][lane];
                up_sent = true;
                dirty |= 1u;
            }
            if (v == wave + 1 && (n & kSentTop)) {
                down = S.h[round][v][0][lane];
                down_sent = true;
                dirty |= 1u << (kRW - 1);
            }
        }
        round ^= 1;
        return notes == 0;
    };
    bool settled = false;
    if (wave == 0 && dirty == 0) flush();
    while (dirty == 0 && !settled) settled = exchange(0);  // nothing to load yet
    if (!settled) {
        load();
        do {
            unsigned note = 0;
            if (dirty) {
                const unsigned had = touched;
                touched = 0;
#pragma unroll
                for (int k = 0; k < kRW; k++)
                    if ((dirty >> k) & 1u) evaluate(k);
#pragma unroll
                for (int k = kRW - 1; k >= 0; k--)
                    if ((dirty >> k) & 1u) evaluate(k);
                if (wave > 0 && (touched & 1u)) {
                    S.h[round][wave][0][lane] = h[0];
                    note |= kSentTop;
                }
                if (wave < kWaves - 1 && ((touched >> (kRW - 1)) & 1u)) {
                    S.h[round][wave][1][lane] = h[kRW - 1];
                    note |= kSentBottom;
                }
                if (dirty) note |= kGoing;
                touched |= had;
            }
            settled = exchange(note);
        } while (!settled);
    }
    if (touched) {
#pragma unroll
        for (int k = 0; k < kRW; k++) {
            if (!((touched >> k) & 1u)) continue;
            const int r = r0 + k;
            if (w[k] < inf) {  // NoData cells keep their value
                p.w[(long long)r * p.pitch + c] = w[k];
                if (lane == 0 || lane == 63) p.edge[edge_index(p, ty, tx, lane != 0, wave * kRW + k)] = w[k];
            }
        }
        if (lane == 0) {
            // a changed side row matters to the rows beside it and next to
            // that: the band's own and, from its first or last row, the next
            const unsigned bands = 1u << wave | (touched & 1u) << wave >> 1 | (touched >> (kRW - 1) & 1u) << wave << 1;
            const unsigned lb = cols & 1ull ? bands : 0u, rb = cols >> 63 ? bands : 0u;
            unsigned o = (lb & ((1u << kWaves) - 1u)) * kLeft | (rb & ((1u << kWaves) - 1u)) * kRight;
            if (wave == 0 && first) o |= kTop | (first & 1ull ? kTopLeft : 0u) | (first >> 63 ? kTopRight : 0u);
            if (wave == kWaves - 1 && last)
                o |= kBottom | (last & 1ull ? kBottomLeft : 0u) | (last >> 63 ? kBottomRight : 0u);
            if (o) atomicOr(&S.out[parity], o);
        }
    }
}

// After the barrier that ends a visit: flags the tiles around it (wave 0).
__device__ __forceinline__ void flag_around(const FillParams &p, int tile, unsigned out, int pass, Flagged &flagged)
{
    const int lane = threadIdx.x & 63;
    const int ty = tile / p.tiles_x, tx = tile - ty * p.tiles_x;
    {
        // lanes 0-8: the tiles around, each with the side of it that changed
        const int dy = lane / 3 - 1, dx = lane % 3 - 1;
        unsigned f = 0;
        if (lane == 0) f = out & kTopLeft ? kBottomRight : 0u;
        if (lane == 1) f = out & kTop ? kBottom : 0u;
        if (lane == 2) f = out & kTopRight ? kBottomLeft : 0u;
        if (lane == 3) f = (out >> 0 & 15u) * kRight;
        if (lane == 5) f = (out >> 4 & 15u) * kLeft;
        if (lane == 6) f = out & kBottomLeft ? kTopRight : 0u;
        if (lane == 7) f = out & kBottom ? kTop : 0u;
        if (lane == 8) f = out & kBottomRight ? kTopLeft : 0u;
        const int nty = ty + dy, ntx = tx + dx;
        const bool need = f != 0 && nty >= 0 && nty < p.tiles_y && ntx >= 0 && ntx < p.tiles_x;
        const int t = nty * p.tiles_x + ntx;
        if (need) {
            flagged.tile = t;
            flagged.old = flag_tile(p, t, f, pass + 1);
        }
    }
}

// FIRST: pass 0, which does nothing for a DEM that is refused (the host
// learns it from the same words, passes later): the DEM is left as the init
// kernel made it, and the later lists stay empty.
template <int RW, bool FIRST>
__global__ __launch_bounds__(64 * (kTH / RW), RW == 8 ? 5 : 3) void fill_pass_kernel(FillParams p, int pass)
{
    __shared__ FillShared<RW> S;
    const int lane = threadIdx.x & 63;
    // the sublists' lengths, one per lane, and where each ends in the whole list
    const unsigned len = p.count[(pass % 3) * kSetWords + lane * kSubStride];
    unsigned end = len;
#pragma unroll
    for (int off = 1; off < kSub; off <<= 1) {
        const unsigned o = (unsigned)__shfl_up((int)end, off);
        if (lane >= off) end += o;
    }
    unsigned n = (unsigned)__builtin_amdgcn_readlane((int)end, kSub - 1);
    if (FIRST && fill_refused(p.range[0], p.range[1], p.nodata)) n = 0;
    if (blockIdx.x == 0 && threadIdx.x < kSub) {
        // the counters that pass + 1 fills (pass - 1 read them)
        p.count[((pass + 2) % 3) * kSetWords + lane * kSubStride] = 0;
        if (lane == 0 && n != 0) *p.ran = (unsigned)pass + 1u;
    }
    // A fixed stride over the list, whose neighbours are tiles kSub apart.
    // The grid is what fits on the GPU at once, so no workgroup starts late
    // with a full share.
    const unsigned stride = gridDim.x;
    unsigned e = blockIdx.x;
    if (e >= n) return;  // the whole workgroup
    const int *list = p.list + (long long)(pass & 1) * kSub * p.sub_cap;
    auto entry = [&](unsigned i) -> int {
        const int sub = __builtin_popcountll(__builtin_amdgcn_ballot_w64(end <= i));  // sublists that end before i
        const unsigned at = i - (unsigned)__builtin_amdgcn_readlane((int)(end - len), sub);
        return list[(long long)sub * p.sub_cap + at];
    };
    int tile = __builtin_amdgcn_readfirstlane(entry(e));
    int ahead = e + stride < n ? entry(e + stride) : 0;
    if (threadIdx.x == 0) {
        unsigned *f = visit_flags(p, tile, pass);
        S.start[0] = *f;
        S.out[0] = 0;
        *f = 0;
    }
    __syncthreads();
    Flagged flagged;
    for (int parity = 0; e < n; e += stride, parity ^= 1) {
        const unsigned start = (unsigned)__builtin_amdgcn_readfirstlane((int)S.start[parity]);
        // the next visit's flags and the list entry of the one after are
        // requested now, so that no visit waits for them
        const bool more = e + stride < n;
        const int next_tile = __builtin_amdgcn_readfirstlane(ahead);
        unsigned next_start = 0;
        if (more && threadIdx.x == 0) next_start = *visit_flags(p, next_tile, pass);
        if (e + 2 * stride < n) ahead = entry(e + 2 * stride);
        fill_tile<RW>(p, tile, start, parity, pass, S, flagged);
        if (more && threadIdx.x == 0) {
            S.start[parity ^ 1] = next_start;
            S.out[parity ^ 1] = 0;
            *visit_flags(p, next_tile, pass) = 0;
        }
        // the next visit reuses the LDS; what a visit leaves there is read
        // right after the barrier and written again only after the next one
        __syncthreads();
        if (threadIdx.x < 64) {
            const unsigned out = (unsigned)__builtin_amdgcn_readfirstlane((int)S.out[parity]);
            if (out != 0) flag_around(p, tile, out, pass, flagged);
        }
        tile = next_tile;
    }
    if (threadIdx.x < 64 && flagged.old == 0) append_tile(p, flagged.tile, pass + 1);
}

}  // namespace

}  // namespace pargo

using pargo::fail;

extern "C" int pargo_pit_remove(pargo_ctx *ctx, const pargo_grid *g, const float *dem, double *filled_out,
                                int *passes_out)
{
    if (!ctx) return PARGO_E_INVALID;
    if (!g || !dem || !filled_out) return fail(ctx, PARGO_E_INVALID, "pargo_pit_remove: null argument");
    if (g->rows < 1 || g->cols < 1) return fail(ctx, PARGO_E_INVALID, "empty grid (%d x %d)", g->rows, g->cols);
    const long long pitch = g->pitch ? g->pitch : g->cols;
    if (pitch < g->cols) return fail(ctx, PARGO_E_INVALID, "pitch %lld < cols %d", pitch, g->cols);
    if (std::isnan(g->nodata)) return fail(ctx, PARGO_E_INVALID, "NaN NoData is not supported");
    int rc = pargo::bind(ctx);
    if (rc) return rc;
    pargo::FillParams p{};
    p.dem = dem;
    p.w = filled_out;
    p.pitch = pitch;
    p.rows = g->rows;
    p.cols = g->cols;
    p.tiles_x = (g->cols + pargo::kTW - 1) / pargo::kTW;
    p.tiles_y = (g->rows + pargo::kTH - 1) / pargo::kTH;
    p.nodata = g->nodata;
    // the reference keeps a cell when fabs(dem - noData) > 1e-6
    // (pitRemoveOperator.cpp:40,53): NoData is the float interval with
    // fabs <= 1e-6
    pargo::nodata_interval(g->nodata, 0.000001, &p.nd_lo, &p.nd_hi, true);
    if (p.nd_lo > p.nd_hi) {
        p.nd_lo = INFINITY;
        p.nd_hi = -INFINITY;
    }
    p.opens = !(g->nodata == INFINITY);
    const int ntiles = p.tiles_x * p.tiles_y;
    constexpr int kBatch = 8;      // passes between checks
    constexpr int kMaxPasses = 1 << 20;
    // scratch: the range check's two words and the passes that had work, the
    // list counters, then the flags, the two worklists and the tiles' edge
    // columns
    const size_t counters = 64 + 3 * (size_t)pargo::kSetWords;
    p.sub_cap = (ntiles + pargo::kSub - 1) / pargo::kSub;
    const size_t words = counters + 2 * (size_t)ntiles + 2 * (size_t)pargo::kSub * p.sub_cap;
    const size_t edge_off = (sizeof(unsigned) * words + 255) / 256 * 256;
    rc = pargo::ensure_scratch(ctx, edge_off + sizeof(double) * 2 * pargo::kTH * (size_t)ntiles);
    if (rc) return rc;
    rc = pargo::ensure_report(ctx);
    if (rc) return rc;
    unsigned *scr = static_cast<unsigned *>(ctx->scratch);
    p.range = scr;
    p.ran = scr + 2;
    p.count = scr + 64;
    p.flags = scr + counters;
    p.list = reinterpret_cast<int *>(p.flags + 2 * (size_t)ntiles);
    p.edge = reinterpret_cast<double *>(static_cast<char *>(ctx->scratch) + edge_off);

    hipLaunchKernelGGL(pargo::fill_reset_kernel, dim3((std::max(2 * ntiles, 3 * pargo::kSetWords) + 255) / 256), dim3(256), 0,
                       ctx->stream, p, 2 * ntiles);
    hipLaunchKernelGGL(pargo::fill_init_kernel, dim3((p.tiles_x + 3) / 4, p.tiles_y), dim3(256), 0, ctx->stream, p);
    // a fixed grid walks each pass's worklist: as many workgroups as are
    // resident at once
    const int cus = ctx->num_cu > 0 ? ctx->num_cu : 256;
    int per_cu = 0;
    const bool tall = ntiles >= pargo::kTallTiles;
    const int pass_threads = tall ? 128 : 256;
    auto *const first_kernel = tall ? pargo::fill_pass_kernel<16, true> : pargo::fill_pass_kernel<8, true>;
    auto *const pass_kernel = tall ? pargo::fill_pass_kernel<16, false> : pargo::fill_pass_kernel<8, false>;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, pass_kernel, pass_threads, 0) != hipSuccess || per_cu < 1)
        per_cu = 4;
    const int pass_blocks = std::min(ntiles, cus * per_cu);
    // Passes are launched a batch ahead of the one whose outcome is waited
    // for, so that the GPU does not idle while the host learns it (about 30 us
    // a batch); passes with nothing on their list, 8 to 15 of them at the end,
    // take 2 us each (4.5 with the grid of a large raster).
    auto launch = [&](int first) -> int {
        for (int k = first; k < first + kBatch; k++)
            hipLaunchKernelGGL(k == 0 ? first_kernel : pass_kernel, dim3(pass_blocks), dim3(pass_threads), 0, ctx->stream, p,
                               k);
        const int slot = first / kBatch & 1;
        PARGO_HIP(ctx, hipMemcpyAsync(static_cast<unsigned *>(ctx->report) + 4 * slot, scr, 3 * sizeof(unsigned),
                                      hipMemcpyDeviceToHost, ctx->stream));
        PARGO_HIP(ctx, hipEventRecord(ctx->report_event[slot], ctx->stream));
        return PARGO_OK;
    };
    int pass = 0, ran = 0;
    auto settle = [&]() -> int {
        int rc = launch(0);
        if (rc) return rc;
        for (;;) {
            rc = launch(pass + kBatch);
            if (rc) return rc;
            const int slot = pass / kBatch & 1;
            PARGO_HIP(ctx, hipEventSynchronize(ctx->report_event[slot]));
            const unsigned *h = static_cast<const unsigned *>(ctx->report) + 4 * slot;  // range, passes with work
            rc = pargo::check_launch(ctx, "pargo_pit_remove");
            if (rc) return rc;
            if (pass == 0 && pargo::fill_refused(h[0], h[1], g->nodata)) {
                if (h[1])
                    return fail(ctx, PARGO_E_INVALID, "the DEM holds %u NaN cells: the reference never settles there", h[1]);
                return fail(ctx, PARGO_E_UNSUPPORTED,
                            "NoData %.17g lies inside the range of filled values [%.17g, 10000]: the reference's "
                            "result would depend on its sweep order",
                            g->nodata, pargo::lowest_filled(h[0]));
            }
            pass += kBatch;
            ran = (int)h[2];
            if (ran < pass) return PARGO_OK;  // the batch's last pass had nothing to do
            if (pass >= kMaxPasses)
                return fail(ctx, PARGO_E_NONTERM, "depression filling did not settle within %d passes", kMaxPasses);
        }
    };
    rc = settle();
    if (rc) {
        // the passes of the batch ahead read the DEM and write the output:
        // the caller gets both back only when they have ended
        hipStreamSynchronize(ctx->stream);
        return rc;
    }
    // The batch ahead of the one that settled is not waited for: its lists are
    // empty, so it touches the context's memory only (with the wait the
    // 1501 x 2003 chain took 772 us instead of 731).
    if (passes_out) *passes_out = ran;
    return PARGO_OK;
}
