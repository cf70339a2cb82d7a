// sca.hip -- D8 contributing area (scad8) on the device.
//
// The reference (apps/hydrology/scad8/scaOperator.cpp:37-131, run by
// RasterOperator::Work, gpro/rasterOperator.h:170-216) sweeps the grid in
// row-major order three times: NoData/initial values, then the number of
// neighbours draining into each cell ("degree"), then ONE accumulation sweep
// in which a cell pulls the area of every inflowing neighbour whose degree
// is 0 (a cell nothing drains into) or -1 (finished earlier in the same
// sweep).  Every accumulation sweep ends with Termination = 1
// (scaOperator.cpp:126), so Work stops after that single sweep.
//
// What one sweep computes, stated without the sweep order:
//   In(c)   = neighbours u whose code points at c, unless c's own code
//             points back at u (scaOperator.cpp:71,94);
//   source  = interior valid cell with In empty (degree 0 after sweep 2);
//   avail(u,c) = u is a source, or u precedes c in row-major order
//             (u is the NW, N, NE or W neighbour) and u is done;
//   done(c) = every u in In(c) is avail(u,c);
//   sca(c)  = 1 + sum of sca(u) over avail(u,c).
// Border cells are never visited: their degree keeps the layer's NoData
// value, so a border cell draining inward is never available.
// The last work cell runs the pull loop even when its degree is <= 0
// (scaOperator.cpp:86): a NoData cell there adds its available inflows to
// NoData.
//
// The "converge" variant repeats the accumulation sweep until nothing
// changes, which lifts the row-major restriction: every inflow is pending
// and sca(c) = 1 + sum over done inflows.
//
// Device formulation: the dependencies that matter (non-source inflows the
// cell waits for) form a forest, each cell feeding at most its one target.
// A 16-bit static word per cell holds what following it needs:
//   bits  0-3   npend: inflows the cell waits for
//   bits  4-7   nsrc: inflows from sources (each adds 1)
//   bit   8     an inflow can never be available (border, or behind in
//               the one-sweep order)
//   bit   9     feeds: the cell is one of its target's pending inflows
//   bits 10-13  the cell's code (window index of its target)
//   bit  14     the cell has an area (interior, not NoData)
// The forest is solved tile by tile (64 x 32 cells) in LDS, where a hop to
// the next cell is one LDS atomic, and only what crosses tile edges goes
// through memory.  Inside a tile every cell has an accumulator (the sum of
// its done inflows' areas, the inflows still awaited, how many were not
// done); a walk starts at each cell that waits for nothing and feeds, adds
// its cell to the target's accumulator and goes on from there if nothing
// else is awaited.
//   1. sca_local_kernel forms the static words and runs the tile's walks
//      with every inflow from outside taken as an arrival of area 0 that is
//      done.  A cell through which the tile is left (an exit, a perimeter
//      cell) then holds what its tile contributes, the number of inflows
//      from outside upstream of it, and whether anything inside the tile
//      keeps it from being done.  Its area when they have arrived is that
//      sum plus theirs, and it is done when they all are, so an exit is one
//      node of a graph whose links are "the exit that a walk entering here
//      leaves through", found by following each entry to the tile's edge.
//   2. sca_link_kernel resolves each exit's successor, the exit of the tile
//      it enters.
//   3. sca_cross_kernel walks that graph: a hop is one 64-bit atomic on the
//      successor's word (sum, awaited, not done), with the successor's own
//      link read beside it.
//   4. sca_final_kernel runs the tile's walks once more, now with the areas
//      that arrive from outside, and writes the areas.
// Cells that never complete (a cycle of codes, which the converging mode
// admits for arbitrary codes) keep the sum of the done inflows they
// received, which is their area.
//
// Measured on the headline DEM's codes: 16384^2 in the reference mode 1.96 ms
// (local 0.89, link 0.07, cross 0.12, final 0.87), 5003 x 7001 in the
// converging mode 0.34 ms, and 0.11 ms for the codes of a filled 1501 x 2003
// DEM, whose paths are long.  One walk over the whole raster with a global
// atomic or a static word read per hop (33 bytes of HBM traffic, up to 1336
// hops in a row) took 4.24, 1.21 and 1.15 ms.
#include <algorithm>
#include <cmath>

#include "internal.h"
#include "sca_swar.h"

namespace pargo {

namespace {

constexpr unsigned kNone = 15;
constexpr int kTileC = 64, kTileR = 32;  // cells per workgroup: 64 x 32
constexpr int kTileN = kTileC * kTileR;

// Perimeter slots of a tile: top row 0-63, bottom row 64-127, then the left
// and the right column without the corners.
constexpr int kSlots = 2 * kTileC + 2 * (kTileR - 2), kSlotStride = 192;
static_assert(kSlots <= kSlotStride && kSlots <= 256, "one thread per slot");
__device__ __forceinline__ int slot_of(int r, int c)
{
    return r == 0 ? c : r == kTileR - 1 ? kTileC + c : (c == 0 ? 2 * kTileC : 2 * kTileC + kTileR - 2) + r - 1;
}
__device__ __forceinline__ int cell_of_slot(int s)
{
    if (s < kTileC) return s;
    if (s < 2 * kTileC) return (kTileR - 1) * kTileC + s - kTileC;
    s -= 2 * kTileC;
    return s < kTileR - 2 ? (s + 1) * kTileC : (s - (kTileR - 2) + 1) * kTileC + kTileC - 1;
}

// A tile's accumulators in sca_local_kernel, 32 bits: sum of areas (at most
// the tile's cells and the 196 sources that can drain into it), inflows from
// outside upstream (at most 196), not-done arrivals, arrivals awaited.
constexpr int kLocExt = 12, kLocBad = 20, kLocPend = 24;
constexpr unsigned kLocSum = (1u << kLocExt) - 1;
static_assert(kTileN + 2 * (kTileC + kTileR) + 4 <= (int)kLocSum, "areas inside a tile fit their field");
// In sca_final_kernel, 64 bits: sum of areas, not-done arrivals, awaited.
constexpr int kFinBad = 40, kFinPend = 44;
constexpr unsigned long long kFinSum = (1ull << kFinBad) - 1, kFinArea = 1ull << 63;  // kFinArea: the cell has one
// An exit's word: sum of areas, arrivals awaited (255: not an exit, or never
// complete), not-done arrivals, and a flag for the exits that await nothing
// from the start.
constexpr int kExitPend = 40, kExitBad = 48;
constexpr unsigned long long kExitStart = 1ull << 63, kExitNever = 255ull << kExitPend;
constexpr unsigned kNoExit = 0xffffffffu;

__device__ __forceinline__ unsigned flow_of(unsigned b) { return (b <= 8u && b != 4u) ? b : kNone; }
__device__ __forceinline__ unsigned excl_of(unsigned b)
{
    if (b <= 8u) return b;
    if ((b & 0xF0u) == PARGO_FLOW_EXCL && (b & 15u) <= 8u) return b & 15u;
    return kNone;
}
__device__ __forceinline__ bool is_valid(unsigned b) { return b != PARGO_FLOW_NODATA && b != PARGO_FLOW_INERT; }

struct ScaParams {
    const uint8_t *__restrict__ flow;
    const uint32_t *__restrict__ mask;  // may be null
    double *__restrict__ area;
    uint16_t *__restrict__ st;          // static words, tile by tile
    unsigned long long *__restrict__ exits;  // [tiles][kSlotStride] exit words
    unsigned *__restrict__ next;        // [tiles][kSlotStride]: the perimeter cell an exit enters, then its successor
    uint8_t *__restrict__ link;         // [tiles][kSlotStride]: slot of the exit reached from a perimeter cell (255: none)
    uint8_t *__restrict__ ext;          // [tiles][kSlotStride]: pending inflows of a perimeter cell from outside
    unsigned *__restrict__ last_done;   // done flags of the 3 x 3 cells ending at (rows-1, cols-1)
    long long pitch;
    int rows, cols, mask_words;
    int tiles_x, ntiles;
    int converge;
    double nodata;
    int w, h, slots;  // with kNarrow: cells and slots a tile has memory for
};

// Memory of a raster that is one column (of at most 32 cells) or one row (of
// at most 16) of tiles: at a full tile's 6784 bytes a raster of one column
// would take 212 bytes a cell.  Such a raster keeps static words for the
// cells a tile holds and slots for the sides that have a tile beyond them
// only, 2.4 to 2.9 bytes a cell.  Its kernels are the same but for these
// addresses, and are compiled into a code object of their own
// (sca_narrow.hip): beside them in one object, the kernels of full tiles ran
// 0.3 % slower (5003 x 7001 layer 397.0 -> 398.4 us).
#ifdef PARGO_SCA_NARROW
constexpr bool kNarrow = true;
#else
constexpr bool kNarrow = false;
#endif
constexpr int kNarrowCols = kTileC / 2, kNarrowRows = kTileR / 2;
// A perimeter cell's slot in memory; of the sides without a tile beyond them
// none is asked for.
__device__ __forceinline__ unsigned mem_slot(const ScaParams &p, int r, int c)
{
    if (!kNarrow) return (unsigned)slot_of(r, c);
    return (unsigned)(p.tiles_x == 1 ? (r == 0 ? c : p.w + c) : (c == 0 ? r : p.h + r));
}
// Whether a perimeter cell has one (all of a full tile's have).
__device__ __forceinline__ bool has_slot(const ScaParams &p, int r, int c)
{
    if (!kNarrow) return true;
    return p.tiles_x == 1 ? (r == 0 || r == kTileR - 1) && c < p.w : (c == 0 || c == kTileC - 1) && r < p.h;
}

__device__ __forceinline__ unsigned npend_of(unsigned s) { return s & 15u; }
__device__ __forceinline__ unsigned nsrc_of(unsigned s) { return (s >> 4) & 15u; }
__device__ __forceinline__ bool poisoned_of(unsigned s) { return (s >> 8) & 1u; }
__device__ __forceinline__ bool feeds_of(unsigned s) { return (s >> 9) & 1u; }
__device__ __forceinline__ int code_of(unsigned s) { return (int)(s >> 10) & 15; }
__device__ __forceinline__ bool area_of(unsigned s) { return (s >> 14) & 1u; }

__device__ __forceinline__ unsigned load_class(const ScaParams &p, int r, int c)
{
    if (r < 0 || r >= p.rows || c < 0 || c >= p.cols) return PARGO_FLOW_NODATA;
    if (p.mask && ((p.mask[(long long)r * p.mask_words + (c >> 5)] >> (c & 31)) & 1u)) return PARGO_FLOW_NODATA;
    return p.flow[(long long)r * p.pitch + c];
}

// Static words of a 64 x 32 tile.  Classes of the tile plus a 2-cell halo go
// to LDS, then the inflow mask of the tile plus a 1-cell halo (bit j set when
// the neighbour at window position j < 4 ? j : j + 1 drains into the cell and
// is not excluded; a cell needs to know which of its inflows are sources, and
// whether its target counts it).  Tiles are dealt to the 8 XCDs in contiguous
// runs (workgroup g runs on XCD g % 8), so neighbouring tiles share their
// halo lines in one L2.
__device__ __forceinline__ int win_of_bit(int j) { return j < 4 ? j : j + 1; }
__device__ __forceinline__ int bit_of_win(int k) { return k < 4 ? k : k - 1; }

__device__ __forceinline__ int xcd_tile(const ScaParams &p)
{
    const int per = (p.ntiles + 7) / 8, g = blockIdx.x;  // tiles per XCD
    return (g & 7) * per + (g >> 3);
}

typedef uint32_t u32_b1 __attribute__((aligned(1)));  // one dword load at any byte address on gfx950

// A tile at least 2 cells from every border whose class rows can be read
// as words, four cells per word (sca_swar.h): columns c0 - 8 .. c0 + 71 of
// each row (the bound leaves a word more on either side).
__device__ __forceinline__ bool sca_swar_tile(const ScaParams &p, int r0, int c0)
{
    return r0 >= 2 && r0 + kSwarTileR + 2 <= p.rows && c0 >= 11 && c0 + 76 <= p.cols;
}

// The static words of such a tile, four cells per lane: the same words as the
// per-cell code of general_words, with half its VALU instructions and a sixth
// of its LDS accesses.
__device__ __forceinline__ void swar_words(const ScaParams &p, SwarTile &T, uint16_t *stw, int r0, int c0)
{
    const int tid = threadIdx.x;
    {
        constexpr int N = kSwarClsRows * kSwarClsWords, PER = (N + 255) / 256;
        uint32_t v[PER], mw[PER];
        // every load of the thread is issued before the first is used
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int i = tid + 256 * k;
            v[k] = mw[k] = 0;
            if (i < N) {
                const int rr = i / kSwarClsWords, w = i - rr * kSwarClsWords;
                const int r = r0 - 2 + rr, col = c0 - 8 + 4 * w;
                v[k] = *reinterpret_cast<const u32_b1 *>(p.flow + (long long)r * p.pitch + col);
                if (p.mask) mw[k] = p.mask[(long long)r * p.mask_words + (col >> 5)] >> (col & 31);
            }
        }
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int i = tid + 256 * k;
            if (i < N) {
                const int rr = i / kSwarClsWords, w = i - rr * kSwarClsWords;
                const uint32_t b = p.mask ? swar_select(swar_bits_to_mask(mw[k]), swar_splat(PARGO_FLOW_NODATA), v[k]) : v[k];
                T.cls[rr][w] = b;
                T.tgt[rr][w] = swar_flow_of(b);
            }
        }
    }
    __syncthreads();
    // Two words, eight cells, at a time: the four words of a row they need
    // are two aligned 64-bit reads (the compiler joined the three words of a
    // single one into unaligned 96-bit reads, and the LDS spent 7,000 cycles
    // a tile on those, 60 % of them stalled on the alignment).
    struct Four {
        SwarRow lo, hi;  // around the first and the second word of the pair
    };
    auto four = [](const uint32_t *row, int w) -> Four {
        const uint2 a = *reinterpret_cast<const uint2 *>(row + w), b = *reinterpret_cast<const uint2 *>(row + w + 2);
        return Four{{a.x, a.y, b.x}, {a.y, b.x, b.y}};
    };
    static_assert(kSwarClsWords % 2 == 0 && kSwarInmWords % 2 == 0, "rows keep the 8-byte alignment");
    for (int i = tid; i < kSwarInmRows * (kSwarInmWords / 2); i += 256) {
        const int lr = i / (kSwarInmWords / 2), q = 2 * (i - lr * (kSwarInmWords / 2));
        const Four b = four(T.cls[lr + 1], q);
        const Four t0 = four(T.tgt[lr], q), t1 = four(T.tgt[lr + 1], q), t2 = four(T.tgt[lr + 2], q);
        *reinterpret_cast<uint2 *>(&T.inm[lr][q]) =
            make_uint2(swar_inflow_rows(b.lo.b, t0.lo, t1.lo, t2.lo), swar_inflow_rows(b.hi.b, t0.hi, t1.hi, t2.hi));
    }
    __syncthreads();
    {
        const int tr = tid >> 3, g = 2 * (tid & 7);
        const uint2 b = *reinterpret_cast<const uint2 *>(&T.cls[tr + 2][g + 2]);
        const uint2 f = *reinterpret_cast<const uint2 *>(&T.tgt[tr + 2][g + 2]);
        const Four m0 = four(T.inm[tr], g), m1 = four(T.inm[tr + 1], g), m2 = four(T.inm[tr + 2], g);
        const SwarCells u = swar_cells_rows(b.x, f.x, m0.lo, m1.lo, m2.lo, p.converge != 0);
        const SwarCells v = swar_cells_rows(b.y, f.y, m0.hi, m1.hi, m2.hi, p.converge != 0);
        *reinterpret_cast<uint4 *>(stw + 8 * tid) = make_uint4(u.s01, u.s23, v.s01, v.s23);
    }
}

// Per-cell form, for tiles near the raster's edge.
struct GeneralTile {
    uint8_t cls[kTileR + 4][kTileC + 4];  // classes, halo 2
    uint8_t tgt[kTileR + 4][kTileC + 4];  // flow_of(class): window index of the target, kNone if none
    uint8_t inm[kTileR + 2][kTileC + 2];  // inflow masks, halo 1
};

__device__ __forceinline__ void general_words(const ScaParams &p, GeneralTile &T, uint16_t *stw, int r0, int c0)
{
    constexpr int CW = kTileC + 4, CH = kTileR + 4, NW = kTileC + 2, NH = kTileR + 2;
    const int tid = threadIdx.x;
    auto &cls = T.cls;
    auto &tgt = T.tgt;
    auto &inm = T.inm;
    {
        // every load of the thread is issued before the first store to LDS,
        // so that their latencies overlap
        constexpr int PER = (CH * CW + 255) / 256;
        unsigned v[PER];
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int i = tid + k * 256;
            v[k] = PARGO_FLOW_NODATA;
            if (i < CH * CW) {
                const int r = r0 - 2 + i / CW, c = c0 - 2 + i % CW;
                if (r >= 0 && r < p.rows && c >= 0 && c < p.cols) {
                    const unsigned b = p.flow[(long long)r * p.pitch + c];
                    const unsigned nd = p.mask ? (p.mask[(long long)r * p.mask_words + (c >> 5)] >> (c & 31)) & 1u : 0u;
                    v[k] = nd ? (unsigned)PARGO_FLOW_NODATA : b;
                }
            }
        }
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int i = tid + k * 256;
            if (i < CH * CW) {
                cls[i / CW][i % CW] = (uint8_t)v[k];
                tgt[i / CW][i % CW] = (uint8_t)flow_of(v[k]);
            }
        }
    }
    __syncthreads();
    for (int i = tid; i < NH * NW; i += 256) {
        const int lr = i / NW + 1, lc = i % NW + 1;  // position in cls
        const unsigned b = cls[lr][lc];
        unsigned m = 0;
        if (is_valid(b)) {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const int k = win_of_bit(j);
                m |= (tgt[lr + k / 3 - 1][lc + k % 3 - 1] == (unsigned)(8 - k)) ? 1u << j : 0u;
            }
            // the excluded window position (at most one) takes no inflow
            const unsigned ex = excl_of(b);
            if (ex != kNone && ex != 4u) m &= ~(1u << bit_of_win((int)ex));
        }
        inm[lr - 1][lc - 1] = (uint8_t)m;
    }
    __syncthreads();
    for (int i = tid; i < kTileR * kTileC; i += 256) {
        const int tr = i / kTileC, tc = i % kTileC;
        const int r = r0 + tr, c = c0 + tc;
        unsigned s = 0;
        if (r < p.rows && c < p.cols) {
            const bool interior = r >= 1 && r <= p.rows - 2 && c >= 1 && c <= p.cols - 2;
            const unsigned b = cls[tr + 2][tc + 2];
            if (interior && b == PARGO_FLOW_INERT) {
                s = 1u << 14;
            } else if (interior && b != PARGO_FLOW_NODATA) {
                const unsigned mine = inm[tr + 1][tc + 1];
                // per inflow bit j: the neighbour is interior (intn), is a
                // source (srcn: nothing drains into it), may be waited for
                // (it precedes the cell in the one-sweep order, or any in
                // the converging mode).  Eight unconditional reads and mask
                // arithmetic, so that no wave loops over its busiest cell.
                unsigned srcn = 0, intn = 0xFFu;
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const int k = win_of_bit(j);
                    srcn |= (inm[tr + 1 + k / 3 - 1][tc + 1 + k % 3 - 1] == 0 ? 1u : 0u) << j;
                }
                // only a cell next to the border has neighbours outside the interior
                if (r <= 1 || r >= p.rows - 2 || c <= 1 || c >= p.cols - 2) {
                    intn = 0;
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        const int k = win_of_bit(j);
                        const int ur = r + k / 3 - 1, uc = c + k % 3 - 1;
                        intn |= (ur >= 1 && ur <= p.rows - 2 && uc >= 1 && uc <= p.cols - 2 ? 1u : 0u) << j;
                    }
                }
                const unsigned waitable = p.converge ? 0xFFu : 0x0Fu;  // window bits 0-3: NW, N, NE, W
                const unsigned in_int = mine & intn;
                const unsigned nsrc = __builtin_popcount(in_int & srcn);
                const unsigned npend = __builtin_popcount(in_int & ~srcn & waitable);
                const unsigned poison = ((mine & ~intn) | (in_int & ~srcn & ~waitable)) != 0 ? 1u : 0u;
                const unsigned f = flow_of(b);
                unsigned feeds = 0;
                if (f != kNone && mine != 0 && (p.converge || f > 4)) {
                    // the target counts this cell when its inflow mask has it
                    const int trr = r + (int)f / 3 - 1, tcc = c + (int)f % 3 - 1;
                    const bool t_interior = trr >= 1 && trr <= p.rows - 2 && tcc >= 1 && tcc <= p.cols - 2;
                    const unsigned tm = inm[tr + 1 + (int)f / 3 - 1][tc + 1 + (int)f % 3 - 1];
                    feeds = (t_interior && ((tm >> bit_of_win(8 - (int)f)) & 1u)) ? 1u : 0u;
                }
                s = npend | (nsrc << 4) | (poison << 8) | (feeds << 9) | ((f == kNone ? 0u : f) << 10) | (1u << 14);
            }
        }
        stw[i] = (uint16_t)s;
    }
}

// One step of a walk: the cell that `idx` (tile row * kTileC + column) with
// code k drains to, -1 outside the tile.
__device__ __forceinline__ int step_to(int idx, int k)
{
    const int r = (idx >> 6) + (int)((unsigned)k / 3u) - 1, c = (idx & 63) + (int)((unsigned)k % 3u) - 1;
    static_assert(kTileC == 64, "a tile row is 64 cells");
    return (unsigned)r < (unsigned)kTileR && (unsigned)c < (unsigned)kTileC ? r * kTileC + c : -1;
}

// Where a walk goes from a cell: the next cell's index in the tile, or
// kLeaves + the cell's slot when it drains out of the tile, or kEnds.
constexpr unsigned kLeaves = 0x8000u, kEnds = 0xffffu;
__device__ __forceinline__ unsigned next_of(int idx, unsigned s)
{
    if (!feeds_of(s)) return kEnds;
    const int t = step_to(idx, code_of(s));
    return t >= 0 ? (unsigned)t : kLeaves + (unsigned)slot_of(idx >> 6, idx & 63);
}

// The cells where walks start, gathered into one list so that they fill as
// few waves as they can (30 to 60 of a tile's cells start a walk, and a hop
// costs a wave the same for one lane as for 64).  A start that is not on the
// perimeter has a source inside the tile draining to it.
constexpr int kStarts = kTileN / 2 + 512;
static_assert(kStarts >= kTileN / 2 + kSlots, "every start has a place");
struct StartList {
    uint16_t cell[kStarts];
    unsigned n;
};
// A thread's cells from here on: column `lane` of tile rows wave + 4k.
__device__ __forceinline__ int my_cell(int k) { return ((int)(threadIdx.x >> 6) + 4 * k) * kTileC + (int)(threadIdx.x & 63); }
// Adds the thread's cells k with bit k of `m` set (all lanes call).
__device__ __forceinline__ void add_starts(StartList &L, unsigned m)
{
    if (__builtin_amdgcn_ballot_w64(m != 0) == 0) return;
    // the lanes' counts, up to 8 each, summed bit by bit over the lanes below
    unsigned before = 0, total = 0;
    const unsigned n = (unsigned)__builtin_popcount(m);
#pragma unroll
    for (int bit = 0; bit < 4; bit++) {
        const unsigned long long b = __builtin_amdgcn_ballot_w64((n >> bit) & 1u);
        before += __builtin_amdgcn_mbcnt_hi((unsigned)(b >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)b, 0u)) << bit;
        total += (unsigned)__builtin_popcountll(b) << bit;
    }
    unsigned at = 0;
    if ((threadIdx.x & 63) == 0) at = atomicAdd(&L.n, total);
    at = (unsigned)__builtin_amdgcn_readfirstlane((int)at) + before;
    for (; m; m &= m - 1) L.cell[at++] = (uint16_t)my_cell(__builtin_ctz(m));
}
// next_of for a cell whose next cell lies in the tile (perimeter cells are
// set by next_of afterwards): the index plus the code's offset, by a byte
// lookup for codes 0..7 (the centre, code 4, never feeds).
__device__ __forceinline__ unsigned next_inside(int idx, unsigned s)
{
    const unsigned code = (s >> 10) & 15u;
    const int off = code == 8u ? 65 : (int)(int8_t)__builtin_amdgcn_perm(0x403F0100u, 0xFFC1C0BFu, code);
    return feeds_of(s) ? (unsigned)(idx + off) & 0xFFFFu : kEnds;
}

union LocalShared {
    SwarTile swar;
    GeneralTile general;
    unsigned acc[kTileN];  // once the static words are formed
};

__global__ __launch_bounds__(256) void sca_local_kernel(ScaParams p)
{
    __shared__ LocalShared S;
    __shared__ __align__(16) uint16_t stw[kTileN], nxt[kTileN];
    __shared__ StartList starts;
    __shared__ uint8_t entry[kSlotStride];
    __shared__ unsigned entries;
    const int tid = threadIdx.x;
    const int tile = xcd_tile(p);
    if (tile >= p.ntiles) return;  // the whole workgroup
    if (tid == 0) starts.n = entries = 0;
    const int ty = tile / p.tiles_x, tx = tile - ty * p.tiles_x;
    const int r0 = ty * kTileR, c0 = tx * kTileC;
    static_assert(kSwarTileR == kTileR && kSwarTileC == kTileC, "one tile shape");
    const bool inner = sca_swar_tile(p, r0, c0);
    if (inner) swar_words(p, S.swar, stw, r0, c0);
    else general_words(p, S.general, stw, r0, c0);
    __syncthreads();
    const unsigned long long slot0 = (unsigned long long)tile * (kNarrow ? p.slots : kSlotStride);
    // the pending inflows of this thread's perimeter cell from outside the tile
    const int pcell = tid < kSlots ? cell_of_slot(tid) : 0;
    unsigned ext = 0;
    if (tid < kSlots) {
        const int lr = pcell >> 6, lc = pcell & 63;
        auto inm_at = [&](int r, int c) -> unsigned {
            return inner ? reinterpret_cast<const uint8_t *>(S.swar.inm[r + 1])[c + 4] : S.general.inm[r + 1][c + 1];
        };
        // inflows from outside that may be waited for, of a cell that waits
        // at all: bits 0-2 come from the row above, 5-7 from the row below,
        // 0, 3, 5 from the left and 2, 4, 7 from the right
        unsigned m = (stw[pcell] & 15u) ? inm_at(lr, lc) : 0u;
        m &= (lr == 0 ? 0x07u : 0u) | (lr == kTileR - 1 ? 0xE0u : 0u) | (lc == 0 ? 0x29u : 0u) | (lc == kTileC - 1 ? 0x94u : 0u);
        if (!p.converge) m &= 0x0Fu;
        for (; m; m &= m - 1) {
            const int j = __builtin_ctz(m);
            const unsigned k = (unsigned)win_of_bit(j);
            const int ur = lr + (int)(k / 3u) - 1, uc = lc + (int)(k % 3u) - 1, gr = r0 + ur, gc = c0 + uc;
            const bool interior = inner || (gr >= 1 && gr <= p.rows - 2 && gc >= 1 && gc <= p.cols - 2);
            if (interior && inm_at(ur, uc) != 0) ext |= 1u << j;
        }
    }
    const unsigned next_ = (unsigned)__builtin_popcount(ext);
    // the static words go out as they are; the tile keeps them with the
    // awaited inflows from inside only
    if constexpr (kNarrow) {
        for (int i = tid; i < kTileN; i += 256)
            if ((i >> 6) < p.h && (i & 63) < p.w) p.st[((long long)tile * p.h + (i >> 6)) * p.w + (i & 63)] = stw[i];
    } else {
        const uint4 words = *reinterpret_cast<const uint4 *>(stw + 8 * tid);
        *reinterpret_cast<uint4 *>(p.st + (long long)tile * kTileN + 8 * tid) = words;
    }
    unsigned s[kTileN / 256];
#pragma unroll
    for (int k = 0; k < kTileN / 256; k++) {
        s[k] = stw[my_cell(k)];
        nxt[my_cell(k)] = (uint16_t)next_inside(my_cell(k), s[k]);
    }
    if (ext) entry[atomicAdd(&entries, 1u)] = (uint8_t)tid;
    __syncthreads();  // the classes and masks are read
#pragma unroll
    for (int k = 0; k < kTileN / 256; k++)
        S.acc[my_cell(k)] = (1u + nsrc_of(s[k])) | ((unsigned)poisoned_of(s[k]) << kLocBad) | (npend_of(s[k]) << kLocPend);
    __syncthreads();
    if (tid < kSlots) nxt[pcell] = (uint16_t)next_of(pcell, stw[pcell]);
    if (ext) S.acc[pcell] += (next_ << kLocExt) - (next_ << kLocPend);
    __syncthreads();
    {
        unsigned m = 0;  // cells that wait for nothing and feed
#pragma unroll
        for (int k = 0; k < kTileN / 256; k++)
            m |= (unsigned)(feeds_of(s[k]) && (S.acc[my_cell(k)] >> kLocPend) == 0) << k;
        add_starts(starts, m);
    }
    __syncthreads();
    for (unsigned i = tid; i < starts.n; i += 256) {
        unsigned t = starts.cell[i], v = S.acc[t];
        t = nxt[t];
        while (t < kLeaves) {
            // areas, and inflows from outside, go on only with a done cell
            const unsigned add = ((v >> kLocBad) & 15u ? 1u << kLocBad : v & ((1u << kLocBad) - 1)) - (1u << kLocPend);
            const unsigned after = nxt[t];
            v = atomicAdd(&S.acc[t], add) + add;
            if ((v >> kLocPend) != 0) break;  // others are on their way
            t = after;
        }
    }
    // the exit that each entry leads to (by the waves that walk least); a
    // cycle of codes leads to none
    for (unsigned i = (unsigned)tid ^ 192u; i < entries; i += 256) {
        const unsigned slot = entry[i];
        unsigned t = (unsigned)cell_of_slot((int)slot);
        for (int n = 0; n < kTileN && t < kLeaves; n++) t = nxt[t];
        unsigned at = slot, exit = t >= kLeaves && t != kEnds ? t - kLeaves : 255u;
        if constexpr (kNarrow) {
            const int in = cell_of_slot((int)slot);
            at = mem_slot(p, in >> 6, in & 63);
            if (exit != 255u) {
                const int out = cell_of_slot((int)exit);
                exit = mem_slot(p, out >> 6, out & 63);
            }
        }
        p.link[slot0 + at] = (uint8_t)exit;
    }
    __syncthreads();
    if (kNarrow ? tid < kSlots && has_slot(p, pcell >> 6, pcell & 63) : tid < kSlotStride) {
        unsigned long long x = kExitNever;
        unsigned to = kNoExit;
        if (tid < kSlots) {
            const unsigned s = stw[pcell], v = S.acc[pcell], t = nxt[pcell];
            const int k = code_of(s);
            if (t >= kLeaves && t != kEnds) {
                const int gr = r0 + (pcell >> 6) + k / 3 - 1, gc = c0 + (pcell & 63) + k % 3 - 1;
                const int beside = (gr / kTileR) * p.tiles_x + gc / kTileC;
                to = (unsigned)beside * (unsigned)(kNarrow ? p.slots : kSlotStride) +
                     mem_slot(p, gr % kTileR, gc % kTileC);
                if ((v >> kLocPend) == 0) {
                    const unsigned n = (v >> kLocExt) & 255u;
                    if ((v >> kLocBad) & 15u) x = kExitStart | (1ull << kExitBad);  // not done, whatever arrives
                    else x = (v & kLocSum) | ((unsigned long long)n << kExitPend) | (n == 0 ? kExitStart : 0ull);
                }
            }
        }
        const unsigned at = kNarrow ? mem_slot(p, pcell >> 6, pcell & 63) : (unsigned)tid;
        p.exits[slot0 + at] = x;
        p.next[slot0 + at] = to;
        p.ext[slot0 + at] = (uint8_t)ext;
    }
}

// Each exit's successor: the exit that the perimeter cell it enters leads
// to, none if that one awaits nothing (it is not done whatever arrives) or
// never completes.
__global__ __launch_bounds__(256) void sca_link_kernel(ScaParams p, unsigned n)
{
    const unsigned i = blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    const unsigned to = p.next[i];
    if (to == kNoExit) return;
    const unsigned slot = p.link[to];
    unsigned x = kNoExit;
    if (slot != 255u) {
        const unsigned per = (unsigned)(kNarrow ? p.slots : kSlotStride);
        x = to / per * per + slot;
        const unsigned pend = (unsigned)(p.exits[x] >> kExitPend) & 255u;
        if (pend == 0 || pend == 255u) x = kNoExit;
    }
    p.next[i] = x;
}

// Walks over the exits: kCrossPer slots per lane, each lane going on to its
// next slot when its walk has ended.
constexpr int kCrossPer = 8;

__global__ __launch_bounds__(256) void sca_cross_kernel(ScaParams p, unsigned n)
{
    const unsigned base = blockIdx.x * (256u * kCrossPer) + threadIdx.x;
    unsigned starts = 0;
    unsigned long long w[kCrossPer];
#pragma unroll
    for (int k = 0; k < kCrossPer; k++) {
        const unsigned i = base + 256u * k;
        // an exit that awaits something changes while others arrive, but its
        // start flag does not
        w[k] = i < n ? __atomic_load_n(&p.exits[i], __ATOMIC_RELAXED) : 0ull;
    }
#pragma unroll
    for (int k = 0; k < kCrossPer; k++) starts |= (unsigned)((w[k] & kExitStart) != 0) << k;
    unsigned at = kNoExit;
    unsigned long long v = 0;
    for (;;) {
        if (at == kNoExit) {
            if (starts == 0) break;
            const int k = __builtin_ffs((int)starts) - 1;
            starts &= starts - 1;
            const unsigned i = base + 256u * (unsigned)k;
            at = p.next[i];
            v = 0;
#pragma unroll
            for (int q = 0; q < kCrossPer; q++)
                if (q == k) v = w[q];
        }
        if (at != kNoExit) {
            const unsigned after = p.next[at];
            const unsigned long long add =
                ((v >> kExitBad) & 255ull ? 1ull << kExitBad : v & ((1ull << kExitPend) - 1)) - (1ull << kExitPend);
            v = atomicAdd(&p.exits[at], add) + add;
            at = ((v >> kExitPend) & 255ull) == 0 ? after : kNoExit;
        }
    }
}

__global__ __launch_bounds__(256) void sca_final_kernel(ScaParams p)
{
    __shared__ unsigned long long acc[kTileN];
    __shared__ __align__(16) uint16_t nxt[kTileN];
    __shared__ StartList starts;
    const int tid = threadIdx.x;
    const int tile = xcd_tile(p);
    if (tile >= p.ntiles) return;  // the whole workgroup
    if (tid == 0) starts.n = 0;
    const int ty = tile / p.tiles_x, tx = tile - ty * p.tiles_x;
    const int r0 = ty * kTileR, c0 = tx * kTileC;
    uint4 words;
    if constexpr (!kNarrow) words = *reinterpret_cast<const uint4 *>(p.st + (long long)tile * kTileN + 8 * tid);
    const int pcell = tid < kSlots ? cell_of_slot(tid) : 0;
    // What arrives at this thread's perimeter cell from outside.  The words
    // of its first three inflows are all requested before one is looked at;
    // more than three drain only into a few corners.
    const unsigned long long slot0 = (unsigned long long)tile * (kNarrow ? p.slots : kSlotStride);
    auto static_word = [&](int i) -> unsigned {  // of cell i of the tile
        if constexpr (!kNarrow) return p.st[(long long)tile * kTileN + i];
        return (i >> 6) < p.h && (i & 63) < p.w ? p.st[((long long)tile * p.h + (i >> 6)) * p.w + (i & 63)] : 0u;
    };
    const unsigned mine = kNarrow ? mem_slot(p, pcell >> 6, pcell & 63) : (unsigned)tid;
    const unsigned ext = tid < kSlots && has_slot(p, pcell >> 6, pcell & 63) ? p.ext[slot0 + mine] : 0u;
    const unsigned pword = tid < kSlots ? static_word(pcell) : 0u;
    unsigned long long arrived = 0;
    if (ext) {
        auto word = [&](unsigned e) -> unsigned long long {  // of the lowest inflow in e
            const unsigned k = (unsigned)win_of_bit(__builtin_ctz(e));
            const unsigned gr = (unsigned)(r0 + (pcell >> 6) - 1) + k / 3u, gc = (unsigned)(c0 + (pcell & 63) - 1) + k % 3u;
            return p.exits[(unsigned long long)((gr / kTileR) * (unsigned)p.tiles_x + gc / kTileC) *
                               (unsigned)(kNarrow ? p.slots : kSlotStride) +
                           mem_slot(p, (int)(gr % kTileR), (int)(gc % kTileC))];
        };
        auto arrival = [&](unsigned long long x) -> unsigned long long {
            if (((x >> kExitPend) & 255ull) != 0) return 0;  // never complete
            return ((x >> kExitBad) & 255ull ? 1ull << kFinBad : x & kFinSum) - (1ull << kFinPend);
        };
        unsigned e = ext;
        unsigned long long x[3];
#pragma unroll
        for (int q = 0; q < 3; q++) {
            x[q] = kExitNever;
            if (e) x[q] = word(e);
            e &= e - 1;
        }
        for (; e; e &= e - 1) arrived += arrival(word(e));
#pragma unroll
        for (int q = 0; q < 3; q++) arrived += arrival(x[q]);
    }
    if constexpr (kNarrow) {
        for (int i = tid; i < kTileN; i += 256) nxt[i] = (uint16_t)static_word(i);
    } else {
        *reinterpret_cast<uint4 *>(nxt + 8 * tid) = words;
    }
    __syncthreads();
    unsigned s[kTileN / 256];
#pragma unroll
    for (int k = 0; k < kTileN / 256; k++) {
        s[k] = nxt[my_cell(k)];  // each cell's word is read and written by one thread
        nxt[my_cell(k)] = (uint16_t)next_inside(my_cell(k), s[k]);
        acc[my_cell(k)] = area_of(s[k]) ? kFinArea | (1ull + nsrc_of(s[k])) |
                                              ((unsigned long long)poisoned_of(s[k]) << kFinBad) |
                                              ((unsigned long long)npend_of(s[k]) << kFinPend)
                                        : 0ull;
    }
    __syncthreads();
    if (tid < kSlots) nxt[pcell] = (uint16_t)next_of(pcell, pword);
    if (ext) acc[pcell] += arrived;
    __syncthreads();
    {
        unsigned m = 0;  // cells that wait for nothing and feed
#pragma unroll
        for (int k = 0; k < kTileN / 256; k++)
            m |= (unsigned)(feeds_of(s[k]) && ((acc[my_cell(k)] >> kFinPend) & 15ull) == 0) << k;
        add_starts(starts, m);
    }
    __syncthreads();
    for (unsigned i = tid; i < starts.n; i += 256) {
        unsigned t = starts.cell[i];
        unsigned long long v = acc[t];
        t = nxt[t];
        while (t < kLeaves) {
            const unsigned long long add = ((v >> kFinBad) & 15ull ? 1ull << kFinBad : v & kFinSum) - (1ull << kFinPend);
            const unsigned after = nxt[t];
            v = atomicAdd(&acc[t], add) + add;
            if (((v >> kFinPend) & 15ull) != 0) break;  // others are on their way
            t = after;
        }
    }
    __syncthreads();
    const int lane = tid & 63, wave = tid >> 6, c = c0 + lane;
    if (c >= p.cols) return;
#pragma unroll
    for (int k = 0; k < kTileR / 4; k++) {
        const int tr = wave + 4 * k, r = r0 + tr;
        if (r >= p.rows) break;
        const unsigned long long v = acc[tr * kTileC + lane];
        const double a = v & kFinArea ? (double)(v & kFinSum) : p.nodata;
        __builtin_nontemporal_store(a, &p.area[(long long)r * p.pitch + c]);
        if (r >= p.rows - 3 && c >= p.cols - 3)
            p.last_done[(r - (p.rows - 3)) * 3 + (c - (p.cols - 3))] = (v >> kFinBad) == kFinArea >> kFinBad ? 1u : 0u;
    }
}

// The reference's last work cell (rows-2, cols-2) always runs the pull
// loop (scaOperator.cpp:86-108).  When it is NoData (or a cell that takes no
// inflow) it adds, in window order, the area of every interior inflowing
// neighbour that is done; all of those precede it in row-major order.
__global__ void sca_last_cell_kernel(ScaParams p)
{
    const int r = p.rows - 2, c = p.cols - 2;
    const unsigned b = load_class(p, r, c);
    if (is_valid(b)) return;
    double v = b == PARGO_FLOW_NODATA ? p.nodata : 1.0;
    for (int k = 0; k < 9; k++) {
        if (k == 4) continue;
        const int ur = r + k / 3 - 1, uc = c + k % 3 - 1;
        if (ur < 1 || ur > p.rows - 2 || uc < 1 || uc > p.cols - 2) continue;
        if (flow_of(load_class(p, ur, uc)) != (unsigned)(8 - k)) continue;
        if (p.last_done[(ur - (p.rows - 3)) * 3 + (uc - (p.cols - 3))]) v += p.area[(long long)ur * p.pitch + uc];
    }
    p.area[(long long)r * p.pitch + c] = v;
}

#ifndef PARGO_SCA_NARROW
// Reference D8 layer (double) to flow classes: NoData when
// fabs(v - nodata) < 1e-6, valid when > 1e-6 (scaOperator.cpp:48,71), and
// neither (NaN) marks a cell that takes no inflow.  A valid cell flows to
// window index k when v == k; it rejects inflow from window cell k when
// dir + v == 8 in double for dir = 8 - k (scaOperator.cpp:71,94).
// A whole number 0..8 needs no search; the others that can satisfy either
// equation lie strictly between -1 and 9.
__device__ __forceinline__ unsigned classify(double v, double nodata)
{
    const double dv = fabs(v - nodata);
    if (dv < 0.000001) return PARGO_FLOW_NODATA;
    if (!(dv > 0.000001)) return PARGO_FLOW_INERT;
    if (!(v > -1.0 && v < 9.0)) return PARGO_FLOW_NONE;
    const int whole = (int)v;
    if ((double)whole == v) return whole == 4 ? (unsigned)PARGO_FLOW_NONE : (unsigned)whole;
    unsigned ex = kNone;
    for (int dir = 0; dir <= 8; dir++)
        if (dir != 4 && (double)dir + v == 8.0) ex = 8u - (unsigned)dir;
    return ex != kNone ? PARGO_FLOW_EXCL | ex : (unsigned)PARGO_FLOW_NONE;
}

// Memory-bound (9 bytes a cell): four cells a lane, as two 16-byte loads and
// one 4-byte store (5003 x 7001: 56 us, one cell a lane took 101).
typedef double f64x2_a8 __attribute__((ext_vector_type(2), aligned(8)));

__global__ __launch_bounds__(256) void d8_classify_kernel(const double *__restrict__ d8, uint8_t *__restrict__ out,
                                                          long long pitch, int rows, int cols, double nodata)
{
    const int c = (blockIdx.x * 256 + threadIdx.x) * 4, r = blockIdx.y;
    if (c >= cols) return;
    const long long i = (long long)r * pitch + c;
    if (c + 4 <= cols) {
        const f64x2_a8 a = *reinterpret_cast<const f64x2_a8 *>(d8 + i), b = *reinterpret_cast<const f64x2_a8 *>(d8 + i + 2);
        const unsigned w = classify(a.x, nodata) | classify(a.y, nodata) << 8 | classify(b.x, nodata) << 16 |
                           classify(b.y, nodata) << 24;
        *reinterpret_cast<u32_b1 *>(out + i) = w;
    } else {
        for (int k = 0; c + k < cols; k++) out[i + k] = (uint8_t)classify(d8[i + k], nodata);
    }
}

// NoData values the flow classes cannot carry: the reference would treat
// NoData cells holding a code as draining, and border degrees equal to 0 or
// -1 as available.
bool sca_nodata_ok(double nodata)
{
    if (std::isnan(nodata)) return false;
    for (int k = -1; k <= 8; k++)
        if (std::fabs(nodata - (double)k) <= 0.000002) return false;
    return true;
}

#endif

}  // namespace

#ifdef PARGO_SCA_NARROW
int sca_narrow
#else
static int sca_full
#endif
    (pargo_ctx *ctx, const pargo_grid *g, const uint8_t *flow, const uint32_t *nodata_mask, int mode, double *sca_out)
{
    const int tiles_x = (g->cols + kTileC - 1) / kTileC;
    const long long ntiles = (long long)tiles_x * ((g->rows + kTileR - 1) / kTileR);
    ScaParams p{};
    p.w = kNarrow ? std::min(g->cols, kTileC) : kTileC;
    p.h = kNarrow ? std::min(g->rows, kTileR) : kTileR;
    p.slots = !kNarrow ? kSlotStride : 2 * (tiles_x == 1 ? p.w : p.h);
    // scratch: the last-cell flags, the exit words of the perimeter slots, the
    // tiles' static words (2 bytes per cell, an even number of them) and, per
    // slot again, its successor, the entry's exit and its inflows from outside
    constexpr size_t head = 256;
    const size_t slots = (size_t)ntiles * p.slots, cells = ((size_t)ntiles * p.w * p.h + 1) & ~(size_t)1;
    const int rc = ensure_scratch(ctx, head + cells * sizeof(uint16_t) + slots * (8 + 4 + 1 + 1));
    if (rc) return rc;
    char *scr = static_cast<char *>(ctx->scratch);
    p.flow = flow;
    p.mask = nodata_mask;
    p.area = sca_out;
    p.last_done = reinterpret_cast<unsigned *>(scr);
    p.exits = reinterpret_cast<unsigned long long *>(scr + head);
    p.st = reinterpret_cast<uint16_t *>(p.exits + slots);
    p.next = reinterpret_cast<unsigned *>(p.st + cells);
    p.link = reinterpret_cast<uint8_t *>(p.next + slots);
    p.ext = p.link + slots;
    p.pitch = g->pitch ? g->pitch : g->cols;
    p.rows = g->rows;
    p.cols = g->cols;
    p.mask_words = (g->cols + 31) / 32;
    p.tiles_x = tiles_x;
    p.ntiles = (int)ntiles;
    p.converge = mode == PARGO_SCA_CONVERGE;
    p.nodata = g->nodata;
    const dim3 tiles(8 * (unsigned)((ntiles + 7) / 8)), threads(256);
    const unsigned n = (unsigned)slots;
    hipLaunchKernelGGL(sca_local_kernel, tiles, threads, 0, ctx->stream, p);
    hipLaunchKernelGGL(sca_link_kernel, dim3((n + 255u) / 256u), threads, 0, ctx->stream, p, n);
    constexpr unsigned per = 256u * kCrossPer;
    hipLaunchKernelGGL(sca_cross_kernel, dim3((n + per - 1) / per), threads, 0, ctx->stream, p, n);
    hipLaunchKernelGGL(sca_final_kernel, tiles, threads, 0, ctx->stream, p);
    if (mode == PARGO_SCA_REFERENCE && g->rows >= 3 && g->cols >= 3)
        hipLaunchKernelGGL(sca_last_cell_kernel, dim3(1), dim3(1), 0, ctx->stream, p);
    return check_launch(ctx, "pargo_sca_d8");
}

}  // namespace pargo

#ifndef PARGO_SCA_NARROW

using pargo::fail;

extern "C" int pargo_d8_classify(pargo_ctx *ctx, const pargo_grid *g, const double *d8, uint8_t *flow_out)
{
    if (!ctx) return PARGO_E_INVALID;
    if (!g || !d8 || !flow_out) return fail(ctx, PARGO_E_INVALID, "pargo_d8_classify: null argument");
    if (g->rows < 1 || g->cols < 1) return fail(ctx, PARGO_E_INVALID, "empty grid (%d x %d)", g->rows, g->cols);
    const long long pitch = g->pitch ? g->pitch : g->cols;
    if (pitch < g->cols) return fail(ctx, PARGO_E_INVALID, "pitch %lld < cols %d", pitch, g->cols);
    if (!pargo::sca_nodata_ok(g->nodata))
        return fail(ctx, PARGO_E_INVALID,
                    "D8 NoData value %.17g is NaN or within 2e-6 of a code in -1..8, which the flow classes "
                    "cannot represent",
                    g->nodata);
    int rc = pargo::bind(ctx);
    if (rc) return rc;
    dim3 grid((g->cols + 1023) / 1024, g->rows);
    hipLaunchKernelGGL(pargo::d8_classify_kernel, grid, dim3(256), 0, ctx->stream, d8, flow_out, pitch, g->rows,
                       g->cols, g->nodata);
    return pargo::check_launch(ctx, "pargo_d8_classify");
}

extern "C" int pargo_sca_d8(pargo_ctx *ctx, const pargo_grid *g, const uint8_t *flow, const uint32_t *nodata_mask,
                            int mode, double *sca_out)
{
    if (!ctx) return PARGO_E_INVALID;
    if (!g || !flow || !sca_out) return fail(ctx, PARGO_E_INVALID, "pargo_sca_d8: null argument");
    if (g->rows < 1 || g->cols < 1) return fail(ctx, PARGO_E_INVALID, "empty grid (%d x %d)", g->rows, g->cols);
    if (mode != PARGO_SCA_REFERENCE && mode != PARGO_SCA_CONVERGE)
        return fail(ctx, PARGO_E_INVALID, "unknown SCA mode %d", mode);
    const long long pitch = g->pitch ? g->pitch : g->cols;
    if (pitch < g->cols) return fail(ctx, PARGO_E_INVALID, "pitch %lld < cols %d", pitch, g->cols);
    if ((long long)g->rows * g->cols >= (1ll << 40))
        return fail(ctx, PARGO_E_INVALID, "grid of %lld cells exceeds the 2^40 area counter",
                    (long long)g->rows * g->cols);
    if (!pargo::sca_nodata_ok(g->nodata))
        return fail(ctx, PARGO_E_INVALID,
                    "D8 NoData value %.17g is NaN or within 2e-6 of a code in -1..8, which the flow classes "
                    "cannot represent",
                    g->nodata);
    int rc = pargo::bind(ctx);
    if (rc) return rc;
    const int tiles_x = (g->cols + pargo::kTileC - 1) / pargo::kTileC;
    const long long ntiles = (long long)tiles_x * ((g->rows + pargo::kTileR - 1) / pargo::kTileR);
    if (ntiles > (1ll << 24))
        return fail(ctx, PARGO_E_INVALID, "grid of %d x %d cells needs %lld tiles, more than 2^24", g->rows, g->cols,
                    ntiles);
    const bool narrow = g->cols <= pargo::kNarrowCols || g->rows <= pargo::kNarrowRows;
    return (narrow ? pargo::sca_narrow : pargo::sca_full)(ctx, g, flow, nodata_mask, mode, sca_out);
}

#endif
