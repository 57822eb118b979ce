// batch.hpp -- device code of the batched path shared by its translation
// units: the item descriptor, tile placement, and the smoothing and raster
// kernels as templates on the scale and the tile shape.  fused.hip holds the
// tables, the graph kernel and the host side; raster_tiles.hip is built once
// per tile shape and instantiates the kernels of that shape.
#pragma once

#include <type_traits>

#include "common.hpp"
#include "geom.hpp"
#include "graph.hpp"
#include "hull_table.hpp"
#include "pixel.hpp"
#include "strips.hpp"

namespace dpx {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

[[maybe_unused]] constexpr int kMaxScale = 15;
[[maybe_unused]] constexpr int kKeys = 4096;

__host__ __device__ constexpr int mask_kmin(int S) { return -(S / 2) - 1; }
__host__ __device__ constexpr int mask_w(int S) { return 2 * S + 2; }

struct DevItem {
    uint64_t in_off, out_off, g_off;
    int32_t W, H, stride, ch;
    uint32_t flags;
    int32_t out_stride, scale, subdivide;
    int32_t aligned16;  // output rows 16-byte aligned
    int32_t graph_w4;   // graph rows 4-byte aligned (W % 4 == 0)
    uint64_t pal_off;   // DPX_INDEXED: the palette's byte offset in the input arena
    uint64_t rows_off;  // subdivision: byte offset of the item's cell rows (kf_smooth)
};


// Summary of a cell's coverage rows at scale S: bit 0 = it covers every
// sample of its own square; bit 1 + (dy+1)*3 + (dx+1) = it covers a sample of
// the neighbouring square at (dx, dy).  The rows are those of samples y0 .. y0 +
// n - 1, their bits the samples from x0.
__host__ __device__ inline uint32_t coverage_info(const uint32_t* rows, int S, int x0, int y0, int n)
{
    const int c0 = -x0;  // bit of the own square's first column
    const uint32_t own = ((1u << S) - 1u) << c0;
    uint32_t info = 0;
    bool full = true;
    for (int r = 0; r < n; r++) {
        int ky = y0 + r;
        int dy = ky < 0 ? -1 : (ky >= S ? 1 : 0);
        uint32_t row = rows[r];
        if (dy == 0 && (row & own) != own) full = false;
        if (row & ((1u << c0) - 1u)) info |= 1u << (1 + (dy + 1) * 3 + 0);
        if ((row & own) && dy != 0) info |= 1u << (1 + (dy + 1) * 3 + 1);
        if (row >> (c0 + S)) info |= 1u << (1 + (dy + 1) * 3 + 2);
    }
    return info | (full ? 1u : 0u);
}

// Cell masks: what a cell shows of the 3x3 cells around it, per cell the
// samples of all its rows at once.  Mask j = (1 - dy) * 3 + (1 - dx) is what
// the cell contributes as candidate (dx, dy) of the cell at (-dx, -dy) from
// it: up to 4x bit ky * S + q of 16, from 5x bit q of byte ky (sample q of row
// ky).  The masks of the table's keys follow its rows (kt_cell: 2 or 8 bytes
// a mask); a smoothed cell's are written by kf_smooth (2 or S bytes a mask,
// then the summary's low byte) in place of its rows.
constexpr int kMaxCellScale = 8, kMaxCellScale16 = 4;
__host__ __device__ constexpr size_t cell_table_bytes(int S)
{
    return S > kMaxCellScale ? 0 : (size_t)kKeys * 9 * (S <= kMaxCellScale16 ? 2 : 8);
}

// The rows of the nine masks of a cell with coverage rows `row(r)`, samples Y0 ..
// of N, their bits the samples from X0: put(j, ky, bits), those without any
// left out.
template <int S, int X0, int Y0, int N, class R, class F>
__host__ __device__ inline void cell_mask_rows(R row, F put)
{
#pragma unroll
    for (int j = 0; j < 9; j++) {
        const int dy = 1 - j / 3, dx = 1 - j % 3, sh = -dx * S - X0;
#pragma unroll
        for (int ky = 0; ky < S; ky++) {
            const int r = ky - dy * S - Y0;
            if (r < 0 || r >= N) continue;
            put(j, ky, (sh >= 0 ? (row(r) >> sh) : (row(r) << -sh)) & ((1u << S) - 1u));
        }
    }
}

// A cell whose own square it covers fully, and into which none of the four
// cells drawn after it (up-left, up, up-right, right) reaches, shows its own
// colour on all of its S*S output pixels.
__device__ inline bool simple_cell(uint32_t own, uint32_t upl, uint32_t up, uint32_t upr, uint32_t right)
{
    return (own & 1u) && !((upl >> 3) & 1u) && !((up >> 2) & 1u) && !((upr >> 1) & 1u) && !((right >> 4) & 1u);
}

// ---------------------------------------------------------------------------
// work distribution: block -> (item, tile column, tile row).  When every item
// of a launch has the same tile grid, the launch grid is (tile columns, tile
// rows, items) and the block index says it all; otherwise the grid is 1-D
// over all tiles and a map built on the host gives each block its item and
// tile: tile_map[b] = (item, tile row << 16 | tile column).
// ---------------------------------------------------------------------------
struct TileAt {
    int item, tx, ty;
};

// The blocks are permuted in groups of 8 * RUN: the hardware hands consecutive
// blocks to the 8 XCDs in turn, and within a group XCD x is given the RUN
// consecutive tiles x * RUN .. x * RUN + RUN - 1 (a row of horizontally
// adjacent tiles), so the input and graph lines that adjacent tiles share are
// fetched into one XCD's L2 once, not into several.  Blocks past the last
// whole group keep their place.
template <int RUN>
__device__ inline TileAt locate_tile(const uint2* __restrict__ tile_map, int grid3d)
{
    const uint32_t n = gridDim.x * gridDim.y * gridDim.z;
    uint32_t b = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    if (b < n / (8 * RUN) * (8 * RUN)) {
        const uint32_t w = b % (8 * RUN);
        b += (w % 8) * RUN + w / 8 - w;
    }
    if (grid3d) {
        const uint32_t plane = gridDim.x * gridDim.y, r = b % plane;
        return TileAt{ (int)(b / plane), (int)(r % gridDim.x), (int)(r / gridDim.x) };
    }
    const uint2 m = tile_map[b];
    return TileAt{ (int)m.x, (int)(m.y & 0xFFFFu), (int)(m.y >> 16) };
}

// ---------------------------------------------------------------------------
// kf_raster: heuristic crossing resolution, cells and the gather raster of a
// tile of cells
// ---------------------------------------------------------------------------
// Raster tiles of TX x (256 / TX) cells, one own cell per thread of a
// 256-thread block (32x8 by default; 16x16 and 64x4 are the other shapes an
// item may be given).
template <int TX>
struct TileShape {
    static constexpr int X = TX, Y = 256 / TX;
    static_assert(X * Y == 256 && X % 4 == 0, "one own cell per thread, whole words per row");
    static constexpr int CX = X + 2, CY = Y + 2;       // candidate cells, halo 1
    static constexpr int DW = X / 4 + 2, DB = 4 * DW;  // data words / bytes of a window row
    static constexpr int WW = DW + 2, WB = 4 * WW;     // words / bytes of a window row
    static constexpr int GY = Y + 2, AY = GY + 2;      // resolved rows, snapshot rows
    // the window loads and the decision clear take one word per thread
    static_assert(AY * WW <= 256 && (GY + 1) * WW <= 256, "a window fits one pass of 256 threads");
};
constexpr int kDefaultTileX = 32;
constexpr uint16_t kNoCell = 0xFFFF;

// LDS windows of the raster tile hold graph bytes in rows of WW 32-bit
// words; word w of a row holds x = x0 - 8 + 4w .. x0 - 5 + 4w.  Words
// 1..DW (x0 - 4 .. x0 + X + 3) carry data, words 0 and DW + 1 stay zero.
// Resolved rows y0 - 1 .. y0 + Y (GY rows: the candidate cells' rows, whose
// keys take the bytes left and right of them too); resolving them reads one
// more snapshot row on each side (AY rows).
#define DPX_TILE_NAMES(TX)                                                                                 \
    using TS = TileShape<TX>;                                                                              \
    constexpr int RTX = TS::X, RTY = TS::Y, RCX = TS::CX, RCY = TS::CY, RWW = TS::WW, RWB = TS::WB;        \
    constexpr int GY = TS::GY, AY = TS::AY, RDW = TS::DW, RDB = TS::DB;                                    \
    (void)RTX; (void)RTY; (void)RCX; (void)RCY; (void)RWW; (void)RWB; (void)GY; (void)AY; (void)RDW; (void)RDB

// Per-cell coverage of smoothed cells (kf_smooth -> kf_raster<S, true>): up to
// 8x the nine cell masks and the coverage summary, from 9x cover_h(S) words of
// sample rows and one of summary; cell (x, y) of an item at word (y * W + x) *
// rows_words(S) of its range.
__host__ __device__ constexpr int rows_words(int S) { return (int)cell_row_words(S); }

// The bytes of pixels (x .. x + 3, y) of a graph of the item, 0 where they
// lie outside the frame (x is a multiple of 4).  One load at any alignment
// also where the rows are not whole words (byte by byte, 64 smoothed frames of
// 251x223 took 168 us a batch at 2x, not 161, and 444 at 8x, not 437); it
// stays inside the item's slot, whose size is rounded up to 256 bytes.
__device__ inline uint32_t graph_word(const DevItem& it, const uint8_t* __restrict__ g, int x, int y)
{
    if ((unsigned)x >= (unsigned)it.W || (unsigned)y >= (unsigned)it.H) return 0u;
    const uint32_t off = (uint32_t)(y * it.W + x);
    if (it.graph_w4) return *reinterpret_cast<const uint32_t*>(g + off);
    const uint32_t at = min(off, (((uint32_t)(it.W * it.H) + 255u) & ~255u) - 4u);
    uint32_t v;
    __builtin_memcpy(&v, g + at, 4);
    v >>= 8u * (off - at);
    const int n = it.W - x;
    return n < 4 ? v & ((1u << (8 * n)) - 1u) : v;
}


// The snapshot rows ay0 .. ay0 + AY - 1 of a tile's window into LDS.
template <int TX>
__device__ inline void tile_snapshot_load(const DevItem& it, const uint8_t* __restrict__ aux, int x0, int ay0,
                                          uint32_t* s_aux32, int t)
{
    DPX_TILE_NAMES(TX);
    static_assert(AY * RWW <= 256, "a word a thread");
    if (t < AY * RWW) {
        const int r = t / RWW, w = t % RWW;
        s_aux32[t] = w >= 1 && w <= RDW ? graph_word(it, aux, x0 - 8 + 4 * w, ay0 + r) : 0u;
    }
}

// Heuristic crossing resolution (ambiguous_cross_Kernel) of a tile's window,
// after tile_snapshot_load and a barrier.  Only the pixels of crossed 2x2
// blocks (both diagonals present) change, and in the symmetric snapshot the
// block with lower-left pixel p is crossed iff p has bit 2 and its right
// neighbour bit 0.  1: list the crossed blocks of the window, four origins
// of a row per thread; 2: decide each listed block once
// (processHeuristics2), the walks reading the snapshot in LDS where they can
// and in HBM beyond the window; 3: remove the losing diagonals, four
// positions per thread, into s_g32 (resolved rows y0 - 1 .. y0 + RTY), and
// the tile's own resolved bytes into gfin when it is given.  s_p32 must
// have been cleared and *s_nblk zeroed before the barrier.
//
// The curve walks of the decisions (up to 31 steps) leave the small window
// on line-heavy frames, and each step outside it is a dependent HBM read.
// With WALK, a tile that has crossed blocks first loads a larger walk window
// of the snapshot into s_walk (an LDS buffer of WalkWindow<TX>::BYTES that
// the kernel uses only later): kWalkEX more bytes on each side and kWalkEY
// more rows above and below, so that no walk (at most 31 steps from a node
// next to a block of the small window) leaves it.  It costs every such tile
// 7-10 KB more reads, which a full batch pays in HBM time (20% of the
// 256x224 batch); it pays where dense crossing lattices make long walks the
// tile's critical path (640x480 frames at 8x), and the autotuner picks it
// per workload class.
constexpr int kWalkEX = 32, kWalkEY = 32;
template <int TX>
struct WalkWindow {
    static constexpr int B = TileShape<TX>::DB + 2 * kWalkEX;    // bytes per row (a multiple of 4)
    static constexpr int R = TileShape<TX>::AY + 2 * kWalkEY;    // rows
    static constexpr int BYTES = B * R;
};

template <int TX, bool WALK>
__device__ inline void tile_resolve(const DevItem& it, const uint8_t* __restrict__ aux, uint8_t* __restrict__ gfin,
                                    int x0, int y0, int ay0, const uint32_t* s_aux32, uint32_t* s_p32,
                                    uint16_t* s_blk, int* s_nblk, uint32_t* s_g32, uint32_t* s_walk, int t)
{
    DPX_TILE_NAMES(TX);
    using WW_ = WalkWindow<TX>;
    for (int k = t; k < (GY + 1) * RDW; k += 256) {
        const int r = k / RDW, w = k % RDW + 1;  // word w of snapshot row r: origins of blocks on rows r, r + 1
        const uint32_t* a = s_aux32 + r * RWW + w;
        uint32_t D = a[0];
        uint32_t cross = (D >> 2) & __builtin_amdgcn_alignbyte(a[1], D, 1) & 0x01010101u;
        while (cross) {
            int q = __builtin_ctz(cross) >> 3;
            cross &= cross - 1;
            s_blk[atomicAdd(s_nblk, 1)] = (uint16_t)(r * RWB + 4 * w + q);
        }
    }
    __syncthreads();
    const int nblk = *s_nblk;
    const bool walk_win = WALK && nblk > 0;  // uniform over the block
    const int ex0 = x0 - 4 - kWalkEX, ey0 = ay0 - kWalkEY;  // the walk window's first byte and row
    if (walk_win) {
        // all of a thread's loads are issued before the first is waited for
        // (a loop that stores each into LDS before the next load waits a
        // memory latency per iteration: 17 us instead of 2 for a tile)
        if (it.graph_w4) {  // x0 and kWalkEX are multiples of 4: whole words inside or outside the frame
            constexpr int NW = WW_::R * (WW_::B / 4), PER = (NW + 255) / 256;
            uint32_t v[PER];
#pragma unroll
            for (int q = 0; q < PER; q++) {
                const int k = t + 256 * q;
                const int r = k / (WW_::B / 4), w = k % (WW_::B / 4);
                const int x = ex0 + 4 * w, y = ey0 + r;
                v[q] = 0;
                if (k < NW && (unsigned)x < (unsigned)it.W && (unsigned)y < (unsigned)it.H)
                    v[q] = *reinterpret_cast<const uint32_t*>(aux + (uint32_t)(y * it.W + x));
            }
#pragma unroll
            for (int q = 0; q < PER; q++)
                if (t + 256 * q < NW) s_walk[t + 256 * q] = v[q];
        } else {
            constexpr int PER = (WW_::BYTES + 255) / 256;
            uint8_t* s8 = reinterpret_cast<uint8_t*>(s_walk);
            uint8_t v[PER];
#pragma unroll
            for (int q = 0; q < PER; q++) {
                const int k = t + 256 * q;
                const int x = ex0 + k % WW_::B, y = ey0 + k / WW_::B;
                v[q] = 0;
                if (k < WW_::BYTES && (unsigned)x < (unsigned)it.W && (unsigned)y < (unsigned)it.H)
                    v[q] = aux[(uint32_t)(y * it.W + x)];
            }
#pragma unroll
            for (int q = 0; q < PER; q++)
                if (t + 256 * q < WW_::BYTES) s8[t + 256 * q] = v[q];
        }
        __syncthreads();
    }
    {
        // (the window is read by words, so that the compiler keeps the LDS
        // and HBM reads apart instead of merging them into one generic load)
        auto get = [&](int gx, int gy) -> uint32_t {
            bool win;
            uint32_t v;
            if (walk_win) {
                const int wx = gx - ex0, wy = gy - ey0;
                win = (unsigned)wx < (unsigned)WW_::B && (unsigned)wy < (unsigned)WW_::R;
                const int c = win ? wy * WW_::B + wx : 0;
                v = (s_walk[c >> 2] >> (8 * (c & 3))) & 0xFFu;
            } else {
                const int wx = gx - (x0 - 4), wy = gy - ay0;
                win = (unsigned)wx < (unsigned)RDB && (unsigned)wy < (unsigned)AY;
                const int c = win ? wy * RWB + wx + 4 : 0;
                v = (s_aux32[c >> 2] >> (8 * (c & 3))) & 0xFFu;
            }
            if (!win) v = aux[(uint32_t)(gy * it.W + gx)];
            return v;
        };
        uint8_t* p8 = reinterpret_cast<uint8_t*>(s_p32);
        for (int k = t; k < nblk; k += 256) {
            int e = s_blk[k];
            int r = e / RWB, c = e % RWB;
            // 1: "/" loses (bits 2 and 5), 2: "\" loses (bits 0 and 7)
            p8[e] = remove_slash(get, x0 - 8 + c, ay0 + r) ? 1 : 2;
        }
    }
    __syncthreads();
    for (int k = t; k < GY * RDW; k += 256) {
        const int r = k / RDW, w = k % RDW + 1;  // word w of resolved row r (snapshot row r + 1)
        const int y = ay0 + 1 + r, x = x0 - 8 + 4 * w;
        const uint32_t* pa = s_p32 + (r + 1) * RWW + w;  // decisions of the blocks with origin on row y
        const uint32_t* pb = pa - RWW;                   // ... on row y - 1
        uint32_t A = pa[0], Al = __builtin_amdgcn_alignbyte(A, pa[-1], 3);
        uint32_t B = pb[0], Bl = __builtin_amdgcn_alignbyte(B, pb[-1], 3);
        uint32_t clear = ((A & 0x01010101u) << 2) |        // up-right block: "/"
                         ((Al >> 1) & 0x01010101u) |        // up-left block: "\"
                         ((Bl & 0x01010101u) << 5) |        // down-left block: "/"
                         (((B >> 1) & 0x01010101u) << 7);  // down-right block: "\"
        uint32_t res = s_aux32[(r + 1) * RWW + w] & ~clear;
        s_g32[r * RWW + w] = res;
        // the resolved graph of the tile's own cells, when the caller keeps it
        if (gfin && y >= y0 && y < y0 + RTY && w >= 2 && w <= RDW - 1 && y < it.H && x < it.W) {
            uint8_t* dst = gfin + it.g_off + (uint32_t)(y * it.W + x);
            const int n = it.W - x;
            if (n >= 4) __builtin_memcpy(dst, &res, 4);  // (one store at any alignment)
            else
                for (int q = 0; q < n; q++) dst[q] = (uint8_t)(res >> (8 * q));
        }
    }
}

// The resolved rows y0 - 1 .. y0 + RTY of a tile's window, read from the
// resolved graph written by kf_smooth (words laid out as in s_g32).
template <int TX>
__device__ inline void tile_resolved_load(const DevItem& it, const uint8_t* __restrict__ gfin, int x0, int y0,
                                          uint32_t* s_g32, int t)
{
    DPX_TILE_NAMES(TX);
    static_assert(GY * RWW <= 256, "a word a thread");
    if (t < GY * RWW) {
        const int r = t / RWW, w = t % RWW;
        s_g32[t] = w >= 1 && w <= RDW ? graph_word(it, gfin + it.g_off, x0 - 8 + 4 * w, y0 - 1 + r) : 0u;
    }
}

// ---------------------------------------------------------------------------
// kf_smooth: crossing resolution, cells and corner-cutting subdivision of a
// tile of cells (subdivision_Kernel kernel.cu:216-261 on the cells_Kernel
// hulls, then triangulate_Kernel's ear clipping, kernel.cu:264-282), each
// own cell once.  Writes the tile's resolved graph bytes to gfin and, for
// every smoothed (non-internal) cell, the coverage of its triangles at scale S
// with its summary to `rows` (rows_words(S) words per cell: its cell masks up
// to 8x, its rows from 9x).
// Internal cells (node 90) keep their hull (kernel.cu:231): the raster takes
// their rows from the table.
//
// Bound by instructions, so each part does the least a lane can do: hulls
// are one table word each, held in registers; a cell's T-junction colours
// are read side by side; the rows come from the polygon's edges, only where
// an edge crosses a row, toggled into an LDS column; and the ear clipping,
// which is needed only to know that it cuts the whole polygon (else the
// triangles cut so far are the cell), runs for the few polygons for which
// that is not plain, gathered into the first lanes.  The cells are listed by
// the size of their hull, so that the lanes of a wave end together.  16 frames
// of 640x480 at 8x: 293 us (606 with every row of every edge visited, every
// cell clipped, and hulls and colours read per vertex); 64 of 251x223 at 4x:
// 127 (334).
// ---------------------------------------------------------------------------
// Blocks a CU, for which the registers are allotted: as many as their LDS
// leaves room for (a wave waits for two thirds of its time, most of it at
// barriers).  One block more than before takes 16 frames of 640x480 at 8x from
// 616 to 566 us a batch, at 6x 477 to 449 and at 4x 291 to 275, 64 of 251x223
// at 4x 235 to 220; 8 blocks at 4x spill: 233.
constexpr int smooth_blocks(int S, bool walk) { return walk ? 3 : S <= 4 ? 7 : S <= 6 ? 6 : S <= 8 ? 5 : 3; }

template <int S, int TX, bool WALK>
__global__ __launch_bounds__(256, smooth_blocks(S, WALK)) void kf_smooth(const DevItem* __restrict__ items, const uint2* __restrict__ tile_map,
                                                 int grid3d, const uint8_t* __restrict__ in,
                                                 const uint8_t* __restrict__ gaux, uint8_t* __restrict__ gfin,
                                                 uint32_t* __restrict__ rows)
{
    DPX_TILE_NAMES(TX);
    constexpr int X0 = cover_x0(S), Y0 = cover_y0(S), COLS = cover_w(S), ROWS = cover_h(S), RW = rows_words(S);
    static_assert(COLS <= 32, "a row of samples is a word");
    constexpr int PITCH = 257;  // of the rows: adjacent rows of a cell in adjacent banks
    __shared__ int s_nblk;
    __shared__ uint8_t s_list[RTX * RTY];
    __shared__ int s_bin[16];  // own cells to smooth per hull size
    __shared__ int s_nlist, s_nclip;
    __shared__ uint8_t s_clip[RTX * RTY];  // columns whose polygon is clipped
    __shared__ uint8_t s_m[RTX * RTY];     // vertices of a column's polygon; 0 once its clipping has failed; at last its summary
    // vertex k of column t at [k * 256 + t]; a hull has at most 8 vertices,
    // its smoothed polygon at most 16, within the cells around (-64 .. 127)
    __shared__ uint16_t s_poly[16 * 256];
    // sample row r of column t at [r * PITCH + t], then its masks; first the walk window
    constexpr int COV = (S > kMaxCellScale || ROWS > RW ? ROWS : RW) * PITCH, WALK_WORDS = WALK ? WalkWindow<TX>::BYTES / 4 : 0;
    // What is needed until the polygons are made lies where the rows come
    // after them (the walk window is read meanwhile and keeps it apart): a
    // block more fits each CU.
    constexpr int HULL_WORDS = RCX * RCY * (int)(sizeof(HullBits) / 4), AUX_WORDS = AY * RWW, P_WORDS = (GY + 1) * RWW;
    constexpr int G_WORDS = GY * RWW, EARLY = HULL_WORDS + AUX_WORDS + P_WORDS + G_WORDS + ((GY + 1) * RDB + 1) / 2;
    constexpr int LATE = COV > WALK_WORDS ? COV : WALK_WORDS;
    __shared__ __align__(8) uint32_t s_cov[WALK ? LATE + EARLY + 1 : LATE > EARLY ? LATE : EARLY];
    uint32_t* s_early = s_cov + (WALK ? (LATE + 1) / 2 * 2 : 0);
    HullBits* s_hull = reinterpret_cast<HullBits*>(s_early);
    uint32_t* s_aux32 = s_early + HULL_WORDS;
    uint32_t* s_p32 = s_aux32 + AUX_WORDS;
    uint32_t* s_g32 = s_p32 + P_WORDS;
    uint16_t* s_blk = reinterpret_cast<uint16_t*>(s_g32 + G_WORDS);
    const uint8_t* s_g = reinterpret_cast<const uint8_t*>(s_g32);

    const int t = threadIdx.x;
    const TileAt at = locate_tile<8>(tile_map, grid3d);
    const DevItem it = items[at.item];
    const int x0 = at.tx * RTX, y0 = at.ty * RTY;
    const uint8_t* aux = gaux + it.g_off;
    const int ay0 = y0 - 2;
    if (t == 0) {
        s_nclip = 0;
        s_nblk = 0;
    }
    if (t < 16) s_bin[t] = 0;
    if (t < (GY + 1) * RWW) s_p32[t] = 0;
    tile_snapshot_load<TX>(it, aux, x0, ay0, s_aux32, t);
    __syncthreads();
    tile_resolve<TX, WALK>(it, aux, gfin, x0, y0, ay0, s_aux32, s_p32, s_blk, &s_nblk, s_g32, s_cov, t);
    __syncthreads();
    // hulls of the own cells and of their neighbours: cell (x0 - 1 + lx,
    // y0 - 1 + ly) at resolved row ly, byte lx + 7
#pragma unroll
    for (int q = 0; q < (RCX * RCY + 255) / 256; q++) {
        const int k = t + 256 * q;
        if (k >= RCX * RCY) break;
        const int lx = k % RCX, ly = k / RCX;
        const int c = ly * RWB + lx + 7;
        s_hull[k] = kHullTable[cell_key(s_g[c], s_g[c - 1], s_g[c + 1])];
    }
    __syncthreads();
    // own cells to smooth: in the frame and not internal, largest hulls first
    int my_n = -1, my_rank = 0;
    {
        const int cx = t % RTX, cy = t / RTX;
        if (x0 + cx < it.W && y0 + cy < it.H && s_g[(cy + 1) * RWB + cx + 8] != 90) {
            my_n = hull_count(s_hull[(cy + 1) * RCX + cx + 1]);
            my_rank = atomicAdd(&s_bin[15 - my_n], 1);
        }
    }
    __syncthreads();
    if (t < 16) {
        const int own = s_bin[t];
        int acc = own;
#pragma unroll
        for (int d = 1; d < 16; d <<= 1) {
            const int v = __shfl_up(acc, d);
            if (t >= d) acc += v;
        }
        s_bin[t] = acc - own;
        if (t == 15) s_nlist = acc;
    }
    __syncthreads();
    if (my_n >= 0) s_list[s_bin[15 - my_n] + my_rank] = (uint8_t)t;
    __syncthreads();
    const int nlist = s_nlist;
    if (nlist == 0) return;  // (uniform)
    uint16_t* P = s_poly + t;  // this lane's columns
    uint32_t* C = s_cov + t;
    int m = 0, wsum = 0;
    if (t < nlist) {
        const int own = s_list[t];
        const int cx = own % RTX, cy = own / RTX;
        const int x = x0 + cx, y = y0 + cy;
        const uint32_t node = s_g[(cy + 1) * RWB + cx + 8];
        const int hk = (cy + 1) * RCX + cx + 1;
        const HullBits h = s_hull[hk];
        const ImgView im{ in + it.in_off, it.W, it.H, it.stride, it.ch, it.flags,
                          (it.flags & DPX_INDEXED) ? in + it.pal_off : nullptr };
        const uint32_t corners = tj_corners(tj_view(im), x, y);
        auto nbr = [&](int e) { return s_hull[hk + edy(e) * RCX + edx(e)]; };
        auto tj = [&](int x4, int y4) -> bool { return tj_kept(corners, x4, y4); };
        subdivide_hull_emit(h, node, nbr, tj, [&](int px, int py) {
            P[256 * m] = (uint16_t)(((uint32_t)px & 0xFFu) | ((uint32_t)py << 8));
            m++;
        });
    }
    __syncthreads();
    if (t < nlist) {
#pragma unroll
        for (int r = 0; r < ROWS; r++) C[PITCH * r] = 0;
        // seen from its pixel's centre almost every cell goes round once
        // (no clipping is needed to know that it is cut wholly); the others
        // are clipped, their vertices counter-clockwise as ear_clip takes them
        if (!poly_star(P, 256, m, 32, 32)) {
            if (poly_shape(P, 256, m).area2 <= 0)
                for (int lo = 0, hi = m - 1; lo < hi; lo++, hi--) {
                    const uint16_t tmp = P[256 * lo];
                    P[256 * lo] = P[256 * hi];
                    P[256 * hi] = tmp;
                }
            s_clip[atomicAdd(&s_nclip, 1)] = (uint8_t)t;
        }
        wsum = poly_rows_cross<ROWS, COLS>(P, 256, m, 2 * S, X0, Y0,
                                           [&](int r, uint32_t mask) { atomicXor(&C[PITCH * r], mask); });
        s_m[t] = (uint8_t)m;
    }
    __syncthreads();
    if (t < s_nclip) {
        const int c = s_clip[t];
        if (ear_clip_ring<16>(s_poly + c, 256, (int)s_m[c], true, [](uint16_t, uint16_t, uint16_t) {}) > 2) s_m[c] = 0;
    }
    __syncthreads();
    if (t < nlist) {
        int bits = 0;
#pragma unroll
        for (int r = 0; r < ROWS; r++) bits += __builtin_popcount(C[PITCH * r]);
        if (s_m[t] == 0 || wsum != bits) {
            // not cut wholly, or a winding other than 0 and 1 (none in the
            // synthetic workloads): the rows of each ear as it is cut
            uint32_t cov[ROWS];
#pragma unroll
            for (int r = 0; r < ROWS; r++) cov[r] = 0;
            ear_clip_ring<16>(P, 256, m, true, [&](uint16_t A, uint16_t B, uint16_t E) {
                // units of 1/(128 S) of a cell; counter-clockwise (an ear's cross is positive)
                tri_rect_or<ROWS, COLS>(vert_x(A) * 2 * S, vert_y(A) * 2 * S, vert_x(B) * 2 * S, vert_y(B) * 2 * S,
                                        vert_x(E) * 2 * S, vert_y(E) * 2 * S, X0, Y0, cov);
            });
#pragma unroll
            for (int r = 0; r < ROWS; r++) C[PITCH * r] = cov[r];
        }
        uint32_t cov[ROWS];
#pragma unroll
        for (int r = 0; r < ROWS; r++) cov[r] = C[PITCH * r];
        const uint32_t info = coverage_info(cov, S, X0, Y0, ROWS);
        if constexpr (S <= kMaxCellScale) {
            uint32_t word[RW] = {};
            cell_mask_rows<S, X0, Y0, ROWS>([&](int r) { return cov[r]; },
                                            [&](int j, int ky, uint32_t bits) {
                                                const int at = S <= kMaxCellScale16 ? 16 * j + ky * S : 8 * (j * S + ky);
                                                word[at / 32] |= bits << (at % 32);
                                            });
            constexpr int at = S <= kMaxCellScale16 ? 16 * 9 : 8 * 9 * S;
            word[at / 32] |= (info & 0xFFu) << (at % 32);
#pragma unroll
            for (int r = 0; r < RW; r++) C[PITCH * r] = word[r];
        } else {
            s_m[t] = (uint8_t)info;
        }
    }
    __syncthreads();
    // the words of a cell by adjacent lanes
    uint32_t* dst = rows + it.rows_off / 4;
    for (int k = t; k < nlist * RW; k += 256) {
        const int c = k / RW, r = k - c * RW, own = s_list[c];
        const uint32_t cell = (uint32_t)(y0 + own / RTX) * (uint32_t)it.W + (uint32_t)(x0 + own % RTX);
        if constexpr (S > kMaxCellScale) dst[(size_t)cell * RW + r] = r == ROWS ? s_m[c] : s_cov[PITCH * r + c];
        else dst[(size_t)cell * RW + r] = s_cov[PITCH * r + c];
    }
}

// `items` are the items of one (scale, subdivision) group, in launch order.
// With SUB the resolved graph comes from gfin and the coverage rows of the
// smoothed cells from `cell_rows` (kf_smooth ran before); without, the kernel
// resolves the crossings itself from the snapshot.
template <int S, bool SUB, int TX, bool WALK>
__global__ __launch_bounds__(256) void kf_raster(const DevItem* __restrict__ items, const uint2* __restrict__ tile_map,
                                                 int grid3d,
                                                 const uint8_t* __restrict__ in, const uint8_t* __restrict__ gaux,
                                                 uint8_t* __restrict__ gfin, const uint32_t* __restrict__ cell_rows,
                                                 const uint32_t* __restrict__ mask_table,
                                                 const uint8_t* __restrict__ info_table, uint8_t* __restrict__ out)
{
    DPX_TILE_NAMES(TX);
    constexpr int MW = mask_w(S), KMIN = mask_kmin(S), RW = rows_words(S);
    // the grid of smoothed cells' rows; the table's are shifted to its columns
    constexpr int SY0 = cover_y0(S), ROWS = cover_h(S), X0 = SUB ? cover_x0(S) : KMIN;
    static_assert(KMIN >= X0 && last_sample(S, 80) - X0 < 32, "a hull's samples stay in the word");
    __shared__ uint32_t s_aux32[SUB ? 1 : AY * RWW];
    __shared__ uint32_t s_p32[SUB ? 1 : (GY + 1) * RWW];  // decisions of crossed blocks, by origin
    __shared__ uint16_t s_blk[SUB ? 1 : (GY + 1) * RDB];  // crossed blocks: origin byte index in the window
    __shared__ int s_nblk;
    __shared__ uint32_t s_g32[GY * RWW];
    static_assert(kKeys == 256 * 16, "16 summaries a thread");
    __shared__ u32x4 s_itab[SUB ? 1 : 256];
    __shared__ uint16_t s_key[RCX * RCY];
    __shared__ uint8_t s_info[RCX * RCY];  // coverage summary bits 0..4 (simple_cell)
    __shared__ uint32_t s_col[RCX * RCY];
    __shared__ uint32_t s_src[SUB ? RCX * RCY : 1];  // smoothed candidates: word offset of their masks in the item's (from 9x: their cell)
    __shared__ uint16_t s_list[RTX * RTY];  // own cells that need the candidate search
    __shared__ int s_nlist;
    // resolved pixels of the first listed cells, so that every own
    // cell's rows are stored together (a line is then written by one store
    // instruction instead of being split between the direct and searched
    // cells).  A pixel is kept as its colour; from S = 5 a tile whose listed
    // cells would overflow that keeps each row's winners instead (see
    // Winners: one word a row up to 8x, where every cell of the tile fits,
    // else two), and looks the colours up when it stores them.
    constexpr bool CODES = S >= 5;
    constexpr int ROW_WORDS = S <= 8 ? 1 : 2;  // of a row's packed winners
    constexpr int PX_WORDS = 2048, PX_CELLS = PX_WORDS / (S * S), PX_CODE_CELLS = PX_WORDS / (S * ROW_WORDS);
    static_assert(PX_CELLS >= 1, "at least one buffered cell");
    __shared__ uint32_t s_px[PX_WORDS];
    // the winners of listed cells' pixels, as two words a cell up to
    // 4x, a word a row from 5x (tiles that do not keep them in s_px)
    constexpr bool MASKS = SUB ? S <= kMaxCellScale : S >= 3 && S <= 7;
    __shared__ uint32_t s_plane[!MASKS ? 1 : S <= kMaxCellScale16 ? 2 * RTX * RTY : PX_CELLS * S];
    __shared__ uint16_t s_idx[RTX * RTY];  // list index of a listed own cell, else kOwnColour
    constexpr uint32_t kOwnColour = 0xFFFF;  // the cell shows its own colour only
    const uint8_t* s_g = reinterpret_cast<const uint8_t*>(s_g32);

    const int t = threadIdx.x;
    const TileAt at = locate_tile<8>(tile_map, grid3d);
    const DevItem it = items[at.item];
    const int x0 = at.tx * RTX, y0 = at.ty * RTY;
    const uint8_t* aux = gaux + it.g_off;
    // (an item's coverage is less than 2^32 words up to 8x, checked on the host; from 9x, and a batch's, it may be more)
    const uint32_t* item_rows = SUB ? cell_rows + it.rows_off / 4 : nullptr;
    auto smoothed_cell = [&](uint32_t src) {
        if constexpr (S <= kMaxCellScale) return item_rows + src;
        else return item_rows + (size_t)src * RW;
    };
    const int ay0 = y0 - 2;  // first snapshot row

    if (t == 0) {
        s_nlist = 0;
        s_nblk = 0;
    }
    // The snapshot bytes (or the resolved ones), the candidates' colours and
    // the table of summaries (in LDS, so that a cell's summary is not another
    // round trip after its key: 1024 frames at 4x 852 -> 836 us, 16 of 640x480
    // at 8x 256 -> 242) are independent loads: issue them together.
    if constexpr (!SUB) s_itab[t] = reinterpret_cast<const u32x4*>(info_table)[t];
    if constexpr (SUB) {
        tile_resolved_load<TX>(it, gfin, x0, y0, s_g32, t);
    } else {
        if (t < (GY + 1) * RWW) s_p32[t] = 0;
        tile_snapshot_load<TX>(it, aux, x0, ay0, s_aux32, t);
    }
    {
        // a colour is one 4-byte load at any alignment, through a descriptor
        // of the item's rows that answers 0 past their end (the cells outside
        // the frame, whose colours nothing reads); the last pixel of a frame
        // of 3-byte pixels, whose word would end past the item, is read by
        // bytes instead (see word_crosses).  Three or four byte loads
        // a colour, each tested for the frame: 1024 frames of 256x224 at 4x
        // 836 us a batch against 799, 64 console frames 75.9 against 71.6.
        const uint32_t in_end = (uint32_t)(it.H - 1) * (uint32_t)it.stride + (uint32_t)(it.W * it.ch);
        const auto src = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(in + it.in_off), 0, in_end, 0x00020000);
        const bool topdown = it.flags & DPX_TOPDOWN, indexed = it.flags & DPX_INDEXED;
        const uint32_t* pal = reinterpret_cast<const uint32_t*>(in + it.pal_off);
        // colorPos (kernel.cu:98-101): the three bytes reversed unless RGB,
        // and the fourth or 255
        const uint32_t order = ((it.flags & DPX_RGB) ? 0x00020100u : 0x00000102u) |
                               (indexed || it.ch == 4 ? 0x03000000u : 0x0D000000u);
        constexpr int PER = (RCX * RCY + 255) / 256;
        uint32_t c[PER];
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const int k = t + 256 * q, x = x0 - 1 + k % RCX, y = y0 - 1 + k / RCX;
            const bool inside = k < RCX * RCY && (unsigned)x < (unsigned)it.W && (unsigned)y < (unsigned)it.H;
            const int row = topdown ? it.H - 1 - y : y;
            // row * stride < 2^31 (checked on the host); the stride itself may exceed 2^24
            const uint32_t off = (uint32_t)row * (uint32_t)it.stride + __umul24(x, it.ch);
            if (indexed) {
                c[q] = __builtin_amdgcn_raw_buffer_load_b8(src, (int)(inside ? off : ~0u), 0, 0);
            } else {
                const bool last = word_crosses(off, in_end, it.ch);
                c[q] = __builtin_amdgcn_raw_buffer_load_b32(src, (int)(inside && !last ? off : ~0u), 0, 0);
                if (inside && last)
                    c[q] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b8(src, (int)off, 0, 0) |
                           (uint32_t)__builtin_amdgcn_raw_buffer_load_b8(src, (int)off + 1, 0, 0) << 8 |
                           (uint32_t)__builtin_amdgcn_raw_buffer_load_b8(src, (int)off + 2, 0, 0) << 16;
            }
        }
#pragma unroll
        for (int q = 0; q < PER; q++) {
            if (indexed) c[q] = pal[c[q]];
            if (t + 256 * q < RCX * RCY) s_col[t + 256 * q] = __builtin_amdgcn_perm(0u, c[q], order);
        }
    }
    __syncthreads();
    if constexpr (!SUB) {
        __shared__ uint32_t s_walk[WALK ? WalkWindow<TX>::BYTES / 4 : 1];
        tile_resolve<TX, WALK>(it, aux, gfin, x0, y0, ay0, s_aux32, s_p32, s_blk, &s_nblk, s_g32, s_walk, t);
        __syncthreads();
    }
    // candidate cells: key and coverage summary.  Candidate (lx, ly) is the
    // cell at (x0 - 1 + lx, y0 - 1 + ly): resolved row ly, byte lx + 7.
    // (unrolled, so that a thread's table loads are all in flight at once)
#pragma unroll
    for (int q = 0; q < (RCX * RCY + 255) / 256; q++) {
        const int k = t + 256 * q;
        if (k >= RCX * RCY) break;
        int lx = k % RCX, ly = k / RCX;
        int x = x0 - 1 + lx, y = y0 - 1 + ly;
        uint16_t key = kNoCell;
        uint8_t info = 0;
        if ((unsigned)x < (unsigned)it.W && (unsigned)y < (unsigned)it.H) {
            int c = ly * RWB + lx + 7;
            key = (uint16_t)cell_key(s_g[c], s_g[c - 1], s_g[c + 1]);
            if constexpr (SUB) {
                // a smoothed cell's rows and summary come from kf_smooth;
                // an internal one (node 90) keeps its hull: the table's
                uint32_t src = 0xFFFFFFFFu;
                if ((key & 0xFFu) != 90) {
                    constexpr int at = S > kMaxCellScale ? 32 * ROWS : S <= kMaxCellScale16 ? 16 * 9 : 8 * 9 * S;
                    src = (uint32_t)y * (uint32_t)it.W + (uint32_t)x;
                    if constexpr (S <= kMaxCellScale) src *= RW;
                    info = (uint8_t)((smoothed_cell(src)[at / 32] >> (at % 32)) & 0x1Fu);
                } else {
                    info = info_table[key] & 0x1Fu;
                }
                s_src[k] = src;
            } else {
                info = reinterpret_cast<const uint8_t*>(s_itab)[key] & 0x1Fu;
            }
        }
        s_key[k] = key;
        s_info[k] = info;
    }
    __syncthreads();

    // Output pixels are written once and not read back by the kernels:
    // non-temporal stores keep them from displacing the graph and table lines
    // the other tiles' loads need in the caches.
    const int OH = it.H * S;
    auto store_row = [&](int gx, int Y, const uint32_t* col) {
        int row = out_topdown(it.flags) ? (OH - 1 - Y) : Y;
        uint8_t* dst = out + it.out_off + (size_t)row * it.out_stride + (size_t)gx * S * 4;
        if constexpr (S % 4 == 0) {
            if (it.aligned16) {
#pragma unroll
                for (int q = 0; q < S; q += 4) {
                    u32x4 v = { col[q], col[q + 1], col[q + 2], col[q + 3] };
                    __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(dst + 4 * q));
                }
                return;
            }
        }
        if constexpr (S % 2 == 0) {
            if ((reinterpret_cast<uintptr_t>(dst) & 7) == 0) {
#pragma unroll
                for (int q = 0; q < S; q += 2) {
                    u32x2 v = { col[q], col[q + 1] };
                    __builtin_nontemporal_store(v, reinterpret_cast<u32x2*>(dst + 4 * q));
                }
                return;
            }
        }
#pragma unroll
        for (int q = 0; q < S; q++) __builtin_nontemporal_store(col[q], reinterpret_cast<uint32_t*>(dst + 4 * q));
    };

    // Own cells, one per thread: a cell whose S*S pixels all show its own
    // colour is written directly, the others are listed for the candidate
    // search, which resolves their pixels into LDS first.
    const int cx = t % RTX, cy = t / RTX;
    const int kown = (cy + 1) * RCX + cx + 1;
    const bool mine = x0 + cx < it.W && y0 + cy < it.H;
    const bool simple = mine && simple_cell(s_info[kown], s_info[kown + RCX - 1], s_info[kown + RCX],
                                            s_info[kown + RCX + 1], s_info[kown + 1]);
    {
        uint32_t i = kOwnColour;
        if (mine && !simple) {
            i = (uint32_t)atomicAdd(&s_nlist, 1);
            s_list[i] = (uint16_t)t;
        }
        s_idx[t] = (uint16_t)i;
    }
    __syncthreads();

    // One unit = one output row (S pixels) of a listed cell, resolved
    // against the 3x3 candidates in draw order (highest cell index first).
    constexpr uint32_t FULL = (S >= 32) ? 0xFFFFFFFFu : ((1u << S) - 1u);
    const int nunits = s_nlist * S;
    const bool codes = CODES && s_nlist > PX_CELLS;  // uniform over the block
    const int px_cells = codes ? PX_CODE_CELLS : PX_CELLS;
    auto fetch_rows = [&](int u, uint32_t* rows) {
        int own = s_list[u / S], ky = u % S;
        int ux = own % RTX, uy = own / RTX;
        // an own cell that covers its whole square takes every pixel the
        // cells drawn after it leave: the candidates drawn before it (left,
        // down-left, down, down-right) can win none, and are not fetched
        const bool own_full = s_info[(uy + 1) * RCX + ux + 1] & 1u;
#pragma unroll
        for (int dy = 1; dy >= -1; dy--) {
#pragma unroll
            for (int dx = 1; dx >= -1; dx--) {
                int k = (uy + 1 + dy) * RCX + (ux + 1 + dx);
                uint32_t row = 0;
                const bool before_own = dy < 0 || (dy == 0 && dx < 0);
                if (!(own_full && before_own) && s_key[k] != kNoCell) {
                    const int r = ky - dy * S - KMIN;
                    if constexpr (SUB) {
                        const uint32_t src = s_src[k];
                        const int rs = ky - dy * S - SY0;
                        if (src != 0xFFFFFFFFu) {
                            if (rs >= 0 && rs < ROWS) row = smoothed_cell(src)[rs];
                        } else if (r >= 0 && r < MW) {
                            row = mask_table[(uint32_t)s_key[k] * MW + r] << (KMIN - X0);
                        }
                    } else if (r >= 0 && r < MW) {
                        row = mask_table[(uint32_t)s_key[k] * MW + r];
                    }
                }
                rows[(1 - dy) * 3 + (1 - dx)] = row;
            }
        }
    };
    // The winning candidate of every pixel of a row, as bit planes: pixel q's
    // is the one at (1 - dx, 1 - dy) = (x0 + 2 x1, y0 + 2 y1) of bits q, or
    // none (dx digit 3).  A candidate then costs three instructions for all
    // of the row's pixels, and a pixel one product of four bits with their
    // places in s_col, not a choice between nine colours: 170 -> 64
    // instructions a row at 6x.
    struct Winners {
        uint32_t w[ROW_WORDS];
    };
    auto winners = [&](const uint32_t* rows) {
        uint32_t seen = 0, won[9];
#pragma unroll
        for (int j = 0; j < 9; j++) {
            const int sh = (j % 3 - 1) * S - X0;
            const uint32_t bits = (sh >= 0 ? (rows[j] >> sh) : (rows[j] << -sh)) & FULL;
            won[j] = bits & ~seen;
            seen |= bits;
        }
        const uint32_t none = FULL & ~seen;
        const uint32_t px0 = won[1] | won[4] | won[7] | none, px1 = won[2] | won[5] | won[8] | none;
        const uint32_t py0 = won[3] | won[4] | won[5], py1 = won[6] | won[7] | won[8];
        Winners r;
        if constexpr (ROW_WORDS == 1) {
            r.w[0] = px0 | px1 << 8 | py0 << 16 | py1 << 24;
        } else {
            r.w[0] = px0 | px1 << 16;
            r.w[1] = py0 | py1 << 16;
        }
        return r;
    };
    // pixel q's colour; last: the cell's last candidate's place in s_col (dx = dy = 1)
    auto winner_colour = [&](const Winners& r, int q, int last) -> uint32_t {
        uint32_t off;
        bool none;
        if constexpr (ROW_WORDS == 1) {
            const uint32_t bits = (r.w[0] >> q) & 0x01010101u;
            off = __builtin_amdgcn_udot4(bits, 1u | 2u << 8 | (uint32_t)RCX << 16 | (uint32_t)(2 * RCX) << 24, 0u, false);
            none = (bits & 0x0101u) == 0x0101u;
        } else {
            const uint32_t x = (r.w[0] >> q) & 0x00010001u, y = (r.w[1] >> q) & 0x00010001u;
            off = (x & 3u) + (x >> 15) + (uint32_t)RCX * ((y & 3u) + (y >> 15));
            none = x == 0x00010001u;
        }
        const uint32_t c = s_col[last - (int)off];
        return none ? 0xFF000000u : c;
    };
    auto resolve_unit = [&](int u, const uint32_t* rows) {
        const int own = s_list[u / S], ky = u % S;
        const int ux = own % RTX, uy = own / RTX, last = (uy + 2) * RCX + ux + 2;
        const Winners w = winners(rows);
        if constexpr (CODES) {
            if (codes && u / S < PX_CODE_CELLS) {
#pragma unroll
                for (int k = 0; k < ROW_WORDS; k++) s_px[u * ROW_WORDS + k] = w.w[k];
                return;
            }
        }
        uint32_t col[S];
#pragma unroll
        for (int q = 0; q < S; q++) col[q] = winner_colour(w, q, last);
        if (!codes && u / S < PX_CELLS) {
#pragma unroll
            for (int q = 0; q < S; q++) s_px[u * S + q] = col[q];
        } else {
            store_row(x0 + ux, (y0 + uy) * S + ky, col);  // beyond the buffer: written directly
        }
    };

    if constexpr (MASKS) {
        // 3x to 7x, with subdivision 1x to 8x: a listed cell's winners are picked for all its pixels at
        // once, from nine independent loads of the cell-mask table: one thread
        // a cell up to 4x, two (four rows each) from 5x.  A tile that keeps
        // winners is then resolved, else one thread per row of a listed cell
        // looks its colours up.  Rows that each fetch and resolve their own
        // nine table rows do the first part S times over: per batch at 4x,
        // 1024 frames of 256x224 884 -> 850 us, 64 console frames 83 -> 77,
        // 128 indexed frames 141 -> 133; at 6x, 4096 sprites 129 -> 120, 8
        // frames of 640x480 97 -> 83.  At 8x the stores bound the batch
        // either way, and the rows, spread over more threads, keep them
        // flowing (16 frames of 640x480: 256 us against 264).  With
        // subdivision kf_smooth writes masks too, and 16 frames of 640x480
        // take 644 -> 617 us at 8x, 501 -> 476 at 6x and 336 -> 292 at 4x.
        constexpr int TB = S <= kMaxCellScale16 ? 2 : 4;  // bytes of a thread's masks
        constexpr int PARTS = S <= kMaxCellScale16 ? 1 : 2;
        const uint8_t* cell_table = reinterpret_cast<const uint8_t*>(mask_table + kKeys * MW);
        const int nparts = s_nlist * PARTS;
        for (int p = t; p < nparts; p += 256) {
            const int i = p / PARTS, h = p % PARTS, own = s_list[i];
            const int ux = own % RTX, uy = own / RTX;
            uint32_t m[9];
#pragma unroll
            for (int j = 0; j < 9; j++) {
                const int k = (uy + 2 - j / 3) * RCX + (ux + 2 - j % 3);
                const uint32_t key = s_key[k];
                m[j] = 0;
                if (key != kNoCell) {
                    const uint8_t* src = cell_table + ((key * 9 + j) * PARTS + h) * TB;
                    if constexpr (SUB) {
                        if (s_src[k] != 0xFFFFFFFFu)
                            src = reinterpret_cast<const uint8_t*>(smoothed_cell(s_src[k])) + j * (PARTS == 1 ? 2 : S) + 4 * h;
                    }
                    __builtin_memcpy(&m[j], src, TB);
                }
            }
            uint32_t seen = 0;
#pragma unroll
            for (int j = 0; j < 9; j++) {
                const uint32_t won = m[j] & ~seen;
                seen |= m[j];
                m[j] = won;
            }
            const uint32_t px0 = m[1] | m[4] | m[7] | ~seen, px1 = m[2] | m[5] | m[8] | ~seen;
            const uint32_t py0 = m[3] | m[4] | m[5], py1 = m[6] | m[7] | m[8];
            if constexpr (PARTS == 1) {
                s_plane[2 * i] = __builtin_amdgcn_perm(px1, px0, 0x05040100u);
                s_plane[2 * i + 1] = py0 | py1 << 16;
            } else {
                uint32_t* words = (codes ? s_px : s_plane) + i * S + 4 * h;  // (every cell fits the former)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    // byte r of the four planes: row 4 h + r
                    const uint32_t two = (uint32_t)(4 + r) << 8 | (uint32_t)r;
                    const uint32_t w = __builtin_amdgcn_perm(px1, px0, 0x0C0C0000u | two) |
                                       __builtin_amdgcn_perm(py1, py0, two << 16 | 0x0C0Cu);
                    if (r < S - 4 || h == 0) words[r] = w;
                }
            }
        }
        __syncthreads();
        if (!codes) {
            for (int u = t; u < nunits; u += 256) {
                const int i = u / S, ky = u % S, own = s_list[i];
                const int ux = own % RTX, uy = own / RTX, last = (uy + 2) * RCX + ux + 2;
                Winners r;
                if constexpr (S <= kMaxCellScale16)
                    r.w[0] = __builtin_amdgcn_perm(s_plane[2 * i + 1] >> (ky * S), s_plane[2 * i] >> (ky * S), 0x06040200u);
                else
                    r.w[0] = s_plane[u];
                uint32_t col[S];
#pragma unroll
                for (int q = 0; q < S; q++) col[q] = winner_colour(r, q, last);
                if (i < PX_CELLS) {
#pragma unroll
                    for (int q = 0; q < S; q++) s_px[u * S + q] = col[q];
                } else {
                    store_row(x0 + ux, (y0 + uy) * S + ky, col);  // beyond the buffer: written directly
                }
            }
            __syncthreads();
        }
    } else if constexpr (!SUB && S <= 2) {
        // 1x and 2x: one thread per listed cell, the candidates' samples of
        // it from the cell-mask table (nine independent loads), resolved in
        // the same draw order as the rows of the other scales.  Measured: 2x
        // frames 8-11% faster than with row units; at 4x a thread resolving
        // 16 pixels alone lengthens sparse tiles (-3.5% on 16-colour frames).
        const uint16_t* cell_table = reinterpret_cast<const uint16_t*>(mask_table + kKeys * MW);
        const int nlist = s_nlist;
        for (int i = t; i < nlist; i += 256) {
            const int own = s_list[i];
            const int ux = own % RTX, uy = own / RTX;
            uint32_t m[9], c[9];
#pragma unroll
            for (int j = 0; j < 9; j++) {
                const int k = (uy + 2 - j / 3) * RCX + (ux + 2 - j % 3);
                const uint32_t key = s_key[k];
                m[j] = key != kNoCell ? cell_table[key * 9 + j] : 0u;
                c[j] = s_col[k];
            }
            uint32_t col[S * S];
#pragma unroll
            for (int p = 0; p < S * S; p++) col[p] = 0xFF000000u;
            uint32_t assigned = 0;
#pragma unroll
            for (int j = 0; j < 9; j++) {
                const uint32_t nb = m[j] & ~assigned;
#pragma unroll
                for (int p = 0; p < S * S; p++) col[p] = ((nb >> p) & 1u) ? c[j] : col[p];
                assigned |= nb;
            }
            if (i < PX_CELLS) {
#pragma unroll
                for (int p = 0; p < S * S; p++) s_px[i * S * S + p] = col[p];
            } else {
#pragma unroll
                for (int ky = 0; ky < S; ky++) store_row(x0 + ux, (y0 + uy) * S + ky, col + ky * S);
            }
        }
        __syncthreads();
    } else if (nunits > 0) {  // uniform: read from LDS after the barrier
        for (int u = t; u < nunits; u += 256) {
            uint32_t rows[9];
            fetch_rows(u, rows);
            resolve_unit(u, rows);
        }
        __syncthreads();
    }

    // At S = 1, 2 and 4 one output row of a cell is one store and the lanes
    // of a wave store adjacent cells, so each thread stores its own cell.  At
    // the other scales that would make every store instruction strided (S * 4
    // bytes between lanes, each line written in pieces by several
    // instructions), so the tile's rows are stored in chunks, adjacent lanes
    // adjacent chunks: of 4 pixels (16 bytes) where the rows are so aligned,
    // else of CW pixels inside one cell.  A thread goes from chunk to chunk
    // by 256, which moves it dr rows and dj chunks on (one row more where
    // that passes the row's end): the tile's cells in the frame, whatever
    // their number, keep every lane busy, and a chunk's cell and pixel take
    // two small products.  Searched cells beyond the pixel buffer were stored
    // by the search itself; their chunks are skipped, or where a chunk may
    // span two cells such tiles keep the per-cell stores (so do tiles at 5x
    // to 7x whose rows allow only chunks of one or two pixels and whose cells
    // overflow the buffer: there the chunks' own work outweighs the
    // coalescing).  With the winners above, per batch: 16 640x480 frames at 8x
    // 339 -> 259 us, 4096 sprites at 6x 164 -> 142, 64 console frames at 6x
    // 207 -> 151, at 12x 726 -> 570; chunks read two and four at a time
    // measured the same.
    constexpr int CW = (S % 4 == 0) ? 4 : ((S % 2 == 0) ? 2 : 1);
    // pixel (kx, ky) of listed cell i, own cell (lx, ly), from the buffer;
    // use_codes (std::true_type: the tile keeps rows' winners) is fixed per
    // tile, outside the store loops
    auto buffered = [&](auto use_codes, int i, int kx, int ky, int lx, int ly) -> uint32_t {
        if constexpr (decltype(use_codes)::value) {
            Winners r;
#pragma unroll
            for (int k = 0; k < ROW_WORDS; k++) r.w[k] = s_px[(i * S + ky) * ROW_WORDS + k];
            return winner_colour(r, kx, (ly + 2) * RCX + lx + 2);
        } else {
            return s_px[(i * S + ky) * S + kx];
        }
    };
    bool chunked = false, wide = false;
    if constexpr (S != 1 && S != 2 && S != 4) {
        const uintptr_t align = reinterpret_cast<uintptr_t>(out + it.out_off) | (uintptr_t)it.out_stride;
        wide = (align & 15) == 0 && (S % 4 == 0 || s_nlist <= px_cells);
        chunked = (align & (4 * CW - 1)) == 0 && (CW == 4 || S >= 9 || s_nlist <= px_cells);
    }
    // floor(v / S) for v < 2^12 (an exact reciprocal to 16 bits suffices)
    auto over_s = [](int v) { return (int)(__umul24((unsigned)v, 65536u / S + 1u) >> 16); };
    auto store_chunks = [&](auto use_codes, auto width) {
        constexpr int N = decltype(width)::value;  // pixels of a chunk
        const int ncx = min(RTX, it.W - x0), rows = min(RTY, it.H - y0) * S, rowpx = ncx * S;
        const int cpr = (rowpx + N - 1) / N;  // chunks of a row
        // (quotients below 2^9 from a reciprocal, half a unit clear of the next)
        const float inv = __builtin_amdgcn_rcpf((float)cpr);
        const int dr = (int)(256.5f * inv), dj = 256 - dr * cpr;
        int row = (int)(((float)t + 0.5f) * inv), j = t - row * cpr;
        const bool down = out_topdown(it.flags);
        const ptrdiff_t pitch = down ? -(ptrdiff_t)it.out_stride : (ptrdiff_t)it.out_stride;
        uint8_t* dst = out + it.out_off + (size_t)(down ? OH - 1 - y0 * S : y0 * S) * it.out_stride +
                       (size_t)x0 * S * 4 + row * pitch + j * (4 * N);
        const ptrdiff_t step = dr * pitch + dj * (4 * N), wrap = pitch - cpr * (4 * N);
        while (row < rows) {
            const int px0 = N * j, la = over_s(px0), kx = px0 - la * S, ly = over_s(row), ky = row - ly * S;
            const uint32_t ia = s_idx[ly * RTX + la], va = s_col[(ly + 1) * RCX + la + 1];
            uint32_t col[N];
            bool stored = false;  // by the search
            if constexpr (S % N == 0) {  // one cell
#pragma unroll
                for (int q = 0; q < N; q++) col[q] = va;
                if (ia != kOwnColour) {
                    stored = (int)ia >= px_cells;
                    if (!stored) {
#pragma unroll
                        for (int q = 0; q < N; q++) col[q] = buffered(use_codes, (int)ia, kx + q, ky, la, ly);
                    }
                }
            } else {
                // the chunk's second cell; past the frame's last column the
                // pixels are not stored and take that column's cell
                const int lb = min(la + 1, ncx - 1), split = S - kx;
                const uint32_t ib = s_idx[ly * RTX + lb], vb = s_col[(ly + 1) * RCX + lb + 1];
#pragma unroll
                for (int q = 0; q < N; q++) col[q] = q >= split ? vb : va;
                if (ia != kOwnColour || ib != kOwnColour) {
#pragma unroll
                    for (int q = 0; q < N; q++) {
                        const bool inb = q >= split;
                        const uint32_t i = inb ? ib : ia;
                        if (i != kOwnColour)
                            col[q] = buffered(use_codes, (int)i, inb ? q - split : kx + q, ky, inb ? lb : la, ly);
                    }
                }
            }
            if (!stored) {
                if constexpr (N == 4) {
                    if (S % 4 == 0 || px0 + 3 < rowpx) {
                        u32x4 v = { col[0], col[1], col[2], col[3] };
                        __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(dst));
                    } else {
#pragma unroll
                        for (int q = 0; q < 4; q++)
                            if (px0 + q < rowpx)
                                __builtin_nontemporal_store(col[q], reinterpret_cast<uint32_t*>(dst + 4 * q));
                    }
                } else if constexpr (N == 2) {
                    u32x2 v = { col[0], col[1] };
                    __builtin_nontemporal_store(v, reinterpret_cast<u32x2*>(dst));
                } else {
                    __builtin_nontemporal_store(col[0], reinterpret_cast<uint32_t*>(dst));
                }
            }
            row += dr;
            j += dj;
            dst += step;
            if (j >= cpr) {
                j -= cpr;
                row++;
                dst += wrap;
            }
        }
    };
    // A thread's own cell, simple or buffered, through one sequence of store
    // instructions for the whole wave: with separate branches for the two
    // kinds, a wave holding both issues every row store twice, each writing
    // part of the same lines.
    auto store_cell = [&](auto use_codes, int i) {
        const uint32_t c = s_col[kown];
#pragma unroll
        for (int ky = 0; ky < S; ky++) {
            uint32_t col[S];
#pragma unroll
            for (int q = 0; q < S; q++) {
                const uint32_t b = buffered(use_codes, i, q, ky, cx, cy);
                col[q] = simple ? c : b;
            }
            store_row(x0 + cx, (y0 + cy) * S + ky, col);
        }
    };
    if constexpr (S != 1 && S != 2 && S != 4) {
        using Wide = std::integral_constant<int, 4>;
        using Narrow = std::integral_constant<int, CW>;
        if (wide || chunked) {
            if constexpr (CODES) {
                if (codes) {
                    if (wide) store_chunks(std::true_type{}, Wide{});
                    else store_chunks(std::true_type{}, Narrow{});
                    return;
                }
            }
            if (wide) store_chunks(std::false_type{}, Wide{});
            else store_chunks(std::false_type{}, Narrow{});
            return;
        }
    }
    if (mine) {
        const int i = simple ? 0 : s_idx[t];  // a simple cell reads entry 0 and ignores it
        if (simple || i < px_cells) {         // listed cells beyond the buffer: stored by the search
            if constexpr (CODES) {
                if (codes) {
                    store_cell(std::true_type{}, i);
                    return;
                }
            }
            store_cell(std::false_type{}, i);
        }
    }
}


using RasterFn = void (*)(const DevItem*, const uint2*, int, const uint8_t*, const uint8_t*, uint8_t*,
                          const uint32_t*, const uint32_t*, const uint8_t*, uint8_t*);
using SmoothFn = void (*)(const DevItem*, const uint2*, int, const uint8_t*, const uint8_t*, uint8_t*, uint32_t*);

// The raster and smoothing kernels of scale S (1..15), per tile shape (one
// translation unit each: raster_tiles.hip).
// walk: the variants that load the walk window (tile_resolve's WALK)
RasterFn pick_raster_t16(int S, bool sub, bool walk);
RasterFn pick_raster_t32(int S, bool sub, bool walk);
RasterFn pick_raster_t64(int S, bool sub, bool walk);
SmoothFn pick_smooth_t16(int S, bool walk);
SmoothFn pick_smooth_t32(int S, bool walk);
SmoothFn pick_smooth_t64(int S, bool walk);

inline RasterFn pick_raster(int S, bool sub, int tx, bool walk = false)
{
    return tx == 16 ? pick_raster_t16(S, sub, walk) : tx == 64 ? pick_raster_t64(S, sub, walk)
                                                              : pick_raster_t32(S, sub, walk);
}
inline SmoothFn pick_smooth(int S, int tx, bool walk = false)
{
    return tx == 16 ? pick_smooth_t16(S, walk) : tx == 64 ? pick_smooth_t64(S, walk) : pick_smooth_t32(S, walk);
}

}  // namespace dpx
