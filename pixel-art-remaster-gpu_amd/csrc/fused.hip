// fused.hip -- the batched path: many frames or sprites of uneven size
// through two fused kernels, three with subdivision.
//
//   kf_graph   strip of 62 columns of a row block, one wave: lane words (YUV
//              fields + class) once per pixel, similarity in four directions
//              (the other four by symmetry) and the trivial crossing removal
//              on row masks in scalar registers -> snapshot graph (1 B/px)
//   kf_raster  tile of 32x8 cells (or 16x16, 64x4): heuristic crossing
//              resolution on the snapshot (crossed blocks listed and decided
//              once), cell keys and coverage summaries in LDS; cells whose S*S
//              pixels are all their own colour are simple, the rest are
//              listed and resolved (cell by cell at 1x to 7x, row by row from
//              8x) against the 3x3 candidate cells in draw order; then every
//              row of the tile's output is stored once, simple and resolved
//              pixels by the same store instructions.
//
// Coverage of an unsmoothed cell depends only on its 12-bit key and the
// scale, so it is precomputed once per scale into a table of sample-row
// bitmasks (kt_mask): bit b of row r of key k says whether sample
// (kmin+b, kmin+r) of the cell's local sample grid is covered, kmin =
// -(S/2)-1, MW = 2S+2 rows and columns (a hull lies within -0.25 .. 1.25 of
// the cell); into a summary byte per key (kt_info, coverage_info's low bits);
// and at 1x to 8x into each key's sample mask of each neighbour cell (kt_cell).
//
// With subdivision, kf_smooth runs between the two: it resolves the crossings
// of each tile, smooths its non-internal cells (polygons in LDS, each own
// cell once) and writes their coverage, as cell masks up to 8x and as sample
// rows from 9x; the raster (kf_raster<S, true>) then reads the resolved graph
// and that coverage, and resolves no crossings.
#include <dlfcn.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <string>
#include <type_traits>
#include <vector>

#include "batch.hpp"
#include "strips.hpp"

namespace dpx {

// ---------------------------------------------------------------------------
// tables
// ---------------------------------------------------------------------------
// Coverage bits of one sample row of a polygon given in 1/64 units and
// already ear-clipped (tri, nt).  Units of the test: 1/(128 S) of a cell.
__device__ inline uint32_t coverage_row(const int* x, const int* y, const uint8_t* tri, int nt, int S, int r)
{
    const int kmin = mask_kmin(S), mw = mask_w(S);
    int sy = (2 * (kmin + r) + 1) * 64;
    uint32_t bits = 0;
    for (int t = 0; t < nt; t++) {
        int ax = x[tri[3 * t]] * 2 * S, ay = y[tri[3 * t]] * 2 * S;
        int bx = x[tri[3 * t + 1]] * 2 * S, by = y[tri[3 * t + 1]] * 2 * S;
        int cx = x[tri[3 * t + 2]] * 2 * S, cy = y[tri[3 * t + 2]] * 2 * S;
        int ymin = min(ay, min(by, cy)), ymax = max(ay, max(by, cy));
        if (sy < ymin || sy > ymax) continue;
        for (int b = 0; b < mw; b++) {
            int sx = (2 * (kmin + b) + 1) * 64;
            if (tri_covers(ax, ay, bx, by, cx, cy, sx, sy)) bits |= 1u << b;
        }
    }
    return bits;
}

__global__ void kt_mask(int S, uint32_t* __restrict__ mask)
{
    int gid = blockIdx.x * blockDim.x + threadIdx.x;
    const int mw = mask_w(S);
    if (gid >= kKeys * mw) return;
    int key = gid / mw, r = gid % mw;
    const HullBits h = kHullTable[key];
    const int n = hull_count(h);
    int x[kMaxPoly], y[kMaxPoly];
    for (int t = 0; t < n; t++) { x[t] = 16 * hull_x(h, t); y[t] = 16 * hull_y(h, t); }
    uint8_t tri[3 * kMaxPoly];
    int ok;
    int nt = ear_clip(x, y, n, tri, &ok);
    mask[gid] = coverage_row(x, y, tri, nt, S, r);
}


// The keys' cell masks (cell_mask_rows), after the row table in the same
// allocation: entry key * 9 + j.
template <int S>
__global__ void kt_cell(const uint32_t* __restrict__ mask, uint8_t* __restrict__ cell)
{
    constexpr int TB = S <= kMaxCellScale16 ? 2 : 8;
    const int key = blockIdx.x * blockDim.x + threadIdx.x;
    if (key >= kKeys) return;
    const uint32_t* rows = mask + (size_t)key * mask_w(S);
    uint64_t m[9] = {};
    cell_mask_rows<S, mask_kmin(S), mask_kmin(S), mask_w(S)>(
        [&](int r) { return rows[r]; },
        [&](int j, int ky, uint32_t bits) { m[j] |= (uint64_t)bits << (ky * (TB == 2 ? S : 8)); });
    for (int j = 0; j < 9; j++) __builtin_memcpy(cell + (size_t)(key * 9 + j) * TB, &m[j], TB);
}

using CellFn = void (*)(const uint32_t*, uint8_t*);
inline CellFn pick_cell_table(int S)
{
    static constexpr CellFn fns[kMaxCellScale + 1] = { nullptr,    kt_cell<1>, kt_cell<2>, kt_cell<3>, kt_cell<4>,
                                                       kt_cell<5>, kt_cell<6>, kt_cell<7>, kt_cell<8> };
    return S <= kMaxCellScale ? fns[S] : nullptr;
}

__global__ void kt_info(const uint32_t* __restrict__ mask, int S, uint8_t* __restrict__ info)
{
    int key = blockIdx.x * blockDim.x + threadIdx.x;
    if (key >= kKeys) return;
    info[key] = (uint8_t)coverage_info(mask + (size_t)key * mask_w(S), S, mask_kmin(S), mask_kmin(S), mask_w(S));
}


// ---------------------------------------------------------------------------
// kf_graph: similarity graph + trivial crossing removal
// ---------------------------------------------------------------------------
// One wave marches down the rows of a strip of 64 columns, one column per
// lane, with the lane word (pixel class + YUV fields, see yuv_lanes) of the
// row above in a register and no LDS, barrier or second pass:
//   * a similarity test is two subtractions, one three-input logic operation
//     and a compare; the right neighbours' words come through the DPP shift
//     of the subtraction itself.  Each pixel tests the four edges it owns
//     (up, up-right, right, down-right: similarity is symmetric);
//   * a compare leaves its 64 answers as one bit each in a scalar register
//     pair, so the other four edges (the neighbours' own, one bit further
//     left or one row down) and the trivial removal (a 2x2 block with all
//     four orthogonal edges loses both diagonals, crossCheck_4) are scalar
//     64-bit operations on whole rows, issued beside other waves' vector work;
//   * the eight bits of a pixel's byte are shifted in by add-with-carry, a
//     row mask as the carries.
// The kernel is bound by vector issue (its bytes would take a quarter of its
// time), so what counts is instructions a pixel: 46 against the 95 of 64-wide
// tiles whose lane words and bytes went through LDS.  1024 frames of 256x224:
// 169 -> 105 us, 82% of the vector issue rate; 16 of 640x480: 23 -> 15.6 us;
// 4096 sprites of 8 to 64 pixels: 28 -> 17 us (their tiles were half empty).
//
// The strips are cut as strips.hpp says: 62 columns each (the outer two lanes
// are halo), several row blocks of an item side by side.
// One more bit of each lane's byte: v + v + (the lane's bit of m).  m is the
// result of a scalar operation: a vector compare's result would have to be
// two wait states old, and the compiler does not look into the block for it.
__device__ inline void shift_in(uint32_t& v, uint64_t m)
{
    uint64_t c;
    asm("v_addc_co_u32_e64 %0, %1, %0, %0, %2" : "+v"(v), "=s"(c) : "s"(m));
}

// A row of lane words as the tests take it (see lane_similar): l, l + bias and
// bias - l.
struct LaneRow {
    uint32_t l, plus, minus;
};

// The edges between row a and row b above it: a's up and up-right edges, b's
// right and down-right ones (the lane's pixel as their left end).  One block,
// so that the neighbour's word comes by the DPP shift of the subtraction
// itself (left to the compiler, a shifted word with two uses is moved first)
// and no shifted operand was written less than two instructions before.  The
// shifted operand is an addend or the minuend: a reversed subtraction
// (v_subrev) with a shift shifts its minuend.
struct RowEdges {
    uint64_t up, up_right, right, down_right;
};

__device__ inline RowEdges row_edges(const LaneRow& a, LaneRow& b)
{
    RowEdges e;
    uint32_t u, v, r0, r1, x, y, d0, d1;
#define DPX_RIGHT " wave_shl:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
    asm("v_add_u32_e32 %[bp], %[bias], %[b]\n\t"
        "v_sub_u32_e32 %[bm], %[bias], %[b]\n\t"
        "v_sub_u32_e32 %[u], %[ap], %[b]\n\t"
        "v_sub_u32_e32 %[v], %[bp], %[a]\n\t"
        "v_add_u32_dpp %[d0], %[am], %[b]" DPX_RIGHT
        "v_sub_u32_dpp %[d1], %[ap], %[b]" DPX_RIGHT
        "v_add_u32_dpp %[r0], %[bm], %[b]" DPX_RIGHT
        "v_sub_u32_dpp %[r1], %[bp], %[b]" DPX_RIGHT
        "v_add_u32_dpp %[x], %[bm], %[a]" DPX_RIGHT
        "v_sub_u32_dpp %[y], %[bp], %[a]" DPX_RIGHT
        "v_bitop3_b32 %[u], %[u], %[test], %[v] bitop3:0x80\n\t"
        "v_bitop3_b32 %[d0], %[d0], %[test], %[d1] bitop3:0x80\n\t"
        "v_bitop3_b32 %[r0], %[r0], %[test], %[r1] bitop3:0x80\n\t"
        "v_bitop3_b32 %[x], %[x], %[test], %[y] bitop3:0x80\n\t"
        "v_cmp_eq_u32_e64 %[eu], %[test], %[u]\n\t"
        "v_cmp_eq_u32_e64 %[ed], %[test], %[d0]\n\t"
        "v_cmp_eq_u32_e64 %[er], %[test], %[r0]\n\t"
        "v_cmp_eq_u32_e64 %[ex], %[test], %[x]"
        : [bp] "=&v"(b.plus), [bm] "=&v"(b.minus), [u] "=&v"(u), [v] "=&v"(v), [d0] "=&v"(d0), [d1] "=&v"(d1),
          [r0] "=&v"(r0), [r1] "=&v"(r1), [x] "=&v"(x), [y] "=&v"(y), [eu] "=&s"(e.up), [ed] "=&s"(e.down_right),
          [er] "=&s"(e.right), [ex] "=&s"(e.up_right)
        : [a] "v"(a.l), [ap] "v"(a.plus), [am] "v"(a.minus), [b] "v"(b.l), [bias] "s"(kSimilarBias),
          [test] "s"(kSimilarTest));
#undef DPX_RIGHT
    return e;
}

__device__ inline bool lane_of(uint64_t mask) { return __builtin_amdgcn_inverse_ballot_w64(mask); }

// How pixels become lane words.
enum GraphPixels {
    kPixelsPlain,    // 3 or 4 bytes, blue first, no alpha test
    kPixelsGeneral,  // either order, alpha test
    kPixelsIndexed,  // one byte, the palette's lane words in LDS
};

template <int PIXELS>
__device__ __forceinline__ void graph_strip(const DevItem& it, const GraphSplit sp, uint32_t strip,
                                            const uint8_t* __restrict__ in, const uint32_t* s_pal,
                                            uint8_t* __restrict__ gaux)
{
    constexpr int G = kGraphRows;
    const uint32_t lane = threadIdx.x;
    const bool topdown = it.flags & DPX_TOPDOWN;
    const int W = it.W, H = it.H;
    const StripLane sl = strip_lane(W, sp, strip, lane);
    const bool col = sl.col;
    const int x = sl.x, y0 = sl.y0;
    const uint64_t cols = __builtin_amdgcn_ballot_w64(col);
    const uint64_t mine = cols & 0x7FFFFFFFFFFFFFFEull;  // the columns stored by this strip
    const int y0_first = __builtin_amdgcn_readlane(y0, 0), y0_last = __builtin_amdgcn_readlane(y0, 63);
    const int R = (int)sp.rows + 2;  // row r is y = y0 - 1 + r

    // Pixels are read through a buffer descriptor of the item's rows.  Rows
    // r_lo .. r_hi - 1 lie in the frame for every lane.  Groups that may hold
    // the last pixel of a frame of 3-byte pixels (`tail`: a lane of the strip
    // loads it) leave it out of their word loads and read it by bytes.
    const uint32_t step = strip_step(it.stride, topdown);
    const uint32_t voff = strip_offset(sl, H, it.stride, it.ch, topdown);
    const uint32_t in_end = (uint32_t)(H - 1) * (uint32_t)it.stride + (uint32_t)(W * it.ch);
    const auto src = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(in + it.in_off), 0, in_end, 0x00020000);
    const int r_lo = 1 - y0_first, r_hi = H + 1 - y0_last;
    const bool tail = PIXELS != kPixelsIndexed && it.ch < 4 &&
                      __builtin_amdgcn_ballot_w64(strip_loads_last(sl, W, H, topdown, strip_loaded_rows(sp))) != 0;

    uint32_t px[G];
    auto fetch = [&](int r0) {
        uint32_t o = voff + (uint32_t)(r0 - 1) * step;
        if (tail && group_loads_last(r0, topdown, r_hi)) {  // (as many loads as below)
#pragma unroll
            for (int q = 0; q < G; q++) {
                px[q] = __builtin_amdgcn_raw_buffer_load_b32(src, (int)(word_crosses(o, in_end, 3) ? ~0u : o), 0, 0);
                o += step;
            }
            return;
        }
#pragma unroll
        for (int q = 0; q < G; q++) {
            if constexpr (PIXELS == kPixelsIndexed)
                px[q] = __builtin_amdgcn_raw_buffer_load_b8(src, (int)o, 0, 0);
            else
                px[q] = __builtin_amdgcn_raw_buffer_load_b32(src, (int)o, 0, 0);
            o += step;
        }
    };
    // the pixels of a group once more, by bytes
    auto fetch_bytes = [&](int r0) {
        const uint32_t o = voff + (uint32_t)(r0 - 1) * step;
#pragma unroll
        for (int q = 0; q < G; q++) {
            px[q] = 0;
#pragma unroll
            for (int k = 0; k < 3; k++)
                px[q] |= (uint32_t)__builtin_amdgcn_raw_buffer_load_b8(src, (int)(o + (uint32_t)q * step) + k, 0, 0)
                         << (8 * k);
        }
    };

    // Lane words (see luma_sum and lane_fields for the steps).
    const uint32_t cls = col ? kLaneOpaque : 0u, cls_clear = col ? kLaneTransparent : 0u;
    const uint32_t order = (it.flags & DPX_RGB) ? 0x03000102u : 0x03020100u;
    const uint32_t clear_below = ((it.flags & DPX_ALPHA) && it.ch == 4) ? 1u << 24 : 0u;
    const uint32_t col_mask = col ? ~0u : 0u;
    auto lane_words = [&](uint32_t* v) {
        if constexpr (PIXELS == kPixelsIndexed) {
#pragma unroll
            for (int q = 0; q < G; q++) v[q] = s_pal[v[q]] & col_mask;
        } else {
            uint32_t y[G];
            uint64_t whole[G];
#pragma unroll
            for (int q = 0; q < G; q++) {
                if constexpr (PIXELS == kPixelsGeneral) v[q] = __builtin_amdgcn_perm(0u, v[q], order);
                const uint32_t n = luma_sum(v[q]);
                y[q] = luma_quotient(n);
                whole[q] = __builtin_amdgcn_ballot_w64(luma_whole(n));
            }
            uint64_t any = 0;
#pragma unroll
            for (int q = 0; q < G; q++) any |= whole[q];
            if (any) {
#pragma unroll
                for (int q = 0; q < G; q++)
                    if (whole[q])
                        y[q] = (uint32_t)luma((int)(v[q] & 0xFFu), (int)((v[q] >> 8) & 0xFFu),
                                              (int)((v[q] >> 16) & 0xFFu));
            }
#pragma unroll
            for (int q = 0; q < G; q++) {
                uint32_t f = lane_fields(v[q], y[q]) | cls;
                if constexpr (PIXELS == kPixelsGeneral) f = v[q] < clear_below ? cls_clear : f;
                v[q] = f;
            }
        }
    };

    // The bytes are stored through a buffer descriptor of the item's graph:
    // lanes whose pixel is not this strip's to write get an offset past its
    // end, which the hardware drops, so that a group of rows has no branch
    // and its rows overlap.
    const uint32_t goff = (uint32_t)y0 * (uint32_t)W + (uint32_t)x;
    const auto out = __builtin_amdgcn_make_buffer_rsrc(gaux + it.g_off, 0, W * H, 0x00020000);
    uint64_t every = ~0ull;
    asm("" : "+s"(every));  // (kept an operand, see shift_in)

    LaneRow a = {};                           // row r - 1
    uint64_t ra = 0, dra = 0, ua = 0, ura = 0;  // row r - 1's R and kept DR; row r - 2's U and kept UR
    const uint32_t gput = lane_of(mine) ? goff : ~0u;

    fetch(0);
    // Loads and stores return in one order, so that waiting for a group's
    // pixels need not wait for the stores issued after them, if their number
    // is always the same: every pass below issues G stores, and so does the
    // way into the loop (dropped).
#pragma unroll
    for (int q = 0; q < G; q++) __builtin_amdgcn_raw_buffer_store_b8((uint8_t)0, out, -1, 0, 0);
    for (int r0 = 0; r0 < R; r0 += G) {
        if (tail && group_loads_last(r0, topdown, r_hi)) fetch_bytes(r0);
        uint32_t w[G];
#pragma unroll
        for (int q = 0; q < G; q++) w[q] = px[q];
        if (r0 + G < R) fetch(r0 + G);
        lane_words(w);
        if (r0 < r_lo || r0 + G > r_hi) {
#pragma unroll
            for (int q = 0; q < G; q++) w[q] = (unsigned)(y0 - 1 + r0 + q) < (unsigned)H ? w[q] : 0u;
        }
        RowEdges ed[G];
#pragma unroll
        for (int q = 0; q < G; q++) {
            LaneRow b;
            b.l = w[q];
            ed[q] = row_edges(a, b);
            a = b;
        }
        uint32_t byte[G];
#pragma unroll
        for (int q = 0; q < G; q++) {
            const uint64_t u = ed[q].up & every, rt = ed[q].right & every;
            const uint64_t full = u & ra & rt & (u >> 1);  // blocks with lower-left pixels in row r - 1
            const uint64_t urk = ed[q].up_right & ~full, drk = ed[q].down_right & ~full;
            byte[q] = lane_of(dra) ? 1u : 0u;
            shift_in(byte[q], ua);
            shift_in(byte[q], ura << 1);
            shift_in(byte[q], ra);
            shift_in(byte[q], ra << 1);
            shift_in(byte[q], urk);
            shift_in(byte[q], u);
            shift_in(byte[q], drk << 1);
            ra = rt;
            dra = drk;
            ua = u;
            ura = urk;
        }
        // byte[q] is row r0 + q - 1's; rows 1 .. R - 2 in the frame are stored
        uint32_t to[G];
#pragma unroll
        for (int q = 0; q < G; q++) to[q] = gput;
        if (r0 < r_lo + 1 || r0 < 2 || r0 + G > min(r_hi + 1, R)) {
#pragma unroll
            for (int q = 0; q < G; q++)
                to[q] = r0 + q >= 2 && r0 + q < R && (unsigned)(y0 - 2 + r0 + q) < (unsigned)H ? gput : ~0u;
        }
#pragma unroll
        for (int q = 0; q < G; q++)
            __builtin_amdgcn_raw_buffer_store_b8((uint8_t)byte[q], out, (int)to[q], (int)((uint32_t)max(r0 + q - 2, 0) * (uint32_t)W), 0);
    }
}

__global__ __launch_bounds__(64) void kf_graph(const DevItem* __restrict__ items, const uint2* __restrict__ tile_map,
                                               int grid3d, int max_rows, const uint8_t* __restrict__ in,
                                               uint8_t* __restrict__ gaux)
{
    __shared__ uint32_t s_pal[256];
    // runs of 8 strips per XCD: the lines that neighbouring strips' rows share
    // are fetched once into one L2
    const TileAt at = locate_tile<8>(tile_map, grid3d);
    const DevItem it = items[at.item];
    const uint32_t strip = (uint32_t)at.ty << 16 | (uint32_t)at.tx;
    const GraphSplit sp = graph_split(it.W, it.H, max_rows);
    if (strip >= sp.strips) return;  // (an item of fewer strips than the launch has for each)
    if (it.flags & DPX_INDEXED) {
        // the lane words of the 256 palette entries
        const uint32_t order = (it.flags & DPX_RGB) ? 0x03000102u : 0x03020100u;
        for (int k = threadIdx.x; k < 256; k += 64) {
            const uint32_t e = __builtin_amdgcn_perm(0u, reinterpret_cast<const uint32_t*>(in + it.pal_off)[k], order);
            uint32_t lw = yuv_lanes(yuv_pack((int)(e & 0xFFu), (int)((e >> 8) & 0xFFu), (int)((e >> 16) & 0xFFu))) |
                          kLaneOpaque;
            if ((it.flags & DPX_ALPHA) && (e >> 24) == 0) lw = kLaneTransparent;
            s_pal[k] = lw;
        }
        __syncthreads();
        graph_strip<kPixelsIndexed>(it, sp, strip, in, s_pal, gaux);
    } else if (it.flags & (DPX_RGB | DPX_ALPHA)) {
        graph_strip<kPixelsGeneral>(it, sp, strip, in, s_pal, gaux);
    } else {
        graph_strip<kPixelsPlain>(it, sp, strip, in, s_pal, gaux);
    }
}

}  // namespace dpx


// ---------------------------------------------------------------------------
// context
// ---------------------------------------------------------------------------
// The launch plan of the last batch.  A batch whose items and output
// alignment equal the last one's reuses it (no validation, grouping, tile
// maps or descriptor comparison): for thousands of sprites that host work
// takes longer than the kernels.
struct PlanGroup {
    int scale;
    bool sub;
    int tx;  // raster tile width (cells): 16, 32 or 64
    dim3 grid;
    int grid3d;
    size_t off_items, off_map;  // in the descriptor buffer
    bool walk;  // the crossing walks read a larger LDS window (tile_resolve's WALK)
};
struct BatchPlan {
    bool valid = false;
    std::vector<dpx_item> items;
    uintptr_t out_mod = 0;  // d_out % 16
    dim3 ggrid;
    int g3d = 0;
    int grows = dpx::kGraphMinRows;  // rows of kf_graph's blocks
    size_t off_items = 0, off_gmap = 0;
    std::vector<PlanGroup> groups;
};

struct dpx_context {
    BatchPlan plan;
    int device = 0;
    uint32_t* d_mask[dpx::kMaxScale + 1] = {};
    uint8_t* d_info[dpx::kMaxScale + 1] = {};
    uint8_t *d_gaux = nullptr, *d_gfin = nullptr;
    size_t g_cap = 0;
    uint32_t* d_rows = nullptr;  // cell rows of smoothed cells (kf_smooth)
    size_t rows_cap = 0;
    uint8_t* d_desc = nullptr;
    size_t desc_cap = 0;
    uint8_t* h_pinned = nullptr;
    size_t pinned_cap = 0;
    hipEvent_t upload_done = nullptr;
    bool upload_pending = false;
    std::vector<uint8_t> last_desc;
    std::vector<uint64_t> g_offsets;
    bool keep_graph = false;  // write the resolved graphs (dpx_context_keep_graph)
    bool last_kept = false;   // the last batch wrote them
    // raster tile width per (size class, scale, subdivision); 0: the default
    int8_t tile_pick[3][dpx::kMaxScale + 1][2] = {};
    // walk window per (size class, scale, subdivision): DPX_WALK_AUTO (the
    // tuned choice: DPX_WALK_ALWAYS where tuning.json asks for the window,
    // else none), DPX_WALK_ALWAYS or DPX_WALK_NEVER
    int8_t walk_pick[3][dpx::kMaxScale + 1][2] = {};
    std::mutex mu;
    // kernel timing: 3 events per recorded batch (start, after graph, end)
    bool timing = false;
    std::vector<hipEvent_t> ev_pool;
    size_t ev_used = 0;
    dpx_batch_times acc{};
};

namespace {

using namespace dpx;

// Size class of an item for the tile picks.
int size_class(int W, int H)
{
    if (W <= 64 && H <= 64) return DPX_CLASS_SPRITE;
    if (W <= 512 && H <= 512) return DPX_CLASS_FRAME;
    return DPX_CLASS_LARGE;
}

int item_tile(const dpx_context* ctx, const dpx_item& a)
{
    const int t = ctx->tile_pick[size_class(a.width, a.height)][a.scale][a.subdivide ? 1 : 0];
    return t ? t : kDefaultTileX;
}

int item_walk(const dpx_context* ctx, const dpx_item& a)
{
    return ctx->walk_pick[size_class(a.width, a.height)][a.scale][a.subdivide ? 1 : 0];
}

// The tile picks of a tuning file: a JSON object whose "picks" array holds
// objects {"class": "sprite" | "frame" | "large", "scale": 1..15,
// "subdivide": 0 | 1, "tile": 16 | 32 | 64, "walk": 0 | 1} (other keys are
// ignored; "walk": 1 picks the walk window for every launch of the key).
// Returns the number of picks applied.
int load_tuning(dpx_context* ctx, const char* path)
{
    FILE* f = fopen(path, "rb");
    if (!f) return 0;
    std::string text;
    char buf[4096];
    size_t n;
    while ((n = fread(buf, 1, sizeof(buf), f)) > 0) text.append(buf, n);
    fclose(f);
    const size_t picks = text.find("\"picks\"");
    if (picks == std::string::npos) return 0;
    int applied = 0;
    for (size_t a = text.find('{', picks); a != std::string::npos; a = text.find('{', a + 1)) {
        const size_t b = text.find('}', a);
        if (b == std::string::npos) break;
        const std::string obj = text.substr(a, b - a);
        auto num = [&](const char* key, int* v) {
            const size_t k = obj.find(key);
            if (k == std::string::npos) return false;
            const size_t c = obj.find(':', k);
            if (c == std::string::npos) return false;
            *v = atoi(obj.c_str() + c + 1);
            return true;
        };
        int cls = -1, scale = 0, sub = 0, tile = 0, walk = 0;
        if (obj.find("\"sprite\"") != std::string::npos) cls = DPX_CLASS_SPRITE;
        else if (obj.find("\"frame\"") != std::string::npos) cls = DPX_CLASS_FRAME;
        else if (obj.find("\"large\"") != std::string::npos) cls = DPX_CLASS_LARGE;
        if (cls < 0 || !num("\"scale\"", &scale) || !num("\"tile\"", &tile)) continue;
        num("\"subdivide\"", &sub);
        num("\"walk\"", &walk);
        if (scale < 1 || scale > kMaxScale || (tile != 16 && tile != 32 && tile != 64)) continue;
        ctx->tile_pick[cls][scale][sub ? 1 : 0] = (int8_t)tile;
        ctx->walk_pick[cls][scale][sub ? 1 : 0] = (int8_t)(walk == 1 ? DPX_WALK_ALWAYS : DPX_WALK_AUTO);
        applied++;
    }
    return applied;
}

// The tuning file: $DPX_TUNING, else tuning.json in the package directory
// (one level above the directory of this library).
std::string tuning_path()
{
    if (const char* e = getenv("DPX_TUNING")) return e;
    Dl_info info;
    if (dladdr(reinterpret_cast<const void*>(&tuning_path), &info) && info.dli_fname) {
        std::string p = info.dli_fname;
        const size_t slash = p.rfind('/');
        p = slash == std::string::npos ? std::string(".") : p.substr(0, slash);
        return p + "/../tuning.json";
    }
    return "tuning.json";
}

int ensure_mask(dpx_context* ctx, int S)
{
    if (ctx->d_mask[S] && ctx->d_info[S]) return DPX_OK;
    size_t n = (size_t)kKeys * mask_w(S);
    const size_t cell_bytes = cell_table_bytes(S);
    if (!ctx->d_mask[S]) DPX_HIP(hipMalloc(&ctx->d_mask[S], n * sizeof(uint32_t) + cell_bytes));
    if (!ctx->d_info[S]) DPX_HIP(hipMalloc(&ctx->d_info[S], kKeys));
    hipLaunchKernelGGL(kt_mask, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, 0, S, ctx->d_mask[S]);
    if (cell_bytes)
        hipLaunchKernelGGL(pick_cell_table(S), dim3(kKeys / 256), dim3(256), 0, 0, ctx->d_mask[S],
                           reinterpret_cast<uint8_t*>(ctx->d_mask[S] + n));
    hipLaunchKernelGGL(kt_info, dim3(kKeys / 256), dim3(256), 0, 0, ctx->d_mask[S], S, ctx->d_info[S]);
    DPX_HIP(hipGetLastError());
    DPX_HIP(hipDeviceSynchronize());
    return DPX_OK;
}

struct Group {
    int scale;
    bool sub;
    int tx = kDefaultTileX;
    int walk = DPX_WALK_AUTO;
    std::vector<DevItem> dev;  // the group's items, in launch order
    std::vector<uint2> map;    // tile map of a 1-D launch
    dim3 grid;
    int grid3d = 0;
};

size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

// Growth of the context's device buffers.  A buffer the device may still be
// reading is only replaced after the device is idle.
int grow_graph(dpx_context* ctx, size_t need)
{
    if (need <= ctx->g_cap) return DPX_OK;
    DPX_HIP(hipDeviceSynchronize());
    (void)hipFree(ctx->d_gaux);
    (void)hipFree(ctx->d_gfin);
    ctx->d_gaux = ctx->d_gfin = nullptr;
    ctx->g_cap = 0;
    size_t cap = align_up(need + need / 4, 1 << 20);
    DPX_HIP(hipMalloc(&ctx->d_gaux, cap));
    DPX_HIP(hipMalloc(&ctx->d_gfin, cap));
    ctx->g_cap = cap;
    return DPX_OK;
}

int grow_rows(dpx_context* ctx, size_t need)
{
    if (need <= ctx->rows_cap) return DPX_OK;
    DPX_HIP(hipDeviceSynchronize());
    (void)hipFree(ctx->d_rows);
    ctx->d_rows = nullptr;
    ctx->rows_cap = 0;
    size_t cap = align_up(need + need / 4, 1 << 20);
    DPX_HIP(hipMalloc(&ctx->d_rows, cap));
    ctx->rows_cap = cap;
    return DPX_OK;
}

int grow_desc(dpx_context* ctx, size_t need)
{
    if (need <= ctx->desc_cap) return DPX_OK;
    if (ctx->upload_pending) {
        DPX_HIP(hipEventSynchronize(ctx->upload_done));
        ctx->upload_pending = false;
    }
    DPX_HIP(hipDeviceSynchronize());
    (void)hipFree(ctx->d_desc);
    ctx->d_desc = nullptr;
    if (ctx->h_pinned) (void)hipHostFree(ctx->h_pinned);
    ctx->h_pinned = nullptr;
    ctx->desc_cap = ctx->pinned_cap = 0;
    ctx->last_desc.clear();
    ctx->plan.valid = false;  // its descriptors are gone with the buffer
    size_t cap = align_up(need * 2, 1 << 16);
    DPX_HIP(hipMalloc(&ctx->d_desc, cap));
    DPX_HIP(hipHostMalloc(&ctx->h_pinned, cap, hipHostMallocDefault));
    ctx->desc_cap = cap;
    ctx->pinned_cap = cap;
    return DPX_OK;
}

// Descriptor bytes of a batch of up to n items of up to `pixels` pixels: the
// items twice (all, and per group), each array 64-byte aligned, with room for
// one group per (scale, subdivision) pair, and kf_graph's map of strips, which
// items of the same tile grid need as well when their strips differ.  (Groups
// of mixed sizes add raster tile maps and may grow the buffer.)
size_t desc_bytes(size_t n, size_t pixels)
{
    return 2 * n * sizeof(DevItem) + graph_strips_bound(n, pixels) * sizeof(uint2) + 64 * (2 * 2 * (kMaxScale + 1) + 4);
}

// Launch grid of a kernel with TX x TY tiles over `dev`: (tile columns, tile
// rows, items) when all items have the same tile grid, else 1-D over all
// tiles with a map from block to (item, tile row << 16 | tile column).
// *grid3d tells the kernel which.  Tile columns and rows fit 16 bits: items
// are at most 32768 pixels wide and high.
dim3 tile_grid(const std::vector<DevItem>& dev, int TX, int TY, int* grid3d, std::vector<uint2>* map)
{
    const unsigned tx0 = (unsigned)(dev[0].W + TX - 1) / TX, ty0 = (unsigned)(dev[0].H + TY - 1) / TY;
    bool same = dev.size() <= 65535;
    for (const DevItem& d : dev)
        same = same && (unsigned)(d.W + TX - 1) / TX == tx0 && (unsigned)(d.H + TY - 1) / TY == ty0;
    map->clear();
    *grid3d = same ? 1 : 0;
    if (same) return dim3(tx0, ty0, (unsigned)dev.size());
    size_t total = 0;
    for (const DevItem& d : dev) total += (size_t)((unsigned)(d.W + TX - 1) / TX) * ((unsigned)(d.H + TY - 1) / TY);
    map->resize(total);
    uint2* at = map->data();
    for (size_t k = 0; k < dev.size(); k++) {
        const unsigned tx = (unsigned)(dev[k].W + TX - 1) / TX, ty = (unsigned)(dev[k].H + TY - 1) / TY;
        for (unsigned y = 0; y < ty; y++)
            for (unsigned x = 0; x < tx; x++) *at++ = make_uint2((unsigned)k, y << 16 | x);
    }
    return dim3((unsigned)total, 1, 1);
}

// The same for kf_graph's strips: (strips, 1, items) when all items have nearly
// as many as the most, else 1-D with a map to (item, strip).  The waves past an
// item's last strip end at once; an eighth of them costs less than a map, which
// is uploaded whenever the items change (64 frames of 248 to 256 columns at 2x,
// other items each call: 78 us with a map; five of 640 and 639 columns:
// 59).
dim3 strip_grid(const std::vector<DevItem>& dev, int max_rows, int* grid3d, std::vector<uint2>* map)
{
    std::vector<uint32_t> strips(dev.size());
    uint32_t total = 0, most = 0;
    for (size_t k = 0; k < dev.size(); k++) {
        const bool as_before = k && dev[k].W == dev[k - 1].W && dev[k].H == dev[k - 1].H;
        strips[k] = as_before ? strips[k - 1] : graph_split(dev[k].W, dev[k].H, max_rows).strips;
        most = std::max(most, strips[k]);
        total += strips[k];
    }
    map->clear();
    *grid3d = dev.size() <= 65535 && (uint64_t)most * dev.size() <= (uint64_t)total + total / 8 ? 1 : 0;
    if (*grid3d) return dim3(most, 1, (unsigned)dev.size());
    map->resize(total);
    uint2* at = map->data();
    for (size_t k = 0; k < dev.size(); k++)
        for (uint32_t q = 0; q < strips[k]; q++) *at++ = make_uint2((unsigned)k, q);
    return dim3(total, 1, 1);
}

}  // namespace

extern "C" int dpx_context_create(int device, dpx_context** out)
{
    DPX_CHECK(out, DPX_EINVAL, "null output pointer");
    *out = nullptr;
    if (int rc = require_device()) return rc;
    DPX_HIP(hipSetDevice(device));
    dpx_context* ctx = new dpx_context();
    ctx->device = device;
    auto cleanup = [&](int rc) {
        dpx_context_destroy(ctx);
        return rc;
    };
    if (hipEventCreateWithFlags(&ctx->upload_done, hipEventDisableTiming) != hipSuccess)
        return cleanup(fail(DPX_EHIP, "event creation failed"));
    load_tuning(ctx, tuning_path().c_str());
    *out = ctx;
    return DPX_OK;
}

extern "C" void dpx_context_destroy(dpx_context* ctx)
{
    if (!ctx) return;
    (void)hipSetDevice(ctx->device);
    (void)hipDeviceSynchronize();
    for (auto* m : ctx->d_mask) (void)hipFree(m);
    for (auto* m : ctx->d_info) (void)hipFree(m);
    (void)hipFree(ctx->d_gaux);
    (void)hipFree(ctx->d_gfin);
    (void)hipFree(ctx->d_rows);
    (void)hipFree(ctx->d_desc);
    if (ctx->h_pinned) (void)hipHostFree(ctx->h_pinned);
    if (ctx->upload_done) (void)hipEventDestroy(ctx->upload_done);
    for (auto e : ctx->ev_pool) (void)hipEventDestroy(e);
    delete ctx;
}

extern "C" int dpx_context_reserve(dpx_context* ctx, int max_items, int64_t max_item_pixels, int scale)
{
    DPX_CHECK(ctx && max_items > 0 && max_item_pixels > 0, DPX_EINVAL, "bad arguments");
    DPX_CHECK(scale >= 0 && scale <= kMaxScale, DPX_EINVAL, "scale %d outside 0..%d", scale, kMaxScale);
    std::lock_guard<std::mutex> lock(ctx->mu);
    DPX_HIP(hipSetDevice(ctx->device));
    if (int rc = grow_graph(ctx, (size_t)max_items * align_up((size_t)max_item_pixels, 256))) return rc;
    if (int rc = grow_desc(ctx, desc_bytes((size_t)max_items, (size_t)max_item_pixels))) return rc;
    if (scale > 0)
        if (int rc = ensure_mask(ctx, scale)) return rc;
    return DPX_OK;
}

namespace dpx {
int context_reserve_rows(dpx_context* ctx, size_t bytes)
{
    std::lock_guard<std::mutex> lock(ctx->mu);
    DPX_HIP(hipSetDevice(ctx->device));
    return grow_rows(ctx, bytes);
}
}  // namespace dpx

extern "C" int dpx_context_set_tile(dpx_context* ctx, int size_class, int scale, int subdivide, int tile_w)
{
    DPX_CHECK(ctx, DPX_EINVAL, "null context");
    DPX_CHECK(size_class >= 0 && size_class <= 2, DPX_EINVAL, "size class %d", size_class);
    DPX_CHECK(scale >= 1 && scale <= kMaxScale, DPX_EINVAL, "scale %d outside 1..%d", scale, kMaxScale);
    DPX_CHECK(tile_w == 0 || tile_w == 16 || tile_w == 32 || tile_w == 64, DPX_EINVAL, "tile width %d", tile_w);
    std::lock_guard<std::mutex> lock(ctx->mu);
    ctx->tile_pick[size_class][scale][subdivide ? 1 : 0] = (int8_t)tile_w;
    ctx->plan.valid = false;  // the next batch plans its groups again
    return DPX_OK;
}

extern "C" int dpx_context_get_tile(dpx_context* ctx, int size_class, int scale, int subdivide, int* tile_w)
{
    DPX_CHECK(ctx && tile_w, DPX_EINVAL, "bad arguments");
    DPX_CHECK(size_class >= 0 && size_class <= 2, DPX_EINVAL, "size class %d", size_class);
    DPX_CHECK(scale >= 1 && scale <= kMaxScale, DPX_EINVAL, "scale %d outside 1..%d", scale, kMaxScale);
    std::lock_guard<std::mutex> lock(ctx->mu);
    const int t = ctx->tile_pick[size_class][scale][subdivide ? 1 : 0];
    *tile_w = t ? t : kDefaultTileX;
    return DPX_OK;
}

extern "C" int dpx_context_set_walk(dpx_context* ctx, int size_class, int scale, int subdivide, int walk)
{
    DPX_CHECK(ctx, DPX_EINVAL, "null context");
    DPX_CHECK(size_class >= 0 && size_class <= 2, DPX_EINVAL, "size class %d", size_class);
    DPX_CHECK(scale >= 1 && scale <= kMaxScale, DPX_EINVAL, "scale %d outside 1..%d", scale, kMaxScale);
    DPX_CHECK(walk == DPX_WALK_AUTO || walk == DPX_WALK_ALWAYS || walk == DPX_WALK_NEVER, DPX_EINVAL,
              "walk window mode %d", walk);
    std::lock_guard<std::mutex> lock(ctx->mu);
    ctx->walk_pick[size_class][scale][subdivide ? 1 : 0] = (int8_t)walk;
    ctx->plan.valid = false;  // the next batch plans its groups again
    return DPX_OK;
}

extern "C" int dpx_context_get_walk(dpx_context* ctx, int size_class, int scale, int subdivide, int* walk)
{
    DPX_CHECK(ctx && walk, DPX_EINVAL, "bad arguments");
    DPX_CHECK(size_class >= 0 && size_class <= 2, DPX_EINVAL, "size class %d", size_class);
    DPX_CHECK(scale >= 1 && scale <= kMaxScale, DPX_EINVAL, "scale %d outside 1..%d", scale, kMaxScale);
    std::lock_guard<std::mutex> lock(ctx->mu);
    *walk = ctx->walk_pick[size_class][scale][subdivide ? 1 : 0];
    return DPX_OK;
}

extern "C" int dpx_context_keep_graph(dpx_context* ctx, int enable)
{
    DPX_CHECK(ctx, DPX_EINVAL, "null context");
    std::lock_guard<std::mutex> lock(ctx->mu);
    ctx->keep_graph = enable != 0;
    return DPX_OK;
}

extern "C" int dpx_batch_graph(dpx_context* ctx, const uint8_t** d_graph, const uint64_t** offsets_host)
{
    DPX_CHECK(ctx && d_graph && offsets_host, DPX_EINVAL, "bad arguments");
    DPX_CHECK(ctx->last_kept, DPX_EINVAL, "the last batch wrote no graphs (see dpx_context_keep_graph)");
    *d_graph = ctx->d_gfin;
    *offsets_host = ctx->g_offsets.data();
    return DPX_OK;
}

// Validates item k and fills its device descriptor; its graph bytes start
// at g_off of the graph scratch.
static int make_dev_item(const dpx_item& a, int k, const uint8_t* d_out, uint64_t g_off, DevItem& d)
{
    using namespace dpx;
    DPX_CHECK(a.width > 0 && a.height > 0 && a.width <= 32768 && a.height <= 32768, DPX_EINVAL,
              "item %d: bad size %dx%d", k, a.width, a.height);
    DPX_CHECK((a.flags & ~kKnownFlags) == 0, DPX_EINVAL, "item %d: unknown flags 0x%x", k, a.flags & ~kKnownFlags);
    const bool indexed = a.flags & DPX_INDEXED;
    DPX_CHECK(indexed ? a.channels == 1 : (a.channels == 3 || a.channels == 4), DPX_EINVAL, "item %d: channels %d%s",
              k, a.channels, indexed ? " (indexed frames have 1)" : "");
    DPX_CHECK(!indexed || a.palette_offset % 4 == 0, DPX_EINVAL, "item %d: palette offset %llu not a multiple of 4", k,
              (unsigned long long)a.palette_offset);
    DPX_CHECK(a.stride >= a.width * a.channels, DPX_EINVAL, "item %d: stride %d", k, a.stride);
    DPX_CHECK((int64_t)a.stride * a.height < (int64_t)1 << 31, DPX_EINVAL, "item %d: input larger than 2 GiB", k);
    DPX_CHECK(a.scale >= 1 && a.scale <= kMaxScale, DPX_EINVAL, "item %d: scale %d outside 1..%d", k, a.scale,
              kMaxScale);
    DPX_CHECK(a.out_stride >= 4 * a.width * a.scale && a.out_stride % 4 == 0 && a.out_offset % 4 == 0, DPX_EINVAL,
              "item %d: output layout (stride %d, offset %llu)", k, a.out_stride, (unsigned long long)a.out_offset);
    DPX_CHECK(!a.subdivide || (uint64_t)a.width * a.height * (2 * a.scale + 3) < ((uint64_t)1 << 32), DPX_EINVAL,
              "item %d: %dx%d at scale %d with subdivision exceeds 2^32 cell-row words", k, a.width, a.height, a.scale);
    memset(&d, 0, sizeof(d));
    d.in_off = a.in_offset;
    d.out_off = a.out_offset;
    d.g_off = g_off;
    d.W = a.width;
    d.H = a.height;
    d.stride = a.stride;
    d.ch = a.channels;
    d.flags = a.flags;
    d.pal_off = indexed ? a.palette_offset : 0;
    d.out_stride = a.out_stride;
    d.scale = a.scale;
    d.subdivide = a.subdivide ? 1 : 0;
    d.aligned16 = (a.out_stride % 16 == 0) && (a.out_offset % 16 == 0) && (reinterpret_cast<uintptr_t>(d_out) % 16 == 0);
    d.graph_w4 = a.width % 4 == 0;
    return DPX_OK;
}

// Validates the items and builds a launch plan: device items, graph tiles,
// raster groups by (scale, subdivision), the descriptor blob (offsets in the
// plan refer to it) and the graph scratch bytes the batch needs.
static int build_plan(dpx_context* ctx, const uint8_t* d_out, const dpx_item* items, int n_items, BatchPlan& plan,
                      std::vector<uint8_t>& blob, std::vector<uint64_t>* g_offsets, size_t* graph_bytes,
                      size_t* rows_bytes)
{
    using namespace dpx;
    plan.valid = false;
    std::vector<DevItem> dev(n_items);
    if (g_offsets) g_offsets->assign(n_items, 0);
    std::map<int, Group> groups;
    uint64_t goff = 0, roff = 0;
    for (int k = 0; k < n_items; k++) {
        const dpx_item& a = items[k];
        DevItem& d = dev[k];
        if (int rc = make_dev_item(a, k, d_out, goff, d)) return rc;
        if (g_offsets) (*g_offsets)[k] = goff;
        goff += align_up((size_t)a.width * a.height, 256);
        if (d.subdivide) {
            d.rows_off = roff;
            roff += align_up((size_t)a.width * a.height * rows_words(a.scale) * 4, 256);
        }
        const int tx = item_tile(ctx, a), wk = item_walk(ctx, a);
        const int gkey = wk << 12 | tx << 8 | a.scale << 1 | d.subdivide;
        Group& grp = groups[gkey];
        grp.tx = tx;
        grp.walk = wk;
        grp.scale = a.scale;
        grp.sub = d.subdivide;
        grp.dev.push_back(d);
    }
    for (auto& kv : groups)
        if (int rc = ensure_mask(ctx, kv.second.scale)) return rc;

    // launch grids
    int g3d = 0;
    std::vector<uint2> gmap;
    uint64_t pixels = 0;
    for (const DevItem& d : dev) pixels += (uint64_t)d.W * d.H;
    plan.grows = graph_rows(pixels);
    const dim3 ggrid = strip_grid(dev, plan.grows, &g3d, &gmap);
    for (auto& kv : groups)
        kv.second.grid = tile_grid(kv.second.dev, kv.second.tx, 256 / kv.second.tx, &kv.second.grid3d, &kv.second.map);

    // descriptor blob: items | graph tile map | per group (items, tile map)
    blob.clear();
    auto put = [&](const void* p, size_t n) {
        size_t off = align_up(blob.size(), 64);
        blob.resize(off + n);
        if (n) memcpy(blob.data() + off, p, n);
        return off;
    };
    plan.off_items = put(dev.data(), dev.size() * sizeof(DevItem));
    plan.off_gmap = put(gmap.data(), gmap.size() * sizeof(uint2));
    plan.ggrid = ggrid;
    plan.g3d = g3d;
    plan.groups.clear();
    for (auto& kv : groups) {
        const Group& grp = kv.second;
        size_t a = put(grp.dev.data(), grp.dev.size() * sizeof(DevItem));
        size_t b = put(grp.map.data(), grp.map.size() * sizeof(uint2));
        const bool walk = grp.walk == DPX_WALK_ALWAYS;
        plan.groups.push_back(PlanGroup{ grp.scale, grp.sub, grp.tx, grp.grid, grp.grid3d, a, b, walk });
    }
    plan.items.assign(items, items + n_items);
    plan.out_mod = reinterpret_cast<uintptr_t>(d_out) % 16;
    *graph_bytes = goff;
    *rows_bytes = roff;
    plan.valid = true;
    return DPX_OK;
}

// The context's own plan for dpx_batch_run: built into the context's
// descriptor buffer (uploaded on `stream` when it differs from the one
// already on the device) and its graph scratch.
static int make_plan(dpx_context* ctx, const uint8_t* d_out, const dpx_item* items, int n_items, hipStream_t stream)
{
    BatchPlan& plan = ctx->plan;
    std::vector<uint8_t> blob;
    size_t gbytes = 0, rbytes = 0;
    if (int rc = build_plan(ctx, d_out, items, n_items, plan, blob, &ctx->g_offsets, &gbytes, &rbytes)) return rc;
    plan.valid = false;
    // graph and cell-row arenas (grown only when a batch needs more)
    if (int rc = grow_graph(ctx, gbytes)) return rc;
    if (int rc = grow_rows(ctx, rbytes)) return rc;
    if (blob != ctx->last_desc) {
        if (ctx->upload_pending) {
            DPX_HIP(hipEventSynchronize(ctx->upload_done));
            ctx->upload_pending = false;
        }
        if (int rc = grow_desc(ctx, blob.size())) return rc;
        memcpy(ctx->h_pinned, blob.data(), blob.size());
        DPX_HIP(hipMemcpyAsync(ctx->d_desc, ctx->h_pinned, blob.size(), hipMemcpyHostToDevice, stream));
        DPX_HIP(hipEventRecord(ctx->upload_done, stream));
        ctx->upload_pending = true;
        ctx->last_desc.swap(blob);
    }
    plan.valid = true;
    return DPX_OK;
}

// The kernels of one batch: kf_graph, then one kf_raster per (scale,
// subdivision) group.  `desc` holds the plan's descriptor blob.
struct LaunchArgs {
    const uint8_t* desc;
    uint8_t* gaux;
    uint8_t* gfin;  // the resolved graph (written by kf_smooth for subdivided items)
    bool keep;      // the raster of the other items writes the resolved graph too
    uint32_t* rows;  // cell rows of smoothed cells
};

// Dynamic LDS of a raster launch, which the kernel does not use: at 8x it
// leaves five blocks a CU in place of eight (as the walk window does by
// itself).  There the stores bound the batch, and fewer blocks storing at once
// get more of them through: 4096 sprites 204 -> 189 us a batch, 64 console
// frames 206 -> 195, 32 of 256x224 at 8x 346 -> 337.  Below 8x fewer blocks
// are slower (4x by 10%), above it neither way holds for all content.
constexpr unsigned raster_pad(int S, bool sub, bool walk) { return S == 8 && !sub && !walk ? 10 * 1024 : 0; }

static int launch_plan(dpx_context* ctx, const BatchPlan& plan, const LaunchArgs& la, const uint8_t* d_in,
                       uint8_t* d_out, hipStream_t stream, hipEvent_t ev_mid)
{
    const DevItem* d_items = reinterpret_cast<const DevItem*>(la.desc + plan.off_items);
    const uint2* d_gmap = reinterpret_cast<const uint2*>(la.desc + plan.off_gmap);
    hipLaunchKernelGGL(kf_graph, plan.ggrid, dim3(64), 0, stream, d_items, d_gmap, plan.g3d, plan.grows, d_in, la.gaux);
    if (ev_mid) DPX_HIP(hipEventRecord(ev_mid, stream));
    for (const PlanGroup& pg : plan.groups) {
        RasterFn fn = pick_raster(pg.scale, pg.sub, pg.tx, pg.walk);
        DPX_CHECK(fn, DPX_EINVAL, "no raster kernel for scale %d", pg.scale);
        const DevItem* d_gitems = reinterpret_cast<const DevItem*>(la.desc + pg.off_items);
        const uint2* d_rmap = reinterpret_cast<const uint2*>(la.desc + pg.off_map);
        if (pg.sub) {
            SmoothFn sf = pick_smooth(pg.scale, pg.tx, pg.walk);
            DPX_CHECK(sf && la.gfin && la.rows, DPX_EINVAL, "no smoothing buffers for scale %d", pg.scale);
            hipLaunchKernelGGL(sf, pg.grid, dim3(256), 0, stream, d_gitems, d_rmap, pg.grid3d, d_in, la.gaux, la.gfin,
                               la.rows);
        }
        hipLaunchKernelGGL(fn, pg.grid, dim3(256), raster_pad(pg.scale, pg.sub, pg.walk), stream, d_gitems, d_rmap,
                           pg.grid3d, d_in, la.gaux,
                           (pg.sub || la.keep) ? la.gfin : nullptr, la.rows, ctx->d_mask[pg.scale],
                           ctx->d_info[pg.scale], d_out);
    }
    DPX_HIP(hipGetLastError());
    return DPX_OK;
}

extern "C" int dpx_batch_run(dpx_context* ctx, const uint8_t* d_in, uint8_t* d_out, const dpx_item* items,
                             int n_items, void* stream_)
{
    DPX_CHECK(ctx && d_in && d_out && items && n_items > 0, DPX_EINVAL, "bad arguments");
    std::lock_guard<std::mutex> lock(ctx->mu);
    hipStream_t stream = as_stream(stream_);
    DPX_HIP(hipSetDevice(ctx->device));
    const BatchPlan& plan = ctx->plan;
    if (!(plan.valid && plan.items.size() == (size_t)n_items &&
          plan.out_mod == reinterpret_cast<uintptr_t>(d_out) % 16 &&
          memcmp(plan.items.data(), items, (size_t)n_items * sizeof(dpx_item)) == 0))
        if (int rc = make_plan(ctx, d_out, items, n_items, stream)) return rc;

    hipEvent_t ev[3] = {};
    if (ctx->timing) {
        while (ctx->ev_pool.size() < ctx->ev_used + 3) {
            hipEvent_t e;
            DPX_HIP(hipEventCreate(&e));
            ctx->ev_pool.push_back(e);
        }
        for (int q = 0; q < 3; q++) ev[q] = ctx->ev_pool[ctx->ev_used + q];
        ctx->ev_used += 3;
        DPX_HIP(hipEventRecord(ev[0], stream));
    }
    LaunchArgs la{ ctx->d_desc, ctx->d_gaux, ctx->d_gfin, ctx->keep_graph, ctx->d_rows };
    if (int rc = launch_plan(ctx, plan, la, d_in, d_out, stream, ev[1])) return rc;
    ctx->last_kept = ctx->keep_graph;
    if (ctx->timing) DPX_HIP(hipEventRecord(ev[2], stream));
    return DPX_OK;
}

// ---------------------------------------------------------------------------
// plans: a batch layout fixed once, with descriptors and graph scratch of its
// own, launched directly or as a HIP graph the library builds
// ---------------------------------------------------------------------------
struct dpx_plan {
    dpx_context* ctx = nullptr;
    BatchPlan plan;
    uint8_t* d_desc = nullptr;
    uint8_t* d_gaux = nullptr;
    uint8_t* d_gfin = nullptr;
    uint32_t* d_rows = nullptr;
    uint32_t flags = 0;
    std::mutex mu;
    // DPX_PLAN_GRAPH: the kernels as graph nodes (kf_graph, then per group
    // kf_smooth when it subdivides and kf_raster); the input and output
    // pointers of the instantiated graph are updated in place when they change
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    std::vector<hipGraphNode_t> nodes;
    std::vector<std::pair<int, int>> node_kind;  // (0 graph / 1 smooth / 2 raster, group)
    const uint8_t* g_in = nullptr;
    uint8_t* g_out = nullptr;
    std::vector<uint64_t> g_offsets;  // per item, in d_gfin
};

namespace {

void plan_free(dpx_plan* p)
{
    if (!p) return;
    if (p->exec) (void)hipGraphExecDestroy(p->exec);
    if (p->graph) (void)hipGraphDestroy(p->graph);
    (void)hipFree(p->d_desc);
    (void)hipFree(p->d_gaux);
    (void)hipFree(p->d_gfin);
    (void)hipFree(p->d_rows);
    delete p;
}

// Kernel node parameters of one of the plan's kernels for (d_in, d_out);
// `a` keeps the argument values the parameter pointers refer to.
struct NodeArgs {
    const DevItem* items;
    const uint2* map;
    int g3d;
    int grows;
    const uint8_t* in;
    const uint8_t* gaux_c;
    uint8_t* gaux;
    uint8_t* gfin;
    const uint32_t* rows_c;
    uint32_t* rows;
    const uint32_t* mask;
    const uint8_t* info;
    uint8_t* out;
    void* ptrs[10];
};

hipKernelNodeParams node_params(dpx_plan* p, int kind, int group, const uint8_t* d_in, uint8_t* d_out, NodeArgs& a)
{
    hipKernelNodeParams np;
    memset(&np, 0, sizeof(np));
    np.blockDim = dim3(256);
    a.in = d_in;
    a.out = d_out;
    a.gaux = p->d_gaux;
    a.gaux_c = p->d_gaux;
    if (kind == 0) {
        a.items = reinterpret_cast<const DevItem*>(p->d_desc + p->plan.off_items);
        a.map = reinterpret_cast<const uint2*>(p->d_desc + p->plan.off_gmap);
        a.g3d = p->plan.g3d;
        a.grows = p->plan.grows;
        void* v[6] = { &a.items, &a.map, &a.g3d, &a.grows, &a.in, &a.gaux };
        memcpy(a.ptrs, v, sizeof(v));
        np.func = reinterpret_cast<void*>(kf_graph);
        np.gridDim = p->plan.ggrid;
        np.blockDim = dim3(64);
    } else {
        const PlanGroup& pg = p->plan.groups[group];
        a.items = reinterpret_cast<const DevItem*>(p->d_desc + pg.off_items);
        a.map = reinterpret_cast<const uint2*>(p->d_desc + pg.off_map);
        a.g3d = pg.grid3d;
        a.gfin = (pg.sub || (p->flags & DPX_PLAN_KEEP_GRAPH)) ? p->d_gfin : nullptr;
        a.rows = p->d_rows;
        a.rows_c = p->d_rows;
        if (kind == 1) {
            void* v[7] = { &a.items, &a.map, &a.g3d, &a.in, &a.gaux_c, &a.gfin, &a.rows };
            memcpy(a.ptrs, v, sizeof(v));
            np.func = reinterpret_cast<void*>(pick_smooth(pg.scale, pg.tx, pg.walk));
        } else {
            a.mask = p->ctx->d_mask[pg.scale];
            a.info = p->ctx->d_info[pg.scale];
            void* v[10] = { &a.items, &a.map, &a.g3d, &a.in, &a.gaux_c, &a.gfin, &a.rows_c, &a.mask, &a.info, &a.out };
            memcpy(a.ptrs, v, sizeof(v));
            np.func = reinterpret_cast<void*>(pick_raster(pg.scale, pg.sub, pg.tx, pg.walk));
            np.sharedMemBytes = raster_pad(pg.scale, pg.sub, pg.walk);
        }
        np.gridDim = pg.grid;
    }
    np.kernelParams = a.ptrs;
    return np;
}

int plan_build_graph(dpx_plan* p, const uint8_t* d_in, uint8_t* d_out)
{
    DPX_HIP(hipGraphCreate(&p->graph, 0));
    p->node_kind.assign(1, { 0, 0 });
    for (int g = 0; g < (int)p->plan.groups.size(); g++) {
        if (p->plan.groups[g].sub) p->node_kind.push_back({ 1, g });
        p->node_kind.push_back({ 2, g });
    }
    p->nodes.assign(p->node_kind.size(), nullptr);
    for (size_t k = 0; k < p->nodes.size(); k++) {
        NodeArgs a;
        memset(&a, 0, sizeof(a));
        const int kind = p->node_kind[k].first;
        hipKernelNodeParams np = node_params(p, kind, p->node_kind[k].second, d_in, d_out, a);
        DPX_CHECK(np.func, DPX_EINVAL, "no kernel for a group of the plan");
        // kf_smooth and the rasters of groups without subdivision follow the
        // graph kernel; a group's raster after subdivision follows its kf_smooth
        hipGraphNode_t dep = (kind == 2 && k > 0 && p->node_kind[k - 1].first == 1) ? p->nodes[k - 1] : p->nodes[0];
        DPX_HIP(hipGraphAddKernelNode(&p->nodes[k], p->graph, k ? &dep : nullptr, k ? 1 : 0, &np));
    }
    DPX_HIP(hipGraphInstantiate(&p->exec, p->graph, nullptr, nullptr, 0));
    p->g_in = d_in;
    p->g_out = d_out;
    return DPX_OK;
}

}  // namespace

extern "C" int dpx_plan_create(dpx_context* ctx, const dpx_item* items, int n_items, uint64_t out_align,
                               uint32_t flags, dpx_plan** out)
{
    DPX_CHECK(out, DPX_EINVAL, "null output pointer");
    *out = nullptr;
    DPX_CHECK(ctx && items && n_items > 0, DPX_EINVAL, "bad arguments");
    DPX_CHECK((flags & ~(uint32_t)(DPX_PLAN_GRAPH | DPX_PLAN_KEEP_GRAPH)) == 0, DPX_EINVAL, "unknown plan flags 0x%x",
              flags);
    std::lock_guard<std::mutex> lock(ctx->mu);
    DPX_HIP(hipSetDevice(ctx->device));
    auto* p = new dpx_plan();
    p->ctx = ctx;
    p->flags = flags;
    std::vector<uint8_t> blob;
    size_t gbytes = 0, rbytes = 0;
    // out_align stands for d_out modulo 16 (only the alignment of the output
    // arena enters the plan)
    const uint8_t* fake_out = reinterpret_cast<const uint8_t*>((uintptr_t)(out_align % 16) + 16);
    int rc = build_plan(ctx, fake_out, items, n_items, p->plan, blob, nullptr, &gbytes, &rbytes);
    const bool want_gfin = (flags & DPX_PLAN_KEEP_GRAPH) || rbytes > 0;
    if (rc == DPX_OK && (hipMalloc(&p->d_desc, blob.size()) != hipSuccess ||
                         hipMalloc(&p->d_gaux, std::max<size_t>(gbytes, 256)) != hipSuccess ||
                         (want_gfin && hipMalloc(&p->d_gfin, std::max<size_t>(gbytes, 256)) != hipSuccess) ||
                         (rbytes > 0 && hipMalloc(&p->d_rows, rbytes) != hipSuccess)))
        rc = fail(DPX_ENOMEM, "plan allocation failed (%zu descriptor, %zu graph and %zu cell-row bytes)", blob.size(),
                  gbytes, rbytes);
    if (rc == DPX_OK && hipMemcpy(p->d_desc, blob.data(), blob.size(), hipMemcpyHostToDevice) != hipSuccess)
        rc = fail(DPX_EHIP, "descriptor upload failed");
    if (rc != DPX_OK) {
        plan_free(p);
        return rc;
    }
    *out = p;
    return DPX_OK;
}

extern "C" int dpx_plan_run(dpx_plan* p, const uint8_t* d_in, uint8_t* d_out, void* stream_)
{
    DPX_CHECK(p && d_in && d_out, DPX_EINVAL, "bad arguments");
    DPX_CHECK(reinterpret_cast<uintptr_t>(d_out) % 16 == p->plan.out_mod, DPX_EINVAL,
              "d_out %% 16 = %u, the plan was made for %u", (unsigned)(reinterpret_cast<uintptr_t>(d_out) % 16),
              (unsigned)p->plan.out_mod);
    std::lock_guard<std::mutex> lock(p->mu);
    hipStream_t stream = as_stream(stream_);
    DPX_HIP(hipSetDevice(p->ctx->device));
    if (!(p->flags & DPX_PLAN_GRAPH)) {
        LaunchArgs la{ p->d_desc, p->d_gaux, p->d_gfin, (p->flags & DPX_PLAN_KEEP_GRAPH) != 0, p->d_rows };
        return launch_plan(p->ctx, p->plan, la, d_in, d_out, stream, nullptr);
    }
    if (!p->exec) {
        if (int rc = plan_build_graph(p, d_in, d_out)) return rc;
    } else if (p->g_in != d_in || p->g_out != d_out) {
        for (size_t k = 0; k < p->nodes.size(); k++) {
            NodeArgs a;
            memset(&a, 0, sizeof(a));
            hipKernelNodeParams np = node_params(p, p->node_kind[k].first, p->node_kind[k].second, d_in, d_out, a);
            DPX_HIP(hipGraphExecKernelNodeSetParams(p->exec, p->nodes[k], &np));
        }
        p->g_in = d_in;
        p->g_out = d_out;
    }
    DPX_HIP(hipGraphLaunch(p->exec, stream));
    return DPX_OK;
}

extern "C" int dpx_plan_graph(dpx_plan* p, const uint8_t** d_graph, const uint64_t** offsets_host)
{
    DPX_CHECK(p && d_graph && offsets_host, DPX_EINVAL, "bad arguments");
    DPX_CHECK(p->flags & DPX_PLAN_KEEP_GRAPH, DPX_EINVAL, "the plan was made without DPX_PLAN_KEEP_GRAPH");
    std::lock_guard<std::mutex> lock(p->mu);
    if (p->g_offsets.empty()) {
        uint64_t off = 0;
        for (const dpx_item& a : p->plan.items) {
            p->g_offsets.push_back(off);
            off += align_up((size_t)a.width * a.height, 256);
        }
    }
    *d_graph = p->d_gfin;
    *offsets_host = p->g_offsets.data();
    return DPX_OK;
}

extern "C" void dpx_plan_destroy(dpx_plan* p)
{
    if (!p) return;
    (void)hipSetDevice(p->ctx->device);
    (void)hipDeviceSynchronize();
    plan_free(p);
}

extern "C" int dpx_batch_timing(dpx_context* ctx, int enable)
{
    DPX_CHECK(ctx, DPX_EINVAL, "null context");
    std::lock_guard<std::mutex> lock(ctx->mu);
    ctx->timing = enable != 0;
    return DPX_OK;
}

extern "C" int dpx_batch_timing_read(dpx_context* ctx, dpx_batch_times* out)
{
    DPX_CHECK(ctx && out, DPX_EINVAL, "bad arguments");
    std::lock_guard<std::mutex> lock(ctx->mu);
    for (size_t b = 0; b + 3 <= ctx->ev_used; b += 3) {
        hipEvent_t* ev = &ctx->ev_pool[b];
        DPX_HIP(hipEventSynchronize(ev[2]));
        float t01, t12;
        DPX_HIP(hipEventElapsedTime(&t01, ev[0], ev[1]));
        DPX_HIP(hipEventElapsedTime(&t12, ev[1], ev[2]));
        ctx->acc.graph_ms += t01;
        ctx->acc.raster_ms += t12;
        ctx->acc.batches++;
    }
    ctx->ev_used = 0;
    *out = ctx->acc;
    ctx->acc = dpx_batch_times{};
    return DPX_OK;
}

// ---------------------------------------------------------------------------
// dpx_batch_run_noalloc: the batched path with every buffer beyond the
// caller's input and output in one static device array, `scratch`, so that a
// call allocates nothing.  Layout (all offsets 256-byte aligned):
//   tables     per scale 1..15 the coverage rows (with the cell masks at 1x to
//              8x) and the coverage summaries, built on the first call
//              on each device;
//   items      the batch's device items, in item order and grouped by
//              (scale, subdivision);
//   tile maps  block -> (item, tile) of the graph launch and of the raster
//              launches;
//   graph      the post-trivial snapshot graph, 1 byte per pixel.
// A call's descriptors reach the device as kernel arguments (k_na_put,
// kNaPutChunk items per launch), not as a copy from host memory.
// ---------------------------------------------------------------------------
namespace {

constexpr size_t na_align(size_t v) { return (v + 255) / 256 * 256; }
constexpr size_t na_mask_bytes(int S)
{
    return na_align((size_t)kKeys * mask_w(S) * 4 + cell_table_bytes(S));
}
constexpr size_t na_info_bytes() { return na_align((size_t)kKeys); }
constexpr size_t na_mask_off(int S)
{
    size_t o = 0;
    for (int s = 1; s < S; s++) o += na_mask_bytes(s) + na_info_bytes();
    return o;
}
constexpr size_t na_info_off(int S) { return na_mask_off(S) + na_mask_bytes(S); }

constexpr int kNaMaxItems = 4096;
constexpr int kNaTX = kDefaultTileX, kNaTY = 256 / kDefaultTileX;  // raster tiles (the default shape)
constexpr size_t kNaGraphTiles = 65536, kNaRasterTiles = 524288;
// Limits are counted in graph tiles of 64x32 pixels.  The map holds two strips
// a tile: blocks of 32 rows never take more ((blocks * (W + 1) + 60) / 62
// strips against blocks * ceil(W / 64) tiles), and lower blocks are used only
// where their strips fit too.
constexpr int kNaGX = 64, kNaGY = 32;
constexpr size_t kNaGraphStrips = 2 * kNaGraphTiles;
constexpr size_t kNaGraphBytes = 48u << 20;
constexpr size_t kNaOffItems = na_mask_off(kMaxScale + 1);
constexpr size_t kNaOffGroupItems = kNaOffItems + na_align(kNaMaxItems * sizeof(DevItem));
constexpr size_t kNaOffGmap = kNaOffGroupItems + na_align(kNaMaxItems * sizeof(DevItem));
constexpr size_t kNaOffRmap = kNaOffGmap + na_align(kNaGraphStrips * sizeof(uint2));
constexpr size_t kNaOffGraph = kNaOffRmap + na_align(kNaRasterTiles * sizeof(uint2));
constexpr size_t kNaScratchBytes = kNaOffGraph + kNaGraphBytes;
static_assert(kNaScratchBytes < (64u << 20), "scratch stays under 64 MiB");

static __device__ __align__(256) uint8_t scratch[kNaScratchBytes];

// One item of a k_na_put launch: its descriptor, its slots in the item
// arrays and the first entries of its strips and tiles in the two maps.
struct NaPut {
    DevItem d;
    uint32_t index;  // in the item array (the graph launch's items)
    uint32_t gslot;  // in the grouped item array
    uint32_t gpos;   // gslot - the group's first slot (the raster launch's items)
    uint32_t gstrip, rtile;
    uint32_t strips;
};
constexpr int kNaPutChunk = 32;
struct NaPutArgs {
    NaPut it[kNaPutChunk];
};
static_assert(sizeof(NaPutArgs) <= 4000, "kernel arguments stay under 4 KB");

// A block per item.  (One block that took the items in turn: 17 us a launch of
// 32, and 21 when each item's strips were counted here.)
__global__ __launch_bounds__(256) void k_na_put(NaPutArgs a, DevItem* __restrict__ items,
                                                DevItem* __restrict__ group_items, uint2* __restrict__ gmap,
                                                uint2* __restrict__ rmap)
{
    const NaPut& p = a.it[blockIdx.x];
    if (threadIdx.x == 0) {
        items[p.index] = p.d;
        group_items[p.gslot] = p.d;
    }
    for (uint32_t t = threadIdx.x; t < p.strips; t += blockDim.x) gmap[p.gstrip + t] = make_uint2(p.index, t);
    const uint32_t rx = (uint32_t)(p.d.W + kNaTX - 1) / kNaTX, ry = (uint32_t)(p.d.H + kNaTY - 1) / kNaTY;
    for (uint32_t t = threadIdx.x; t < rx * ry; t += blockDim.x)
        rmap[p.rtile + t] = make_uint2(p.gpos, (t / rx) << 16 | (t % rx));
}

constexpr int kNaMaxDevices = 64;
std::mutex g_na_mu;
uint8_t* g_na_ptr[kNaMaxDevices] = {};  // each device's address of `scratch`

// Set-up on the first call on a device: the array's address on this device
// and its tables, built on `stream` and waited for (later calls on any
// stream read them).
int na_setup(int dev, hipStream_t stream, uint8_t** out)
{
    std::lock_guard<std::mutex> lock(g_na_mu);
    if (!g_na_ptr[dev]) {
        uint8_t* ptr = nullptr;
        DPX_HIP(hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch)));
        DPX_CHECK(ptr, DPX_EHIP, "no device address for the scratch array");
        for (int S = 1; S <= kMaxScale; S++) {
            uint32_t* mask = reinterpret_cast<uint32_t*>(ptr + na_mask_off(S));
            const size_t n = (size_t)kKeys * mask_w(S);
            hipLaunchKernelGGL(kt_mask, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, S, mask);
            if (S <= kMaxCellScale)
                hipLaunchKernelGGL(pick_cell_table(S), dim3(kKeys / 256), dim3(256), 0, stream, mask,
                                   reinterpret_cast<uint8_t*>(mask + n));
            hipLaunchKernelGGL(kt_info, dim3(kKeys / 256), dim3(256), 0, stream, mask, S,
                               ptr + na_info_off(S));
        }
        DPX_HIP(hipGetLastError());
        DPX_HIP(hipStreamSynchronize(stream));
        g_na_ptr[dev] = ptr;
    }
    *out = g_na_ptr[dev];
    return DPX_OK;
}

}  // namespace

extern "C" int dpx_batch_run_noalloc(const uint8_t* d_in, uint8_t* d_out, const dpx_item* items, int n_items,
                                     void* stream_)
{
    DPX_CHECK(d_in && d_out && items && n_items > 0, DPX_EINVAL, "bad arguments");
    DPX_CHECK(n_items <= kNaMaxItems, DPX_EINVAL, "%d items: dpx_batch_run_noalloc takes at most %d", n_items,
              kNaMaxItems);
    hipStream_t stream = as_stream(stream_);
    int dev = 0;
    DPX_HIP(hipGetDevice(&dev));
    DPX_CHECK(dev >= 0 && dev < kNaMaxDevices, DPX_ENODEV, "device %d", dev);
    // pass 1: validate, graph bytes and tiles, per group (2 * scale + sub)
    // its item and tile counts
    uint32_t gcount[2 * (kMaxScale + 1)] = {}, gtiles[2 * (kMaxScale + 1)] = {};
    size_t gbytes = 0, graph_tiles = 0, raster_tiles = 0;
    uint64_t pixels = 0;
    for (int k = 0; k < n_items; k++) {
        DevItem d;
        if (int rc = make_dev_item(items[k], k, d_out, 0, d)) return rc;
        DPX_CHECK(!d.subdivide, DPX_EINVAL,
                  "item %d: subdivision needs per-cell row buffers; dpx_batch_run_noalloc takes items without it", k);
        gbytes += align_up((size_t)d.W * d.H, 256);
        graph_tiles += (size_t)((d.W + kNaGX - 1) / kNaGX) * ((d.H + kNaGY - 1) / kNaGY);
        pixels += (uint64_t)d.W * d.H;
        const size_t rt = (size_t)((d.W + kNaTX - 1) / kNaTX) * ((d.H + kNaTY - 1) / kNaTY);
        raster_tiles += rt;
        const int g = 2 * d.scale + d.subdivide;
        gcount[g]++;
        gtiles[g] += (uint32_t)std::min<size_t>(rt, 0xFFFFFFFFu);
    }
    DPX_CHECK(gbytes <= kNaGraphBytes, DPX_EINVAL,
              "batch needs %zu graph bytes: dpx_batch_run_noalloc holds at most %zu (one byte per pixel, each item "
              "rounded up to 256)", gbytes, kNaGraphBytes);
    DPX_CHECK(graph_tiles <= kNaGraphTiles && raster_tiles <= kNaRasterTiles, DPX_EINVAL,
              "batch has %zu graph and %zu raster tiles: dpx_batch_run_noalloc holds at most %zu and %zu", graph_tiles,
              raster_tiles, kNaGraphTiles, kNaRasterTiles);
    auto count_strips = [&](int rows) {
        size_t n = 0;
        for (int k = 0; k < n_items; k++) n += graph_split(items[k].width, items[k].height, rows).strips;
        return n;
    };
    int grows = graph_rows(pixels);
    size_t graph_strips = count_strips(grows);
    if (graph_strips > kNaGraphStrips) graph_strips = count_strips(grows = kNaGY);
    uint8_t* base = nullptr;
    if (int rc = na_setup(dev, stream, &base)) return rc;
    DevItem* d_items = reinterpret_cast<DevItem*>(base + kNaOffItems);
    DevItem* d_gitems = reinterpret_cast<DevItem*>(base + kNaOffGroupItems);
    uint2* d_gmap = reinterpret_cast<uint2*>(base + kNaOffGmap);
    uint2* d_rmap = reinterpret_cast<uint2*>(base + kNaOffRmap);
    uint8_t* d_graph = base + kNaOffGraph;
    // groups in ascending (scale, subdivision): first item slot and tile
    uint32_t gslot0[2 * (kMaxScale + 1)], gtile0[2 * (kMaxScale + 1)];
    uint32_t slot = 0, tile = 0;
    for (int g = 0; g < 2 * (kMaxScale + 1); g++) {
        gslot0[g] = slot;
        gtile0[g] = tile;
        slot += gcount[g];
        tile += gtiles[g];
    }
    // pass 2: descriptors to the device, kNaPutChunk items per launch
    uint32_t gnext[2 * (kMaxScale + 1)] = {}, gtnext[2 * (kMaxScale + 1)] = {};
    NaPutArgs args;
    memset(&args, 0, sizeof(args));
    uint64_t goff = 0;
    uint32_t gt = 0;
    int n_put = 0;
    for (int k = 0; k < n_items; k++) {
        NaPut& p = args.it[n_put++];
        (void)make_dev_item(items[k], k, d_out, goff, p.d);  // (validated in pass 1)
        const int g = 2 * p.d.scale + p.d.subdivide;
        p.index = (uint32_t)k;
        p.gpos = gnext[g]++;
        p.gslot = gslot0[g] + p.gpos;
        p.gstrip = gt;
        p.rtile = gtile0[g] + gtnext[g];
        p.strips = graph_split(p.d.W, p.d.H, grows).strips;
        gt += p.strips;
        gtnext[g] += (uint32_t)(((p.d.W + kNaTX - 1) / kNaTX) * ((p.d.H + kNaTY - 1) / kNaTY));
        goff += align_up((size_t)p.d.W * p.d.H, 256);
        if (n_put == kNaPutChunk || k == n_items - 1) {
            hipLaunchKernelGGL(k_na_put, dim3(n_put), dim3(256), 0, stream, args, d_items, d_gitems, d_gmap, d_rmap);
            n_put = 0;
        }
    }
    hipLaunchKernelGGL(kf_graph, dim3((unsigned)graph_strips), dim3(64), 0, stream, d_items, d_gmap, 0,
                       grows, d_in, d_graph);
    for (int g = 0; g < 2 * (kMaxScale + 1); g++) {
        if (!gcount[g]) continue;
        const int S = g / 2;
        RasterFn fn = pick_raster(S, g % 2, kNaTX);
        DPX_CHECK(fn, DPX_EINVAL, "no raster kernel for scale %d", S);
        hipLaunchKernelGGL(fn, dim3(gtiles[g]), dim3(256), raster_pad(S, g % 2, false), stream,
                           d_gitems + gslot0[g], d_rmap + gtile0[g], 0, d_in, d_graph, nullptr, nullptr,
                           reinterpret_cast<const uint32_t*>(base + na_mask_off(S)),
                           base + na_info_off(S), d_out);
    }
    DPX_HIP(hipGetLastError());
    return DPX_OK;
}

