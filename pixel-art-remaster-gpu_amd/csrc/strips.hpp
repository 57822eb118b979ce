// strips.hpp -- how kf_graph cuts a launch into strips, and which bytes a
// strip's pixel loads ask for.  Host and device: the plan counts the strips,
// the kernel walks them, and the index arithmetic is checked on the CPU.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

namespace dpx {

// A strip's outer two lanes are its halo, so a strip yields 62 columns.  62
// does not divide the widths of frames, so strips do not start over at a
// frame's edge: an item's rows are cut into blocks of equal height, laid side
// by side with one empty column before each, and the strips are cut from that
// row of columns; a strip that holds the end of one block and the start of
// the next works on both (lanes are independent but for the shift, and the
// empty column belongs to the outside class).  256x224 in 4 blocks: 17
// strips, 16.6 of them used.
// Pixels are loaded kGraphRows rows at a time, one such group ahead (two
// groups ahead: 109 -> 113 us, for the registers' copies).
constexpr int kStripCols = 62;
constexpr int kGraphRows = 4;
// Rows of a launch's row blocks.  A wave alone takes 0.25 us a row, and each
// block re-reads two halo rows, so blocks are as tall as leaves about
// kGraphWaves strips, five waves a SIMD: measured at 2 / 6 / 14 / 30 / 56
// rows, one 256x224 frame takes 3.7 / 4.7 / 6.0 / 9.2 / 15.1 us, 64 console
// frames (4.2 Mpixel) 22 / 15.1 / 13.8 / 15.8 / 19.8, 128 of 320x224 59 / 31
// / 22.6 / 21.1 / 22.9 and 1024 of 256x224 274 / 162 / 119 / 116 / 105.
// Heights of 4 k + 2 make whole groups with the halo.
constexpr uint64_t kGraphWaves = 4800;
constexpr int kGraphMinRows = 2, kGraphMaxRows = 58;

inline int graph_rows(uint64_t pixels)
{
    const int rows = (int)std::min<uint64_t>(pixels / (kStripCols * kGraphWaves), kGraphMaxRows);
    return std::max((rows + 2) / kGraphRows * kGraphRows - 2, kGraphMinRows);
}

struct GraphSplit {
    uint32_t blocks, rows, strips;
};

__host__ __device__ inline GraphSplit graph_split(int W, int H, int max_rows)
{
    GraphSplit s;
    s.blocks = ((uint32_t)H + (uint32_t)max_rows - 1) / (uint32_t)max_rows;
    s.rows = ((uint32_t)H + s.blocks - 1) / s.blocks;
    s.blocks = ((uint32_t)H + s.rows - 1) / s.rows;  // (blocks of s.rows rows that hold a row)
    // columns 1 .. blocks * (W + 1) - 1 of the row of blocks carry pixels
    s.strips = (s.blocks * ((uint32_t)W + 1) - 1 + kStripCols - 1) / kStripCols;
    return s;
}

// No batch of up to n items of up to `pixels` pixels has more strips.  With
// row blocks of r = graph_rows(T) rows, T the batch's pixels, an item of W x H
// has at most (W + 61) / 62 strips where H <= r, and else, as ceil(H / r) < 2 H
// / r and H <= W H, fewer than (4 W H / r + 61) / 62; and T / r is at most 3 *
// kStripCols * kGraphWaves below the height's cap, T / kGraphMaxRows on it.
inline size_t graph_strips_bound(size_t n, size_t pixels)
{
    const size_t total = n * pixels, per_rows = std::min<size_t>(total / kGraphMinRows, 3 * kStripCols * kGraphWaves);
    return (n * (std::min<size_t>(pixels, 32768) + 61) + 4 * std::max<size_t>(per_rows, total / kGraphMaxRows)) /
               kStripCols + 1;
}

// The column of a lane of a strip: whether it carries pixels, its x and its
// block's first row.  The empty column before a block stands on the block's
// first column, lanes past the last block on its last; neither is stored.
struct StripLane {
    bool col;
    int x, y0;
};

__host__ __device__ inline StripLane strip_lane(int W, const GraphSplit& sp, uint32_t strip, uint32_t lane)
{
    const uint32_t p = strip * kStripCols + lane, blk = p / ((uint32_t)W + 1), c = p % ((uint32_t)W + 1);
    StripLane l;
    l.col = blk < sp.blocks && c != 0;
    l.x = l.col ? (int)c - 1 : (blk < sp.blocks ? 0 : W - 1);
    l.y0 = (int)((blk < sp.blocks ? blk : sp.blocks - 1) * sp.rows);
    return l;
}

// Pixels are read through a buffer descriptor of the item's rows, which
// answers 0 for offsets from its end on (rows above or below the frame).  Row
// r of a lane's block is y = y0 - 1 + r; it lies at off + (r - 1) * step
// modulo 2^32.  Byte offsets within an item fit 31 bits (checked on the host).
__host__ __device__ inline uint32_t strip_offset(const StripLane& l, int H, int stride, int ch, bool topdown)
{
    return (uint32_t)(topdown ? H - 1 - l.y0 : l.y0) * (uint32_t)stride + (uint32_t)(l.x * ch);
}
__host__ __device__ inline uint32_t strip_step(int stride, bool topdown) { return (uint32_t)(topdown ? -stride : stride); }

// The 4-byte load of a pixel at `off` that begins inside the rows and ends past
// them (the last pixel of a frame of 3-byte pixels).  It is not issued (~0u
// lies past any item's end): what the descriptor does with the bytes past its
// end is the hardware's to say, and the item may end where the caller's memory
// does.  The pixel is read by bytes.
__host__ __device__ inline bool word_crosses(uint32_t off, uint32_t end, int ch) { return off == end - 3u && ch < 4; }

// Does a lane load that pixel in one of its groups (the rows past its block's
// halo that fill the last group among them)?  `rows`: of its block, halo and
// filling included, as strip_loaded_rows gives them.
__host__ __device__ inline int strip_loaded_rows(const GraphSplit& sp)
{
    return ((int)sp.rows + 2 + kGraphRows - 1) / kGraphRows * kGraphRows;
}
__host__ __device__ inline bool strip_loads_last(const StripLane& l, int W, int H, bool topdown, int rows)
{
    return l.x == W - 1 && (topdown ? l.y0 <= 1 : l.y0 + rows >= H + 1);
}
// ... and may it be in the group from row r0 on?  r_hi: H + 1 - y0 of the
// strip's last block, one past the last row of it that lies in the frame.
__host__ __device__ inline bool group_loads_last(int r0, bool topdown, int r_hi)
{
    return topdown ? r0 < 2 : r0 + kGraphRows >= r_hi;
}

}  // namespace dpx
