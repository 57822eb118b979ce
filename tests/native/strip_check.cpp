// The bytes that kf_graph's strips and kf_raster's colours ask for
// (strips.hpp), enumerated on the host: over frame sizes, strides, row orders
// and block heights, every 4-byte load lies inside the item or begins past its
// end, where the buffer descriptor answers 0; the pixels left out are read by
// bytes inside the item; and every pixel of a frame is stored by exactly one
// lane of one strip.  Prints the loads looked at and those left out.
#include <stdio.h>

#include <vector>

#include "strips.hpp"
using namespace dpx;

static long loads = 0, left_out = 0;

// The load of a pixel: does it stay inside, or begin past the end?
static bool word_ok(uint32_t off, uint32_t end) { return off >= end || (uint64_t)off + 4 <= end; }

static bool check(int W, int H, int ch, int stride, bool topdown, int max_rows)
{
    const GraphSplit sp = graph_split(W, H, max_rows);
    const uint32_t end = (uint32_t)(H - 1) * (uint32_t)stride + (uint32_t)(W * ch);
    std::vector<int> stored((size_t)W * H, 0);
    for (uint32_t strip = 0; strip < sp.strips; strip++) {
        StripLane l[64];
        bool tail = false;
        for (uint32_t k = 0; k < 64; k++) {
            l[k] = strip_lane(W, sp, strip, k);
            tail = tail || (ch < 4 && strip_loads_last(l[k], W, H, topdown, strip_loaded_rows(sp)));
        }
        const int R = (int)sp.rows + 2, r_hi = H + 1 - l[63].y0;
        for (int r0 = 0; r0 < R; r0 += kGraphRows) {
            const bool bytes = tail && group_loads_last(r0, topdown, r_hi);
            for (int k = 0; k < 64; k++)
                for (int q = 0; q < kGraphRows; q++) {
                    const int r = r0 + q, y = l[k].y0 - 1 + r;
                    uint32_t o = strip_offset(l[k], H, stride, ch, topdown) +
                                 (uint32_t)(r - 1) * strip_step(stride, topdown);
                    const bool in_frame = y >= 0 && y < H;
                    const uint32_t want = (uint32_t)(topdown ? H - 1 - y : y) * (uint32_t)stride + (uint32_t)(l[k].x * ch);
                    if (in_frame ? o != want : o < end) {
                        printf("%dx%d stride %d strip %u lane %d row %d: offset %u\n", W, H, stride, strip, k, r, o);
                        return false;
                    }
                    loads++;
                    if (bytes && word_crosses(o, end, ch)) {
                        left_out++;
                        if (o + 3 != end) return false;  // three bytes, the item's last
                        o = ~0u;
                    }
                    if (!word_ok(o, end)) {
                        printf("%dx%d stride %d %s rows %d strip %u lane %d row %d: word at %u of %u\n", W, H, stride,
                               topdown ? "top-down" : "bottom-up", max_rows, strip, k, r, o, end);
                        return false;
                    }
                    if (l[k].col && k > 0 && k < 63 && r >= 1 && r < R - 1 && in_frame) stored[(size_t)y * W + l[k].x]++;
                }
        }
    }
    for (int n : stored)
        if (n != 1) return false;
    // the raster's colours
    for (int y = 0; y < H; y++)
        for (int x = 0; x < W; x++) {
            const uint32_t o = (uint32_t)y * (uint32_t)stride + (uint32_t)(x * ch);
            if (!word_ok(word_crosses(o, end, ch) ? ~0u : o, end) || (word_crosses(o, end, ch) && o + 3 != end)) {
                printf("%dx%d stride %d pixel %d,%d: word at %u of %u\n", W, H, stride, x, y, o, end);
                return false;
            }
        }
    return true;
}

int main()
{
    const int widths[] = { 1, 2, 3, 5, 8, 30, 61, 62, 63, 64, 65, 124, 131, 200 };
    const int heights[] = { 1, 2, 3, 4, 5, 6, 7, 9, 13, 14, 29, 31, 57, 58, 59, 60, 61, 62, 63, 116, 117, 119 };
    for (int W : widths)
        for (int H : heights)
            for (int ch = 3; ch <= 4; ch++)
                for (int pad : { 0, 1, 2, 3, 7 })
                    for (int topdown = 0; topdown < 2; topdown++)
                        for (int rows = 2; rows <= 58; rows += 4)
                            if (!check(W, H, ch, W * ch + pad, topdown, rows)) return 1;
    printf("%ld %ld\n", loads, left_out);
    return 0;
}
