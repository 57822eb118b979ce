// How far a smoothed vertex can lie from its cell: subdivide_hull_emit over all
// pairs of a cell's key and a neighbour's, both kinds of corner, against the
// bounds that the sample grid of smoothed cells is made for (common.hpp).
// Prints the extremes met.
#include <hip/hip_runtime.h>
#include <stdio.h>

#include <algorithm>
#include <vector>

#include "common.hpp"
#include "geom.hpp"
using namespace dpx;

int main()
{
    struct Key {
        HullBits h;
        uint32_t node;
    };
    std::vector<Key> keys;     // own: hull and node
    std::vector<HullBits> hulls;  // a neighbour's: hull
    for (uint32_t key = 0; key < 4096; key++) {
        int hx[2 * kMaxPts], hy[2 * kMaxPts];
        const HullBits h = hull_pack(hx, hy, cell_hull(key, hx, hy));
        keys.push_back(Key{ h, key & 0xFFu });
        bool met = false;
        for (const HullBits& o : hulls) met = met || (o.xs == h.xs && o.ys == h.ys);
        if (!met) hulls.push_back(h);
    }
    int x_lo = 0, x_hi = 64, y_lo = 0, y_hi = 64;
    for (const Key& k : keys)
        for (const HullBits& o : hulls)
            for (int kept = 0; kept < 2; kept++)
                subdivide_hull_emit(k.h, k.node, [&](int) { return o; }, [&](int, int) { return kept != 0; },
                                    [&](int x, int y) {
                                        x_lo = std::min(x_lo, x);
                                        x_hi = std::max(x_hi, x);
                                        y_lo = std::min(y_lo, y);
                                        y_hi = std::max(y_hi, y);
                                    });
    printf("%d %d %d %d\n", x_lo, x_hi, y_lo, y_hi);
    // and the grid holds every sample within those bounds, in a word a row
    for (int S = 1; S <= 15; S++) {
        for (int k = -2 * S; k < 3 * S; k++) {
            const int at = (2 * k + 1) * 32;  // 64 S times the sample's place
            const bool col = at >= x_lo * S && at <= x_hi * S, row = at >= y_lo * S && at <= y_hi * S;
            if (col != (k >= cover_x0(S) && k < cover_x0(S) + cover_w(S)) ||
                row != (k >= cover_y0(S) && k < cover_y0(S) + cover_h(S)) || cover_w(S) > 32)
                return 1;
        }
        // (the cells around a sample's are its candidates)
        if (cover_x0(S) < -S || cover_y0(S) < -S || cover_x0(S) + cover_w(S) > 2 * S || cover_y0(S) + cover_h(S) > 2 * S)
            return 1;
    }
    return 0;
}
