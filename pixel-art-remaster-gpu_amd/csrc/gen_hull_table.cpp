// gen_hull_table.cpp -- run at build time: writes the hulls of the 4096 cell
// keys (geom.hpp's cell_hull) packed as HullBits, so that no kernel and no
// first call has to compute them.
#include <stdio.h>

#include "geom.hpp"

int main()
{
    for (uint32_t key = 0; key < 4096; key++) {
        int hx[2 * dpx::kMaxPts], hy[2 * dpx::kMaxPts];
        const int n = dpx::cell_hull(key, hx, hy);
        if (n < 3 || n > 8) return 1;
        for (int t = 0; t < n; t++)
            if (hx[t] < -1 || hx[t] > 5 || hy[t] < -1 || hy[t] > 5) return 1;
        const dpx::HullBits h = dpx::hull_pack(hx, hy, n);
        printf("{0x%xu, 0x%xu},%c", h.xs, h.ys, key % 8 == 7 ? '\n' : ' ');
    }
    return 0;
}
