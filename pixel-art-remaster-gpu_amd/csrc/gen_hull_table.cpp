// gen_hull_table.cpp -- run at build time: writes the hulls of the 4096 cell
// keys (geom.hpp's cell_hull) as one 64-bit word each, so that no kernel and
// no first call has to compute them: point t at bits 6t (x + 1, 3 bits) and
// 6t + 3 (y + 1, 3 bits), in quarter units, and the vertex count at bit 48.
#include <stdio.h>
#include <stdlib.h>

#include "geom.hpp"

int main()
{
    for (uint32_t key = 0; key < 4096; key++) {
        int hx[2 * dpx::kMaxPts], hy[2 * dpx::kMaxPts];
        const int n = dpx::cell_hull(key, hx, hy);
        if (n < 3 || n > 8) return 1;
        uint64_t w = (uint64_t)n << 48;
        for (int t = 0; t < n; t++) {
            if (hx[t] < -1 || hx[t] > 6 || hy[t] < -1 || hy[t] > 6) return 1;
            w |= (uint64_t)(uint32_t)(hx[t] + 1) << (6 * t) | (uint64_t)(uint32_t)(hy[t] + 1) << (6 * t + 3);
        }
        printf("0x%llxull,%c", (unsigned long long)w, key % 8 == 7 ? '\n' : ' ');
    }
    return 0;
}
