// cell_triangles (geom.hpp) for every kind of vertex count a diagram may hold:
// min(count - 2, 15) in 64 bits, never below 0.
#include <stdint.h>
#include <stdio.h>

#include "geom.hpp"

int main()
{
    auto check = [](int64_t n) {
        const int64_t want = n - 2 < 0 ? 0 : n - 2 > dpx::kCellSize / 3 ? dpx::kCellSize / 3 : n - 2;
        if (dpx::cell_triangles((int)n) == want) return true;
        printf("%lld: %d\n", (long long)n, dpx::cell_triangles((int)n));
        return false;
    };
    for (int64_t d = 0; d < 100000; d++)
        if (!check(INT32_MIN + d) || !check(INT32_MAX - d) || !check(d - 50000)) return 1;
    printf("ok\n");
    return 0;
}
