// Polygons with coordinates up to kEarLimit (geom.hpp): poly_shape calls strict
// what is strictly convex in 64 bits, and ear_clip_ring gives ear_clip's
// triangles, for those also without the inside tests.  Wide rings, thin ones
// and arbitrary polygons, many with vertices at the limit itself.  Prints the
// polygons and the strictly convex ones.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdio.h>

#include <algorithm>
#include <random>
#include <vector>

#include "geom.hpp"
using namespace dpx;

#ifndef LIMIT
#define LIMIT kEarLimit
#endif

int main()
{
    std::mt19937 rng(3);
    auto uni = [&](int a, int b) { return (int)(rng() % (unsigned)(b - a + 1)) + a; };
    long polygons = 0, strict = 0;
    for (int it = 0; it < 400000; it++) {
        const int n = uni(3, 16), kind = uni(0, 3);
        std::vector<int> x(n), y(n);
        if (kind < 3) {  // around a ring, a thin one, the edge of the square
            std::vector<double> a(n);
            for (double& v : a) v = uni(0, 62831) / 10000.0;
            std::sort(a.begin(), a.end());
            const double r = LIMIT * (uni(50, 100) / 100.0), h = kind == 1 ? uni(5, 100) / 100.0 : 1.0;
            for (int k = 0; k < n; k++) {
                const double s = kind == 2 ? LIMIT / std::max(fabs(cos(a[k])), fabs(sin(a[k]))) : r;
                x[k] = std::clamp((int)lrint(s * cos(a[k])), -LIMIT, LIMIT);
                y[k] = std::clamp((int)lrint(s * h * sin(a[k])), -LIMIT, LIMIT);
            }
        } else {
            for (int k = 0; k < n; k++) {
                x[k] = uni(0, 2) ? uni(-LIMIT, LIMIT) : uni(0, 1) ? LIMIT : -LIMIT;
                y[k] = uni(0, 2) ? uni(-LIMIT, LIMIT) : uni(0, 1) ? LIMIT : -LIMIT;
            }
        }
        if (uni(0, 1)) std::reverse(x.begin(), x.end()), std::reverse(y.begin(), y.end());
        uint8_t tri[3 * kMaxPoly];
        int ok;
        const int nt = ear_clip(x.data(), y.data(), n, tri, &ok);
        std::vector<uint32_t> P(n), want;
        for (int k = 0; k < n; k++) P[k] = ((uint32_t)x[k] & 0xFFFFu) | ((uint32_t)y[k] << 16);
        for (int k = 0; k < 3 * nt; k++) want.push_back(P[tri[k]]);
        const PolyShape s = poly_shape(P.data(), 1, n);
        // strictly convex: every other vertex strictly on one side of every edge
        bool left = true, right = true;
        for (int e = 0; e < n; e++)
            for (int k = 0; k < n; k++) {
                const int f = (e + 1) % n;
                if (k == e || k == f) continue;
                const int64_t c = (int64_t)(x[f] - x[e]) * (y[k] - y[e]) - (int64_t)(y[f] - y[e]) * (x[k] - x[e]);
                left = left && c > 0;
                right = right && c < 0;
            }
        if (s.strict && !left && !right) {
            printf("polygon %d of %d vertices: not strictly convex\n", it, n);
            return 1;
        }
        if (s.area2 <= 0) std::reverse(P.begin(), P.end());
        for (int pass = 0; pass < (s.strict ? 2 : 1); pass++) {
            std::vector<uint32_t> got;
            ear_clip_ring<16>(P.data(), 1, n, pass == 0, [&](uint32_t a, uint32_t b, uint32_t c) {
                got.push_back(a);
                got.push_back(b);
                got.push_back(c);
            });
            if (got != want) {
                printf("polygon %d of %d vertices, kind %d, pass %d: other triangles\n", it, n, kind, pass);
                return 1;
            }
        }
        polygons++;
        strict += s.strict;
    }
    printf("%ld %ld\n", polygons, strict);
    return 0;
}
