// ear_clip_ring (geom.hpp) against ear_clip on random polygons of 3..16
// vertices on the 1/64 lattice (star-shaped ones, some with straight corners,
// and arbitrary, mostly self-crossing ones): the same triangles in the same
// order, and the same number of vertices left; for the strictly convex ones
// of poly_shape also without the inside tests; convex and star-shaped ones
// are cut wholly.  subdivide_hull_emit against subdivide_cell_emit for random
// keys of a cell and its neighbours.  And tj_corners (pixel.hpp) against
// tjunction at every lattice point of a cell, for the frame formats.  Prints
// the number of polygons, of strictly convex ones, and of cells.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdio.h>

#include <algorithm>
#include <random>
#include <vector>

#include "geom.hpp"
#include "pixel.hpp"
using namespace dpx;

int main()
{
    std::mt19937 rng(7);
    auto uni = [&](int a, int b) { return (int)(rng() % (unsigned)(b - a + 1)) + a; };
    long polygons = 0, strict = 0, cells = 0;
    for (int it = 0; it < 400000; it++) {
        const int n = uni(3, 16), kind = uni(0, 3);
        std::vector<int> x(n), y(n);
        if (kind < 3) {
            std::vector<double> a(n);
            for (double& v : a) v = uni(0, 6283) / 1000.0;
            std::sort(a.begin(), a.end());
            for (int k = 0; k < n; k++) {
                const double r = kind == 0 ? 50 : kind == 1 ? uni(10, 60) : uni(20, 60);
                x[k] = 32 + (int)lrint(r * cos(a[k]));
                y[k] = 32 + (int)lrint(r * sin(a[k]));
                if (kind == 2) x[k] = x[k] / 16 * 16, y[k] = y[k] / 16 * 16;
            }
        } else {
            for (int k = 0; k < n; k++) x[k] = uni(-22, 86), y[k] = uni(-22, 86);
        }
        if (uni(0, 1)) std::reverse(x.begin(), x.end()), std::reverse(y.begin(), y.end());
        uint8_t tri[3 * kMaxPoly];
        int ok;
        const int nt = ear_clip(x.data(), y.data(), n, tri, &ok);
        std::vector<uint32_t> P(n);
        for (int k = 0; k < n; k++) P[k] = ((uint32_t)x[k] & 0xFFFFu) | ((uint32_t)y[k] << 16);
        std::vector<uint32_t> want;
        for (int k = 0; k < 3 * nt; k++) want.push_back(P[tri[k]]);
        const PolyShape s = poly_shape(P.data(), 1, n);
        if (s.area2 <= 0) std::reverse(P.begin(), P.end());
        for (int pass = 0; pass < 2; pass++) {
            if (pass == 1 && !s.strict) continue;
            std::vector<uint32_t> got;
            const int left = ear_clip_ring<16>(P.data(), 1, n, pass == 0, [&](uint32_t a, uint32_t b, uint32_t c) {
                got.push_back(a);
                got.push_back(b);
                got.push_back(c);
            });
            if (got != want || left != n - nt || ((s.convex || poly_star(P.data(), 1, n, 32, 32)) && left != 2)) {
                printf("polygon %d (n %d, kind %d) pass %d: %zu of %zu corners, %d left, convex %d\n", it, n, kind, pass,
                       got.size(), want.size(), left, (int)s.convex);
                return 1;
            }
        }
        polygons++;
        strict += s.strict;
    }
    struct Points {
        int x[32], y[32], n;
    };
    for (int it = 0; it < 300000; it++) {
        Points own, nb[8];
        auto make = [&](Points& p, uint32_t key) { p.n = cell_hull(key, p.x, p.y); };
        const uint32_t key = (uint32_t)uni(0, 4095), node = key & 0xFFu, corners = (uint32_t)uni(0, 31);
        make(own, key);
        for (Points& p : nb) make(p, (uint32_t)uni(0, 4095));
        std::vector<int> want, got;
        auto tj = [&](int x, int y) { return tj_kept(corners, x, y); };
        subdivide_cell_emit((const int*)own.x, (const int*)own.y, own.n, node,
                            [&](int e, auto f) { return f((const int*)nb[e].x, (const int*)nb[e].y, nb[e].n); }, tj,
                            [&](int x, int y) { want.push_back(x), want.push_back(y); });
        subdivide_hull_emit(hull_pack(own.x, own.y, own.n), node,
                            [&](int e) { return hull_pack(nb[e].x, nb[e].y, nb[e].n); }, tj,
                            [&](int x, int y) { got.push_back(x), got.push_back(y); });
        if (got != want) {
            printf("key %u: %zu and %zu coordinates\n", key, got.size(), want.size());
            return 1;
        }
        for (int v : got)
            if (v < -64 || v > 127) {
                printf("key %u: coordinate %d\n", key, v);
                return 1;
            }
    }
    for (int it = 0; it < 400; it++) {
        const int W = uni(1, 12), H = uni(1, 9), fmt = uni(0, 3), ch = fmt == 1 ? 4 : fmt == 3 ? 1 : 3;
        const int stride = W * ch + uni(0, 5), colours = uni(1, 3);
        std::vector<uint8_t> img((size_t)stride * H), pal(1024);
        for (uint8_t& v : img) v = (uint8_t)uni(0, colours);
        for (size_t k = 0; k < pal.size(); k++) pal[k] = (uint8_t)uni(0, 1);
        const ImgView im{ img.data(), W, H, stride, ch, fmt == 2 ? (uint32_t)DPX_TOPDOWN : fmt == 3 ? (uint32_t)DPX_INDEXED : 0u,
                          fmt == 3 ? pal.data() : nullptr };
        const TjView v = tj_view(im);
        for (int j = 0; j < H; j++)
            for (int i = 0; i < W; i++) {
                const uint32_t c = tj_corners(v, i, j);
                cells++;
                for (int y4 = -1; y4 <= 6; y4++)
                    for (int x4 = -1; x4 <= 6; x4++)
                        if (tj_kept(c, x4, y4) != tjunction(v, i, j, x4, y4)) {
                            printf("cell %d,%d of %dx%d format %d vertex %d,%d\n", i, j, W, H, fmt, x4, y4);
                            return 1;
                        }
            }
    }
    printf("%ld %ld %ld\n", polygons, strict, cells);
    return 0;
}
