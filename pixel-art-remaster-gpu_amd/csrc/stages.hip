// stages.hip -- the per-stage kernels (one kernel per stage of kernel.cu's
// sequence, intermediates in HBM in the reference's formats), the stage entry
// points of the C ABI, the plain per-frame path and the launch_kernel drop-in.
//
// The graph kernels take 16x16 threads, one per pixel; the kernels that read
// and write whole cells (45 slots, 360 bytes) take runs or tiles of cells,
// staged in LDS and written as contiguous ranges; the raster and the window
// take tiles of output pixels.  The formats are the reference's; the batched
// path in fused.hip, which has none of them in HBM, is the fast one.
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <numeric>
#include <type_traits>

#include "common.hpp"
#include "geom.hpp"
#include "graph.hpp"
#include "hull_table.hpp"
#include "pixel.hpp"

namespace dpx {
namespace {

constexpr int kB = 16;

dim3 grid2(int W, int H) { return dim3((unsigned)((W + kB - 1) / kB), (unsigned)((H + kB - 1) / kB)); }

__device__ inline bool in_frame(int i, int j, int W, int H) { return i >= 0 && j >= 0 && i < W && j < H; }

// graph_Kernel (kernel.cu:140-159): 8 similarity bits per pixel
__global__ void k_graph(ImgView im, uint8_t* __restrict__ graph)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    int j = blockIdx.y * blockDim.y + threadIdx.y;
    if (i >= im.W || j >= im.H) return;
    Yuv c = yuv_of(load_px(im, i, j), im.flags, colour_channels(im));
    uint32_t g = 0;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        int ni = i + edx(e), nj = j + edy(e);
        if (!in_frame(ni, nj, im.W, im.H)) continue;
        if (similar(c, yuv_of(load_px(im, ni, nj), im.flags, colour_channels(im)))) g |= 1u << e;
    }
    graph[(size_t)j * im.W + i] = (uint8_t)g;
}

__device__ inline void gather_nb(const uint8_t* g, int W, int H, int i, int j, uint32_t* nb)
{
#pragma unroll
    for (int e = 0; e < 8; e++) {
        int ni = i + edx(e), nj = j + edy(e);
        nb[e] = in_frame(ni, nj, W, H) ? (uint32_t)g[(size_t)nj * W + ni] : 0u;
    }
}

// trivial_cross_Kernel (kernel.cu:162-177), in place: reads orthogonal bits,
// clears the pixel's own diagonal bits only.
__global__ void k_trivial(uint8_t* graph, int W, int H)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    int j = blockIdx.y * blockDim.y + threadIdx.y;
    if (i >= W || j >= H) return;
    uint32_t nb[8];
    gather_nb(graph, W, H, i, j, nb);
    uint8_t* p = &graph[(size_t)j * W + i];
    uint32_t c = *p;
    *p = (uint8_t)(c & ~trivial_clear_mask(c, nb));
}

// ambiguous_cross_Kernel (kernel.cu:180-189): decisions on the snapshot aux
__global__ void k_heuristic(uint8_t* __restrict__ graph, const uint8_t* __restrict__ aux, int W, int H)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    int j = blockIdx.y * blockDim.y + threadIdx.y;
    if (i >= W || j >= H) return;
    uint32_t nb[8];
    gather_nb(aux, W, H, i, j, nb);
    size_t idx = (size_t)j * W + i;
    uint32_t c = aux[idx];
    // a caller's graph may hold links that leave the frame (the similarity
    // stage never makes one): a walk reaching past the edge finds a node
    // without links there and stops
    auto get = [=](int x, int y) -> uint32_t {
        return (unsigned)x < (unsigned)W && (unsigned)y < (unsigned)H ? aux[(size_t)y * W + x] : 0u;
    };
    graph[idx] = (uint8_t)(c & ~heuristic_clear_mask(get, i, j, c, nb));
}

// The kernels below write whole cells of 45 slots (360 bytes).  A thread
// that writes its own cell's slots puts every lane of a store on a line of
// its own, so the cells' values go to LDS first and a block then writes its
// kRun cells as one contiguous range, adjacent lanes adjacent slots.
constexpr int kRun = 64;

__device__ inline dpx_point hull_point(HullBits h, int t)
{
    dpx_point p;
    p.x = 0.25f * (float)hull_x(h, t);
    p.y = 0.25f * (float)hull_y(h, t);
    return p;
}

// cells_Kernel (kernel.cu:192-213): hull points in 45-slot cells.  Slots past
// the closing point are written as (0,0).  Bound by its writes (20.6 MB for
// 256x224); 8 us there; the
// hulls computed in per-thread arrays took 59.
__global__ __launch_bounds__(256) void k_cells(const uint8_t* __restrict__ graph, size_t N,
                                               dpx_point* __restrict__ diagram, int32_t* __restrict__ edge_count)
{
    __shared__ HullBits s_h[kRun];
    const size_t c0 = (size_t)blockIdx.x * kRun;
    const int t = threadIdx.x, cells = (int)(N - c0 < kRun ? N - c0 : kRun);
    if (t < cells) {
        const size_t idx = c0 + t;
        const uint32_t left = idx > 0 ? graph[idx - 1] : 0u;
        const uint32_t right = idx + 1 < N ? graph[idx + 1] : 0u;
        const HullBits h = kHullTable[cell_key(graph[idx], left, right)];
        s_h[t] = h;
        edge_count[idx] = hull_count(h);
    }
    __syncthreads();
    dpx_point* d = diagram + c0 * kCellSize;
    for (int k = t; k < cells * kCellSize; k += 256) {
        const int c = k / kCellSize, q = k - c * kCellSize;
        const HullBits h = s_h[c];
        const int n = hull_count(h);
        dpx_point p = { 0.0f, 0.0f };
        if (q <= n) p = hull_point(h, q == n ? 0 : q);
        d[k] = p;
    }
}

__device__ inline int load_quarter(const dpx_point* c, int n, int* x, int* y)
{
    for (int t = 0; t < n; t++) {
        x[t] = (int)(c[t].x * 4.0f);
        y[t] = (int)(c[t].y * 4.0f);
    }
    return n;
}

// One cell of subdivision_Kernel in per-thread arrays: any vertex counts and
// coordinates that a caller's diagram may hold.
__device__ __noinline__ int subdivide_any(ImgView im, uint32_t node, int i, int j, int n,
                                          dpx_point* __restrict__ diagram, const dpx_point* __restrict__ daux,
                                          const int32_t* __restrict__ eaux)
{
    const int W = im.W, idx = j * W + i;
    int hx[2 * kMaxPts], hy[2 * kMaxPts];
    load_quarter(&daux[(size_t)idx * kCellSize], n, hx, hy);
    TjView tv = tj_view(im);
    auto nbr = [&](int e, int* lx, int* ly) -> int {
        int q = idx + edy(e) * W + edx(e);
        lx[0] = ly[0] = 0;
        if (q < 0 || q >= W * im.H) return 1;  // (a link that leaves the frame)
        int ln = eaux[q];
        if (ln > 2 * kMaxPts - 1) ln = 2 * kMaxPts - 1;
        if (ln < 1) return 1;
        return load_quarter(&daux[(size_t)q * kCellSize], ln, lx, ly);
    };
    auto tj = [&](int x4, int y4) -> bool { return tjunction(tv, i, j, x4, y4); };
    int ox[kMaxPoly], oy[kMaxPoly];
    int m = subdivide_cell(hx, hy, n, node, nbr, tj, ox, oy);
    dpx_point* c = &diagram[(size_t)idx * kCellSize];
    for (int t = 0; t < m; t++) {
        dpx_point p;
        p.x = (float)ox[t] * (1.0f / 64.0f);
        p.y = (float)oy[t] * (1.0f / 64.0f);
        c[t] = p;
    }
    return m;
}

// x | y << 16; false when one lies outside -limit .. limit (at most 32767)
__device__ inline bool pack_point(int x, int y, int limit, uint32_t* w)
{
    *w = ((uint32_t)x & 0xFFFFu) | ((uint32_t)y << 16);
    return x >= -limit && x <= limit && y >= -limit && y <= limit;
}
__device__ inline int point_x(uint32_t w) { return (int)(int16_t)(w & 0xFFFFu); }
__device__ inline int point_y(uint32_t w) { return (int)w >> 16; }

// subdivision_Kernel (kernel.cu:216-261) on the snapshots daux/eaux, a tile
// of 32x8 cells per block: the hulls of the tile and the cells around it in
// LDS (up to 8 vertices, as the cells stage makes them), the new points from
// LDS to the diagram.  A cell with other hulls around it, or a link that
// leaves the frame, takes subdivide_any.  (All cells through per-thread
// arrays: 58 us for 256x224; so 28.)
constexpr int kSubX = 32, kSubY = 8, kSubPitch = 9;  // (9 words a hull: no bank is shared by adjacent cells)
__global__ __launch_bounds__(256) void k_subdivide(ImgView im, const uint8_t* __restrict__ graph,
                                                   dpx_point* __restrict__ diagram,
                                                   const dpx_point* __restrict__ daux,
                                                   int32_t* __restrict__ edge_count,
                                                   const int32_t* __restrict__ eaux)
{
    constexpr int CX = kSubX + 2, CY = kSubY + 2;
    constexpr uint8_t ANY = 255;
    __shared__ uint32_t s_hull[CX * CY * kSubPitch];
    __shared__ uint8_t s_n[CX * CY];
    __shared__ uint32_t s_new[16 * 256];  // point k of cell t at [k * 256 + t]
    __shared__ uint8_t s_m[256];
    const int t = threadIdx.x, W = im.W, H = im.H;
    const int x0 = blockIdx.x * kSubX, y0 = blockIdx.y * kSubY;
    for (int k = t; k < CX * CY; k += 256) {
        const int x = x0 - 1 + k % CX, y = y0 - 1 + k / CX;
        int n = 1;  // (outside the frame: never asked for, see below)
        if (in_frame(x, y, W, H)) n = eaux[y * W + x];
        s_n[k] = n < 1 || n > 8 ? ANY : (uint8_t)n;
    }
    __syncthreads();
    // (all of a thread's loads before the first is waited for)
    constexpr int PER = (CX * CY * 8 + 255) / 256;
    dpx_point p[PER];
#pragma unroll
    for (int k = 0; k < PER; k++) {
        const int c = (t >> 3) + 32 * k, q = t & 7, x = x0 - 1 + c % CX, y = y0 - 1 + c / CX;
        p[k] = dpx_point{ 0.0f, 0.0f };
        if (c < CX * CY && in_frame(x, y, W, H) && s_n[c] != ANY && q < s_n[c])
            p[k] = daux[(size_t)(y * W + x) * kCellSize + q];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; k++) {
        const int c = (t >> 3) + 32 * k, q = t & 7;
        if (c < CX * CY) {
            uint32_t w;
            // (the new points are 16 times as large and have to fit as well)
            if (!pack_point((int)(p[k].x * 4.0f), (int)(p[k].y * 4.0f), 1024, &w)) s_n[c] = ANY;
            s_hull[c * kSubPitch + q] = w;
        }
    }
    __syncthreads();
    const int cx = t % kSubX, cy = t / kSubX, i = x0 + cx, j = y0 + cy;
    const int own = (cy + 1) * CX + cx + 1;
    s_m[t] = 0;
    if (i < W && j < H) {
        const int idx = j * W + i;
        const uint32_t node = graph[idx];
        const int n = eaux[idx];
        // subdivide_cell emits up to 2n points into kMaxPoly slots; real hulls
        // have at most 8 vertices, larger caller-supplied counts leave the
        // cell, and so do internal nodes (kernel.cu:231)
        if (node != 90 && n >= 3 && n <= kMaxPoly / 2) {
            bool any = false;
#pragma unroll
            for (int e = 0; e < 8; e++)
                if (bit(node, e))
                    any = any || !in_frame(i + edx(e), j + edy(e), W, H) || s_n[own + edy(e) * CX + edx(e)] == ANY;
            if (any || s_n[own] == ANY) {
                edge_count[idx] = subdivide_any(im, node, i, j, n, diagram, daux, eaux);
            } else {
                struct PointsX {
                    const uint32_t* p;
                    __device__ int operator[](int k) const { return point_x(p[k]); }
                };
                struct PointsY {
                    const uint32_t* p;
                    __device__ int operator[](int k) const { return point_y(p[k]); }
                };
                const uint32_t corners = tj_corners(tj_view(im), i, j);
                const uint32_t* h = s_hull + own * kSubPitch;
                auto nbr = [&](int e, auto f) {
                    const int c = own + edy(e) * CX + edx(e);
                    const uint32_t* q = s_hull + c * kSubPitch;
                    return f(PointsX{ q }, PointsY{ q }, (int)s_n[c]);
                };
                auto tj = [&](int x4, int y4) -> bool { return tj_kept(corners, x4, y4); };
                int m = 0;
                subdivide_cell_emit(PointsX{ h }, PointsY{ h }, n, node, nbr, tj, [&](int px, int py) {
                    s_new[256 * m + t] = ((uint32_t)px & 0xFFFFu) | ((uint32_t)py << 16);
                    m++;
                });
                edge_count[idx] = m;
                s_m[t] = (uint8_t)m;
            }
        }
    }
    __syncthreads();
    for (int k = t; k < 256 * 16; k += 256) {
        const int c = k >> 4, q = k & 15;
        if (q >= s_m[c]) continue;
        const uint32_t w = s_new[256 * q + c];
        dpx_point p;
        p.x = (float)point_x(w) * (1.0f / 64.0f);
        p.y = (float)point_y(w) * (1.0f / 64.0f);
        diagram[(size_t)((y0 + c / kSubX) * W + x0 + c % kSubX) * kCellSize + q] = p;
    }
}

// One cell of triangulate_Kernel in per-thread arrays: any vertex counts and coordinates.
__device__ __noinline__ void triangulate_any(dpx_point* __restrict__ c, int n, float fi, float fj)
{
    int x[kMaxPoly], y[kMaxPoly];
    uint8_t tri[3 * kMaxPoly];
    int nt = 0, ok = 0;
    if (n >= 3 && n <= kMaxPoly) {
        for (int t = 0; t < n; t++) {
            x[t] = (int)(c[t].x * 64.0f);
            y[t] = (int)(c[t].y * 64.0f);
        }
        nt = ear_clip(x, y, n, tri, &ok);
    }
    for (int t = 0; t < kCellSize; t++) {
        dpx_point p;
        if (t < 3 * nt) {
            p.x = (float)x[tri[t]] * (1.0f / 64.0f) + fi;
            p.y = (float)y[tri[t]] * (1.0f / 64.0f) + fj;
        } else {
            p.x = fi;
            p.y = fj;
        }
        c[t] = p;
    }
}

// triangulate_Kernel (kernel.cu:264-282): ear clipping, then every slot gets
// the pixel offset; unwritten slots stay at the pixel origin.  A block takes
// kTriRun cells, a lane a cell; the polygons (up to 16 vertices, twice a
// hull's) lie in LDS.  Cells go to the lanes by the work they are, so that a
// wave's lanes end together: those that need the inside tests by their
// vertices, then the strictly convex ones, whose waves skip the tests.
// Other cells take triangulate_any.  Bound by the instructions of the tests.
// (28 us for 256x224.  All cells through per-thread arrays: 109, every vertex
// read a round trip to memory; vertices shifted in LDS: 56.)
constexpr int kTriRun = 256, kTriBlock = 1024;  // (all threads read and write, the first kTriRun clip)
struct alignas(16) TriSlots {
    float x, y;  // the pixel
    int n;       // slots of triangles; -1: the cell takes triangulate_any
    int pad;
};
__global__ __launch_bounds__(kTriBlock) void k_triangulate(dpx_point* __restrict__ diagram,
                                                         const int32_t* __restrict__ edge_count, int W, size_t N)
{
    constexpr int MAXN = 16, MAXV = 3 * (MAXN - 2);
    __shared__ uint32_t s_poly[MAXN * kTriRun];  // vertex k of cell t at [k * kTriRun + t]
    __shared__ uint32_t s_tri[MAXV * kTriRun];   // triangle corners likewise
    __shared__ uint8_t s_n[kTriRun], s_any[kTriRun];
    __shared__ uint16_t s_list[kTriRun];  // cell (| kStrict) of each lane
    __shared__ int s_bin[64];
    __shared__ TriSlots s_slots[kTriRun];
    constexpr uint16_t kStrict = 0x8000;
    const size_t c0 = (size_t)blockIdx.x * kTriRun;
    const int t = threadIdx.x, cells = (int)(N - c0 < kTriRun ? N - c0 : kTriRun);
    dpx_point* d = diagram + c0 * kCellSize;
    int n_own = 0;
    if (t < kTriRun) {
        if (t < cells) n_own = edge_count[c0 + t];
        s_n[t] = (uint8_t)(n_own >= 3 && n_own <= MAXN ? n_own : 0);
        s_any[t] = n_own > MAXN;
    }
    if (t < 64) s_bin[t] = 0;
    __syncthreads();
    {
        // (all of a thread's loads before the first is waited for: a loop
        // that stores each waits a memory latency per vertex)
        constexpr int PER = kTriRun * MAXN / kTriBlock;
        dpx_point p[PER];
        const int q = t % MAXN;
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int c = t / MAXN + k * (kTriBlock / MAXN);
            p[k] = dpx_point{ 0.0f, 0.0f };
            if (q < s_n[c]) p[k] = d[c * kCellSize + q];
        }
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int c = t / MAXN + k * (kTriBlock / MAXN);
            uint32_t w;
            if (!pack_point((int)(p[k].x * 64.0f), (int)(p[k].y * 64.0f), kEarLimit, &w)) s_any[c] = 1;
            s_poly[q * kTriRun + c] = w;
        }
    }
    __syncthreads();
    int bin = 2 * MAXN + 1, rank = 0;  // (nothing to cut)
    bool strict = false;
    if (t < kTriRun) {
        if (s_n[t] && !s_any[t]) {
            uint32_t* P = s_poly + t;
            const int n = s_n[t];
            const PolyShape shape = poly_shape(P, kTriRun, n);
            strict = shape.strict;
            if (shape.area2 <= 0)
                for (int lo = 0, hi = n - 1; lo < hi; lo++, hi--) {
                    const uint32_t tmp = P[kTriRun * lo];
                    P[kTriRun * lo] = P[kTriRun * hi];
                    P[kTriRun * hi] = tmp;
                }
            bin = (strict ? MAXN : 0) + MAXN - n;
        }
        rank = atomicAdd(&s_bin[bin], 1);
    }
    __syncthreads();
    if (t < 64) {
        const int own = s_bin[t];
        int at = own;
#pragma unroll
        for (int e = 1; e < 64; e <<= 1) {
            const int v = __shfl_up(at, e);
            if (t >= e) at += v;
        }
        s_bin[t] = at - own;
    }
    __syncthreads();
    if (t < kTriRun) s_list[s_bin[bin] + rank] = (uint16_t)t | (strict ? kStrict : (uint16_t)0);
    __syncthreads();
    if (t < kTriRun) {
        const int c = s_list[t] & 0xFF;
        const bool test = !(s_list[t] & kStrict);
        const int n = s_any[c] ? 0 : s_n[c];
        uint32_t* T = s_tri + c;
        int written = 0;
        if (n)
            ear_clip_ring<MAXN>(s_poly + c, kTriRun, n, test, [&](uint32_t A, uint32_t B, uint32_t C) {
                T[kTriRun * written] = A;
                T[kTriRun * (written + 1)] = B;
                T[kTriRun * (written + 2)] = C;
                written += 3;
            });
        const size_t idx = c0 + c, j = idx / (size_t)W;
        s_slots[c] = TriSlots{ (float)(int)(idx - j * (size_t)W), (float)(int)j, s_any[c] ? -1 : written, 0 };
    }
    __syncthreads();
    for (int k = t; k < cells * kCellSize; k += kTriBlock) {
        const int c = k / kCellSize, q = k - c * kCellSize;
        const TriSlots sl = s_slots[c];
        if (sl.n < 0) continue;
        dpx_point p = { sl.x, sl.y };
        if (q < sl.n) {
            const uint32_t w = s_tri[q * kTriRun + c];
            p.x = (float)point_x(w) * (1.0f / 64.0f) + sl.x;
            p.y = (float)point_y(w) * (1.0f / 64.0f) + sl.y;
        }
        d[k] = p;
    }
    if (t < cells && s_any[t]) triangulate_any(d + t * kCellSize, n_own, s_slots[t].x, s_slots[t].y);
}

// color_kernel (kernel.cu:67-104) + position_kernel (kernel.cu:109-137), a
// run of cells per block, adjacent lanes adjacent slots (256x224: 9 us; a thread per
// cell: 55)
__global__ __launch_bounds__(256) void k_export_vbo(ImgView im, const dpx_point* __restrict__ diagram,
                                                    const int32_t* __restrict__ edge_count,
                                                    dpx_point* __restrict__ pos, dpx_uchar4* __restrict__ color)
{
    __shared__ uint32_t s_rgba[kRun];
    __shared__ int s_valid[kRun];
    const size_t N = (size_t)im.W * im.H, c0 = (size_t)blockIdx.x * kRun;
    const int t = threadIdx.x, cells = (int)(N - c0 < kRun ? N - c0 : kRun);
    if (t < cells) {
        const size_t idx = c0 + t;
        s_rgba[t] = cell_rgba(load_px(im, (int)(idx % (size_t)im.W), (int)(idx / (size_t)im.W)), colour_channels(im));
        s_valid[t] = (edge_count[idx] - 2) * 3;
    }
    __syncthreads();
    for (int k = t; k < cells * kCellSize; k += 256) {
        const int c = k / kCellSize, q = k - c * kCellSize;
        const size_t s = c0 * kCellSize + k;
        if (color) {
            const uint32_t rgba = s_rgba[c];
            dpx_uchar4 c4;
            c4.x = (uint8_t)(rgba & 0xFF);
            c4.y = (uint8_t)((rgba >> 8) & 0xFF);
            c4.z = (uint8_t)((rgba >> 16) & 0xFF);
            c4.w = (uint8_t)(rgba >> 24);
            color[s] = c4;
        }
        if (pos) {
            dpx_point p = { -100.0f, -100.0f };
            if (q < s_valid[c]) p = diagram[s];
            pos[s] = p;
        }
    }
}

// ---------------------------------------------------------------------------
// glDrawArrays(GL_TRIANGLES) in VBO order (simpleVBO.cpp:281) as a gather,
// for the frame's raster and for the GLUT window (display()
// callbacks.cpp:39-72, renderCuda simpleVBO.cpp:185-440): a sample takes the
// colour of the highest-index cell (the last one drawn) with a triangle that
// covers it.  Cells reach at most three quarters of a cell past their unit
// square, so the cells around the sample's own are the candidates.
//
// All coordinates are whole numbers of a unit such that a cell is `unit` of
// them: 1/(128 scale) of a cell for the raster, 1/(512 sc) for the window
// (sc the scale in hundredths).  Sample s of output pixel (X, Y) lies at
// (step X + ox[s], step Y + oy[s]) and a 1/64-lattice vertex v at v unit / 64.
// Window point (X + ox/8, Y + oy/8) is image point ((8 (X - tx) + ox) * 100)
// / (8 * sc), i.e. (8 (X - tx) + ox) * 6400 units.
// ---------------------------------------------------------------------------
struct TriGeom {
    int unit, step;         // of a cell, of an output pixel
    long long ox[4], oy[4]; // samples of pixel (0, 0)
    int W, H;               // output pixels
    int topdown;            // output row 0 is the top one
    int quads;              // each image pixel as its square
};

__device__ inline long long floor_div(long long a, long long b)  // b > 0
{
    long long q = a / b;
    return (a % b != 0 && a < 0) ? q - 1 : q;
}

// The colour of a pixel from its samples': averaged per channel, halves rounded up.
template <int NS>
__device__ inline uint32_t tri_average(const uint32_t* col)
{
    if constexpr (NS == 1) return col[0];
    uint32_t color = 0;
#pragma unroll
    for (int b = 0; b < 4; b++) {
        uint32_t sum = NS / 2;
#pragma unroll
        for (int s = 0; s < NS; s++) sum += (col[s] >> (8 * b)) & 0xFFu;
        color |= (sum / NS) << (8 * b);
    }
    return color;
}

// A sample's colour over the cells [i0, i1] x [j0, j1] in reverse draw order,
// straight from the diagram and in 64 bits: any scale and any coordinates.
__device__ __noinline__ uint32_t tri_sample_any(ImgView im, const dpx_point* __restrict__ diagram,
                                                const int32_t* __restrict__ edge_count, int unit, int i0, int i1,
                                                int j0, int j1, long long px, long long py)
{
    for (int j = j1; j >= j0; j--)
        for (int i = i1; i >= i0; i--) {
            const size_t k = (size_t)j * im.W + (size_t)i;
            const int nt = cell_triangles(edge_count[k]);
            const dpx_point* c = &diagram[k * kCellSize];
            const float fi = (float)i, fj = (float)j;
            const long long sx = px - (long long)i * unit, sy = py - (long long)j * unit;
            for (int t = 0; t < nt; t++) {
                long long w[6];
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    const dpx_point p = c[3 * t + q];
                    w[2 * q] = (long long)(int)((p.x - fi) * 64.0f) * (unit / 64);
                    w[2 * q + 1] = (long long)(int)((p.y - fj) * 64.0f) * (unit / 64);
                }
                if (tri_covers(w[0], w[1], w[2], w[3], w[4], w[5], sx, sy))
                    return cell_rgba(load_px(im, i, j), colour_channels(im));
            }
        }
    return 0xFF000000u;  // clear colour (0,0,0,1), main.cpp:260
}

// 16 x TY output pixels per block.  The cells around them (`cap` of them fit
// the LDS the launch gave) are read once: each triangle's three edge
// functions e = dx sy - dy sx + k, counter-clockwise and with the tie of the
// coverage rule in k (covered: all three above 0), so that a sample's test of
// a triangle is six multiply-adds; and how far the cells reach beyond their
// squares, which keeps most pixels to one to four of the cells around them.
// A vertex within a smoothed cell's reach, and a sample that lies up to two
// cells and a pixel from its candidates, keep every term in 31 bits and the
// factors in 24; a cell of a caller's diagram beyond that, and scales with more
// cells, take tri_sample_any.  (With half a cell for the reach, dithers of
// nearly similar colours took that in most blocks: the raster of 256x224 at 8x
// 546 us, so 151, the window at 8x 719, so 96.)
// Bound by the instructions of the tests; straight from memory in 64 bits
// the 1200x800 window of a smoothed 256x224 frame took 221 us, so 40.
constexpr int kTris = kCellSize / 3;
constexpr int kTriLow = std::min(kReachXLow, kReachYLow), kTriHigh = std::max(kReachXHigh, kReachYHigh);  // 1/64 units
constexpr long long kTriUnitMost = 512 * 3200, kTriStep = 8 * 6400;  // of the window, the larger ones
static_assert((kTriHigh - kTriLow) * (2 * (2 * kTriUnitMost + kTriStep) + 2 * kTriHigh * kTriUnitMost / 64) < 1LL << 31 &&
              2 * kTriUnitMost + kTriStep < 1 << 23, "an edge function and its factors");
struct TriEdge {
    uint32_t d;  // dx | dy << 16
    int k;
};
constexpr size_t kTriCellBytes = 3 * kTris * sizeof(TriEdge) + sizeof(int);

template <int NS, int TY>
__global__ __launch_bounds__(16 * TY) void k_tri(ImgView im, const dpx_point* __restrict__ diagram,
                                             const int32_t* __restrict__ edge_count, TriGeom v, int cap,
                                             uint8_t* __restrict__ out, int out_stride)
{
    extern __shared__ uint32_t s_dyn[];
    TriEdge* s_edge = reinterpret_cast<TriEdge*>(s_dyn);
    int* s_nt = reinterpret_cast<int*>(s_edge + (size_t)cap * 3 * kTris);
    __shared__ int s_range[4], s_any;
    __shared__ int s_lo, s_hi;  // the least and greatest vertex coordinate, 1/64 units of its cell
    constexpr int NT = 16 * TY;
    const int t = threadIdx.x, X = blockIdx.x * 16 + (t & 15), Y = blockIdx.y * TY + (t >> 4);
    // The cell of the block's first sample (64-bit, one division a wave), and
    // every sample relative to that cell in 32 bits.  A block far outside the
    // image keeps only that it is (its 16 pixels reach at most 64 cells).
    auto origin = [&](int first, const long long* o) {
        long long p = o[0];
#pragma unroll
        for (int s = 1; s < NS; s++) p = min(p, o[s]);
        return floor_div(p + (long long)v.step * first, (long long)v.unit);
    };
    auto near_frame = [](long long c, int n) { return (int)(c < -128 ? -128 : c > n + 64 ? n + 64 : c); };
    const long long oi = origin(X - (t & 15), v.ox), oj = origin(Y - (t >> 4), v.oy);
    const int ni = near_frame(oi, im.W), nj = near_frame(oj, im.H);
    int rx[NS], ry[NS], ci[NS], cj[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) {
        rx[s] = (int)((long long)v.step * (X - (t & 15)) + v.ox[s] - oi * v.unit) + v.step * (t & 15);
        ry[s] = (int)((long long)v.step * (Y - (t >> 4)) + v.oy[s] - oj * v.unit) + v.step * (t >> 4);
        ci[s] = ni + floor_div(rx[s], v.unit);
        cj[s] = nj + floor_div(ry[s], v.unit);
    }
    uint32_t col[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) col[s] = 0xFF000000u;  // clear colour (0,0,0,1), main.cpp:260
    const bool mine = X < v.W && Y < v.H;
    const int cc = colour_channels(im);
    if (v.quads) {
        // the two triangles of pixel (ci, cj) cover [ci, ci+1) x [cj, cj+1)
        // under the coverage rule (left and bottom edges in, right and top out)
#pragma unroll
        for (int s = 0; s < NS; s++)
            if (mine && in_frame(ci[s], cj[s], im.W, im.H)) col[s] = cell_rgba(load_px(im, ci[s], cj[s]), cc);
    } else {
        int i0 = ci[0], i1 = ci[0], j0 = cj[0], j1 = cj[0];
#pragma unroll
        for (int s = 1; s < NS; s++) {
            i0 = min(i0, ci[s]);
            i1 = max(i1, ci[s]);
            j0 = min(j0, cj[s]);
            j1 = max(j1, cj[s]);
        }
        // this pixel's candidates, and (corner threads) the block's; pixels
        // past the output's edge only widen the block's range
        i0 = max(i0 - 1, 0);
        j0 = max(j0 - 1, 0);
        i1 = min(i1 + 1, im.W - 1);
        j1 = min(j1 + 1, im.H - 1);
        if (t == 0) {
            s_range[0] = i0;
            s_range[1] = j0;
            s_any = 0;
            s_lo = 0;
            s_hi = 64;
        }
        if (t == NT - 1) {
            s_range[2] = i1;
            s_range[3] = j1;
        }
        __syncthreads();
        const int bi = s_range[0], bj = s_range[1], nci = s_range[2] - bi + 1, ncj = s_range[3] - bj + 1;
        if (nci > 0 && ncj > 0) {  // (uniform; else no cell lies near this block)
            const int nc = nci * ncj, vs = v.unit / 64;
            if (nc > cap) {
                if (t == 0) s_any = 1;
            } else {
                for (int k = t; k < nc; k += NT)
                    s_nt[k] = cell_triangles(edge_count[(size_t)(bj + k / nci) * im.W + bi + k % nci]);
                __syncthreads();
                int lo = 0, hi = 64;
                bool wide = false;
                for (int k = t; k < nc * kTris; k += NT) {
                    const int c = k / kTris, q = k - c * kTris;
                    if (q >= s_nt[c]) continue;
                    const int i = bi + c % nci, j = bj + c / nci;
                    const dpx_point* p = &diagram[((size_t)j * im.W + i) * kCellSize + 3 * q];
                    int x[3], y[3];
#pragma unroll
                    for (int e = 0; e < 3; e++) {
                        x[e] = (int)((p[e].x - (float)i) * 64.0f);
                        y[e] = (int)((p[e].y - (float)j) * 64.0f);
                        lo = min(lo, min(x[e], y[e]));
                        hi = max(hi, max(x[e], y[e]));
                    }
                    if (lo < kTriLow || hi > kTriHigh) {
                        wide = true;
                        break;
                    }
                    // counter-clockwise; a degenerate triangle covers nothing: edges of zeros
                    const int o = (x[1] - x[0]) * (y[2] - y[0]) - (y[1] - y[0]) * (x[2] - x[0]);
                    if (o < 0) {
                        swap2(&x[1], &x[2]);
                        swap2(&y[1], &y[2]);
                    }
#pragma unroll
                    for (int e = 0; e < 3; e++) {
                        const int f = (e + 1) % 3, dx = o ? x[f] - x[e] : 0, dy = o ? y[f] - y[e] : 0;
                        const int tie = dy < 0 || (dy == 0 && dx > 0) ? 1 : 0;
                        s_edge[(c * kTris + q) * 3 + e] = TriEdge{ ((uint32_t)dx & 0xFFFFu) | ((uint32_t)dy << 16),
                                                                   (dy * x[e] - dx * y[e]) * vs + tie };
                    }
                }
                if (wide) s_any = 1;
                if (lo < 0) atomicMin(&s_lo, lo);
                if (hi > 64) atomicMax(&s_hi, hi);
            }
            __syncthreads();
            if (mine && s_any) {
#pragma unroll 1
                for (int s = 0; s < NS; s++) {
                    int sx = rx[0], sy = ry[0];
#pragma unroll
                    for (int q = 1; q < NS; q++)
                        if (q == s) {
                            sx = rx[q];
                            sy = ry[q];
                        }
                    const uint32_t c = tri_sample_any(im, diagram, edge_count, v.unit, i0, i1, j0, j1,
                                                      (long long)ni * v.unit + sx, (long long)nj * v.unit + sy);
#pragma unroll
                    for (int q = 0; q < NS; q++)
                        if (q == s) col[q] = c;
                }
            } else if (mine) {
                // cells whose reach ends before all of the pixel's samples
                const int lo = s_lo * vs, hi = s_hi * vs;
                int x_lo = rx[0], x_hi = rx[0], y_lo = ry[0], y_hi = ry[0];
#pragma unroll
                for (int s = 1; s < NS; s++) {
                    x_lo = min(x_lo, rx[s]);
                    x_hi = max(x_hi, rx[s]);
                    y_lo = min(y_lo, ry[s]);
                    y_hi = max(y_hi, ry[s]);
                }
                while (i0 <= i1 && x_lo - (i0 - ni) * v.unit > hi) i0++;
                while (i1 >= i0 && x_hi - (i1 - ni) * v.unit < lo) i1--;
                while (j0 <= j1 && y_lo - (j0 - nj) * v.unit > hi) j0++;
                while (j1 >= j0 && y_hi - (j1 - nj) * v.unit < lo) j1--;
                uint32_t left = (1u << NS) - 1u;
                for (int j = j1; j >= j0 && left; j--)
                    for (int i = i1; i >= i0 && left; i--) {
                        const int c = (j - bj) * nci + i - bi, nt = s_nt[c];
                        int sx[NS], sy[NS];
#pragma unroll
                        for (int s = 0; s < NS; s++) {
                            sx[s] = rx[s] - (i - ni) * v.unit;
                            sy[s] = ry[s] - (j - nj) * v.unit;
                        }
                        uint32_t hit = 0;
                        const TriEdge* w = s_edge + c * kTris * 3;
                        for (int q = 0; q < nt && (left & ~hit); q++, w += 3) {
                            int low[NS];
#pragma unroll
                            for (int e = 0; e < 3; e++) {
                                const TriEdge ed = w[e];
                                const int dx = point_x(ed.d), dy = -point_y(ed.d);
#pragma unroll
                                for (int s = 0; s < NS; s++) {
                                    const int f = mad24(dx, sy[s], mad24(dy, sx[s], ed.k));
                                    low[s] = e == 0 ? f : min(low[s], f);
                                }
                            }
#pragma unroll
                            for (int s = 0; s < NS; s++) hit |= low[s] > 0 ? 1u << s : 0u;
                        }
                        hit &= left;
                        if (hit) {
                            const uint32_t rgba = cell_rgba(load_px(im, i, j), cc);
#pragma unroll
                            for (int s = 0; s < NS; s++)
                                if ((hit >> s) & 1u) col[s] = rgba;
                            left &= ~hit;
                        }
                    }
            }
        }
    }
    if (!mine) return;
    const int row = v.topdown ? (v.H - 1 - Y) : Y;
    *reinterpret_cast<uint32_t*>(out + (size_t)row * out_stride + (size_t)X * 4) = tri_average<NS>(col);
}

// A thread per pixel, the cells around all of its samples read once from the
// diagram, each triangle tested against every sample that no cell has covered
// yet.  For views that put so many cells into a block that they do not fit LDS
// (scales below 1), and for one sample a pixel up to 1x, where a tile would set
// up two cells' triangles for each pixel that it tests (256x224 at 1x: the
// raster 39 us, so 31, the window 46, so 30).  SMALL: units of at most
// kTriSmallUnit a cell and places below 2^26, so that they are 32-bit, and so
// are the tests of triangles within four cells of their own.
constexpr int kTriSmallUnit = 4096, kTriSmallVertex = 256;  // (coordinates below 511 * 64 apart: 2 * 32704^2 < 2^31)
constexpr int kTriBatch = 4;
template <int NS, bool SMALL>
__global__ __launch_bounds__(256) void k_tri_far(ImgView im, const dpx_point* __restrict__ diagram,
                                                 const int32_t* __restrict__ edge_count, TriGeom v,
                                                 uint8_t* __restrict__ out, int out_stride)
{
    using Place = std::conditional_t<SMALL, int, long long>;
    const int X = blockIdx.x * 16 + (threadIdx.x & 15), Y = blockIdx.y * 16 + (threadIdx.x >> 4);
    if (X >= v.W || Y >= v.H) return;
    const Place unit = v.unit, u = v.unit / 64;
    Place px[NS], py[NS], i0 = 0, i1 = 0, j0 = 0, j1 = 0;
    uint32_t col[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) {
        px[s] = (Place)v.step * X + (Place)v.ox[s];
        py[s] = (Place)v.step * Y + (Place)v.oy[s];
        col[s] = 0xFF000000u;  // clear colour (0,0,0,1), main.cpp:260
        const Place ci = floor_div(px[s], unit), cj = floor_div(py[s], unit);
        if (s == 0 || ci < i0) i0 = ci;
        if (s == 0 || ci > i1) i1 = ci;
        if (s == 0 || cj < j0) j0 = cj;
        if (s == 0 || cj > j1) j1 = cj;
    }
    // the window may lie far outside the image: clamp to the frame
    i0 = i0 - 1 < 0 ? 0 : i0 - 1;
    j0 = j0 - 1 < 0 ? 0 : j0 - 1;
    i1 = i1 + 1 > im.W - 1 ? im.W - 1 : i1 + 1;
    j1 = j1 + 1 > im.H - 1 ? im.H - 1 : j1 + 1;
    const int cc = colour_channels(im);
    uint32_t left = (1u << NS) - 1u;
    for (Place j = j1; j >= j0 && left; j--)
        for (Place i = i1; i >= i0 && left; i--) {
            const size_t k = (size_t)j * im.W + (size_t)i;
            const int nt = cell_triangles(edge_count[k]);
            const dpx_point* c = &diagram[k * kCellSize];
            const float fi = (float)i, fj = (float)j;
            uint32_t hit = 0;
            for (int t0 = 0; t0 < nt && (left & ~hit); t0 += kTriBatch) {
                // (a batch's loads before its first test: a triangle at a time
                // waits a memory latency for each)
                dpx_point p[3 * kTriBatch];
#pragma unroll
                for (int q = 0; q < 3 * kTriBatch; q++) p[q] = c[min(3 * t0 + q, 3 * nt - 1)];
#pragma unroll
                for (int b = 0; b < kTriBatch; b++) {
                    if (t0 + b >= nt || !(left & ~hit)) break;
                    int w[6], most = 0;
#pragma unroll
                    for (int q = 0; q < 3; q++) {
                        w[2 * q] = (int)((p[3 * b + q].x - fi) * 64.0f);
                        w[2 * q + 1] = (int)((p[3 * b + q].y - fj) * 64.0f);
                    }
                    auto test = [&](auto one) {
                        using T = decltype(one);
#pragma unroll
                        for (int s = 0; s < NS; s++)
                            if (((left & ~hit) >> s) & 1u)
                                if (tri_covers<T>(w[0] * (T)u, w[1] * (T)u, w[2] * (T)u, w[3] * (T)u, w[4] * (T)u,
                                                  w[5] * (T)u, (T)(px[s] - i * unit), (T)(py[s] - j * unit)))
                                    hit |= 1u << s;
                    };
                    if constexpr (SMALL) {
#pragma unroll
                        for (int q = 0; q < 6; q++) most = max(most, max(w[q], -1 - w[q]));
                        if (most < kTriSmallVertex) test(0);
                        else test(0LL);
                    } else {
                        test(0LL);
                    }
                }
            }
            if (hit) {
                const uint32_t rgba = cell_rgba(load_px(im, (int)i, (int)j), cc);
#pragma unroll
                for (int s = 0; s < NS; s++)
                    if ((hit >> s) & 1u) col[s] = rgba;
                left &= ~hit;
            }
        }
    const int row = v.topdown ? (v.H - 1 - Y) : Y;
    *reinterpret_cast<uint32_t*>(out + (size_t)row * out_stride + (size_t)X * 4) = tri_average<NS>(col);
}

void launch_tri(const ImgView& im, const dpx_point* diagram, const int32_t* edge_count, TriGeom v, int samples,
                uint8_t* out, int out_stride, hipStream_t stream)
{
    // the coarsest units in which everything is whole (a vertex lies at a 64th of a cell)
    long long g = std::gcd((long long)(v.unit / 64), (long long)v.step), far_off = 0;
    for (int s = 0; s < samples; s++) g = std::gcd(g, std::gcd(v.ox[s], v.oy[s]));
    v.unit /= (int)g;
    v.step /= (int)g;
    for (int s = 0; s < samples; s++) {
        v.ox[s] /= g;
        v.oy[s] /= g;
        far_off = std::max({ far_off, std::abs(v.ox[s]), std::abs(v.oy[s]) });
    }
    // cells that n output pixels reach on one axis: their own, a part at each
    // end and one around each side
    auto reach = [&](int n) { return ((long long)n * v.step - 1) / v.unit + 4; };
    auto lds_of = [&](int ty) { return (size_t)(reach(16) * reach(ty)) * kTriCellBytes; };
    // tiles of 16 rows where their cells leave room for several blocks a CU
    // (from 2.5x up), else of 4 rows (from 1x up: 48 KB), else no LDS
    const bool tall = v.quads || lds_of(16) <= 40 * 1024;
    const int ty = tall ? 16 : 4, cap = v.quads ? 0 : (int)std::min(reach(16) * reach(ty), 1LL << 20);
    const size_t lds = v.quads ? 0 : lds_of(ty);
    const dim3 grid((unsigned)((v.W + 15) / 16), (unsigned)((v.H + ty - 1) / ty));
    const bool small = v.unit <= kTriSmallUnit && far_off + (long long)v.step * std::max(v.W, v.H) < 1LL << 26;
    if (lds > 60 * 1024 || (samples == 1 && v.unit <= v.step && !v.quads)) {
        const dim3 far((unsigned)((v.W + 15) / 16), (unsigned)((v.H + 15) / 16));
        auto fn = samples == 4 ? (small ? k_tri_far<4, true> : k_tri_far<4, false>) : small ? k_tri_far<1, true> : k_tri_far<1, false>;
        hipLaunchKernelGGL(fn, far, dim3(256), 0, stream, im, diagram, edge_count, v, out, out_stride);
        return;
    }
    auto fn = samples == 4 ? (tall ? k_tri<4, 16> : k_tri<4, 4>) : (tall ? k_tri<1, 16> : k_tri<1, 4>);
    hipLaunchKernelGGL(fn, grid, dim3(16 * ty), lds, stream, im, diagram, edge_count, v, cap, out, out_stride);
}

// ---------------------------------------------------------------------------
// Components: lock-free union-find over the graph's edges.  Roots are hooked
// under smaller roots only, so each component's root is its smallest index.
// ---------------------------------------------------------------------------
__device__ inline int uf_find(int32_t* parent_, int v)
{
    // other threads hook roots and halve paths concurrently: read through volatile
    volatile int32_t* parent = parent_;
    int p = parent[v];
    while (p != v) {
        int gp = parent[p];
        if (gp != p) parent[v] = gp;  // path halving; any ancestor is a valid parent
        v = p;
        p = gp;
    }
    return v;
}

// Components in two levels: each 32x32 tile of nodes is labelled by one
// block with a union-find in LDS over the edges inside the tile (roots are
// the smallest node of each piece, so the tile's pieces come out with their
// smallest global index); the edges that cross tile borders are then united
// in global memory (k_cc_cross), and the final pass takes every node's root.
constexpr int kCcTile = 32;

__device__ inline int uf_find_lds(int* parent_, int v)
{
    volatile int* parent = parent_;
    int p = parent[v];
    while (p != v) {
        int gp = parent[p];
        if (gp != p) parent[v] = gp;  // path halving; any ancestor is a valid parent
        v = p;
        p = gp;
    }
    return v;
}

__global__ __launch_bounds__(256) void k_cc_tile(const uint8_t* __restrict__ graph, int W, int H, int32_t* parent)
{
    __shared__ int s_par[kCcTile * kCcTile];
    const int tx0 = blockIdx.x * kCcTile, ty0 = blockIdx.y * kCcTile;
    for (int k = threadIdx.x; k < kCcTile * kCcTile; k += 256) s_par[k] = k;
    __syncthreads();
    for (int k = threadIdx.x; k < kCcTile * kCcTile; k += 256) {
        const int lx = k % kCcTile, ly = k / kCcTile, i = tx0 + lx, j = ty0 + ly;
        if (i >= W || j >= H) continue;
        const uint32_t g = graph[(size_t)j * W + i];
        // edges towards smaller indices only (each edge once): bits 3, 5, 6, 7
        const int es[4] = { 3, 5, 6, 7 };
        for (int t = 0; t < 4; t++) {
            const int e = es[t];
            if (!bit(g, e)) continue;
            const int nlx = lx + edx(e), nly = ly + edy(e);
            if ((unsigned)nlx >= (unsigned)kCcTile || (unsigned)nly >= (unsigned)kCcTile) continue;  // k_cc_cross
            if (!in_frame(i + edx(e), j + edy(e), W, H)) continue;
            const int u = nly * kCcTile + nlx;
            for (;;) {
                const int ru = uf_find_lds(s_par, u), rv = uf_find_lds(s_par, k);
                if (ru == rv) break;
                const int hi = ru > rv ? ru : rv, lo = ru > rv ? rv : ru;
                if (atomicCAS(&s_par[hi], hi, lo) == hi) break;
            }
        }
    }
    __syncthreads();
    for (int k = threadIdx.x; k < kCcTile * kCcTile; k += 256) {
        const int lx = k % kCcTile, ly = k / kCcTile, i = tx0 + lx, j = ty0 + ly;
        if (i >= W || j >= H) continue;
        int r = k;
        for (int p = s_par[r]; p != r; p = s_par[r]) r = p;
        parent[(size_t)j * W + i] = (ty0 + r / kCcTile) * W + tx0 + r % kCcTile;
    }
}

// The edges between tiles, united in global memory (parents are tile roots
// after k_cc_tile).
__global__ void k_cc_cross(const uint8_t* __restrict__ graph, int W, int H, int32_t* parent)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y * blockDim.y + threadIdx.y;
    if (i >= W || j >= H) return;
    const int lx = i % kCcTile, ly = j % kCcTile;
    if (lx != 0 && ly != 0 && lx != kCcTile - 1) return;  // no backward edge leaves the tile
    const int v = j * W + i;
    const uint32_t g = graph[v];
    const int es[4] = { 3, 5, 6, 7 };
    for (int t = 0; t < 4; t++) {
        const int e = es[t];
        if (!bit(g, e)) continue;
        const int ni = i + edx(e), nj = j + edy(e);
        if (!in_frame(ni, nj, W, H)) continue;
        if (ni / kCcTile == i / kCcTile && nj / kCcTile == j / kCcTile) continue;  // inside: k_cc_tile
        const int u = nj * W + ni;
        for (;;) {
            int ru = uf_find(parent, u), rv = uf_find(parent, v);
            if (ru == rv) break;
            int hi = ru > rv ? ru : rv, lo = ru > rv ? rv : ru;
            if (atomicCAS(&parent[hi], hi, lo) == hi) break;
        }
    }
}

// The root of v without shortening paths: the final pass writes each
// label over its own parent entry (the arrays alias), so it must write no
// other entry -- a halving write could replace a label another thread has
// already set to its root with a non-root ancestor.  Entries it reads are
// then an old parent or the root, both ancestors.
__device__ inline int uf_root(const int32_t* parent_, int v)
{
    const volatile int32_t* parent = parent_;
    int p = parent[v];
    while (p != v) {
        v = p;
        p = parent[v];
    }
    return v;
}

__global__ void k_cc_final(int32_t* parent, int32_t* labels, int N)
{
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < N) labels[k] = uf_root(parent, k);
}

int check_img(const void* p, int W, int H, int stride, int ch, uint32_t flags)
{
    DPX_CHECK(p != nullptr, DPX_EINVAL, "null image pointer");
    DPX_CHECK(W > 0 && H > 0 && W <= 32768 && H <= 32768, DPX_EINVAL, "bad frame size %dx%d", W, H);
    DPX_CHECK((flags & ~kKnownFlags) == 0, DPX_EINVAL, "unknown flags 0x%x", flags & ~kKnownFlags);
    DPX_CHECK(!(flags & DPX_INDEXED), DPX_EINVAL, "indexed frames: batched and serving paths only");
    DPX_CHECK(ch == 3 || ch == 4, DPX_EINVAL, "channels must be 3 or 4, got %d", ch);
    DPX_CHECK(stride >= W * ch, DPX_EINVAL, "stride %d < width*channels %d", stride, W * ch);
    return DPX_OK;
}

}  // namespace

// -------------------------------------------------------------------------
// stage entry points
// -------------------------------------------------------------------------
extern "C" int dpx_stage_similarity_graph(const uint8_t* d_img, int W, int H, int stride, int ch, uint32_t flags,
                                          uint8_t* d_graph, void* stream)
{
    if (int rc = check_img(d_img, W, H, stride, ch, flags)) return rc;
    DPX_CHECK(d_graph, DPX_EINVAL, "null graph pointer");
    ImgView im{ d_img, W, H, stride, ch, flags };
    hipLaunchKernelGGL(k_graph, grid2(W, H), dim3(kB, kB), 0, as_stream(stream), im, d_graph);
    DPX_HIP(hipGetLastError());
    return DPX_OK;
}

extern "C" int dpx_stage_trivial_cross(uint8_t* d_graph, int W, int H, void* stream)
{
    DPX_CHECK(d_graph && W > 0 && H > 0, DPX_EINVAL, "bad arguments");
    hipLaunchKernelGGL(k_trivial, grid2(W, H), dim3(kB, kB), 0, as_stream(stream), d_graph, W, H);
    DPX_HIP(hipGetLastError());
    return DPX_OK;
}

extern "C" int dpx_stage_heuristic_cross(uint8_t* d_graph, uint8_t* d_graph_aux, int W, int H, void* stream)
{
    DPX_CHECK(d_graph && d_graph_aux && W > 0 && H > 0, DPX_EINVAL, "bad arguments");
    DPX_HIP(hipMemcpyAsync(d_graph_aux, d_graph, (size_t)W * H, hipMemcpyDeviceToDevice, as_stream(stream)));
    hipLaunchKernelGGL(k_heuristic, grid2(W, H), dim3(kB, kB), 0, as_stream(stream), d_graph, d_graph_aux, W, H);
    DPX_HIP(hipGetLastError());
    return DPX_OK;
}

extern "C" int dpx_stage_cells(const uint8_t* d_graph, int W, int H, dpx_point* d_diagram, int32_t* d_edge_count,
                               void* stream)
{
    DPX_CHECK(d_graph && d_diagram && d_edge_count && W > 0 && H > 0, DPX_EINVAL, "bad arguments");
    const size_t N = (size_t)W * H;
    hipLaunchKernelGGL(k_cells, dim3((unsigned)((N + kRun - 1) / kRun)), dim3(256), 0, as_stream(stream), d_graph, N,
                       d_diagram, d_edge_count);
    DPX_HIP(hipGetLastError());
    return DPX_OK;
}

extern "C" int dpx_stage_subdivide(const uint8_t* d_img, int W, int H, int stride, int ch, uint32_t flags,
                                   const uint8_t* d_graph, dpx_point* d_diagram, dpx_point* d_diagram_aux,
                                   int32_t* d_edge_count, int32_t* d_edge_count_aux, void* stream)
{
    if (int rc = check_img(d_img, W, H, stride, ch, flags)) return rc;
    DPX_CHECK(d_graph && d_diagram && d_diagram_aux && d_edge_count && d_edge_count_aux, DPX_EINVAL,
              "bad arguments");
    size_t N = (size_t)W * H;
    hipStream_t s = as_stream(stream);
    DPX_HIP(hipMemcpyAsync(d_diagram_aux, d_diagram, N * kCellSize * sizeof(dpx_point), hipMemcpyDeviceToDevice, s));
    DPX_HIP(hipMemcpyAsync(d_edge_count_aux, d_edge_count, N * sizeof(int32_t), hipMemcpyDeviceToDevice, s));
    ImgView im{ d_img, W, H, stride, ch, flags };
    const dim3 tiles((unsigned)((W + kSubX - 1) / kSubX), (unsigned)((H + kSubY - 1) / kSubY));
    hipLaunchKernelGGL(k_subdivide, tiles, dim3(256), 0, s, im, d_graph, d_diagram, d_diagram_aux,
                       d_edge_count, d_edge_count_aux);
    DPX_HIP(hipGetLastError());
    return DPX_OK;
}

extern "C" int dpx_stage_triangulate(dpx_point* d_diagram, const int32_t* d_edge_count, int W, int H, void* stream)
{
    DPX_CHECK(d_diagram && d_edge_count && W > 0 && H > 0, DPX_EINVAL, "bad arguments");
    const size_t N = (size_t)W * H;
    hipLaunchKernelGGL(k_triangulate, dim3((unsigned)((N + kTriRun - 1) / kTriRun)), dim3(kTriBlock), 0,
                       as_stream(stream), d_diagram, d_edge_count, W, N);
    DPX_HIP(hipGetLastError());
    return DPX_OK;
}

extern "C" int dpx_stage_export_vbo(const uint8_t* d_img, int W, int H, int stride, int ch, uint32_t flags,
                                    const dpx_point* d_diagram, const int32_t* d_edge_count, dpx_point* d_pos,
                                    dpx_uchar4* d_color, void* stream)
{
    if (int rc = check_img(d_img, W, H, stride, ch, flags)) return rc;
    DPX_CHECK(d_diagram && d_edge_count && (d_pos || d_color), DPX_EINVAL, "bad arguments");
    ImgView im{ d_img, W, H, stride, ch, flags };
    const size_t N = (size_t)W * H;
    hipLaunchKernelGGL(k_export_vbo, dim3((unsigned)((N + kRun - 1) / kRun)), dim3(256), 0, as_stream(stream), im, d_diagram, d_edge_count,
                       d_pos, d_color);
    DPX_HIP(hipGetLastError());
    return DPX_OK;
}

extern "C" int dpx_stage_rasterize(const uint8_t* d_img, int W, int H, int stride, int ch, uint32_t flags,
                                   const dpx_point* d_diagram, const int32_t* d_edge_count, int scale,
                                   uint8_t* d_out, int out_stride, void* stream)
{
    if (int rc = check_img(d_img, W, H, stride, ch, flags)) return rc;
    DPX_CHECK(d_diagram && d_edge_count && d_out, DPX_EINVAL, "bad arguments");
    DPX_CHECK(scale >= 1 && scale <= 32, DPX_EINVAL, "scale %d outside 1..32", scale);
    DPX_CHECK((long long)W * scale <= 65536 && (long long)H * scale <= 65536, DPX_EINVAL, "output too large");
    DPX_CHECK(out_stride >= 4 * W * scale && out_stride % 4 == 0, DPX_EINVAL, "bad out_stride %d", out_stride);
    ImgView im{ d_img, W, H, stride, ch, flags };
    TriGeom v{};
    v.unit = 128 * scale;
    v.step = 128;
    v.ox[0] = v.oy[0] = 64;
    v.W = W * scale;
    v.H = H * scale;
    v.topdown = out_topdown(flags);
    launch_tri(im, d_diagram, d_edge_count, v, 1, d_out, out_stride, as_stream(stream));
    DPX_HIP(hipGetLastError());
    return DPX_OK;
}

extern "C" int dpx_stage_present(const uint8_t* d_img, int W, int H, int stride, int ch, uint32_t flags,
                                 const dpx_point* d_diagram, const int32_t* d_edge_count, const dpx_view* view,
                                 uint8_t* d_out, int out_stride, void* stream)
{
    if (int rc = check_img(d_img, W, H, stride, ch, flags)) return rc;
    DPX_CHECK(view && d_out, DPX_EINVAL, "bad arguments");
    DPX_CHECK(view->mode == DPX_VIEW_CELLS || view->mode == DPX_VIEW_QUADS, DPX_EINVAL, "unknown view mode %d",
              view->mode);
    DPX_CHECK(view->mode == DPX_VIEW_QUADS || (d_diagram && d_edge_count), DPX_EINVAL,
              "the cells view needs the triangulated diagram");
    DPX_CHECK(view->scale_x100 >= 25 && view->scale_x100 <= 3200, DPX_EINVAL, "scale_x100 %d outside 25..3200",
              view->scale_x100);
    DPX_CHECK(view->translate_x >= -65536 && view->translate_x <= 65536 && view->translate_y >= -65536 &&
                  view->translate_y <= 65536,
              DPX_EINVAL, "translation outside -65536..65536");
    DPX_CHECK(view->width >= 1 && view->width <= 16384 && view->height >= 1 && view->height <= 16384, DPX_EINVAL,
              "window %dx%d outside 1..16384", view->width, view->height);
    DPX_CHECK((view->flags & ~(DPX_VIEW_AA | DPX_VIEW_TOPDOWN)) == 0 && view->reserved == 0, DPX_EINVAL,
              "unknown view flags");
    DPX_CHECK(out_stride >= 4 * view->width && out_stride % 4 == 0, DPX_EINVAL, "bad out_stride %d", out_stride);
    ImgView im{ d_img, W, H, stride, ch, flags };
    const bool aa = view->flags & DPX_VIEW_AA;
    TriGeom v{};
    v.unit = 512 * view->scale_x100;
    v.step = 8 * 6400;
    // rotated 4x grid, or the pixel's centre
    const int sox[4] = { 3, 7, 1, 5 }, soy[4] = { 1, 3, 5, 7 };
    for (int s = 0; s < 4; s++) {
        v.ox[s] = ((aa ? sox[s] : 4) - 8LL * view->translate_x) * 6400;
        v.oy[s] = ((aa ? soy[s] : 4) - 8LL * view->translate_y) * 6400;
    }
    v.W = view->width;
    v.H = view->height;
    v.topdown = (view->flags & DPX_VIEW_TOPDOWN) ? 1 : 0;
    v.quads = view->mode == DPX_VIEW_QUADS;
    launch_tri(im, d_diagram, d_edge_count, v, aa ? 4 : 1, d_out, out_stride, as_stream(stream));
    DPX_HIP(hipGetLastError());
    return DPX_OK;
}

extern "C" int dpx_stage_components(const uint8_t* d_graph, int W, int H, int32_t* d_labels, void* stream)
{
    DPX_CHECK(d_graph && d_labels && W > 0 && H > 0, DPX_EINVAL, "bad arguments");
    int N = W * H;
    hipStream_t s = as_stream(stream);
    // d_labels doubles as the parent array, then receives the roots
    const dim3 tiles((unsigned)((W + kCcTile - 1) / kCcTile), (unsigned)((H + kCcTile - 1) / kCcTile));
    hipLaunchKernelGGL(k_cc_tile, tiles, dim3(256), 0, s, d_graph, W, H, d_labels);
    hipLaunchKernelGGL(k_cc_cross, grid2(W, H), dim3(kB, kB), 0, s, d_graph, W, H, d_labels);
    hipLaunchKernelGGL(k_cc_final, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, s, d_labels, d_labels, N);
    DPX_HIP(hipGetLastError());
    return DPX_OK;
}

}  // namespace dpx

// -------------------------------------------------------------------------
// Plain per-frame path: kernel.cu's sequence with per-call allocation,
// blocking copies and one kernel per stage, plus the raster.
// -------------------------------------------------------------------------
namespace {

// A frame's device buffers, in one allocation: each hipMalloc and hipFree
// takes the driver's time, seven of them longer than the kernels.
struct FrameBuffers {
    uint8_t *img = nullptr, *graph = nullptr, *graph_aux = nullptr, *out = nullptr;
    dpx_point *diagram = nullptr, *diagram_aux = nullptr;
    int32_t *ec = nullptr, *ec_aux = nullptr;
    uint8_t* all = nullptr;
    ~FrameBuffers() { (void)hipFree(all); }
};

// Runs the stages up to triangulation on a frame already in fb.img.
int run_stages(FrameBuffers& fb, int W, int H, int stride, int ch, uint32_t flags, bool subdivide)
{
    using namespace dpx;
    size_t N = (size_t)W * H;
    if (int rc = dpx_stage_similarity_graph(fb.img, W, H, stride, ch, flags, fb.graph, nullptr)) return rc;
    if (int rc = dpx_stage_trivial_cross(fb.graph, W, H, nullptr)) return rc;
    if (int rc = dpx_stage_heuristic_cross(fb.graph, fb.graph_aux, W, H, nullptr)) return rc;
    if (int rc = dpx_stage_cells(fb.graph, W, H, fb.diagram, fb.ec, nullptr)) return rc;
    if (subdivide) {
        if (int rc = dpx_stage_subdivide(fb.img, W, H, stride, ch, flags, fb.graph, fb.diagram, fb.diagram_aux, fb.ec,
                                         fb.ec_aux, nullptr))
            return rc;
    }
    if (int rc = dpx_stage_triangulate(fb.diagram, fb.ec, W, H, nullptr)) return rc;
    (void)N;
    return DPX_OK;
}

int alloc_frame(FrameBuffers& fb, int W, int H, int stride, bool subdivide, size_t out_bytes)
{
    const size_t N = (size_t)W * H;
    size_t bytes = 0;
    auto place = [&](size_t n) {
        const size_t at = bytes;
        bytes += (n + 255) / 256 * 256;
        return at;
    };
    const size_t img = place((size_t)stride * H), graph = place(N), graph_aux = place(N);
    const size_t diagram = place(N * dpx::kCellSize * sizeof(dpx_point)), ec = place(N * sizeof(int32_t));
    const size_t diagram_aux = place(subdivide ? N * dpx::kCellSize * sizeof(dpx_point) : 0);
    const size_t ec_aux = place(subdivide ? N * sizeof(int32_t) : 0), out = place(out_bytes);
    DPX_HIP(hipMalloc(&fb.all, bytes));
    fb.img = fb.all + img;
    fb.graph = fb.all + graph;
    fb.graph_aux = fb.all + graph_aux;
    fb.diagram = reinterpret_cast<dpx_point*>(fb.all + diagram);
    fb.ec = reinterpret_cast<int32_t*>(fb.all + ec);
    fb.diagram_aux = reinterpret_cast<dpx_point*>(fb.all + diagram_aux);
    fb.ec_aux = reinterpret_cast<int32_t*>(fb.all + ec_aux);
    fb.out = fb.all + out;
    return DPX_OK;
}

}  // namespace

extern "C" int dpx_frame(const uint8_t* img, int W, int H, int stride, int ch, const dpx_params* params,
                         uint8_t* out_rgba, int out_stride, uint8_t* graph_out, int32_t* edge_count_out,
                         dpx_point* diagram_out)
{
    using namespace dpx;
    DPX_CHECK(params, DPX_EINVAL, "null params");
    if (int rc = check_img(img, W, H, stride, ch, params->flags)) return rc;
    DPX_CHECK(params->reserved == 0, DPX_EINVAL, "reserved must be 0");
    if (int rc = require_device()) return rc;
    int scale = params->scale;
    bool sub = params->subdivide != 0;
    if (out_rgba) {
        DPX_CHECK(scale >= 1 && scale <= 32, DPX_EINVAL, "scale %d outside 1..32", scale);
        DPX_CHECK(out_stride >= 4 * W * scale, DPX_EINVAL, "bad out_stride %d", out_stride);
    }
    size_t N = (size_t)W * H;
    FrameBuffers fb;
    if (int rc = alloc_frame(fb, W, H, stride, sub, out_rgba ? (size_t)out_stride * H * scale : 0)) return rc;
    DPX_HIP(hipMemcpy(fb.img, img, (size_t)stride * H, hipMemcpyHostToDevice));
    if (int rc = run_stages(fb, W, H, stride, ch, params->flags, sub)) return rc;
    if (out_rgba) {
        if (int rc = dpx_stage_rasterize(fb.img, W, H, stride, ch, params->flags, fb.diagram, fb.ec, scale, fb.out,
                                         out_stride, nullptr))
            return rc;
    }
    DPX_HIP(hipDeviceSynchronize());
    if (out_rgba) DPX_HIP(download(out_rgba, fb.out, (size_t)out_stride * H * scale));
    if (graph_out) DPX_HIP(hipMemcpy(graph_out, fb.graph, N, hipMemcpyDeviceToHost));
    if (edge_count_out) DPX_HIP(hipMemcpy(edge_count_out, fb.ec, N * sizeof(int32_t), hipMemcpyDeviceToHost));
    if (diagram_out) DPX_HIP(download(diagram_out, fb.diagram, N * kCellSize * sizeof(dpx_point)));
    return DPX_OK;
}

extern "C" dpx_point* launch_kernel(dpx_point* pos, dpx_uchar4* colorPos, float time, char* img_data, int img_width,
                                    int img_height, int img_widthstep, int* edge_count_h, char* graph_h,
                                    bool subdivide)
{
    using namespace dpx;
    (void)time;
    int W = img_width, H = img_height;
    if (check_img(img_data, W, H, img_widthstep, 3, 0) || require_device()) return nullptr;
    size_t N = (size_t)W * H;
    FrameBuffers fb;
    if (alloc_frame(fb, W, H, img_widthstep, subdivide, 0)) return nullptr;
    if (hipMemcpy(fb.img, img_data, (size_t)img_widthstep * H, hipMemcpyHostToDevice) != hipSuccess) {
        fail(DPX_EHIP, "image upload failed");
        return nullptr;
    }
    if (run_stages(fb, W, H, img_widthstep, 3, 0, subdivide)) return nullptr;
    if (pos || colorPos) {
        if (dpx_stage_export_vbo(fb.img, W, H, img_widthstep, 3, 0, fb.diagram, fb.ec, pos, colorPos, nullptr))
            return nullptr;
    }
    if (hipDeviceSynchronize() != hipSuccess) {
        fail(DPX_EHIP, "device error in the stage kernels");
        return nullptr;
    }
    dpx_point* diagram_h = (dpx_point*)malloc(N * kCellSize * sizeof(dpx_point));
    if (!diagram_h) {
        fail(DPX_ENOMEM, "host allocation of the diagram failed");
        return nullptr;
    }
    bool ok = true;
    if (edge_count_h)
        ok = ok && hipMemcpy(edge_count_h, fb.ec, N * sizeof(int32_t), hipMemcpyDeviceToHost) == hipSuccess;
    ok = ok && download(diagram_h, fb.diagram, N * kCellSize * sizeof(dpx_point)) == hipSuccess;
    if (graph_h) ok = ok && hipMemcpy(graph_h, fb.graph, N, hipMemcpyDeviceToHost) == hipSuccess;
    if (!ok) {
        free(diagram_h);
        fail(DPX_EHIP, "result download failed");
        return nullptr;
    }
    return diagram_h;
}
