// stages.hip -- the per-stage kernels (one kernel per stage of kernel.cu's
// sequence, intermediates in HBM in the reference's formats), the stage entry
// points of the C ABI, the plain per-frame path and the launch_kernel drop-in.
//
// Launch shape: 16x16 threads, one thread per pixel (or per output pixel for
// the raster).  These kernels favour a direct mapping of the reference's data
// formats over speed; the batched path in fused.hip is the fast one.
#include <stdlib.h>
#include <string.h>

#include "common.hpp"
#include "geom.hpp"
#include "graph.hpp"
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

// cells_Kernel (kernel.cu:192-213): hull points in 45-slot cells.  Slots past
// the closing point are written as (0,0).
__global__ void k_cells(const uint8_t* __restrict__ graph, int W, int H, dpx_point* __restrict__ diagram,
                        int32_t* __restrict__ edge_count)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    int j = blockIdx.y * blockDim.y + threadIdx.y;
    if (i >= W || j >= H) return;
    size_t N = (size_t)W * H, idx = (size_t)j * W + i;
    uint32_t left = idx > 0 ? graph[idx - 1] : 0u;
    uint32_t right = idx + 1 < N ? graph[idx + 1] : 0u;
    int hx[2 * kMaxPts], hy[2 * kMaxPts];
    int n = cell_hull(cell_key(graph[idx], left, right), hx, hy);
    dpx_point* c = &diagram[idx * kCellSize];
    for (int t = 0; t < kCellSize; t++) {
        dpx_point p;
        p.x = t <= n ? 0.25f * (float)hx[t] : 0.0f;
        p.y = t <= n ? 0.25f * (float)hy[t] : 0.0f;
        c[t] = p;
    }
    edge_count[idx] = n;
}

__device__ inline int load_quarter(const dpx_point* c, int n, int* x, int* y)
{
    for (int t = 0; t < n; t++) {
        x[t] = (int)(c[t].x * 4.0f);
        y[t] = (int)(c[t].y * 4.0f);
    }
    return n;
}

// subdivision_Kernel (kernel.cu:216-261) on the snapshots daux/eaux.
__global__ void k_subdivide(ImgView im, const uint8_t* __restrict__ graph, dpx_point* __restrict__ diagram,
                            const dpx_point* __restrict__ daux, int32_t* __restrict__ edge_count,
                            const int32_t* __restrict__ eaux)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    int j = blockIdx.y * blockDim.y + threadIdx.y;
    int W = im.W;
    if (i >= W || j >= im.H) return;
    int idx = j * W + i;
    uint32_t node = graph[idx];
    if (node == 90) return;  // internal node (kernel.cu:231)
    int n = eaux[idx];
    // subdivide_cell emits up to 2n points into kMaxPoly slots; real hulls
    // have at most 8 vertices, larger caller-supplied counts leave the cell
    if (n < 3 || n > kMaxPoly / 2) return;
    int hx[2 * kMaxPts], hy[2 * kMaxPts];
    load_quarter(&daux[(size_t)idx * kCellSize], n, hx, hy);
    TjView tv = tj_view(im);
    auto nbr = [&](int e, int* lx, int* ly) -> int {
        int q = idx + edy(e) * W + edx(e);
        int ln = eaux[q];
        if (ln > 2 * kMaxPts - 1) ln = 2 * kMaxPts - 1;
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
    edge_count[idx] = m;
}

// triangulate_Kernel (kernel.cu:264-282): ear clipping, then every slot gets
// the pixel offset; unwritten slots stay at the pixel origin.
__global__ void k_triangulate(dpx_point* __restrict__ diagram, const int32_t* __restrict__ edge_count, int W,
                              int H)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    int j = blockIdx.y * blockDim.y + threadIdx.y;
    if (i >= W || j >= H) return;
    size_t idx = (size_t)j * W + i;
    dpx_point* c = &diagram[idx * kCellSize];
    int n = edge_count[idx];
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
    float fi = (float)i, fj = (float)j;
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

// color_kernel (kernel.cu:67-104) + position_kernel (kernel.cu:109-137)
__global__ void k_export_vbo(ImgView im, const dpx_point* __restrict__ diagram, const int32_t* __restrict__ edge_count,
                             dpx_point* __restrict__ pos, dpx_uchar4* __restrict__ color)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    int j = blockIdx.y * blockDim.y + threadIdx.y;
    if (i >= im.W || j >= im.H) return;
    size_t idx = (size_t)j * im.W + i;
    uint32_t rgba = cell_rgba(load_px(im, i, j), colour_channels(im));
    dpx_uchar4 c4;
    c4.x = (uint8_t)(rgba & 0xFF);
    c4.y = (uint8_t)((rgba >> 8) & 0xFF);
    c4.z = (uint8_t)((rgba >> 16) & 0xFF);
    c4.w = (uint8_t)(rgba >> 24);
    int valid = (edge_count[idx] - 2) * 3;
    for (int t = 0; t < kCellSize; t++) {
        size_t s = idx * kCellSize + t;
        if (color) color[s] = c4;
        if (pos) {
            dpx_point p;
            if (t < valid) p = diagram[s];
            else { p.x = -100.0f; p.y = -100.0f; }
            pos[s] = p;
        }
    }
}

// glDrawArrays(GL_TRIANGLES) in VBO order (simpleVBO.cpp:281) as a gather:
// each output pixel takes the colour of the highest-index cell (the last one
// drawn) with a triangle covering its centre.  Cells reach at most 0.34 past
// their unit square, so the 3x3 cells around the pixel are the candidates.
__global__ void k_raster_tri(ImgView im, const dpx_point* __restrict__ diagram, const int32_t* __restrict__ edge_count,
                             int scale, uint8_t* __restrict__ out, int out_stride)
{
    int X = blockIdx.x * blockDim.x + threadIdx.x;
    int Y = blockIdx.y * blockDim.y + threadIdx.y;
    int OW = im.W * scale, OH = im.H * scale;
    if (X >= OW || Y >= OH) return;
    int cx = X / scale, cy = Y / scale;
    uint32_t color = 0xFF000000u;  // clear colour (0,0,0,1), main.cpp:260
    bool done = false;
    for (int dy = 1; dy >= -1 && !done; dy--)
        for (int dx = 1; dx >= -1 && !done; dx--) {
            int ci = cx + dx, cj = cy + dy;
            if (!in_frame(ci, cj, im.W, im.H)) continue;
            size_t k = (size_t)cj * im.W + ci;
            int nt = edge_count[k] - 2;
            if (nt > kCellSize / 3) nt = kCellSize / 3;
            int sx = (2 * X + 1) * 64 - ci * 128 * scale, sy = (2 * Y + 1) * 64 - cj * 128 * scale;
            const dpx_point* c = &diagram[k * kCellSize];
            float fi = (float)ci, fj = (float)cj;
            for (int t = 0; t < nt; t++) {
                int v[6];
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    dpx_point p = c[3 * t + q];
                    v[2 * q] = (int)((p.x - fi) * 64.0f) * 2 * scale;
                    v[2 * q + 1] = (int)((p.y - fj) * 64.0f) * 2 * scale;
                }
                if (tri_covers(v[0], v[1], v[2], v[3], v[4], v[5], sx, sy)) {
                    color = cell_rgba(load_px(im, ci, cj), colour_channels(im));
                    done = true;
                    break;
                }
            }
        }
    int row = out_topdown(im.flags) ? (OH - 1 - Y) : Y;
    *reinterpret_cast<uint32_t*>(out + (size_t)row * out_stride + (size_t)X * 4) = color;
}

// ---------------------------------------------------------------------------
// Presentation: the GLUT window (display() callbacks.cpp:39-72, renderCuda
// simpleVBO.cpp:185-440).  Window point (X + ox/8, Y + oy/8) maps to image
// point ((8 (X - tx) + ox) * 100) / (8 * sc), sc the scale in hundredths.  In
// units of 1/(512 sc) of a cell that is (8 (X - tx) + ox) * 6400 and a
// 1/64-lattice vertex v is 64 v * 8 sc: both integers, so coverage is exact.
// ---------------------------------------------------------------------------
struct ViewGeom {
    int mode, sc, tx, ty, W, H, aa, topdown;
};

__device__ inline long long floor_div(long long a, long long b)  // b > 0
{
    long long q = a / b;
    return (a % b != 0 && a < 0) ? q - 1 : q;
}

// colour of the sample at window position (8 X + ox, 8 Y + oy) / 8
__device__ inline uint32_t present_sample(const ImgView& im, const dpx_point* __restrict__ diagram,
                                          const int32_t* __restrict__ edge_count, const ViewGeom& v, int X, int Y,
                                          int ox, int oy)
{
    const long long unit = 512LL * v.sc;  // one cell
    const long long px = (8LL * (X - v.tx) + ox) * 6400, py = (8LL * (Y - v.ty) + oy) * 6400;
    const long long ci = floor_div(px, unit), cj = floor_div(py, unit);
    const int cc = colour_channels(im);
    if (v.mode == DPX_VIEW_QUADS) {
        // the two triangles of pixel (ci, cj) cover [ci, ci+1) x [cj, cj+1)
        // under the coverage rule (left and bottom edges in, right and top out)
        if (ci < 0 || cj < 0 || ci >= im.W || cj >= im.H) return 0xFF000000u;
        return cell_rgba(load_px(im, (int)ci, (int)cj), cc);
    }
    for (int dy = 1; dy >= -1; dy--)
        for (int dx = 1; dx >= -1; dx--) {  // cells in reverse draw order: the first hit wins
            long long i = ci + dx, j = cj + dy;
            if (i < 0 || j < 0 || i >= im.W || j >= im.H) continue;
            size_t k = (size_t)j * im.W + (size_t)i;
            int nt = edge_count[k] - 2;
            if (nt > kCellSize / 3) nt = kCellSize / 3;
            const long long sx = px - i * unit, sy = py - j * unit;
            const dpx_point* c = &diagram[k * kCellSize];
            const float fi = (float)i, fj = (float)j;
            for (int t = 0; t < nt; t++) {
                long long w[6];
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    dpx_point p = c[3 * t + q];
                    w[2 * q] = (long long)(int)((p.x - fi) * 64.0f) * 8 * v.sc;
                    w[2 * q + 1] = (long long)(int)((p.y - fj) * 64.0f) * 8 * v.sc;
                }
                if (tri_covers(w[0], w[1], w[2], w[3], w[4], w[5], sx, sy))
                    return cell_rgba(load_px(im, (int)i, (int)j), cc);
            }
        }
    return 0xFF000000u;  // clear colour (main.cpp:260)
}

// The four antialiasing samples of window pixel (X, Y) in one scan: the
// cells around all four, in reverse draw order, each triangle read once and
// tested against every sample not yet covered.  A cell reaches at most a
// quarter cell beyond its square, so the cells outside a sample's own 3x3
// never cover it and the first cover found is the sample's last in draw
// order, as in present_sample.
__device__ inline void present_samples4(const ImgView& im, const dpx_point* __restrict__ diagram,
                                        const int32_t* __restrict__ edge_count, const ViewGeom& v, int X, int Y,
                                        const int* sox, const int* soy, uint32_t* col)
{
    const long long unit = 512LL * v.sc;
    long long px[4], py[4];
    long long i0 = 0, i1 = 0, j0 = 0, j1 = 0;
#pragma unroll
    for (int s = 0; s < 4; s++) {
        px[s] = (8LL * (X - v.tx) + sox[s]) * 6400;
        py[s] = (8LL * (Y - v.ty) + soy[s]) * 6400;
        col[s] = 0xFF000000u;  // clear colour (main.cpp:260)
        const long long ci = floor_div(px[s], unit), cj = floor_div(py[s], unit);
        if (s == 0 || ci < i0) i0 = ci;
        if (s == 0 || ci > i1) i1 = ci;
        if (s == 0 || cj < j0) j0 = cj;
        if (s == 0 || cj > j1) j1 = cj;
    }
    // the window may lie far outside the image: clamp to the frame
    j0 = j0 - 1 < 0 ? 0 : j0 - 1;
    i0 = i0 - 1 < 0 ? 0 : i0 - 1;
    j1 = j1 + 1 > im.H - 1 ? im.H - 1 : j1 + 1;
    i1 = i1 + 1 > im.W - 1 ? im.W - 1 : i1 + 1;
    const int cc = colour_channels(im);
    uint32_t left = 0xFu;
    for (long long j = j1; j >= j0 && left; j--)
        for (long long i = i1; i >= i0 && left; i--) {
            size_t k = (size_t)j * im.W + (size_t)i;
            int nt = edge_count[k] - 2;
            if (nt > kCellSize / 3) nt = kCellSize / 3;
            const dpx_point* c = &diagram[k * kCellSize];
            const float fi = (float)i, fj = (float)j;
            long long sx[4], sy[4];
#pragma unroll
            for (int s = 0; s < 4; s++) { sx[s] = px[s] - i * unit; sy[s] = py[s] - j * unit; }
            uint32_t hit = 0;
            for (int t = 0; t < nt && (left & ~hit); t++) {
                long long w[6];
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    dpx_point p = c[3 * t + q];
                    w[2 * q] = (long long)(int)((p.x - fi) * 64.0f) * 8 * v.sc;
                    w[2 * q + 1] = (long long)(int)((p.y - fj) * 64.0f) * 8 * v.sc;
                }
#pragma unroll
                for (int s = 0; s < 4; s++)
                    if (((left & ~hit) >> s) & 1u)
                        if (tri_covers(w[0], w[1], w[2], w[3], w[4], w[5], sx[s], sy[s])) hit |= 1u << s;
            }
            if (hit) {
                const uint32_t rgba = cell_rgba(load_px(im, (int)i, (int)j), cc);
#pragma unroll
                for (int s = 0; s < 4; s++)
                    if ((hit >> s) & 1u) col[s] = rgba;
                left &= ~hit;
            }
        }
}

__global__ void k_present(ImgView im, const dpx_point* __restrict__ diagram, const int32_t* __restrict__ edge_count,
                          ViewGeom v, uint8_t* __restrict__ out, int out_stride)
{
    int X = blockIdx.x * blockDim.x + threadIdx.x;
    int Y = blockIdx.y * blockDim.y + threadIdx.y;
    if (X >= v.W || Y >= v.H) return;
    uint32_t color;
    if (!v.aa) {
        color = present_sample(im, diagram, edge_count, v, X, Y, 4, 4);
    } else {
        // rotated 4x grid, averaged per channel with halves rounded up
        const int sox[4] = { 3, 7, 1, 5 }, soy[4] = { 1, 3, 5, 7 };
        uint32_t sum[4] = { 0, 0, 0, 0 }, cs[4];
        if (v.mode == DPX_VIEW_QUADS) {
#pragma unroll
            for (int s = 0; s < 4; s++) cs[s] = present_sample(im, diagram, edge_count, v, X, Y, sox[s], soy[s]);
        } else {
            present_samples4(im, diagram, edge_count, v, X, Y, sox, soy, cs);
        }
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const uint32_t c = cs[s];
#pragma unroll
            for (int b = 0; b < 4; b++) sum[b] += (c >> (8 * b)) & 0xFFu;
        }
        color = 0;
#pragma unroll
        for (int b = 0; b < 4; b++) color |= ((sum[b] + 2) >> 2) << (8 * b);
    }
    int row = v.topdown ? (v.H - 1 - Y) : Y;
    *reinterpret_cast<uint32_t*>(out + (size_t)row * out_stride + (size_t)X * 4) = color;
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
    hipLaunchKernelGGL(k_cells, grid2(W, H), dim3(kB, kB), 0, as_stream(stream), d_graph, W, H, d_diagram,
                       d_edge_count);
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
    hipLaunchKernelGGL(k_subdivide, grid2(W, H), dim3(kB, kB), 0, s, im, d_graph, d_diagram, d_diagram_aux,
                       d_edge_count, d_edge_count_aux);
    DPX_HIP(hipGetLastError());
    return DPX_OK;
}

extern "C" int dpx_stage_triangulate(dpx_point* d_diagram, const int32_t* d_edge_count, int W, int H, void* stream)
{
    DPX_CHECK(d_diagram && d_edge_count && W > 0 && H > 0, DPX_EINVAL, "bad arguments");
    hipLaunchKernelGGL(k_triangulate, grid2(W, H), dim3(kB, kB), 0, as_stream(stream), d_diagram, d_edge_count, W, H);
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
    hipLaunchKernelGGL(k_export_vbo, grid2(W, H), dim3(kB, kB), 0, as_stream(stream), im, d_diagram, d_edge_count,
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
    hipLaunchKernelGGL(k_raster_tri, grid2(W * scale, H * scale), dim3(kB, kB), 0, as_stream(stream), im, d_diagram,
                       d_edge_count, scale, d_out, out_stride);
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
    ViewGeom v{ view->mode, view->scale_x100, view->translate_x, view->translate_y, view->width, view->height,
                (view->flags & DPX_VIEW_AA) ? 1 : 0, (view->flags & DPX_VIEW_TOPDOWN) ? 1 : 0 };
    hipLaunchKernelGGL(k_present, grid2(v.W, v.H), dim3(kB, kB), 0, as_stream(stream), im, d_diagram, d_edge_count, v,
                       d_out, out_stride);
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

struct FrameBuffers {
    uint8_t *img = nullptr, *graph = nullptr, *graph_aux = nullptr, *out = nullptr;
    dpx_point *diagram = nullptr, *diagram_aux = nullptr, *pos = nullptr;
    int32_t *ec = nullptr, *ec_aux = nullptr;
    ~FrameBuffers()
    {
        (void)hipFree(img);
        (void)hipFree(graph);
        (void)hipFree(graph_aux);
        (void)hipFree(out);
        (void)hipFree(diagram);
        (void)hipFree(diagram_aux);
        (void)hipFree(ec);
        (void)hipFree(ec_aux);
    }
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

int alloc_frame(FrameBuffers& fb, int W, int H, int stride, bool subdivide)
{
    size_t N = (size_t)W * H;
    DPX_HIP(hipMalloc(&fb.img, (size_t)stride * H));
    DPX_HIP(hipMalloc(&fb.graph, N));
    DPX_HIP(hipMalloc(&fb.graph_aux, N));
    DPX_HIP(hipMalloc(&fb.diagram, N * dpx::kCellSize * sizeof(dpx_point)));
    DPX_HIP(hipMalloc(&fb.ec, N * sizeof(int32_t)));
    if (subdivide) {
        DPX_HIP(hipMalloc(&fb.diagram_aux, N * dpx::kCellSize * sizeof(dpx_point)));
        DPX_HIP(hipMalloc(&fb.ec_aux, N * sizeof(int32_t)));
    }
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
    if (int rc = alloc_frame(fb, W, H, stride, sub)) return rc;
    DPX_HIP(hipMemcpy(fb.img, img, (size_t)stride * H, hipMemcpyHostToDevice));
    if (int rc = run_stages(fb, W, H, stride, ch, params->flags, sub)) return rc;
    if (out_rgba) {
        DPX_HIP(hipMalloc(&fb.out, (size_t)out_stride * H * scale));
        if (int rc = dpx_stage_rasterize(fb.img, W, H, stride, ch, params->flags, fb.diagram, fb.ec, scale, fb.out,
                                         out_stride, nullptr))
            return rc;
    }
    DPX_HIP(hipDeviceSynchronize());
    if (out_rgba) DPX_HIP(hipMemcpy(out_rgba, fb.out, (size_t)out_stride * H * scale, hipMemcpyDeviceToHost));
    if (graph_out) DPX_HIP(hipMemcpy(graph_out, fb.graph, N, hipMemcpyDeviceToHost));
    if (edge_count_out) DPX_HIP(hipMemcpy(edge_count_out, fb.ec, N * sizeof(int32_t), hipMemcpyDeviceToHost));
    if (diagram_out)
        DPX_HIP(hipMemcpy(diagram_out, fb.diagram, N * kCellSize * sizeof(dpx_point), hipMemcpyDeviceToHost));
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
    if (alloc_frame(fb, W, H, img_widthstep, subdivide)) return nullptr;
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
    ok = ok && hipMemcpy(diagram_h, fb.diagram, N * kCellSize * sizeof(dpx_point), hipMemcpyDeviceToHost) == hipSuccess;
    if (graph_h) ok = ok && hipMemcpy(graph_h, fb.graph, N, hipMemcpyDeviceToHost) == hipSuccess;
    if (!ok) {
        free(diagram_h);
        fail(DPX_EHIP, "result download failed");
        return nullptr;
    }
    return diagram_h;
}
