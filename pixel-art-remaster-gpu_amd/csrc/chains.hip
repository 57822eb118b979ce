// chains.hip -- border chains of a resolved graph (extractBorderPoints
// cc_functions.cu:348-503): dpx_stage_border_chains.
//
// The definition is a sequential scan: a walk starts at each node, in
// row-major order, that is neither internal (90) nor without links nor
// listed; it leaves by the node's first link clockwise from up-left and at
// each node turns clockwise from the link it came in by.  It is a chain when
// it comes back to its start through the link just counter-clockwise of the
// first one; it is abandoned on an internal, listed or discarded node,
// discarding the node it stepped from.  Chain nodes are listed; an abandoned
// walk leaves its start unlisted (the behaviour that reproduces the chains
// recorded in alex_png.txt:1-21).
//
// Where a walk goes does not depend on the marks: the turn rule gives each
// directed link (node s, link e) one successor (the neighbour t, its first
// link clockwise after 7 - e), and on a symmetric graph that is a
// permutation of the directed links whose cycles are the faces of the
// graph's plane embedding; a link into an internal node has no successor,
// which cuts some cycles into paths.  So the links are ranked first, all in
// parallel, and each path or cycle that holds a start (the first link of a
// node) becomes an array of its links' nodes in walk order: a walk is a
// contiguous range of one array.
//
// Which walks run, and where they stop, is then found as a fixpoint instead
// of in scan order.  Give every mark the start of the walk that made it as
// its time.  A walk from s stops at the first node whose mark time is below
// s, and does not run at all when s was listed at a time below s, so the
// outcome of a walk depends on walks of smaller s only: the equations have
// one solution, the sequential scan's, and any iteration that re-evaluates
// what a change can reach arrives at it (by induction over s: once all
// smaller walks are final and seen, s is final at its next evaluation).
// The unit that is evaluated is a path, not a walk: the walks of one path in
// order of s, against the other paths' marks of the round before
// (k_bc_sim).  Most dependences lie inside a path, so few rounds are needed:
// 6 for a 256x224 frame, 14 for a 640x480 one, the last of them on a few
// dozen paths.  k_bc_spread then hands the changed nodes' mark times to the
// other paths through those nodes, and marks a path for the next round only
// if a time changed that one of its walks compares with (below the path's
// last walk `send`); `tau` is the smallest such time, and the next
// evaluation keeps what the walks up to it did.
//
// Bound: the chain of rounds, each two launches of a few microseconds, and
// the ranking's launches in front of them; bytes and arithmetic are small
// (640x480: 272 k links of 12 B).  Measured, against one wave that took the
// walks in scan order (a microsecond a walk): dithered 640x480 frames 6.3 ->
// 0.4-1.2 ms, one in eight, with a face of thousands of abandoned walks, 9-13 ->
// 3.1-3.9 ms; 256x224 game frames 0.60-1.64 -> 0.27-0.80 ms; 64x48 0.29 -> 0.16;
// game frames of 1280x960 39-99 -> 4-42 ms, dithered ones 45-50 -> 1.5-1.6.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <utility>

#include "common.hpp"
#include "geom.hpp"
#include "graph.hpp"

namespace dpx {
namespace {

constexpr int32_t kInf = 0x7FFFFFFF;        // "never" for mark times
constexpr uint32_t kCycle = 0x80000000u;    // flag beside a path's length and on a cycle's ranking key
constexpr uint32_t kStartBit = 0x80000000u; // flag beside a position's node: the node's first link
constexpr int kShort = 512;                 // positions of a path that one wave holds in registers
constexpr int kLong = 8192;                 // positions of a path that fit a block's LDS
constexpr int kSimBlock = 512;
// Frames of more nodes are refused without an aligned scratch (include/depixel.h), though none is used.
constexpr uint32_t kScratchUnalignedNodes = 622336;
constexpr int kGridRounds = 8;  // rounds as launches over the machine; k_bc_finish does the rest

inline size_t round256(size_t v) { return (v + 255) / 256 * 256; }

// Counters (ints, cleared by k_bc_clear).
enum {
    kStatus = 0,   // DPX_EINVAL: a link leaves the frame or has no reverse link
    kLinks = 1,    // directed links of walkable nodes
    kPlaces = 2,   // positions of the path arrays handed out
    kPaths = 3,    // paths with starts
    kLongs = 4,    // ... of more than kShort positions
    kRanked = 8,   // one flag per ranking launch: it changed something
    kWaiting = 32,  // one flag per round: short paths wait for it
    kWaitingLong = kWaiting + kGridRounds + 1,  // long paths waiting, per evaluation of them
    kCounters = kWaitingLong + kGridRounds + 2
};

// Ranking state of a directed link: x = the link 2^k steps on, key = the
// smallest key seen on the way (a path's last link has the smallest: its id
// without kCycle, and points at itself), dist = steps to that link.
struct BcLink {
    uint32_t x, key, dist;
};

// Device arrays.  Per link of a walkable node (id base[node] + rank of the
// link among the node's): apos, its position (-1: its path has no start).
// Per position: A = node | kStartBit, ph = path, E = smallest time at which
// another path marks the node, m = time at which this path does, ring = the
// next position of the same node on this path, T = work times of paths
// beyond kLong.  Per path: off, len (| kCycle), ct = time of its chain, send
// (above), tau (kInf: not waiting), cnt = starts of a long path, S[off ..] =
// their positions in order of the start.  Per node: base, xl = time at which
// a path other than the one it starts on lists it.
struct Bc {
    const uint8_t* g;
    int W, H;
    uint32_t N;
    int32_t* ctr;
    uint32_t* base;
    int32_t* xl;
    int32_t* nflag;   // node changed in this round
    int32_t* nlist;   // k_bc_finish: the changed nodes
    int32_t* dshort;  // k_bc_finish: the short paths that wait
    int32_t* dlong;   // the long paths that wait
    int32_t* longs;   // all long paths
    int32_t *off, *ct, *send, *tau, *cnt;
    uint32_t* len;
    int32_t* apos;
    uint32_t* A;
    int32_t *ph, *E, *m, *ring, *S;
    uint32_t* T;
    BcLink *SA, *SB;
};

__device__ inline bool walkable(uint32_t v) { return v != 0u && v != 90u; }
__device__ inline int link_rank(uint32_t v, int e) { return __builtin_popcount(v & ((1u << e) - 1u)); }

// id of the successor of link (s, e); the link itself at the end of a path
__device__ inline uint32_t bc_succ(const Bc& b, uint32_t s, int e, uint32_t id)
{
    const uint32_t t = s + edy(e) * b.W + edx(e), vt = b.g[t];
    return vt == 90u ? id : b.base[t] + link_rank(vt, cw_turn(vt, 7 - e, +1));
}

// Exclusive prefix of v over a block of BLOCK threads; *total: the sum.
template <int BLOCK>
__device__ inline uint64_t block_prefix(uint64_t v, uint64_t* total)
{
    __shared__ uint64_t s_wave[BLOCK / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint64_t incl = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint64_t t = __shfl_up(incl, d);
        if (lane >= d) incl += t;
    }
    __syncthreads();  // (an earlier call's reads of s_wave)
    if (lane == 63) s_wave[wave] = incl;
    __syncthreads();
    uint64_t before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < BLOCK / 64; w++) {
        const uint64_t t = s_wave[w];
        if (w < wave) before += t;
        all += t;
    }
    *total = all;
    return before + incl - v;
}

__global__ void k_bc_clear(int32_t* ctr)
{
    for (int k = threadIdx.x; k < kCounters; k += blockDim.x) ctr[k] = 0;
}

// Checks the links and gives the links of each block's nodes a range of ids.
constexpr int kNodeBlock = 1024;
__global__ __launch_bounds__(kNodeBlock) void k_bc_base(Bc b)
{
    const uint32_t s = blockIdx.x * (uint32_t)kNodeBlock + threadIdx.x;
    __shared__ uint32_t s_base;
    uint32_t deg = 0;
    if (s < b.N) {
        const uint32_t v = b.g[s];
        if (walkable(v)) {
            deg = __builtin_popcount(v);
            const int i = (int)(s % (uint32_t)b.W), j = (int)(s / (uint32_t)b.W);
            bool ok = true;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                if (!bit(v, e)) continue;
                const int ni = i + edx(e), nj = j + edy(e);
                if ((unsigned)ni >= (unsigned)b.W || (unsigned)nj >= (unsigned)b.H) ok = false;
                else ok = ok && bit(b.g[(uint32_t)nj * (uint32_t)b.W + (uint32_t)ni], 7 - e);
            }
            if (!ok) b.ctr[kStatus] = DPX_EINVAL;
        }
        b.xl[s] = kInf;
        b.nflag[s] = 0;
    }
    uint64_t total;
    const uint64_t before = block_prefix<kNodeBlock>(deg, &total);
    if (threadIdx.x == 0) s_base = (uint32_t)atomicAdd(&b.ctr[kLinks], (int)total);
    __syncthreads();
    if (s < b.N) b.base[s] = s_base + (uint32_t)before;
}

__global__ __launch_bounds__(256) void k_bc_link(Bc b)
{
    const uint32_t s = blockIdx.x * 256u + threadIdx.x;
    if (s >= b.N || b.ctr[kStatus] != 0) return;
    const uint32_t v = b.g[s];
    if (!walkable(v)) return;
    uint32_t id = b.base[s];
#pragma unroll
    for (int e = 0; e < 8; e++) {
        if (!bit(v, e)) continue;
        const uint32_t nx = bc_succ(b, s, e, id);
        b.SA[id] = BcLink{ nx, nx == id ? id : id | kCycle, 0u };
        b.apos[id] = 0;
        id++;
    }
}

// Three rounds of pointer jumping (each link composed with the state it
// points to seven times).  A state covers `len` steps; launch `r` does
// nothing once a launch changed no key: every state is then final in both
// buffers (keys that no further window of `len` steps lowers anywhere on a
// cycle are its smallest; on a path some link still reaches the end as long
// as one does not).
__global__ __launch_bounds__(256) void k_bc_jump(Bc b, const BcLink* __restrict__ in, BcLink* __restrict__ out,
                                                 uint32_t len, int r)
{
    if (b.ctr[kStatus] != 0 || (r > 0 && b.ctr[kRanked + r - 1] == 0)) return;
    const uint32_t n = (uint32_t)b.ctr[kLinks];
    bool changed = false;
    for (uint64_t id = blockIdx.x * 256ull + threadIdx.x; id < n; id += gridDim.x * 256ull) {
        BcLink st = in[id];
        const uint32_t key = st.key;
#pragma unroll
        for (int h = 1; h < 8; h++) {
            const BcLink x = in[st.x];
            if (x.key < st.key) {
                st.key = x.key;
                st.dist = (uint32_t)h * len + x.dist;
            }
            st.x = x.x;
        }
        out[id] = st;
        changed = changed || st.key != key;
    }
    if (changed) b.ctr[kRanked + r] = 1;
}

// Paths that hold a start: flagged at their last link (a cycle's: its
// smallest), in apos until k_bc_place writes that.
__global__ __launch_bounds__(256) void k_bc_starts(Bc b, const BcLink* __restrict__ F)
{
    const uint32_t s = blockIdx.x * 256u + threadIdx.x;
    if (s >= b.N || b.ctr[kStatus] != 0) return;
    const uint32_t v = b.g[s];
    if (!walkable(v)) return;
    b.apos[F[b.base[s] + link_rank(v, cw_first_link(v))].key & ~kCycle] = 1;
}

// Each path with a start takes a number and its range of positions, both
// block by block; info[last link] = (offset, length | kCycle, path or -1).
// The path is known by its first link (its predecessor, the link that turns
// into it from the neighbour across the link just counter-clockwise, belongs
// to an internal node), the cycle by its smallest.
__global__ __launch_bounds__(kNodeBlock) void k_bc_heads(Bc b, const BcLink* __restrict__ F, BcLink* __restrict__ info)
{
    const uint32_t s = blockIdx.x * (uint32_t)kNodeBlock + threadIdx.x;
    __shared__ uint32_t s_place, s_path;
    const uint32_t v = s < b.N && b.ctr[kStatus] == 0 ? b.g[s] : 0u;
    // (bit e: link e is the head of a path with a start)
    uint32_t heads = 0, id0 = 0, n_paths = 0;
    uint64_t n_places = 0;
    auto length = [&](int e, uint32_t id, const BcLink& st) -> uint32_t {
        return st.key & kCycle ? F[bc_succ(b, s, e, id)].dist + 1u : st.dist + 1u;
    };
    if (walkable(v)) {
        id0 = b.base[s];
    }
    if (walkable(v)) {
        uint32_t id = id0;
        BcLink sts[8];
        int has[8];
#pragma unroll
        for (int e = 0; e < 8; e++)
            if (bit(v, e)) sts[e] = F[id0 + link_rank(v, e)];
#pragma unroll
        for (int e = 0; e < 8; e++)
            if (bit(v, e)) has[e] = b.apos[sts[e].key & ~kCycle];
#pragma unroll
        for (int e = 0; e < 8; e++) {
            if (!bit(v, e)) continue;
            const BcLink st = sts[e];
            bool head;
            if (st.key & kCycle) {
                head = st.key == (id | kCycle);
            } else {
                const int a = cw_turn(v, e, -1);
                head = b.g[s + edy(a) * b.W + edx(a)] == 90u;
            }
            if (head) {
                const uint32_t last = st.key & ~kCycle;
                if (has[e]) {
                    heads |= 1u << e;
                    n_paths++;
                    n_places += length(e, id, st);
                } else {
                    info[last] = BcLink{ 0u, 0u, 0xFFFFFFFFu };
                }
            }
            id++;
        }
    }
    uint64_t all_places, all_paths;
    const uint64_t place = block_prefix<kNodeBlock>(n_places, &all_places);
    const uint64_t path = block_prefix<kNodeBlock>(n_paths, &all_paths);
    if (threadIdx.x == 0 && all_paths) {
        s_place = (uint32_t)atomicAdd(&b.ctr[kPlaces], (int)all_places);
        s_path = (uint32_t)atomicAdd(&b.ctr[kPaths], (int)all_paths);
    }
    __syncthreads();
    if (!heads) return;
    uint32_t off = s_place + (uint32_t)place, p = s_path + (uint32_t)path;
    for (int e = 0; e < 8; e++) {
        if (!bit(heads, e)) continue;
        const uint32_t id = id0 + link_rank(v, e);
        const BcLink st = F[id];
        const uint32_t L = length(e, id, st);
        info[st.key & ~kCycle] = BcLink{ off, L | (st.key & kCycle), p };
        b.off[p] = (int32_t)off;
        b.len[p] = L | (st.key & kCycle);
        b.ct[p] = kInf;
        b.send[p] = -1;
        b.tau[p] = -1;
        if (L > (uint32_t)kShort) b.longs[atomicAdd(&b.ctr[kLongs], 1)] = (int32_t)p;
        off += L;
        p++;
    }
}

// Every link takes its place in its path.
__global__ __launch_bounds__(256) void k_bc_place(Bc b, const BcLink* __restrict__ F, const BcLink* __restrict__ info)
{
    const uint32_t s = blockIdx.x * 256u + threadIdx.x;
    if (s >= b.N || b.ctr[kStatus] != 0) return;
    const uint32_t v = b.g[s];
    if (!walkable(v)) return;
    const int fl = cw_first_link(v);
    uint32_t id = b.base[s];
#pragma unroll
    for (int e = 0; e < 8; e++) {
        if (!bit(v, e)) continue;
        const BcLink st = F[id], inf = info[st.key & ~kCycle];
        int32_t a = -1;
        if (inf.dist != 0xFFFFFFFFu) {
            a = (int32_t)(inf.x + (inf.key & ~kCycle) - 1u - st.dist);
            b.A[a] = s | (e == fl ? kStartBit : 0u);
            b.ph[a] = (int32_t)inf.dist;
        }
        b.apos[id] = a;
        id++;
    }
}

// The links of one node: positions and paths (-1: none), n of them.
struct NodeLinks {
    int32_t a[8], p[8];
};
__device__ inline void node_links(const Bc& b, uint32_t s, uint32_t n, NodeLinks& k)
{
    const uint32_t id = b.base[s];
#pragma unroll
    for (uint32_t q = 0; q < 8; q++) k.a[q] = q < n ? b.apos[id + q] : -1;
#pragma unroll
    for (uint32_t q = 0; q < 8; q++) k.p[q] = k.a[q] >= 0 ? b.ph[k.a[q]] : -1;
}

// Times and rings (over the ranking's buffers, which are done with).
__global__ __launch_bounds__(256) void k_bc_times(Bc b)
{
    const uint32_t s = blockIdx.x * 256u + threadIdx.x;
    if (s >= b.N || b.ctr[kStatus] != 0) return;
    const uint32_t v = b.g[s];
    if (!walkable(v)) return;
    NodeLinks k;
    node_links(b, s, __builtin_popcount(v), k);
#pragma unroll
    for (int q = 0; q < 8; q++) {
        if (k.a[q] < 0) continue;
        int next = k.a[q];  // the next link of the same path after q, wrapping
#pragma unroll
        for (int d = 7; d >= 1; d--) {
            const int o = (q + d) & 7;
            if (k.p[o] == k.p[q]) next = k.a[o];
        }
        b.ring[k.a[q]] = next;
        b.m[k.a[q]] = kInf;
        b.E[k.a[q]] = kInf;
    }
}

// The starts of each long path in order of their nodes: a bitmap of a window
// of nodes in LDS, each set bit's rank counted from the words before it.
constexpr int kSortWords = 16384, kSortBlock = 1024;
__global__ __launch_bounds__(kSortBlock) void k_bc_sort(Bc b)
{
    __shared__ uint32_t s_bits[kSortWords];
    __shared__ uint32_t s_lo, s_hi;
    if (b.ctr[kStatus] != 0) return;
    const int n_long = b.ctr[kLongs], t = threadIdx.x;
    for (int q = blockIdx.x; q < n_long; q += gridDim.x) {
        const int p = b.longs[q];
        const uint32_t off = (uint32_t)b.off[p], L = b.len[p] & ~kCycle;
        __syncthreads();
        if (t == 0) {
            s_lo = 0xFFFFFFFFu;
            s_hi = 0u;
        }
        __syncthreads();
        uint32_t lo = 0xFFFFFFFFu, hi = 0u;
        for (uint32_t k = t; k < L; k += kSortBlock) {
            const uint32_t a = b.A[off + k];
            if (!(a & kStartBit)) continue;
            lo = min(lo, a & ~kStartBit);
            hi = max(hi, a & ~kStartBit);
        }
        atomicMin(&s_lo, lo);
        atomicMax(&s_hi, hi);
        __syncthreads();
        lo = s_lo;
        hi = s_hi;
        uint64_t done = 0;  // starts written
        constexpr uint32_t SPAN = kSortWords * 32u;
        for (uint32_t w0 = lo / 32u * 32u; w0 <= hi; w0 += SPAN) {
            for (int k = t; k < kSortWords; k += kSortBlock) s_bits[k] = 0u;
            __syncthreads();
            for (uint32_t k = t; k < L; k += kSortBlock) {
                const uint32_t a = b.A[off + k], s = a & ~kStartBit;
                if ((a & kStartBit) && s >= w0 && s - w0 < SPAN) atomicOr(&s_bits[(s - w0) >> 5], 1u << ((s - w0) & 31u));
            }
            __syncthreads();
            constexpr int PER = kSortWords / kSortBlock;
            uint32_t n = 0;
#pragma unroll
            for (int k = 0; k < PER; k++) n += __builtin_popcount(s_bits[t * PER + k]);
            uint64_t total;
            uint64_t at = done + block_prefix<kSortBlock>(n, &total);
            for (int k = 0; k < PER; k++) {
                uint32_t w = s_bits[t * PER + k];
                while (w) {
                    b.S[off + at++] = (int32_t)(w0 + (uint32_t)(t * PER + k) * 32u + __builtin_ctz(w));
                    w &= w - 1u;
                }
            }
            done += total;
            __syncthreads();
        }
        for (uint32_t k = t; k < (uint32_t)done; k += kSortBlock) {  // the nodes' positions
            const uint32_t s = (uint32_t)b.S[off + k], v = b.g[s];
            b.S[off + k] = b.apos[b.base[s] + link_rank(v, cw_first_link(v))] - (int32_t)off;
        }
        if (t == 0) b.cnt[p] = (int32_t)done;
    }
}

// The smallest v of the wave, in every lane's result.
__device__ inline int wave_min(int v)
{
#define DPX_DPP_MIN(ctrl, rows) v = min(v, __builtin_amdgcn_update_dpp(kInf, v, ctrl, rows, 0xF, false))
    DPX_DPP_MIN(0x111, 0xF);  // row_shr:1, 2, 4, 8: lane 15 of each row holds its row's
    DPX_DPP_MIN(0x112, 0xF);
    DPX_DPP_MIN(0x114, 0xF);
    DPX_DPP_MIN(0x118, 0xF);
    DPX_DPP_MIN(0x142, 0xA);  // row_bcast:15, 31
    DPX_DPP_MIN(0x143, 0xC);
#undef DPX_DPP_MIN
    return __builtin_amdgcn_readlane(v, 63);
}

__device__ inline int32_t take_tau(const Bc& b, int p, int lane)
{
    // (set by atomics of another launch or wave, so read as one)
    const int32_t tau = __hip_atomic_load(&b.tau[p], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (lane == 0) __hip_atomic_store(&b.tau[p], kInf, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return tau;
}

// Where an evaluation leaves the nodes whose times it changed: a flag each
// (k_bc_spread looks at every node's), or also a list (k_bc_finish).
struct NoteFlag {
    __device__ void operator()(const Bc& b, int node) const { b.nflag[node] = 1; }
};
struct NoteList {
    int* n;
    __device__ void operator()(const Bc& b, int node) const
    {
        if (atomicExch(&b.nflag[node], 1) == 0) b.nlist[atomicAdd(n, 1)] = node;
    }
};

// One path of at most 64 J positions, one wave: position lane + 64 j in
// registers.  The next walk is the smallest start left; the first marked
// position after its place is the smallest distance over the lanes.
template <int J, class Note>
__device__ inline void sim_short(const Bc& b, int p, uint32_t off, uint32_t len, Note note)
{
    const int lane = threadIdx.x & 63, L = (int)(len & ~kCycle);
    const bool cyc = len & kCycle;
    const int32_t tau = take_tau(b, p, lane), old_ct = b.ct[p];
    int node[J], tm[J], own[J], st[J], was[J], last = -1;
#pragma unroll
    for (int j = 0; j < J; j++) {
        const int q = lane + 64 * j;
        node[j] = -1;
        tm[j] = own[j] = st[j] = was[j] = kInf;
        if (q < L) {
            const uint32_t a = b.A[off + q];
            node[j] = (int)(a & ~kStartBit);
            tm[j] = b.E[off + q];
            was[j] = b.m[off + q];
            if (a & kStartBit) {
                last = max(last, node[j]);
                if (node[j] > tau && !(b.xl[node[j]] < node[j])) st[j] = node[j];
            }
            if (was[j] <= tau) {
                own[j] = was[j];
                tm[j] = min(tm[j], own[j]);
            }
        }
    }
    int ct = old_ct <= tau ? old_ct : kInf;
    for (int walk = 0; walk < L && ct == kInf; walk++) {  // (at most a start a position)
        int s = st[0];
#pragma unroll
        for (int j = 1; j < J; j++) s = min(s, st[j]);
        s = wave_min(s);
        if (s == kInf) break;
        int P = kInf;  // the start's place
#pragma unroll
        for (int j = 0; j < J; j++)
            if (st[j] == s) {
                P = lane + 64 * j;
                st[j] = kInf;
            }
        P = wave_min(P);
        int d = kInf;  // steps past the node after it to the first marked one
#pragma unroll
        for (int j = 0; j < J; j++) {
            const int q = lane + 64 * j;
            int dq = q - P - 1;
            if (dq < 0) dq += cyc ? L : kInf;  // (q = P itself: L - 1 or more, never the smallest below n)
            if (tm[j] < s && q != P) d = min(d, dq);
        }
        d = wave_min(d);
        const int n = cyc ? L - 1 : L - 1 - P;
        if (d >= n && cyc) {
            ct = s;
            break;
        }
        int prev = P + min(d, n);  // the node before the marked one, or the path's last
        if (prev >= L) prev -= L;
        int v = node[0];
#pragma unroll
        for (int j = 1; j < J; j++)
            if ((prev >> 6) == j) v = node[j];
        v = __builtin_amdgcn_readlane(v, prev & 63);
#pragma unroll
        for (int j = 0; j < J; j++)
            if (node[j] == v) {
                own[j] = min(own[j], s);
                tm[j] = min(tm[j], s);
            }
    }
#pragma unroll
    for (int j = 0; j < J; j++) {
        const int q = lane + 64 * j;
        if (q >= L) continue;
        const int now = min(own[j], ct);
        if (now != was[j]) b.m[off + q] = now;
        if (now != was[j] || ct != old_ct) note(b, node[j]);
    }
    last = -wave_min(-last);
    if (lane == 0) {
        b.ct[p] = ct;
        b.send[p] = ct != kInf ? ct : last;
    }
}

// One path of any length, one block of threads.  Positions' times are kept
// as time << 1 | (1: not this path's own mark).  Wave 0 takes the walks in
// order of their starts.  Up to kLong positions the times lie in LDS with the
// smallest of each 64, so that a walk of any length is three LDS reads: the
// 64 positions around its start, the minima, the 64 positions that hold the
// first marked one (cycles of 6,000 positions with 3,000 walks of 250 steps
// are met in 640x480 frames).  Beyond, the times lie in T and the LDS holds
// the smallest of each 64 << shift of them, and of each 64 of those: a walk is
// two reads of T around LDS reads.  (Game frames of 1280x960 and up have faces
// of 30,000 positions and thousands of walks of that length: reading T ahead
// of each walk, through device-scope atomics, 1280x960 took 50 to 108 ms and
// 1920x1080 7 to 141.)
struct LongLds {
    uint32_t tm[kLong];  // times, or beyond kLong positions the smallest of each 64 << shift
    uint16_t ring[kLong];
    uint32_t bm[kLong / 64];
    int ct;
};

__device__ inline void wave_settle()  // this wave's LDS writes are seen by its next reads
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The place of the first position after P, n of them (wrapping), whose time
// is below st; -1: none.  On the entries of tm.
__device__ inline int first_marked(const LongLds& s, int P, bool cyc, uint32_t st)
{
    const int lane = threadIdx.x & 63, B = P >> 6, pl = P & 63;
    static_assert(kLong / 64 == 128, "two minima a lane");
    const uint64_t own = __ballot((s.tm[64 * B + lane] >> 1) < st);
    const uint64_t after = pl == 63 ? 0ull : own & (~0ull << (pl + 1));
    if (after) return 64 * B + __builtin_ctzll(after);
    const uint64_t m0 = __ballot((s.bm[lane] >> 1) < st), m1 = __ballot((s.bm[64 + lane] >> 1) < st);
    // blocks after B, then (on a cycle) those before it
    auto above = [](uint64_t m, int k) { return k >= 63 ? 0ull : k < 0 ? m : m & (~0ull << (k + 1)); };
    auto below = [](uint64_t m, int k) { return k <= 0 ? 0ull : k >= 64 ? m : m & ((1ull << k) - 1ull); };
    int blk = -1;
    if (const uint64_t a0 = above(m0, B)) blk = __builtin_ctzll(a0);
    else if (const uint64_t a1 = above(m1, B - 64)) blk = 64 + __builtin_ctzll(a1);
    else if (cyc) {
        if (const uint64_t b0 = below(m0, B)) blk = __builtin_ctzll(b0);
        else if (const uint64_t b1 = below(m1, B - 64)) blk = 64 + __builtin_ctzll(b1);
        else {  // what is left of P's own 64
            const uint64_t before = below(own, pl);
            return before ? 64 * B + __builtin_ctzll(before) : -1;
        }
    }
    if (blk < 0) return -1;
    return 64 * blk + __builtin_ctzll(__ballot((s.tm[64 * blk + lane] >> 1) < st));
}

template <bool LDS, int THREADS, class Note>
__device__ inline void sim_long(const Bc& b, int p, uint32_t off, uint32_t len, LongLds& s, Note note)
{
    const int t = threadIdx.x, lane = t & 63, L = (int)(len & ~kCycle);
    const bool cyc = len & kCycle;
    __syncthreads();  // (the block's path before: its LDS, its tau)
    const int32_t tau = __hip_atomic_load(&b.tau[p], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), old_ct = b.ct[p];
    // (T is this block's alone until the kernel ends, and written anew by every evaluation)
    uint32_t* tg = b.T + off;
    auto get = [&](int q) -> uint32_t {
        if constexpr (LDS) return s.tm[q];
        else return __hip_atomic_load(&tg[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    auto put = [&](int q, uint32_t v) {
        if constexpr (LDS) s.tm[q] = v;
        else __hip_atomic_store(&tg[q], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    auto ring = [&](int q) -> int {
        if constexpr (LDS) return s.ring[q];
        else return b.ring[off + q] - (int)off;
    };
    int sb = 6;  // positions of an entry of minima: 1 << sb
    if constexpr (!LDS) {
        while ((uint32_t)(L - 1) >> sb >= (uint32_t)kLong) sb++;
        for (int k = t; k < kLong; k += THREADS) s.tm[k] = 0xFFFFFFFEu;
        __syncthreads();
    }
    const int L64 = (L + 63) / 64 * 64;
    for (int q = t; q < L64; q += THREADS) {  // (whole waves)
        uint32_t v = 0xFFFFFFFFu;
        if (q < L) {
            v = (uint32_t)b.E[off + q] << 1 | 1u;
            const int32_t was = b.m[off + q];
            if (was <= tau) v = min(v, (uint32_t)was << 1);
            if constexpr (LDS) s.ring[q] = (uint16_t)(b.ring[off + q] - (int32_t)off);
            else put(q, v);
        }
        if constexpr (LDS) s.tm[q] = v;
        const uint32_t low = (uint32_t)wave_min((int)(v >> 1)) << 1;
        if (lane == 0) {
            if constexpr (LDS) s.bm[q >> 6] = low;
            else atomicMin(&s.tm[q >> sb], low);
        }
    }
    if constexpr (LDS) {
        for (int k = L64 / 64 + t; k < kLong / 64; k += THREADS) s.bm[k] = 0xFFFFFFFEu;
    } else {
        __syncthreads();
        for (int k = t; k < kLong; k += THREADS) {  // (whole waves)
            const uint32_t low = (uint32_t)wave_min((int)(s.tm[k] >> 1)) << 1;
            if (lane == 0) s.bm[k >> 6] = low;
        }
    }
    __syncthreads();
    if (t < 64) {
        int ct = old_ct <= tau ? old_ct : kInf;
        const int cnt = b.cnt[p];
        // (the next 64 starts are loaded while the ones before run)
        int pos = lane < cnt ? b.S[off + lane] : 0;
        int node = (int)(b.A[off + pos] & ~kStartBit), xl = b.xl[node];
        for (int k = 0; k < cnt && ct == kInf; k += 64) {
            const int cpos = pos, cnode = node, cxl = xl;
            if (k + 64 < cnt) {
                pos = k + 64 + lane < cnt ? b.S[off + k + 64 + lane] : 0;
                node = (int)(b.A[off + pos] & ~kStartBit);
                xl = b.xl[node];
            }
            uint64_t todo = __ballot(k + lane < cnt && cnode > tau && !(cxl < cnode));
            while (todo) {
                const int w = __builtin_ctzll(todo);
                todo &= todo - 1;
                const uint32_t st = (uint32_t)__builtin_amdgcn_readlane(cnode, w);
                const int P = __builtin_amdgcn_readlane(cpos, w);
                int h = -1;  // the first marked position of the walk
                if constexpr (LDS) {
                    h = first_marked(s, P, cyc, st);
                } else {
                    // the first position in lo .. hi - 1 whose time is below st
                    auto scan = [&](int lo, int hi) {
                        for (int c = lo & ~63; c < hi; c += 64) {
                            const int q = c + lane;
                            if (const uint64_t hit = __ballot(q >= lo && q < hi && (get(q) >> 1) < st))
                                return c + (int)__builtin_ctzll(hit);
                        }
                        return -1;
                    };
                    auto end = [&](int e) { return (int)min((uint32_t)L, (uint32_t)(e + 1) << sb); };
                    const int own = P >> sb;
                    h = scan(P + 1, end(own));
                    if (h < 0) {
                        const int blk = first_marked(s, own, cyc, st);
                        if (blk >= 0) h = scan(blk << sb, end(blk));
                        else if (cyc) h = scan(own << sb, P);
                    }
                }
                if (h < 0 && cyc) {
                    ct = (int)st;
                    break;
                }
                const int prev = h < 0 ? L - 1 : h == 0 ? L - 1 : h - 1;
                int q = prev;
                do {  // (uniform: every place of the node on this path)
                    const uint32_t v = get(q);
                    if (lane == 0 && (st << 1) < v) {
                        put(q, st << 1);
                        if constexpr (LDS) {
                            s.bm[q >> 6] = min(s.bm[q >> 6], st << 1);
                        } else {
                            const int e = q >> sb;
                            s.tm[e] = min(s.tm[e], st << 1);
                            s.bm[e >> 6] = min(s.bm[e >> 6], st << 1);
                        }
                    }
                    q = ring(q);
                } while (q != prev);
                wave_settle();
            }
        }
        if (lane == 0) {
            const int pl = b.S[off + cnt - 1];
            s.ct = ct;
            b.ct[p] = ct;
            b.send[p] = ct != kInf ? ct : (int)(b.A[off + pl] & ~kStartBit);
            __hip_atomic_store(&b.tau[p], kInf, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    __syncthreads();
    const int ct = s.ct;
    for (int q = t; q < L; q += THREADS) {
        const uint32_t v = get(q);
        const int now = min((v & 1u) ? kInf : (int)(v >> 1), ct), was = b.m[off + q];
        if (now != was) b.m[off + q] = now;
        if (now != was || ct != old_ct) note(b, (int)(b.A[off + q] & ~kStartBit));
    }
}

template <int THREADS, class Note>
__device__ inline void sim_path_long(const Bc& b, int p, LongLds& s, Note note)
{
    const uint32_t off = (uint32_t)b.off[p], len = b.len[p];
    if ((len & ~kCycle) <= (uint32_t)kLong) sim_long<true, THREADS>(b, p, off, len, s, note);
    else sim_long<false, THREADS>(b, p, off, len, s, note);
}

template <class Note>
__device__ inline void sim_path_short(const Bc& b, int p, Note note)
{
    const uint32_t off = (uint32_t)b.off[p], len = b.len[p];
    if ((len & ~kCycle) <= 64u) sim_short<1>(b, p, off, len, note);
    else sim_short<kShort / 64>(b, p, off, len, note);
}

// Is path p short, and waiting to be evaluated?
__device__ inline bool short_waits(const Bc& b, int p)
{
    return (b.len[p] & ~kCycle) <= (uint32_t)kShort &&
           __hip_atomic_load(&b.tau[p], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != kInf;
}

// Round r: the short paths that wait (in round 0 all of them), kChunk of them
// looked at by a wave, and with slot >= 0 the long ones (slot 0: all).
// Evaluating a long path of thousands of walks takes as long as many rounds
// of the others, whose first rounds change what it sees, so it waits for
// some of them: rounds 0, 1, 4 and 7, then whenever no short path waits
// (640x480: 2-3 evaluations in place of 7-9).
// A wave evaluates the paths of its chunk one after another, 4 us each and
// more: with chunks of 8 a round of a 640x480 frame took 38 us, of 2 it takes
// 11 to 31 (of 1: no better, twice the waves).  Rounds without long paths need
// no LDS and fill the machine.
constexpr int kChunk = 2;
constexpr bool long_round(int r) { return r <= 1 || r % 3 == 1; }
template <bool LONG>
__global__ __launch_bounds__(kSimBlock) void k_bc_sim(Bc b, int r, int slot)
{
    if (b.ctr[kStatus] != 0) return;
    if constexpr (LONG) {
        __shared__ LongLds s;
        const int n_long = slot == 0 ? b.ctr[kLongs] : b.ctr[kWaitingLong + slot];
        for (int k = blockIdx.x; k < n_long; k += gridDim.x)
            sim_path_long<kSimBlock>(b, slot == 0 ? b.longs[k] : b.dlong[k], s, NoteFlag{});
    }
    if (r > 0 && b.ctr[kWaiting + r] == 0) return;
    constexpr int WAVES = kSimBlock / 64;
    const int n = b.ctr[kPaths], lane = threadIdx.x & 63;
    for (int k = (blockIdx.x + (threadIdx.x >> 6) * gridDim.x) * kChunk; k < n; k += gridDim.x * WAVES * kChunk) {
        uint64_t todo = __ballot(lane < kChunk && k + lane < n && short_waits(b, k + lane));
        while (todo) {
            const int p = __builtin_amdgcn_readfirstlane(k + (int)__builtin_ctzll(todo));
            todo &= todo - 1;
            sim_path_short(b, p, NoteFlag{});
        }
    }
}

// A changed node's times, handed to the paths through it; wait(p): path p's
// inputs changed where it looks, and it was not waiting yet.
template <class Wait>
__device__ inline void spread_node(const Bc& b, int s, Wait wait)
{
    const uint32_t v = b.g[s];
    const int fr = link_rank(v, cw_first_link(v));
    NodeLinks k;
    node_links(b, (uint32_t)s, __builtin_popcount(v), k);
    int m[8], ct[8], e_old[8], send[8];
#pragma unroll
    for (int q = 0; q < 8; q++) {
        m[q] = k.a[q] >= 0 ? b.m[k.a[q]] : kInf;
        e_old[q] = k.a[q] >= 0 ? b.E[k.a[q]] : kInf;
        ct[q] = k.p[q] >= 0 ? b.ct[k.p[q]] : kInf;
        send[q] = k.p[q] >= 0 ? b.send[k.p[q]] : -1;
    }
    const int x_old = b.xl[s];
#pragma unroll
    for (int q = 0; q < 8; q++) {
        if (k.a[q] < 0) continue;
        int e_new = kInf, x_new = kInf;
#pragma unroll
        for (int o = 0; o < 8; o++)
            if (k.p[o] != k.p[q]) {
                e_new = min(e_new, m[o]);
                x_new = min(x_new, ct[o]);
            }
        int tau = kInf;
        if (e_new != e_old[q]) {
            b.E[k.a[q]] = e_new;
            if (min(e_new, e_old[q]) < send[q]) tau = min(e_new, e_old[q]);
        }
        if (q == fr && x_new != x_old) {
            b.xl[s] = x_new;
            if ((x_new < s) != (x_old < s) && s <= send[q]) tau = min(tau, s - 1);
        }
        if (tau != kInf && atomicMin(&b.tau[k.p[q]], tau) == kInf) wait(k.p[q]);
    }
    b.nflag[s] = 0;
}

// After round r: every node whose flag is set (after round 0 all of them).
__global__ __launch_bounds__(256) void k_bc_spread(Bc b, int r, int slot)
{
    const uint32_t s = blockIdx.x * 256u + threadIdx.x;
    if (s >= b.N || b.ctr[kStatus] != 0) return;
    if (r == 0 ? !walkable(b.g[s]) : b.nflag[s] == 0) return;
    bool any = false;
    spread_node(b, (int)s, [&](int p) {
        if ((b.len[p] & ~kCycle) > (uint32_t)kShort) b.dlong[atomicAdd(&b.ctr[kWaitingLong + slot], 1)] = p;
        else any = true;
    });
    if (any) b.ctr[kWaiting + r + 1] = 1;
}

// The rounds that are left, in one block: on few paths a block's barrier
// costs less than a launch.  Ends when no path waits: among the short paths
// every round makes at least the smallest walk that is not final (for what the
// long ones last did) so, and each evaluation of the long ones the smallest of
// all.  Frames take a few dozen rounds; paths that still wait after max_rounds
// leave no chains and a status.
constexpr int kFinishBlock = 1024;
__global__ __launch_bounds__(kFinishBlock) void k_bc_finish(Bc b, int slot, uint32_t max_rounds)
{
    __shared__ LongLds s;
    __shared__ int s_short, s_long, s_nodes;
    if (b.ctr[kStatus] != 0) return;
    const int t = threadIdx.x;
    if (t == 0) {
        s_short = 0;
        s_long = b.ctr[kWaitingLong + slot];
    }
    __syncthreads();
    if (b.ctr[kWaiting + kGridRounds])
        for (int p = t, n = b.ctr[kPaths]; p < n; p += kFinishBlock)
            if (short_waits(b, p)) b.dshort[atomicAdd(&s_short, 1)] = p;
    __syncthreads();
    int n_short = s_short, n_long = s_long;
    for (uint32_t round = 0; (n_short | n_long) && round < max_rounds; round++) {  // (uniform)
        __syncthreads();
        if (t == 0) {
            s_nodes = s_short = 0;
            s_long = n_short ? n_long : 0;
        }
        __syncthreads();
        const NoteList note{ &s_nodes };
        if (n_short) {
            for (int k = t >> 6; k < n_short; k += kFinishBlock / 64)
                sim_path_short(b, __builtin_amdgcn_readfirstlane(b.dshort[k]), note);
        } else {
            for (int k = 0; k < n_long; k++) sim_path_long<kFinishBlock>(b, b.dlong[k], s, note);
        }
        __syncthreads();
        for (int k = t; k < s_nodes; k += kFinishBlock)
            spread_node(b, b.nlist[k], [&](int p) {
                if ((b.len[p] & ~kCycle) > (uint32_t)kShort) b.dlong[atomicAdd(&s_long, 1)] = p;
                else b.dshort[atomicAdd(&s_short, 1)] = p;
            });
        __syncthreads();
        n_short = s_short;
        n_long = s_long;
    }
    if (t == 0 && (n_short | n_long)) b.ctr[kStatus] = DPX_EHIP;
}

// The chain a node starts: its length (0: none), its place and its path's range.
__device__ inline uint32_t chain_at(const Bc& b, uint32_t s, uint32_t* off, uint32_t* pos)
{
    if (s >= b.N) return 0u;
    const uint32_t v = b.g[s];
    if (!walkable(v)) return 0u;
    const int a = b.apos[b.base[s] + link_rank(v, cw_first_link(v))];
    const int p = b.ph[a];
    if (b.ct[p] != (int)s) return 0u;
    *off = (uint32_t)b.off[p];
    *pos = (uint32_t)a - *off;
    return b.len[p] & ~kCycle;
}

// Chains and chain nodes of each block of nodes, then of the blocks before it.
__global__ __launch_bounds__(kNodeBlock) void k_bc_count(Bc b, uint64_t* __restrict__ sums)
{
    if (b.ctr[kStatus] != 0) return;
    uint32_t off, pos;
    const uint32_t L = chain_at(b, blockIdx.x * (uint32_t)kNodeBlock + threadIdx.x, &off, &pos);
    uint64_t chains, nodes;
    block_prefix<kNodeBlock>(L ? 1u : 0u, &chains);
    block_prefix<kNodeBlock>(L, &nodes);
    if (threadIdx.x == 0) {
        sums[2 * blockIdx.x] = chains;
        sums[2 * blockIdx.x + 1] = nodes;
    }
}

__global__ __launch_bounds__(kNodeBlock) void k_bc_sums(Bc b, uint64_t* __restrict__ sums, uint32_t n_blocks,
                                                        int max_nodes, int max_chains, int32_t* __restrict__ counts)
{
    const int status = b.ctr[kStatus];
    uint64_t chains = 0, nodes = 0;
    for (uint32_t k0 = 0; k0 < n_blocks && status == 0; k0 += kNodeBlock) {
        const uint32_t k = k0 + threadIdx.x;
        const uint64_t c = k < n_blocks ? sums[2 * k] : 0u, n = k < n_blocks ? sums[2 * k + 1] : 0u;
        uint64_t tc, tn;
        const uint64_t bc = block_prefix<kNodeBlock>(c, &tc), bn = block_prefix<kNodeBlock>(n, &tn);
        if (k < n_blocks) {
            sums[2 * k] = chains + bc;
            sums[2 * k + 1] = nodes + bn;
        }
        chains += tc;
        nodes += tn;
    }
    if (threadIdx.x == 0) {  // (where not all fit, k_bc_write counts those that do)
        const bool fit = chains <= (uint64_t)max_chains && nodes <= (uint64_t)max_nodes;
        counts[0] = fit ? (int32_t)chains : 0;
        counts[1] = fit ? (int32_t)nodes : 0;
        counts[2] = status != 0 ? status : fit ? 0 : DPX_ENOMEM;
    }
}

// The chains in scan order.  Those that fit the caller's arrays are a prefix.
__global__ __launch_bounds__(kNodeBlock) void k_bc_write(Bc b, const uint64_t* __restrict__ sums,
                                                         int32_t* __restrict__ nodes, int32_t* __restrict__ sizes,
                                                         int max_nodes, int max_chains, int32_t* __restrict__ counts)
{
    __shared__ uint32_t s_off[kNodeBlock], s_pos[kNodeBlock], s_len[kNodeBlock], s_at[kNodeBlock];
    if (b.ctr[kStatus] != 0) return;
    const int t = threadIdx.x;
    uint32_t off = 0, pos = 0;
    const uint32_t L = chain_at(b, blockIdx.x * (uint32_t)kNodeBlock + t, &off, &pos);
    uint64_t tc, tn;
    const uint64_t c0 = block_prefix<kNodeBlock>(L ? 1u : 0u, &tc), n0 = block_prefix<kNodeBlock>(L, &tn);
    const uint64_t c = sums[2 * blockIdx.x] + c0, n = sums[2 * blockIdx.x + 1] + n0;
    const bool fits = L && c < (uint64_t)max_chains && n + L <= (uint64_t)max_nodes;
    if (L) {
        s_off[c0] = off;
        s_pos[c0] = pos;
        s_len[c0] = fits ? L : 0u;
        s_at[c0] = (uint32_t)n;
        if (fits) {
            sizes[c] = (int32_t)L;
            if (counts[2] == DPX_ENOMEM) {  // the prefix's last has the largest of both
                atomicMax(&counts[0], (int)c + 1);
                atomicMax(&counts[1], (int)(n + L));
            }
        }
    }
    __syncthreads();
    // short chains by waves, long ones by the block
    for (uint32_t k = t >> 6; k < (uint32_t)tc; k += kNodeBlock / 64) {
        const uint32_t len = s_len[k];
        if (len > 512u) continue;
        for (uint32_t q = t & 63; q < len; q += 64) {
            uint32_t a = s_pos[k] + q;
            if (a >= len) a -= len;
            nodes[s_at[k] + q] = (int32_t)(b.A[s_off[k] + a] & ~kStartBit);
        }
    }
    for (uint32_t k = 0; k < (uint32_t)tc; k++) {
        const uint32_t len = s_len[k];
        if (len <= 512u) continue;
        for (uint32_t q = t; q < len; q += kNodeBlock) {
            uint32_t a = s_pos[k] + q;
            if (a >= len) a -= len;
            nodes[s_at[k] + q] = (int32_t)(b.A[s_off[k] + a] & ~kStartBit);
        }
    }
}

}  // namespace

// dpx_stage_border_chains with a bound on k_bc_finish's rounds (not part of
// the interface: the test of what happens at the bound calls it).
extern "C" int dpx_internal_border_chains(const uint8_t* d_graph, int W, int H, uint8_t* d_scratch, int32_t* d_nodes,
                                          int max_nodes, int32_t* d_sizes, int max_chains, int32_t* d_counts,
                                          void* stream, uint32_t max_rounds)
{
    DPX_CHECK(d_graph && d_scratch && d_nodes && d_sizes && d_counts && W > 0 && H > 0, DPX_EINVAL,
              "bad arguments");
    DPX_CHECK((int64_t)W * H <= (1 << 28), DPX_EINVAL, "frame too large (%dx%d)", W, H);
    DPX_CHECK(max_nodes >= 0 && max_chains >= 0, DPX_EINVAL, "negative capacity");
    const hipStream_t s = as_stream(stream);
    const uint32_t N = (uint32_t)W * (uint32_t)H;
    const size_t E = 8 * (size_t)N;
    // (the scratch's contract, include/depixel.h)
    DPX_CHECK(N <= kScratchUnalignedNodes || reinterpret_cast<uintptr_t>(d_scratch) % 4 == 0, DPX_EINVAL,
              "d_scratch must be 4-byte aligned for a frame of %dx%d", W, H);
    // working memory, in stream order
    const uint32_t node_blocks = (N + kNodeBlock - 1) / kNodeBlock;
    const size_t szLink = round256(E * 4), szRank = round256(E * sizeof(BcLink)), szNode = round256((size_t)N * 4),
                 szLong = round256((E / kShort + 1) * 4), szSums = round256((size_t)node_blocks * 16);
    const size_t szTimes = std::max(2 * szRank, 5 * szLink);
    const size_t bytes = szTimes + 3 * szLink + 11 * szNode + 2 * szLong + szSums + round256(4 * kCounters);
    uint8_t* work = nullptr;
    DPX_HIP(hipMallocAsync(reinterpret_cast<void**>(&work), bytes, s));
    struct FreeAfter {  // freed in stream order on every return below
        void* p;
        hipStream_t s;
        ~FreeAfter() { (void)hipFreeAsync(p, s); }
    } free_after{ work, s };
    uint8_t* at = work;
    auto take = [&](size_t n) {
        uint8_t* p = at;
        at += n;
        return p;
    };
    auto ints = [&](size_t n) { return reinterpret_cast<int32_t*>(take(n)); };
    Bc b{};
    b.g = d_graph;
    b.W = W;
    b.H = H;
    b.N = N;
    // the ranking's buffers (2 x 12 bytes a link), and over them the positions' times
    b.SA = reinterpret_cast<BcLink*>(take(szTimes));
    b.SB = reinterpret_cast<BcLink*>(work + szRank);
    b.E = reinterpret_cast<int32_t*>(work);
    b.m = reinterpret_cast<int32_t*>(work + szLink);
    b.ring = reinterpret_cast<int32_t*>(work + 2 * szLink);
    b.S = reinterpret_cast<int32_t*>(work + 3 * szLink);
    b.T = reinterpret_cast<uint32_t*>(work + 4 * szLink);
    b.apos = ints(szLink);
    b.A = reinterpret_cast<uint32_t*>(take(szLink));
    b.ph = ints(szLink);
    b.base = reinterpret_cast<uint32_t*>(take(szNode));
    b.xl = ints(szNode);
    b.nflag = ints(szNode);
    b.nlist = ints(szNode);
    b.dshort = ints(szNode);
    b.off = ints(szNode);
    b.len = reinterpret_cast<uint32_t*>(take(szNode));
    b.ct = ints(szNode);
    b.send = ints(szNode);
    b.tau = ints(szNode);
    b.cnt = ints(szNode);
    b.dlong = ints(szLong);
    b.longs = ints(szLong);
    uint64_t* sums = reinterpret_cast<uint64_t*>(take(szSums));
    b.ctr = ints(round256(4 * kCounters));

    const dim3 per_node((N + 255) / 256), per_block(node_blocks);
    const dim3 per_link((unsigned)std::min<size_t>((E + 255) / 256, 2048));
    const dim3 sims((unsigned)std::min<uint32_t>((N + kSimBlock / 64 * kChunk - 1) / (kSimBlock / 64 * kChunk), 768));
    hipLaunchKernelGGL(k_bc_clear, dim3(1), dim3(64), 0, s, b.ctr);
    hipLaunchKernelGGL(k_bc_base, per_block, dim3(kNodeBlock), 0, s, b);
    hipLaunchKernelGGL(k_bc_link, per_node, dim3(256), 0, s, b);
    BcLink *cur = b.SA, *oth = b.SB;
    int launches = 0;
    for (uint64_t len = 1; len < E; len *= 8) {
        hipLaunchKernelGGL(k_bc_jump, per_link, dim3(256), 0, s, b, cur, oth, (uint32_t)len, launches++);
        std::swap(cur, oth);
    }
    // (E = 8 N >= 8: at least one launch; the states are in `cur`)
    hipLaunchKernelGGL(k_bc_starts, per_node, dim3(256), 0, s, b, cur);
    hipLaunchKernelGGL(k_bc_heads, per_block, dim3(kNodeBlock), 0, s, b, cur, oth);
    hipLaunchKernelGGL(k_bc_place, per_node, dim3(256), 0, s, b, cur, oth);
    hipLaunchKernelGGL(k_bc_times, per_node, dim3(256), 0, s, b);
    hipLaunchKernelGGL(k_bc_sort, dim3((unsigned)std::min<size_t>(E / kShort + 1, 256)), dim3(kSortBlock), 0, s, b);
    int slot = 0;  // of the long paths that wait
    for (int r = 0; r < kGridRounds; r++) {
        if (long_round(r)) hipLaunchKernelGGL(k_bc_sim<true>, sims, dim3(kSimBlock), 0, s, b, r, slot++);
        else hipLaunchKernelGGL(k_bc_sim<false>, sims, dim3(kSimBlock), 0, s, b, r, -1);
        hipLaunchKernelGGL(k_bc_spread, per_node, dim3(256), 0, s, b, r, slot);
    }
    hipLaunchKernelGGL(k_bc_finish, dim3(1), dim3(kFinishBlock), 0, s, b, slot, max_rounds);
    hipLaunchKernelGGL(k_bc_count, per_block, dim3(kNodeBlock), 0, s, b, sums);
    hipLaunchKernelGGL(k_bc_sums, dim3(1), dim3(kNodeBlock), 0, s, b, sums, node_blocks, max_nodes, max_chains,
                       d_counts);
    hipLaunchKernelGGL(k_bc_write, per_block, dim3(kNodeBlock), 0, s, b, sums, d_nodes, d_sizes, max_nodes, max_chains,
                       d_counts);
    DPX_HIP(hipGetLastError());
    return DPX_OK;
}

extern "C" int dpx_stage_border_chains(const uint8_t* d_graph, int W, int H, uint8_t* d_scratch, int32_t* d_nodes,
                                       int max_nodes, int32_t* d_sizes, int max_chains, int32_t* d_counts,
                                       void* stream)
{
    // (W H is checked there; twice the nodes and one more, far beyond what any graph has been seen to take)
    return dpx_internal_border_chains(d_graph, W, H, d_scratch, d_nodes, max_nodes, d_sizes, max_chains, d_counts, stream,
                                      2u * (uint32_t)W * (uint32_t)H + 1u);
}

}  // namespace dpx
