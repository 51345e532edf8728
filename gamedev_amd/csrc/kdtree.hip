// k-d tree collision search on gfx950: a left-balanced k-d tree over every collision site and an
// exact top-K query per active owner, the reference's COLLISION_SEARCH=kdtree path.
//
// Reference behaviour followed: the tag-update build of kdtree::buildTree_thrust
// (inc/swarm/kdtree/builder_thrust.h:263-318, 418-526; layout helpers helpers.h:95-300; subtree
// domains builder_common.h:205-240; widest dimension box.h:111-125) and col_cache_get (KD)
// (inc/swarm/_col_cache.cuh:15-71) with the bounded max-heap of idx_old_heap
// (inc/swarm/kdtree/index_heap.cuh:11-177) and the closest-corner-tracking traversal
// (inc/swarm/kdtree/traverse-cct.h:26-100).
//
// Layout: a subtree's pivot is the point of rank `left size` among its points, ordered along its split dimension;
// points that tie there keep the order that the level above gave them, and so on up to the input order (the
// stable one; the reference's thrust::sort is not stable, so its layout for equal coordinates is unspecified).
// That order is a comparison of a point's coordinates, the most recently used split dimension first, and of its
// index at last, so no level has to be sorted: subtrees of more than KD_SLOTS points are split by a radix
// selection of the pivot and a partition in any order, smaller ones are finished in LDS by one block each.
// Query: one lane per active owner, owners taken in Morton order so that neighbouring lanes walk
// similar paths; heap and path are columns of LDS. Rows are written in heap order.
#include "gdx_internal.h"
#include "gdx_device.h"

#include <algorithm>
#include <climits>
#include <cmath>

#pragma clang fp contract(off)

namespace gdx {
namespace {

constexpr int KD_BLOCK = 256;
constexpr int KD_QUERY_BLOCK = 64;
constexpr int KD_ACTIVE = 4;                 // flag beside the split dimension in node.w
constexpr int WAVE = 64;

int blocks(long long n, int per) { return static_cast<int>((n + per - 1) / per); }

__device__ __forceinline__ double ld(const field &f, long long i)
{
    return *reinterpret_cast<const double *>(f.base + i*f.stride);
}

// float coordinate -> unsigned key with the same order (-0 and +0 equal, as the comparison is)
__device__ __forceinline__ uint32_t ordered(float x)
{
    uint32_t u = __float_as_uint(x == 0.0f ? 0.0f : x);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ float pick(int d, float x, float y, float z)
{
    const float v = d == 1 ? y : x;
    return d == 2 ? z : v;
}
__device__ __forceinline__ float coord(const float4 &p, int d) { return pick(d, p.x, p.y, p.z); }

struct kd_box
{
    float lo[3], hi[3];
};

// widest extent; a later dimension wins ties
__device__ __forceinline__ int widest(const kd_box &b)
{
    int best = 0;
    float w_best = 0.0f;
#pragma unroll
    for (int d = 0; d < 3; ++d)
    {
        float w = b.hi[d] - b.lo[d];
        if (w < w_best) continue;
        w_best = w;
        best = d;
    }
    return best;
}

// points left of the pivot of a left-balanced subtree of m points
__host__ __device__ __forceinline__ int kd_left(int m)
{
    if (m < 2) return 0;
    const int levels = 32 - __builtin_clz(static_cast<unsigned int>(m));
    const int half = 1 << (levels - 2);
    const int last = m - ((1 << (levels - 1)) - 1);
    return half - 1 + (last < half ? last : half);
}

// ---------------------------------------------------------------------------------------------
// build
// ---------------------------------------------------------------------------------------------
constexpr int KD_LDS_LEVELS = 12, KD_SLOTS = 1 << KD_LDS_LEVELS;      // largest subtree of the LDS part
constexpr int KD_FINISH_BLOCK = 1024;
constexpr int KD_SPLIT_BLOCK = 512, KD_CHUNK = 4096;
constexpr int KD_BINS = 2048;                                         // 11 bits a digit, three digits a coordinate
constexpr int KD_TIES = 1024;
constexpr int KD_INIT_BLOCKS = 512;
constexpr uint32_t KD_SITE = 0x80000000u;                             // active flag beside the point's index

// a subtree before its split: the box of its domain as ordered keys, its points [start, start + size) and the
// order of its points: split dimension | second << 2 | third << 4, 3 for none
struct kd_seg
{
    uint32_t lo[3], hi[3];
    int start, size, order;
};

// a digit's outcome: leading bits of the pivot's key, its rank among the points that share them, their number
struct kd_sel
{
    uint32_t prefix;
    int rank, count;
};

__device__ __forceinline__ float unordered(uint32_t u)
{
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}

// the order of a subtree's points: its widest dimension, then the dimensions used above it, latest first
__device__ __forceinline__ int order_of(const uint32_t lo[3], const uint32_t hi[3], int above)
{
    kd_box b;
#pragma unroll
    for (int d = 0; d < 3; ++d) { b.lo[d] = unordered(lo[d]); b.hi[d] = unordered(hi[d]); }
    const int dim = widest(b), a0 = above & 3, a1 = (above >> 2) & 3;
    if (dim == a0) return above;
    if (dim == a1) return dim | (a0 << 2) | (above & 0x30);
    return dim | (a0 << 2) | (a1 << 4);
}

// whether p comes before q where they tie in the split dimension
__device__ __forceinline__ bool tie_less(const float4 &p, const float4 &q, int order)
{
#pragma unroll
    for (int k = 2; k < 6; k += 2)
    {
        const int d = (order >> k) & 3;
        if (d == 3) break;
        const uint32_t a = ordered(coord(p, d)), b = ordered(coord(q, d));
        if (a != b) return a < b;
    }
    return (__float_as_uint(p.w) & ~KD_SITE) < (__float_as_uint(q.w) & ~KD_SITE);
}

__device__ __forceinline__ void put_node(const float4 &p, int dim, long long tag, float4 *node, int *idx)
{
    const uint32_t w = __float_as_uint(p.w);
    node[tag] = make_float4(p.x, p.y, p.z, __int_as_float(dim | ((w & KD_SITE) ? KD_ACTIVE : 0)));
    idx[tag] = int(w & ~KD_SITE);
}

__global__ __launch_bounds__(KD_BLOCK) void k_kd_init(const float4 *pts, const unsigned char *active, int n,
                                                     int n_phys, float4 *out, unsigned int *world_bits)
{
    __shared__ unsigned int red[6][KD_BLOCK / WAVE];
    // world box of the data: minima of the ordered keys and of their complements, one atomic per block and bound
    unsigned int k[6] = {~0u, ~0u, ~0u, ~0u, ~0u, ~0u};
    for (long long i = (long long)blockIdx.x*KD_BLOCK + threadIdx.x; i < n; i += (long long)gridDim.x*KD_BLOCK)
    {
        float4 p = pts[i];
        const unsigned int o[3] = {ordered(p.x), ordered(p.y), ordered(p.z)};
#pragma unroll
        for (int d = 0; d < 3; ++d) { k[d] = min(k[d], o[d]); k[3 + d] = min(k[3 + d], ~o[d]); }
        p.w = __uint_as_float(uint32_t(i) | (active[X_WEDGE ? int(i) % n_phys : int(i)] ? KD_SITE : 0u));
        out[i] = p;
    }
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
#pragma unroll
    for (int b = 0; b < 6; ++b)
    {
        unsigned int v = k[b];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v = min(v, static_cast<unsigned int>(__shfl_xor(v, o, WAVE)));
        if (lane == 0) red[b][wave] = v;
    }
    __syncthreads();
    if (threadIdx.x < 6)
    {
        int b = threadIdx.x;
        unsigned int v = red[b][0];
        for (int w = 1; w < KD_BLOCK / WAVE; ++w) v = min(v, red[b][w]);
        atomicMin(world_bits + b, v);
    }
}

__global__ void k_kd_root(const unsigned int *world_bits, int n, float *world, kd_seg *seg)
{
    if (threadIdx.x != 0) return;
    kd_seg g;
    for (int d = 0; d < 3; ++d)
    {
        g.lo[d] = world_bits[d];
        g.hi[d] = ~world_bits[3 + d];
        world[d] = unordered(g.lo[d]);
        world[3 + d] = unordered(g.hi[d]);
    }
    g.start = 0;
    g.size = n;
    g.order = order_of(g.lo, g.hi, 63);
    *seg = g;
}

// the bin that holds rank `rank` of `bins`, by the whole block
template <int BLOCK>
__device__ __forceinline__ kd_sel pick_bin(const unsigned int *bins, int rank)
{
    constexpr int PER = KD_BINS / BLOCK;
    __shared__ int total[BLOCK / WAVE];
    __shared__ kd_sel found;
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
    int c[PER], sum = 0;
#pragma unroll
    for (int k = 0; k < PER; ++k) { c[k] = int(bins[threadIdx.x*PER + k]); sum += c[k]; }
    int incl = sum;
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1)
    {
        const int t = __shfl_up(incl, o, WAVE);
        if (lane >= o) incl += t;
    }
    if (lane == WAVE - 1) total[wave] = incl;
    __syncthreads();
    int before = incl - sum;
    for (int w = 0; w < wave; ++w) before += total[w];
    if (rank >= before && rank < before + sum)
    {
        int k = 0;
        while (rank >= before + c[k]) before += c[k++];
        found.prefix = threadIdx.x*PER + k;
        found.rank = rank - before;
        found.count = c[k];
    }
    __syncthreads();
    return found;
}

// the three digits of a key relative to its subtree's lower bound: the leading 11, the next 11 and the last 10
// bits of the subtree's extent
struct kd_digits
{
    int dim, s1, s2;
    uint32_t lo;
};

__device__ __forceinline__ kd_digits digits_of(const kd_seg *g)
{
    kd_digits k;
    k.dim = g->order & 3;
    k.lo = g->lo[k.dim];
    const int bits = 32 - __clz(static_cast<int>(g->hi[k.dim] - k.lo));
    k.s1 = max(bits - 11, 0);
    k.s2 = max(bits - 22, 0);
    return k;
}

// One digit of the radix selection of every subtree's pivot. bins: [3][segs][KD_BINS], sel: [3][segs]; the blocks
// of digit D each find digit D - 1's bin from its counts, which saves a launch between them. A level of 1e6 points
// takes 6 launches and 37 us, against 300 us for the radix sort of (subtree, coordinate) keys: a selection needs
// three reads of the points and one write, whatever the number of subtrees.
template <int D>
__global__ __launch_bounds__(KD_SPLIT_BLOCK) void k_kd_digit(const float4 *points, const kd_seg *seg, int segs,
                                                            int chunks, unsigned int *bins, kd_sel *sel)
{
    __shared__ unsigned int count[KD_BINS];
    const int s = blockIdx.x / chunks, chunk = blockIdx.x % chunks;
    const int start = seg[s].start, size = seg[s].size;
    if ((long long)chunk*KD_CHUNK >= size) return;
    const kd_digits k = digits_of(seg + s);
    uint32_t prefix = 0;
    if constexpr (D > 0)
    {
        const kd_sel last = D == 1 ? kd_sel{0u, kd_left(size), 0} : sel[s];
        kd_sel now = pick_bin<KD_SPLIT_BLOCK>(bins + ((long long)(D - 1)*segs + s)*KD_BINS, last.rank);
        now.prefix |= D == 1 ? 0u : last.prefix << (k.s1 - k.s2);
        prefix = now.prefix;
        if (chunk == 0 && threadIdx.x == 0) sel[(D - 1)*segs + s] = now;
    }
    for (int b = threadIdx.x; b < KD_BINS; b += KD_SPLIT_BLOCK) count[b] = 0u;
    __syncthreads();
    const int begin = chunk*KD_CHUNK, end = min(begin + KD_CHUNK, size);
    for (int i = begin + threadIdx.x; i < end; i += KD_SPLIT_BLOCK)
    {
        const uint32_t rel = ordered(coord(points[start + i], k.dim)) - k.lo;
        if (D == 0) atomicAdd(count + (rel >> k.s1), 1u);
        else if (D == 1 && rel >> k.s1 == prefix) atomicAdd(count + ((rel >> k.s2) & ((1u << (k.s1 - k.s2)) - 1u)), 1u);
        else if (D == 2 && rel >> k.s2 == prefix) atomicAdd(count + (rel & ((1u << k.s2) - 1u)), 1u);
    }
    __syncthreads();
    unsigned int *const to = bins + ((long long)D*segs + s)*KD_BINS;
    for (int b = threadIdx.x; b < KD_BINS; b += KD_SPLIT_BLOCK)
        if (count[b]) atomicAdd(to + b, count[b]);
}

// points below the pivot's coordinate to the front of their subtree's range, those that tie with it behind them,
// the rest at the end, each part in any order; cursors: [segs][4]
__global__ __launch_bounds__(KD_SPLIT_BLOCK) void k_kd_partition(const float4 *points, const kd_seg *seg, int segs,
                                                                int chunks, const unsigned int *bins, kd_sel *sel,
                                                                int *cursors, float4 *out)
{
    constexpr int PER = KD_CHUNK / KD_SPLIT_BLOCK, WAVES = KD_SPLIT_BLOCK / WAVE;
    __shared__ int counts[WAVES][3], base[3];
    const int s = blockIdx.x / chunks, chunk = blockIdx.x % chunks;
    const int start = seg[s].start, size = seg[s].size;
    if ((long long)chunk*KD_CHUNK >= size) return;
    const kd_digits k = digits_of(seg + s);
    const kd_sel last = sel[segs + s];
    const kd_sel ties = pick_bin<KD_SPLIT_BLOCK>(bins + (2ll*segs + s)*KD_BINS, last.rank);
    const uint32_t pivot = (last.prefix << k.s2) | ties.prefix;
    if (chunk == 0 && threadIdx.x == 0) sel[2*segs + s] = ties;
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
    const int begin = chunk*KD_CHUNK;
    float4 p[PER];
    int part[PER], mine[3] = {0, 0, 0};
#pragma unroll
    for (int e = 0; e < PER; ++e)
    {
        const int i = begin + e*KD_SPLIT_BLOCK + int(threadIdx.x);
        part[e] = 3;
        if (i < size)
        {
            p[e] = points[start + i];
            const uint32_t rel = ordered(coord(p[e], k.dim)) - k.lo;
            part[e] = rel < pivot ? 0 : (rel == pivot ? 1 : 2);
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) mine[c] += __popcll(__ballot(part[e] == c));
    }
    if (lane == 0)
    {
#pragma unroll
        for (int c = 0; c < 3; ++c) counts[wave][c] = mine[c];
    }
    __syncthreads();
    if (threadIdx.x < 3)
    {
        int sum = 0;
        for (int w = 0; w < WAVES; ++w) sum += counts[w][threadIdx.x];
        base[threadIdx.x] = sum ? atomicAdd(cursors + 4*s + threadIdx.x, sum) : 0;
    }
    __syncthreads();
    const int below = kd_left(size) - ties.rank;
    int at[3] = {start + base[0], start + below + base[1], start + below + ties.count + base[2]};
    for (int w = 0; w < wave; ++w)
    {
#pragma unroll
        for (int c = 0; c < 3; ++c) at[c] += counts[w][c];
    }
#pragma unroll
    for (int e = 0; e < PER; ++e)
    {
#pragma unroll
        for (int c = 0; c < 3; ++c)
        {
            const unsigned long long m = __ballot(part[e] == c);
            if (part[e] == c) out[at[c] + __popcll(m & ((1ull << lane) - 1ull))] = p[e];
            at[c] += __popcll(m);
        }
    }
}

// Puts the points that tie with a pivot on their sides of it, settles the pivot and describes its children. One
// block per subtree: usually the pivot is alone and nothing is left to order. Up to KD_TIES ties are ranked against
// each other in LDS, more are selected by the digits of the further dimensions and of the index, through `spare`.
__global__ __launch_bounds__(KD_TIES) void k_kd_settle(float4 *points, float4 *spare, const kd_seg *seg, int segs,
                                                      const kd_sel *sel, kd_seg *children, float4 *node, int *idx)
{
    __shared__ float4 ties[KD_TIES];
    __shared__ unsigned int count[KD_BINS];
    __shared__ int side[2];
    const int s = blockIdx.x;
    const kd_seg g = seg[s];
    const kd_sel tie = sel[2*segs + s];
    const int left = kd_left(g.size), t = tie.count;
    float4 *const first = points + g.start + (left - tie.rank);
    if (t > 1 && t <= KD_TIES)
    {
        const int i = threadIdx.x;
        if (i < t) ties[i] = first[i];
        __syncthreads();
        if (i < t)
        {
            const float4 p = ties[i];
            int rank = 0;
            for (int j = 0; j < t; ++j) rank += tie_less(ties[j], p, g.order) ? 1 : 0;
            first[rank] = p;
        }
    }
    else if (t > KD_TIES)
    {
        uint32_t found[3] = {0u, 0u, 0u};
        int rank = tie.rank;
        // key q of a point: the second and third dimension's coordinates, then the index
        auto key = [&](const float4 &p, int q) {
            const int d = q == 2 ? 3 : (g.order >> (2 + 2*q)) & 3;
            if (q == 2) return __float_as_uint(p.w) & ~KD_SITE;
            return d == 3 ? 0u : ordered(coord(p, d));
        };
#pragma unroll
        for (int q = 0; q < 3; ++q)
            for (int shift = 21, width = 11; shift >= 0; shift = shift == 21 ? 10 : shift - 10, width = shift ? 11 : 10)
            {
                for (int b = threadIdx.x; b < KD_BINS; b += KD_TIES) count[b] = 0u;
                __syncthreads();
                for (int i = threadIdx.x; i < t; i += KD_TIES)
                {
                    const float4 p = first[i];
                    bool same = true;
#pragma unroll
                    for (int r = 0; r < q; ++r) same = same && key(p, r) == found[r];
                    const uint32_t v = key(p, q);
                    if (same && (shift == 21 || v >> (shift + width) == found[q]))
                        atomicAdd(count + ((v >> shift) & ((1u << width) - 1u)), 1u);
                }
                __syncthreads();
                const kd_sel now = pick_bin<KD_TIES>(count, rank);
                found[q] = (found[q] << width) | now.prefix;
                rank = now.rank;
            }
        if (threadIdx.x < 2) side[threadIdx.x] = 0;
        __syncthreads();
        float4 *const to = spare + g.start + (left - tie.rank);
        for (int i = threadIdx.x; i < t; i += KD_TIES)
        {
            const float4 p = first[i];
            int c = 0;      // -1 before the pivot, 1 behind it
#pragma unroll
            for (int q = 2; q >= 0; --q)
            {
                const uint32_t v = key(p, q);
                if (v != found[q]) c = v < found[q] ? -1 : 1;
            }
            const int at = c == 0 ? tie.rank : (c < 0 ? atomicAdd(side, 1) : tie.rank + 1 + atomicAdd(side + 1, 1));
            to[at] = p;
        }
        __syncthreads();
        for (int i = threadIdx.x; i < t; i += KD_TIES) first[i] = to[i];
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    const int dim = g.order & 3;
    const float4 p = points[g.start + left];
    put_node(p, dim, segs - 1 + s, node, idx);
    kd_seg l = g, r = g;
    const uint32_t cut = ordered(coord(p, dim));
#pragma unroll
    for (int d = 0; d < 3; ++d)
        if (d == dim) l.hi[d] = r.lo[d] = cut;
    l.size = left;
    r.size = g.size - 1 - left;
    r.start = g.start + left + 1;
    l.order = order_of(l.lo, l.hi, g.order);
    r.order = order_of(r.lo, r.hi, g.order);
    children[2*s] = l;
    children[2*s + 1] = r;
}

// Every subtree of up to KD_SLOTS - 1 points, by one block in LDS. A subtree of r levels owns 2^r slots; they are
// sorted (bitonically, all subtrees of a level at once), the pivot is written to its node and the two sides move
// into the two halves of the slots. Strides of up to 64 stay within a wavefront's slots and need no barrier.
// Bound by LDS latency: 364 compare steps for 12 levels, 229 us for 256 subtrees of 3900 points, one per CU; the
// radix sorts of all points that it stands in for took 300 us for each of the 11 levels.
__global__ __launch_bounds__(KD_FINISH_BLOCK) void k_kd_finish(const float4 *points, const kd_seg *seg, int segs,
                                                              int levels, float4 *node, int *idx)
{
    constexpr uint32_t NONE = ~0u;
    struct part { uint32_t lo[3], hi[3]; int order, size; };
    __shared__ float4 pts[KD_SLOTS];
    __shared__ uint64_t key[KD_SLOTS];                   // ordered coordinate << 32 | point
    __shared__ uint32_t box[6][KD_SLOTS / 2];
    __shared__ int info[KD_SLOTS / 2];                   // order | size << 6
    const int t = threadIdx.x;
    const kd_seg g = seg[blockIdx.x];
    const int slots = 1 << levels;
    for (int i = t; i < slots; i += KD_FINISH_BLOCK)
    {
        uint64_t k = ~0ull;
        if (i < g.size)
        {
            const float4 p = points[g.start + i];
            pts[i] = p;
            k = (uint64_t(ordered(coord(p, g.order & 3))) << 32) | uint32_t(i);
        }
        key[i] = k;
    }
    if (t < 3) { box[t][0] = g.lo[t]; box[3 + t][0] = g.hi[t]; }
    if (t == 0) info[0] = g.order | (g.size << 6);
    __syncthreads();
    for (int r = levels; r >= 1; --r)
    {
        const int span = 1 << r;
        if (r > 1)
            for (int k = 2; k <= span; k <<= 1)
                for (int j = k >> 1; j > 0; j >>= 1)
                {
                    for (int p = t; p < slots / 2; p += KD_FINISH_BLOCK)
                    {
                        const int i = 2*p - (p & (j - 1));
                        const bool up = (i & k) == 0 || k == span;
                        const uint64_t a = key[i], b = key[i + j];
                        bool less = b < a;
                        if (uint32_t(a >> 32) == uint32_t(b >> 32) && uint32_t(a) != NONE && uint32_t(b) != NONE)
                            less = tie_less(pts[uint32_t(b)], pts[uint32_t(a)], info[i >> r] & 63);
                        if (less == up) { key[i] = b; key[i + j] = a; }
                    }
                    if (j > 64 || (j == 1 && k > 64)) __syncthreads();
                    else
                    {
                        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                        __builtin_amdgcn_wave_barrier();
                    }
                }
        __syncthreads();
        // settle the pivots; at r = 1 every subtree is one point and has no children
        const int subtrees = slots >> r;
        part l, h;
        bool split = false;
        for (int q = t; q < subtrees; q += KD_FINISH_BLOCK)
        {
            const int size = info[q] >> 6, order = info[q] & 63, dim = order & 3;
            const int left = kd_left(size);
            const float4 p = size ? pts[uint32_t(key[q*span + left])] : make_float4(0.f, 0.f, 0.f, 0.f);
            if (size) put_node(p, dim, ((long long)(segs + blockIdx.x) << (levels - r)) - 1 + q, node, idx);
            if (r == 1) continue;
            split = true;
#pragma unroll
            for (int d = 0; d < 3; ++d) { l.lo[d] = h.lo[d] = box[d][q]; l.hi[d] = h.hi[d] = box[3 + d][q]; }
            const uint32_t cut = ordered(coord(p, dim));
#pragma unroll
            for (int d = 0; d < 3; ++d)
                if (d == dim) l.hi[d] = h.lo[d] = cut;
            l.size = left;
            h.size = max(size - 1 - left, 0);
            l.order = order_of(l.lo, l.hi, order);
            h.order = order_of(h.lo, h.hi, order);
        }
        if (r == 1) break;
        const int half = span >> 1;
        uint32_t from[KD_SLOTS / KD_FINISH_BLOCK];
#pragma unroll
        for (int e = 0; e < KD_SLOTS / KD_FINISH_BLOCK; ++e)
        {
            const int i = t + e*KD_FINISH_BLOCK;
            from[e] = NONE;
            if (i >= slots) continue;
            const int q = i >> r, pos = i & (half - 1), size = info[q] >> 6, left = kd_left(size);
            const bool right = i & half;
            if (pos < (right ? size - 1 - left : left)) from[e] = uint32_t(key[q*span + pos + (right ? left + 1 : 0)]);
        }
        __syncthreads();
        if (split)
        {
#pragma unroll
            for (int d = 0; d < 3; ++d)
            {
                box[d][2*t] = l.lo[d]; box[3 + d][2*t] = l.hi[d];
                box[d][2*t + 1] = h.lo[d]; box[3 + d][2*t + 1] = h.hi[d];
            }
            info[2*t] = l.order | (l.size << 6);
            info[2*t + 1] = h.order | (h.size << 6);
        }
        __syncthreads();
#pragma unroll
        for (int e = 0; e < KD_SLOTS / KD_FINISH_BLOCK; ++e)
        {
            const int i = t + e*KD_FINISH_BLOCK;
            if (i >= slots) continue;
            uint64_t k = ~0ull;
            if (from[e] != NONE)
                k = (uint64_t(ordered(coord(pts[from[e]], info[i >> (r - 1)] & 3))) << 32) | from[e];
            key[i] = k;
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------------------------
// query
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ float d2_of(float ax, float ay, float az, float bx, float by, float bz)
{
    float dx = ax - bx, dy = ay - by, dz = az - bz;
    return dx*dx + dy*dy + dz*dz;
}

__device__ __forceinline__ float key_d2(uint64_t k) { return __uint_as_float(uint32_t(k >> 32)); }

// nextafterf(x, inf) for x >= 0 or NaN
__device__ __forceinline__ float above(float x)
{
    const uint32_t u = __float_as_uint(x);
    return __uint_as_float(u + (u < 0x7f800000u ? 1u : 0u));
}

// col_site_init's wedge images (src/swarm/col_site_init.cu:42-62): physical points at [0, n), every point
// rotated by -width (image 1) at [n, 2n) and by +width (image 2) at [2n, 3n)
__global__ __launch_bounds__(KD_BLOCK) void k_kd_images(const float4 *pts, int n, float cw, float sw, float4 *out)
{
    const long long i = (long long)blockIdx.x*KD_BLOCK + threadIdx.x;
    if (i >= n) return;
    const float4 p = pts[i];
    out[i] = p;
#pragma unroll
    for (int image = 0; image < 2; ++image)
    {
        const float sa = image == 0 ? -sw : sw;
        out[i + (long long)(image + 1)*n] = make_float4(cw*p.x - sa*p.y, sa*p.x + cw*p.y, p.z, p.w);
    }
}

// max-heap columns in LDS: `cand` takes the place of the entry at `slot` and sinks. The larger child and its
// children are read together, which halves the chain of dependent LDS reads.
__device__ __forceinline__ void sift_from(uint64_t *heap, int slot, uint64_t cand)
{
    for (int child = 2*slot + 1; child < N_K; child = 2*slot + 1)
    {
        uint64_t cv = heap[child*WAVE];
        if (child + 1 < N_K)
        {
            const uint64_t other = heap[(child + 1)*WAVE];
            if (other > cv) { cv = other; ++child; }
        }
        if (cv < cand) break;
        heap[slot*WAVE] = cv;
        slot = child;
    }
    heap[slot*WAVE] = cand;
}

// the same from the root: slots 1 .. N_K - 2 fill their levels, slot N_K - 1 is the only one below them
// returns the new root
__device__ __forceinline__ uint64_t sift_root(uint64_t *heap, uint64_t cand)
{
    int slot = 0;
    bool sinks = true;
    uint64_t root = cand;
#pragma unroll
    for (int l = 1; l < LOG2K; l += 2)
    {
        if (!sinks) continue;
        int child = 2*slot + 1;
        const uint64_t *h = heap + child*WAVE, *g = h + (child + 1)*WAVE;      // children, grandchildren
        const uint64_t a = h[0], b = h[WAVE];
        uint64_t g0 = 0, g1 = 0, g2 = 0, g3 = 0;
        if (l + 1 < LOG2K) { g0 = g[0]; g1 = g[WAVE]; g2 = g[2*WAVE]; g3 = g[3*WAVE]; }
        const bool right = b > a;
        const uint64_t cv = right ? b : a;
        if (right) { ++child; g0 = g2; g1 = g3; }
        sinks = !(cv < cand);
        if (!sinks) continue;
        if (l == 1) root = cv;
        heap[slot*WAVE] = cv;
        slot = child;
        if (l + 1 == LOG2K) continue;
        child = 2*slot + 1 + (g1 > g0 ? 1 : 0);
        const uint64_t gv = g1 > g0 ? g1 : g0;
        sinks = !(gv < cand);
        if (!sinks) continue;
        heap[slot*WAVE] = gv;
        slot = child;
    }
    if (slot == N_K / 2 - 1)
    {
        const uint64_t cv = heap[(N_K - 1)*WAVE];
        if (!(cv < cand)) { heap[slot*WAVE] = cv; slot = N_K - 1; }
    }
    heap[slot*WAVE] = cand;
    return root;
}

// queries: the nq physical particles in Morton order; the tree holds nt records, record r being particle
// r % n_phys at image r / n_phys when n_phys > 0 (a wedge), else particle r
//
// A lane walks the tree alone, so what bounds it is the latency of a chain of node loads and the heap, both of
// which are indexed differently in every lane. Heap and path values live in LDS, one column per lane (no bank
// conflicts whatever the index); as private arrays they were scratch, whose 38 KB per wavefront did not fit the
// caches. The path takes 8 bytes per level: the far child of a path node is the path's sibling one level down,
// so a pending one is a bit, with the plane's coordinate and the distance of the closest corner behind it; the
// corner itself follows from the planes of the far sides that the path is on. 1e6 points, 32 neighbours:
// 13.1 -> 2.6 ms (262 visits and 217 heap insertions per wavefront, 6 wavefronts per CU).
__global__ __launch_bounds__(KD_QUERY_BLOCK) void k_kd_topk(const float4 *__restrict__ node,
                                                           const int *__restrict__ node_idx, int nt, int nq,
                                                           int n_phys, float image_dist_min,
                                                           const float *world, const int *sidx, const float4 *pts,
                                                           const unsigned char *active, const int *pidx_slot,
                                                           const unsigned char *group, bound_state u, int *nbr,
                                                           double *measure, unsigned long long *graph,
                                                           unsigned char *nbr_image)
{
    static_assert(KD_QUERY_BLOCK == WAVE, "one wavefront per block: no column is shared");
    extern __shared__ uint64_t kd_lds[];
    const int lane = threadIdx.x % WAVE;
    uint64_t *const heap = kd_lds + lane;                                            // [N_K] columns
    float2 *const path = reinterpret_cast<float2 *>(kd_lds + N_K*WAVE) + lane;        // [levels of the tree]
    const int m = xcd_block()*KD_QUERY_BLOCK + threadIdx.x;
    const int n = nt;
    const int p = m < nq ? sidx[m] : 0;
    const bool qactive = m < nq && active[p];
    unsigned long long mask = 0ull;
    int g = qactive ? int(group[p]) : -1;
    if (qactive)
    {
        const float4 qp = pts[p];
        const uint64_t empty = (uint64_t(__float_as_uint(qp.w*qp.w)) << 32) | 0xffffffffull;
        // one entry per particle when two of its images can share this ball (_col_cache.cuh:38-41)
        const bool dedup = X_WEDGE && !(image_dist_min < 0.0f || image_dist_min > 2.0f*qp.w);
        for (int k = 0; k < N_K; ++k) heap[k*WAVE] = empty;
        uint64_t top = empty;                                  // the heap's root
        float cull = above(key_d2(top));
        const float wx = fminf(fmaxf(qp.x, world[0]), world[3]);
        const float wy = fminf(fmaxf(qp.y, world[1]), world[4]);
        const float wz = fminf(fmaxf(qp.z, world[2]), world[5]);
        float cx = wx, cy = wy, cz = wz;
        // bit l: the far child of the path's node at level l is still to be visited (pending) or the path goes
        // through it (taken); is_y, is_z: the node's split dimension
        unsigned int pending = 0u, taken = 0u, is_y = 0u, is_z = 0u;
        unsigned int id = 0u;
        int level = 0;
        bool run = !(d2_of(cx, cy, cz, qp.x, qp.y, qp.z) > cull);
        float4 np = node[0];
        int r = node_idx[0];
        while (run)
        {
            const int bits = __float_as_int(np.w);
            const int dim = bits & 3;
            const float d2 = d2_of(np.x, np.y, np.z, qp.x, qp.y, qp.z);
            const float nd = coord(np, dim);
            const bool left_close = coord(qp, dim) < nd;
            const unsigned int lc = 2u*id + 1u;
            const unsigned int near = left_close ? lc : lc + 1u, far = left_close ? lc + 1u : lc;
            // the near child's record is on its way while the heap takes this one
            const unsigned int ahead = min(near, unsigned(n) - 1u);
            const float4 next = node[ahead];
            const int next_r = node_idx[ahead];
            if ((bits & KD_ACTIVE) && __float_as_uint(d2) <= uint32_t(top >> 32))
            {
                const int image = X_WEDGE ? r / n_phys : 0;
                const int j = X_WEDGE ? r - image*n_phys : r;
                const uint64_t cand = (uint64_t(__float_as_uint(d2)) << 32) | uint32_t(3*j + image);
                // a particle already in the heap is replaced only by a nearer image of itself
                // (idx_old_heap::processCandidate, inc/swarm/kdtree/index_heap.cuh:112-175)
                int found = -1;
                if (X_WEDGE && dedup)
                {
                    for (int k = 0; k < N_K; ++k)
                    {
                        const uint32_t ck = uint32_t(heap[k*WAVE]);
                        if (found < 0 && ck != 0xffffffffu && int(ck / 3u) == j) found = k;
                    }
                }
                if (X_WEDGE && found >= 0)
                {
                    if (cand < heap[found*WAVE]) sift_from(heap, found, cand);
                    top = heap[0];
                }
                else if (cand < top)
                {
                    top = sift_root(heap, cand);
                }
                cull = above(key_d2(top));
            }
            const float far_d2 = d2_of(dim == 0 ? nd : cx, dim == 1 ? nd : cy, dim == 2 ? nd : cz, qp.x, qp.y, qp.z);
            if (far < unsigned(n) && far_d2 < cull)
            {
                const unsigned int bit = 1u << level;
                path[level*WAVE] = make_float2(nd, far_d2);
                pending |= bit;
                is_y = dim == 1 ? is_y | bit : is_y & ~bit;
                is_z = dim == 2 ? is_z | bit : is_z & ~bit;
            }
            id = near;
            ++level;
            np = next;
            r = next_r;
            if (id >= unsigned(n))
            {
                // the deepest far child that is still close enough
                while (pending)
                {
                    const int l = 31 - __clz(static_cast<int>(pending));
                    if (path[l*WAVE].y < cull) break;
                    pending &= ~(1u << l);
                }
                run = pending != 0u;
                if (run)
                {
                    const int l = 31 - __clz(static_cast<int>(pending));
                    const unsigned int bit = 1u << l;
                    pending &= ~bit;
                    taken = (taken & (bit - 1u)) | bit;
                    id = (((id + 1u) >> (level - l - 1)) ^ 1u) - 1u;
                    level = l + 1;
                    np = node[id];
                    r = node_idx[id];
                    // its closest corner: in each dimension the plane of the deepest far side that the path is on
                    const unsigned int tx = taken & ~(is_y | is_z), ty = taken & is_y, tz = taken & is_z;
                    cx = tx ? path[(31 - __clz(static_cast<int>(tx)))*WAVE].x : wx;
                    cy = ty ? path[(31 - __clz(static_cast<int>(ty)))*WAVE].x : wy;
                    cz = tz ? path[(31 - __clz(static_cast<int>(tz)))*WAVE].x : wz;
                }
            }
            // one latch: lanes that go down and lanes that go back visit their next nodes together (as two nested
            // loops, which the compiler makes of it otherwise, a wavefront takes 420 visits instead of 260)
            __builtin_amdgcn_wave_barrier();
        }
        const int s = pidx_slot[p];
        float max_d2 = 0.0f;
        int row[N_K];
#pragma unroll
        for (int k = 0; k < N_K; ++k)
        {
            const uint64_t entry = heap[k*WAVE];
            const uint32_t code = uint32_t(entry);
            if (code != 0xffffffffu)
            {
                max_d2 = fmaxf(max_d2, key_d2(entry));
                int jj = int(code) / 3;
                row[k] = pidx_slot[jj];
                mask |= 1ull << group[jj];
            }
            else
            {
                row[k] = -1;
            }
        }
        int4 *dst = reinterpret_cast<int4 *>(nbr + (long long)s*N_K);
#pragma unroll
        for (int t = 0; t < N_K; t += 4)
            dst[t / 4] = make_int4(row[bitrev_slot(t)], row[bitrev_slot(t + 1)], row[bitrev_slot(t + 2)],
                                   row[bitrev_slot(t + 3)]);
        if constexpr (X_WEDGE)
        {
#pragma unroll
            for (int t = 0; t < N_K; ++t)
            {
                const uint32_t code = uint32_t(heap[bitrev_slot(t)*WAVE]);
                nbr_image[(long long)s*N_K + t] = static_cast<unsigned char>(code != 0xffffffffu ? code % 3u : 0u);
            }
        }
        measure[s] = ball_measure(ld(u.y, p), ld(u.z, p), sqrt(static_cast<double>(max_d2)));
    }
    // one atomic per distinct owner group of this wavefront (col_dep_graph.cu:14-60)
    unsigned long long todo = __ballot(qactive);
    while (todo)
    {
        int leader = __ffsll(static_cast<long long>(todo)) - 1;
        int lg = __builtin_amdgcn_readlane(g, leader);
        unsigned long long mine = (g == lg) ? mask : 0ull;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) mine |= __shfl_xor(mine, o, WAVE);
        if (lane == leader) atomicOr(graph + lg, mine);
        todo &= ~__ballot(g == lg);
    }
}

}  // namespace

void kd_build(context &c)
{
    const float4 *src = c.pts.p;
    int n = c.n;
    hipStream_t st = c.stream;
    if constexpr (X_WEDGE)
    {
        if (3ll*n > INT_MAX / 3) throw status_error(12, "wedge k-d node count exceeds the index limit");
        const float width = static_cast<float>(X_MAX - X_MIN);
        const float sw = static_cast<float>(std::sin(static_cast<double>(width)));
        const float cw = static_cast<float>(std::cos(static_cast<double>(width)));
        c.wedge_rec.alloc(size_t(3)*n);
        k_kd_images<<<blocks(n, KD_BLOCK), KD_BLOCK, 0, st>>>(c.pts.p, n, cw, sw, c.wedge_rec.p);
        hip_check(hipGetLastError(), "launch k-d images");
        src = c.wedge_rec.p;
        n *= 3;
    }
    kd_tree &t = c.kd;
    t.n = n;
    t.node.alloc(n);
    t.idx.alloc(n);
    t.world.alloc(6);
    int levels = 0;
    while ((1ll << levels) - 1 < n) ++levels;      // levels of a left-balanced tree of n nodes
    const int top = std::max(0, levels - KD_LDS_LEVELS);
    const size_t seg_words = (size_t(1) << top)*(sizeof(kd_seg) / sizeof(unsigned int));
    const size_t most = size_t(1) << std::max(0, top - 1);      // subtrees of the last level that is split
    t.points[0].alloc(n);
    t.points[1].alloc(top ? n : 0);
    t.segments.alloc(2*seg_words);
    t.counts.alloc(most*(3*KD_BINS + 4 + 3*sizeof(kd_sel) / sizeof(unsigned int)) + 6);
    unsigned int *const wbits = t.counts.p;
    hip_check(hipMemsetAsync(wbits, 0xff, 6*sizeof(unsigned int), st), "k-d world init");
    kd_seg *seg = reinterpret_cast<kd_seg *>(t.segments.p), *next = reinterpret_cast<kd_seg *>(t.segments.p + seg_words);
    k_kd_init<<<std::min(KD_INIT_BLOCKS, blocks(n, KD_BLOCK)), KD_BLOCK, 0, st>>>(src, c.active.p, n, c.n,
                                                                                t.points[0].p, wbits);
    k_kd_root<<<1, 64, 0, st>>>(wbits, n, t.world.p, seg);
    hip_check(hipGetLastError(), "launch k-d init");
    float4 *points = t.points[0].p, *other = t.points[1].p;
    int largest = n;
    for (int L = 0; L < top; ++L)
    {
        const int segs = 1 << L, chunks = blocks(largest, KD_CHUNK);
        unsigned int *const bins = t.counts.p + 6;
        int *const cursors = reinterpret_cast<int *>(bins + size_t(segs)*3*KD_BINS);
        kd_sel *const sel = reinterpret_cast<kd_sel *>(cursors + size_t(segs)*4);
        hip_check(hipMemsetAsync(bins, 0, sizeof(unsigned int)*size_t(segs)*(3*KD_BINS + 4), st), "k-d counts");
        k_kd_digit<0><<<segs*chunks, KD_SPLIT_BLOCK, 0, st>>>(points, seg, segs, chunks, bins, sel);
        k_kd_digit<1><<<segs*chunks, KD_SPLIT_BLOCK, 0, st>>>(points, seg, segs, chunks, bins, sel);
        k_kd_digit<2><<<segs*chunks, KD_SPLIT_BLOCK, 0, st>>>(points, seg, segs, chunks, bins, sel);
        k_kd_partition<<<segs*chunks, KD_SPLIT_BLOCK, 0, st>>>(points, seg, segs, chunks, bins, sel, cursors, other);
        k_kd_settle<<<segs, KD_TIES, 0, st>>>(other, points, seg, segs, sel, next, t.node.p, t.idx.p);
        hip_check(hipGetLastError(), "launch k-d split");
        std::swap(points, other);
        std::swap(seg, next);
        largest = kd_left(largest);
    }
    k_kd_finish<<<1 << top, KD_FINISH_BLOCK, 0, st>>>(points, seg, 1 << top, levels - top, t.node.p, t.idx.p);
    hip_check(hipGetLastError(), "launch k-d finish");
}

void kd_query(context &c)
{
    const int n = c.n;
    float image_dist_min = -1.0f;
    if constexpr (X_WEDGE)
    {
        // _get_image_dist_min (inc/swarm/param_grid.cuh:86-89), each sine rounded once from double
        auto sinf1 = [](float a) { return static_cast<float>(std::sin(static_cast<double>(a))); };
        const float x_min = static_cast<float>(X_MIN), x_max = static_cast<float>(X_MAX);
        image_dist_min = 2.0f*static_cast<float>(Y_MIN)
            *std::fmin(sinf1(static_cast<float>(Z_MIN)), sinf1(static_cast<float>(Z_MAX)))
            *std::fabs(sinf1(0.5f*(x_max - x_min)));
        c.nbr_image.alloc(size_t(std::max(1, c.n_active))*N_K);
    }
    int levels = 0;
    while ((1ll << levels) - 1 < c.kd.n) ++levels;
    const size_t lds = size_t(WAVE)*(N_K*sizeof(uint64_t) + levels*sizeof(float2));
    k_kd_topk<<<xcd_grid(blocks(n, KD_QUERY_BLOCK)), KD_QUERY_BLOCK, lds, c.stream>>>(
        c.kd.node.p, c.kd.idx.p, c.kd.n, n, X_WEDGE ? n : 0, image_dist_min, c.kd.world.p, c.index.idx.p, c.pts.p,
        c.active.p, c.pidx_slot.p, c.group.p, c.user, c.nbr.p, c.measure.p, c.graph.p, c.nbr_image.p);
    hip_check(hipGetLastError(), "launch k-d top-K");
}

}  // namespace gdx
