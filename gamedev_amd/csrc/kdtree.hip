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
// Build: every level sorts (tag, coordinate along the point's split dimension) with the library's
// stable LSD radix sort (the reference's thrust::sort is not stable, so its layout for equal
// coordinates is unspecified; this layout is the stable one), then one thread per array position
// moves its point into the left or right child subtree, or settles it as the subtree's pivot, and
// sets its split dimension to the widest extent of the child subtree's domain.
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

__device__ __forceinline__ int level_of(int node) { return 63 - __clzll(static_cast<long long>(node) + 1ll); }
__device__ __forceinline__ int levels_for(int n) { return level_of(n - 1) + 1; }
__device__ __forceinline__ int full_nodes(int levels) { return (1 << levels) - 1; }

__device__ __forceinline__ int subtree_size(int n, int root)
{
    int levels_sub = levels_for(n) - level_of(root);
    int first = (root + 1) << (levels_sub - 1);
    int on_last = 1 << (levels_sub - 1);
    int last_on_last = first + on_last - 1;
    int missing = min(max(last_on_last - n, 0), on_last);
    return full_nodes(levels_sub) - missing;
}

// array position of a level-L subtree's pivot during step L
__device__ __forceinline__ int pivot_pos(int L, int n, int subtree)
{
    int settled = full_nodes(L);
    int levels_total = levels_for(n);
    int remaining = levels_total - L;
    int earlier = subtree - settled;
    int left_if_full = earlier*full_nodes(remaining);
    int left_on_last_if_full = earlier*(1 << (remaining - 1));
    int total_on_last = n - full_nodes(levels_total - 1);
    int missing = left_on_last_if_full - min(total_on_last, left_on_last_if_full);
    int left_root = 2*subtree + 1;
    return settled + left_if_full - missing + (left_root >= n ? 0 : subtree_size(n, left_root));
}

// ---------------------------------------------------------------------------------------------
// build
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(KD_BLOCK) void k_kd_init(const float4 *pts, int n, float4 *node, int *idx,
                                                     unsigned int *world_bits)
{
    __shared__ unsigned int red[6][KD_BLOCK / WAVE];
    int i = blockIdx.x*KD_BLOCK + threadIdx.x;
    float4 p = pts[min(i, n - 1)];
    if (i < n)
    {
        node[i] = make_float4(p.x, p.y, p.z, __int_as_float(0));
        idx[i] = i;
    }
    // world box of the data: ordered-key minima and maxima, one atomic per block and bound
    unsigned int k[6] = {ordered(p.x), ordered(p.y), ordered(p.z), ordered(p.x), ordered(p.y), ordered(p.z)};
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
#pragma unroll
    for (int b = 0; b < 6; ++b)
    {
        unsigned int v = k[b];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1)
        {
            unsigned int t = __shfl_xor(v, o, WAVE);
            v = (b < 3) ? min(v, t) : max(v, t);
        }
        if (lane == 0) red[b][wave] = v;
    }
    __syncthreads();
    if (threadIdx.x < 6)
    {
        int b = threadIdx.x;
        unsigned int v = red[b][0];
        for (int w = 1; w < KD_BLOCK / WAVE; ++w) v = (b < 3) ? min(v, red[b][w]) : max(v, red[b][w]);
        if (b < 3) atomicMin(world_bits + b, v);
        else atomicMax(world_bits + b, v);
    }
}

__device__ __forceinline__ float unordered(uint32_t u)
{
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}

__global__ void k_kd_world(const unsigned int *world_bits, float *world, int *dim0)
{
    if (threadIdx.x != 0) return;
    kd_box b;
    for (int d = 0; d < 3; ++d) { b.lo[d] = unordered(world_bits[d]); b.hi[d] = unordered(world_bits[3 + d]); }
    for (int d = 0; d < 3; ++d) { world[d] = b.lo[d]; world[3 + d] = b.hi[d]; }
    *dim0 = widest(b);
}

__global__ __launch_bounds__(KD_BLOCK) void k_kd_dim0(float4 *node, int n, const int *dim0)
{
    int i = blockIdx.x*KD_BLOCK + threadIdx.x;
    if (i < n) node[i].w = __int_as_float(*dim0);
}

__global__ __launch_bounds__(KD_BLOCK) void k_kd_keys(const float4 *node, const uint32_t *tag, int n, uint64_t *key,
                                                     int *val, bool tag_only)
{
    int i = blockIdx.x*KD_BLOCK + threadIdx.x;
    if (i >= n) return;
    float4 p = node[i];
    uint64_t t = tag[i];
    key[i] = tag_only ? t : (t << 32) | ordered(coord(p, __float_as_int(p.w)));
    val[i] = i;
}

__global__ __launch_bounds__(KD_BLOCK) void k_kd_gather(const uint64_t *key, const int *val, const float4 *node,
                                                       const int *idx, int n, bool tag_only,
                                                       const unsigned char *active, int n_phys, float4 *node_out,
                                                       int *idx_out, uint32_t *tag_out)
{
    int i = blockIdx.x*KD_BLOCK + threadIdx.x;
    if (i >= n) return;
    int from = val[i];
    float4 p = node[from];
    const int r = idx[from];
    if (tag_only && active[r % n_phys]) p.w = __int_as_float(__float_as_int(p.w) | KD_ACTIVE);
    node_out[i] = p;
    idx_out[i] = r;
    tag_out[i] = tag_only ? uint32_t(key[i]) : uint32_t(key[i] >> 32);
}

// step L of the tag update: positions below the settled count are final; every other point moves
// into its subtree's left or right child, or stays as the subtree's pivot (its node)
__global__ __launch_bounds__(KD_BLOCK) void k_kd_update(float4 *node, uint32_t *tag, int n, int L,
                                                       const float *world)
{
    int g = blockIdx.x*KD_BLOCK + threadIdx.x;
    if (g >= n || g < full_nodes(L)) return;
    int subtree = int(tag[g]);
    kd_box b;
#pragma unroll
    for (int d = 0; d < 3; ++d) { b.lo[d] = world[d]; b.hi[d] = world[3 + d]; }
    for (int cur = subtree; cur > 0;)
    {
        int parent = (cur + 1) / 2 - 1;
        float4 pp = node[parent];
        int d = __float_as_int(pp.w);
        float split = coord(pp, d);
        if (cur & 1) b.hi[d] = fminf(split, b.hi[d]);
        else b.lo[d] = fmaxf(split, b.lo[d]);
        cur = parent;
    }
    int pivot = pivot_pos(L, n, subtree);
    float4 pv = node[pivot];
    int pd = __float_as_int(pv.w);
    float pc = coord(pv, pd);
    if (g < pivot) { subtree = 2*subtree + 1; b.hi[pd] = pc; }
    else if (g > pivot) { subtree = 2*subtree + 2; b.lo[pd] = pc; }
    if (g != pivot) node[g].w = __int_as_float(widest(b));
    tag[g] = uint32_t(subtree);
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
    dbuf<float4> node_b;
    dbuf<int> idx_b;
    dbuf<uint32_t> tag, tag_b;
    dbuf<uint64_t> key;
    dbuf<int> val;
    dbuf<unsigned int> wbits;
    dbuf<int> dim0;
    node_b.alloc(n);
    idx_b.alloc(n);
    tag.alloc(n);
    tag_b.alloc(n);
    key.alloc(n);
    val.alloc(n);
    wbits.alloc(6);
    dim0.alloc(1);
    const unsigned int init[6] = {~0u, ~0u, ~0u, 0u, 0u, 0u};
    hip_check(hipMemcpyAsync(wbits.p, init, sizeof(init), hipMemcpyHostToDevice, st), "k-d world init");
    hip_check(hipMemsetAsync(tag.p, 0, sizeof(uint32_t)*n, st), "k-d tags");
    k_kd_init<<<blocks(n, KD_BLOCK), KD_BLOCK, 0, st>>>(src, n, t.node.p, t.idx.p, wbits.p);
    k_kd_world<<<1, 64, 0, st>>>(wbits.p, t.world.p, dim0.p);
    k_kd_dim0<<<blocks(n, KD_BLOCK), KD_BLOCK, 0, st>>>(t.node.p, n, dim0.p);
    hip_check(hipGetLastError(), "launch k-d init");
    int levels = 0;
    while ((1ll << levels) - 1 < n) ++levels;      // levels of a left-balanced tree of n nodes
    const int deepest = levels - 1;
    auto sort_level = [&](int L, bool tag_only) {
        k_kd_keys<<<blocks(n, KD_BLOCK), KD_BLOCK, 0, st>>>(t.node.p, tag.p, n, key.p, val.p, tag_only);
        // tags of step L are below 2^(L+1); the final pass sorts tags of up to `levels` bits
        int tag_bits = tag_only ? levels : L + 1;
        radix_sort_pairs(key.p, val.p, n, 0, (tag_only ? 0 : 32) + tag_bits, c.scratch, st);
        k_kd_gather<<<blocks(n, KD_BLOCK), KD_BLOCK, 0, st>>>(key.p, val.p, t.node.p, t.idx.p, n, tag_only,
                                                             c.active.p, c.n, node_b.p, idx_b.p, tag_b.p);
        hip_check(hipGetLastError(), "launch k-d sort");
        swap_buf(t.node, node_b);
        swap_buf(t.idx, idx_b);
        swap_buf(tag, tag_b);
    };
    for (int L = 0; L < deepest; ++L)
    {
        sort_level(L, false);
        k_kd_update<<<blocks(n, KD_BLOCK), KD_BLOCK, 0, st>>>(t.node.p, tag.p, n, L, t.world.p);
        hip_check(hipGetLastError(), "launch k-d update");
    }
    sort_level(deepest, true);
    hip_check(hipStreamSynchronize(st), "k-d build");
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
