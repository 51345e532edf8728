// Geometry epoch of the collision operator on gfx950: collision sites, Morton keys, stable radix
// sort, adaptive Morton hierarchy, exact top-K neighbour lists and the KNN ball measure.
//
// Reference behaviour followed: col_site_init (src/swarm/col_site_init.cu:79-118), morton_keygen and
// the hierarchy build (inc/swarm/morton/morton_index.cuh:41-229), the root cube of
// morton_ghost_index::build_index (inc/swarm/morton/morton_ghost.cuh:176-183), col_cache_get
// (inc/swarm/_col_cache.cuh:73-159) and col_space_bin / col_dep_graph (src/swarm/col_space_bin.cu,
// src/swarm/col_dep_graph.cu). The top-K contract is the reference's: the K smallest (d^2, code)
// among active records with d^2 <= q^2, ascending, where code = 3*particle index.
#include "gdx_internal.h"
#include "gdx_device.h"
#include "gdx_topk.h"

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>

#pragma clang fp contract(off)

namespace gdx {

void hip_check(hipError_t e, const char *what)
{
    if (e != hipSuccess) throw status_error(17, std::string(what) + ": " + hipGetErrorString(e));
}

namespace {

constexpr int WAVE = 64;
constexpr int CHUNK = 8;                 // sorted records per chunk box

__device__ __forceinline__ unsigned long long lanemask_lt(int lane) { return (1ull << lane) - 1ull; }

__device__ __forceinline__ double ld(const field &f, long long i)
{
    return *reinterpret_cast<const double *>(f.base + i*f.stride);
}

// ============================================================================================
// device-wide exclusive scan of u32 (reduce, scan partials, downsweep)
// ============================================================================================
constexpr int SCAN_BLOCK = 256;
constexpr int SCAN_ITEMS = 8;
constexpr int SCAN_TILE = SCAN_BLOCK*SCAN_ITEMS;

__device__ __forceinline__ unsigned int block_exclusive(unsigned int v, unsigned int *lds_waves, unsigned int &total)
{
    int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
    unsigned int inc = v;
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1)
    {
        unsigned int t = __shfl_up(inc, o, WAVE);
        if (lane >= o) inc += t;
    }
    if (lane == WAVE - 1) lds_waves[wave] = inc;
    __syncthreads();
    unsigned int base = 0;
    total = 0;
    for (int w = 0; w < SCAN_BLOCK / WAVE; ++w)
    {
        unsigned int x = lds_waves[w];
        if (w < wave) base += x;
        total += x;
    }
    __syncthreads();
    return base + inc - v;
}

__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_reduce(const unsigned int *in, int n, unsigned int *partial)
{
    __shared__ unsigned int waves[SCAN_BLOCK / WAVE];
    long long base = (long long)blockIdx.x*SCAN_TILE + (long long)threadIdx.x*SCAN_ITEMS;
    unsigned int s = 0;
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i) if (base + i < n) s += in[base + i];
    unsigned int total;
    block_exclusive(s, waves, total);
    if (threadIdx.x == 0) partial[blockIdx.x] = total;
}

__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_partials(unsigned int *partial, int m)
{
    __shared__ unsigned int waves[SCAN_BLOCK / WAVE];
    unsigned int carry = 0;
    for (int chunk = 0; chunk < m; chunk += SCAN_TILE)
    {
        unsigned int v[SCAN_ITEMS];
        unsigned int s = 0;
        int base = chunk + threadIdx.x*SCAN_ITEMS;
#pragma unroll
        for (int i = 0; i < SCAN_ITEMS; ++i) { v[i] = (base + i < m) ? partial[base + i] : 0u; s += v[i]; }
        unsigned int total;
        unsigned int ex = block_exclusive(s, waves, total) + carry;
#pragma unroll
        for (int i = 0; i < SCAN_ITEMS; ++i) { if (base + i < m) partial[base + i] = ex; ex += v[i]; }
        carry += total;
    }
}

__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_down(const unsigned int *in, unsigned int *out, int n,
                                                         const unsigned int *partial)
{
    __shared__ unsigned int waves[SCAN_BLOCK / WAVE];
    long long base = (long long)blockIdx.x*SCAN_TILE + (long long)threadIdx.x*SCAN_ITEMS;
    unsigned int v[SCAN_ITEMS];
    unsigned int s = 0;
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i) { v[i] = (base + i < n) ? in[base + i] : 0u; s += v[i]; }
    unsigned int total;
    unsigned int ex = block_exclusive(s, waves, total) + partial[blockIdx.x];
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i) { if (base + i < n) out[base + i] = ex; ex += v[i]; }
}

// ============================================================================================
// stable LSD radix sort of (u64 key, int value) and the stable slot order, 8-bit digits
// ============================================================================================
// A pass is three launches: digit counts per tile, a scan along each digit's row of tiles, and the move. In the
// move a wavefront ranks its own consecutive records round by round without a barrier, then the tile is put in
// order in LDS, so that records of one digit leave in runs. 1e7 records: 106 us a pass (240 MB, 50 us at the copy
// rate) against 180 us in five launches when the whole block ranked 256 records between barriers and wrote them
// one by one; 65536 records: 11 us against 31 us.
constexpr int SORT_BLOCK = 256;
constexpr int SORT_WAVES = SORT_BLOCK / WAVE;
constexpr int RADIX = 256;
constexpr int SORT_ITEMS = 8;             // per thread: runs of 64 bytes at 256 digits, five blocks per CU
constexpr int SORT_ITEMS_SMALL = 2;       // where the larger tile would leave CUs idle
constexpr int SORT_SMALL = 256*SORT_BLOCK*SORT_ITEMS;

static_assert(SORT_BLOCK == SCAN_BLOCK, "the row scan is the scan's");

inline int sort_items(int n) { return n < SORT_SMALL ? SORT_ITEMS_SMALL : SORT_ITEMS; }

// a pass's digit of a key: eight bits, or, of a two-dimensional Morton key, whose every third bit is zero, the
// eight that twelve bits hold
struct key_digit
{
    int shift;
    bool flat;
    __device__ __forceinline__ unsigned operator()(uint64_t key) const
    {
        const unsigned w = unsigned(key >> shift);
        return flat ? (w & 3u) | ((w >> 1) & 12u) | ((w >> 2) & 48u) | ((w >> 3) & 192u) : w & 255u;
    }
};

// rank of the lane's digit among those of the wavefront's earlier records (counted in cnt) and earlier lanes
template <int BITS>
__device__ __forceinline__ unsigned wave_rank(unsigned digit, bool valid, unsigned *cnt, int lane)
{
    unsigned long long peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < BITS; ++b)
    {
        const bool bit = (digit >> b) & 1u;
        const unsigned long long m = __ballot(bit);
        peers &= bit ? m : ~m;
    }
    const unsigned rank = __popcll(peers & lanemask_lt(lane));
    const unsigned before = valid ? cnt[digit] : 0u;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (valid && rank == 0) cnt[digit] = before + __popcll(peers);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    return before + rank;
}

// exclusive prefix over the block's 256 threads
__device__ __forceinline__ uint64_t prefix_256(uint64_t v, uint64_t *waves)
{
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
    uint64_t incl = v;
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1)
    {
        const uint64_t t = __shfl_up(incl, o, WAVE);
        if (lane >= o) incl += t;
    }
    if (lane == WAVE - 1) waves[wave] = incl;
    __syncthreads();
    uint64_t before = incl - v;
    for (int w = 0; w < wave; ++w) before += waves[w];
    return before;
}

template <int ITEMS>
__global__ __launch_bounds__(SORT_BLOCK) void k_radix_hist(const uint64_t *keys, int n, key_digit digit,
                                                          unsigned int *hist, int nblocks)
{
    __shared__ unsigned int cnt[RADIX];
    cnt[threadIdx.x] = 0;
    __syncthreads();
    const long long base = (long long)blockIdx.x*SORT_BLOCK*ITEMS;
#pragma unroll
    for (int r = 0; r < ITEMS; ++r)
    {
        const long long i = base + r*SORT_BLOCK + threadIdx.x;
        if (i < n) atomicAdd(&cnt[digit(keys[i])], 1u);
    }
    __syncthreads();
    hist[(long long)threadIdx.x*nblocks + blockIdx.x] = cnt[threadIdx.x];
}

// one block per digit: exclusive scan of its row of tile counts, and its total
__global__ __launch_bounds__(SORT_BLOCK) void k_radix_rows(unsigned int *hist, int nblocks, unsigned int *totals)
{
    __shared__ unsigned int waves[SCAN_BLOCK / WAVE];
    unsigned int *const row = hist + (long long)blockIdx.x*nblocks;
    unsigned int carry = 0;
    for (int base = 0; base < nblocks; base += SORT_BLOCK)
    {
        const int i = base + threadIdx.x;
        const unsigned int v = i < nblocks ? row[i] : 0u;
        unsigned int total;
        const unsigned int ex = block_exclusive(v, waves, total);
        if (i < nblocks) row[i] = carry + ex;
        carry += total;
    }
    if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

// where a tile's digits go: from the per-wavefront counts, cnt becomes each wavefront's offset inside the tile
// and to[] what a tile position of that digit is moved by; returns with both visible to the block
__device__ __forceinline__ void tile_offsets(unsigned int (*cnt)[RADIX], long long *to, const unsigned int *row_start,
                                             const unsigned int *totals, int digits, int nblocks, uint64_t *waves)
{
    const int t = threadIdx.x;
    __syncthreads();
    unsigned int tile = 0;
#pragma unroll
    for (int w = 0; w < SORT_WAVES; ++w) tile += cnt[w][t];
    const unsigned int all = t < digits ? totals[t] : 0u;
    const uint64_t before = prefix_256((uint64_t(all) << 32) | tile, waves);
    unsigned int run = unsigned(before);
    const unsigned int start = t < digits ? row_start[(long long)t*nblocks + blockIdx.x] : 0u;
    to[t] = (long long)(before >> 32) + start - run;
#pragma unroll
    for (int w = 0; w < SORT_WAVES; ++w)
    {
        const unsigned int c = cnt[w][t];
        cnt[w][t] = run;
        run += c;
    }
    __syncthreads();
}

// vals_in null: the records' values are their positions
template <int ITEMS>
__global__ __launch_bounds__(SORT_BLOCK) void k_radix_scatter(const uint64_t *keys_in, const int *vals_in, int n,
                                                             key_digit digit, const unsigned int *hist,
                                                             const unsigned int *totals, int nblocks,
                                                             uint64_t *keys_out, int *vals_out)
{
    constexpr int TILE = SORT_BLOCK*ITEMS;
    __shared__ unsigned int cnt[SORT_WAVES][RADIX];
    __shared__ long long to[RADIX];
    __shared__ uint64_t waves[SORT_WAVES];
    __shared__ uint64_t tile_key[TILE];
    __shared__ int tile_val[TILE];
    const int t = threadIdx.x, lane = t % WAVE, wave = t / WAVE;
#pragma unroll
    for (int w = 0; w < SORT_WAVES; ++w) cnt[w][t] = 0;
    __syncthreads();
    const long long base = (long long)blockIdx.x*TILE;
    const int count = int(min((long long)TILE, n - base));
    uint64_t key[ITEMS];
    int val[ITEMS];
    unsigned int rank[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r)
    {
        const int i = (wave*ITEMS + r)*WAVE + lane;
        const bool valid = i < count;
        key[r] = valid ? keys_in[base + i] : 0ull;
        val[r] = valid ? (vals_in ? vals_in[base + i] : int(base) + i) : 0;
    }
#pragma unroll
    for (int r = 0; r < ITEMS; ++r)
        rank[r] = wave_rank<8>(digit(key[r]), (wave*ITEMS + r)*WAVE + lane < count, cnt[wave], lane);
    tile_offsets(cnt, to, hist, totals, RADIX, nblocks, waves);
#pragma unroll
    for (int r = 0; r < ITEMS; ++r)
    {
        if ((wave*ITEMS + r)*WAVE + lane >= count) continue;
        const unsigned int at = cnt[wave][digit(key[r])] + rank[r];
        tile_key[at] = key[r];
        tile_val[at] = val[r];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r)
    {
        const int j = r*SORT_BLOCK + t;
        if (j >= count) continue;
        const uint64_t k = tile_key[j];
        const long long at = to[digit(k)] + j;
        keys_out[at] = k;
        vals_out[at] = tile_val[j];
    }
}

// The slot order is one such pass over the sorted records by (inactive, group), read from one byte per particle:
// slots of active owners by group, Morton order inside each; ghosts have no slot. It writes both maps itself,
// where sorting (key, particle) pairs wrote, read back and copied 120 MB more for 1e7 particles: 1.0 -> 0.39 ms.
constexpr int SLOT_INACTIVE = 64, SLOT_DIGITS = SLOT_BINS;
static_assert(SLOT_DIGITS == 2*SLOT_INACTIVE && LOCAL_GROUPS <= SLOT_INACTIVE, "a slot digit holds group and activity");

template <int ITEMS>
__global__ __launch_bounds__(SORT_BLOCK) void k_slot_hist(const int *sidx, const unsigned char *bin, int nr, int n,
                                                         unsigned int *hist, int nblocks)
{
    __shared__ unsigned int cnt[SLOT_DIGITS];
    if (threadIdx.x < SLOT_DIGITS) cnt[threadIdx.x] = 0;
    __syncthreads();
    const long long base = (long long)blockIdx.x*SORT_BLOCK*ITEMS;
    int p[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r)
    {
        const long long i = base + r*SORT_BLOCK + threadIdx.x;
        p[r] = i < nr ? sidx[i] : n;
    }
#pragma unroll
    for (int r = 0; r < ITEMS; ++r)
        if (p[r] < n) atomicAdd(&cnt[bin[p[r]]], 1u);
    __syncthreads();
    if (threadIdx.x < SLOT_DIGITS) hist[(long long)threadIdx.x*nblocks + blockIdx.x] = cnt[threadIdx.x];
}

template <int ITEMS>
__global__ __launch_bounds__(SORT_BLOCK) void k_slot_maps(const int *sidx, const unsigned char *bin, int nr, int n,
                                                         const unsigned int *hist, const unsigned int *totals,
                                                         int nblocks, int *slot_pidx, int *pidx_slot)
{
    constexpr int TILE = SORT_BLOCK*ITEMS;
    __shared__ unsigned int cnt[SORT_WAVES][RADIX];
    __shared__ long long to[RADIX];
    __shared__ uint64_t waves[SORT_WAVES];
    __shared__ int tile_p[TILE];
    __shared__ unsigned char tile_bin[TILE];
    __shared__ int placed;
    const int t = threadIdx.x, lane = t % WAVE, wave = t / WAVE;
#pragma unroll
    for (int w = 0; w < SORT_WAVES; ++w) cnt[w][t] = 0;
    if (t == 0) placed = 0;
    __syncthreads();
    const long long base = (long long)blockIdx.x*TILE;
    int p[ITEMS];
    unsigned int d[ITEMS], rank[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r)
    {
        const long long i = base + (wave*ITEMS + r)*WAVE + lane;
        p[r] = i < nr ? sidx[i] : n;
    }
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) d[r] = p[r] < n ? bin[p[r]] : 0u;
#pragma unroll
    for (int r = 0; r < ITEMS; ++r)
    {
        if (p[r] < n && d[r] >= SLOT_INACTIVE) pidx_slot[p[r]] = -1;
        rank[r] = wave_rank<6>(d[r], p[r] < n && d[r] < SLOT_INACTIVE, cnt[wave], lane);
    }
    tile_offsets(cnt, to, hist, totals, SLOT_INACTIVE, nblocks, waves);
    int mine = 0;
#pragma unroll
    for (int r = 0; r < ITEMS; ++r)
    {
        const bool valid = p[r] < n && d[r] < SLOT_INACTIVE;
        mine += __popcll(__ballot(valid));
        if (!valid) continue;
        const unsigned int at = cnt[wave][d[r]] + rank[r];
        tile_p[at] = p[r];
        tile_bin[at] = static_cast<unsigned char>(d[r]);
    }
    if (lane == 0) atomicAdd(&placed, mine);
    __syncthreads();
    const int count = placed;
#pragma unroll
    for (int r = 0; r < ITEMS; ++r)
    {
        const int j = r*SORT_BLOCK + t;
        if (j >= count) continue;
        const int q = tile_p[j], s = int(to[tile_bin[j]] + j);
        slot_pidx[s] = q;
        pidx_slot[q] = s;
    }
}

// ============================================================================================
// collision sites (src/swarm/col_site_init.cu:79-118) and spatial groups (col_space_bin.cu:11-35)
// ============================================================================================
__device__ __forceinline__ bool is_active(double y, double z)
{
    if (y < Y_MIN || y >= Y_MAX) return false;
#ifdef HALF_DISK
    if (N_Z > 1 && (z < Z_MIN || z > Z_MAX)) return false;
#else
    if (N_Z > 1 && (z < Z_MIN || z >= Z_MAX)) return false;
#endif
    return true;
}

__device__ __forceinline__ int space_bin(double x, double y, double z)
{
    int bin_x = 0;
    int bin_y = static_cast<int>(floor((y - Y_MIN) / (Y_MAX - Y_MIN)*COL_BIN_Y));
    int bin_z = 0;
    if constexpr (N_X > 1) bin_x = static_cast<int>(floor((x - X_MIN) / (X_MAX - X_MIN)*COL_BIN_X));
    if constexpr (N_Z > 1)
    {
        double extent_z = Z_MAX - Z_MIN;
        bin_z = static_cast<int>(floor((z - Z_MIN) / extent_z*COL_BIN_Z));
    }
    bin_x = (bin_x < 0) ? 0 : ((bin_x >= COL_BIN_X) ? COL_BIN_X - 1 : bin_x);
    bin_y = (bin_y < 0) ? 0 : ((bin_y >= COL_BIN_Y) ? COL_BIN_Y - 1 : bin_y);
    bin_z = (bin_z < 0) ? 0 : ((bin_z >= COL_BIN_Z) ? COL_BIN_Z - 1 : bin_z);
    constexpr int count_x = (N_X > 1) ? COL_BIN_X : 1;
    return bin_x + count_x*(bin_y + COL_BIN_Y*bin_z);
}

__global__ __launch_bounds__(256) void k_site_init(bound_state u, int n, float4 *pts, unsigned char *active,
                                                  unsigned char *group, unsigned char *bin, int *bad)
{
    long long i = (long long)blockIdx.x*blockDim.x + threadIdx.x;
    if (i >= n) return;
    double x = ld(u.x, i), y = ld(u.y, i), z = ld(u.z, i);
    bool finite = isfinite(x) && isfinite(y) && isfinite(z) && isfinite(ld(u.size, i)) && isfinite(ld(u.numr, i));
    if (u.vx.base) finite = finite && isfinite(ld(u.vx, i)) && isfinite(ld(u.vy, i)) && isfinite(ld(u.vz, i));
    if (!finite)
    {
        active[i] = 0;
        group[i] = 0;
        bin[i] = SLOT_INACTIVE;
        pts[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        atomicMin(bad, int(i) + 1);
        return;
    }
    bool act = is_active(y, z);
    double R = cyl_R(y, z);
    double Z = cyl_Z(y, z);
    float4 p;
    if (N_X == 1 && N_Z == 1) p = make_float4(static_cast<float>(R), 0.0f, 0.0f, 0.0f);
    else p = make_float4(static_cast<float>(R*cos(x)), static_cast<float>(R*sin(x)), static_cast<float>(Z), 0.0f);
    p.w = act ? static_cast<float>(H_SEARCH*hg(R)*R) : 0.0f;
    pts[i] = p;
    active[i] = static_cast<unsigned char>(act);
    const int g = space_bin(x, y, z);
    group[i] = static_cast<unsigned char>(g);
    bin[i] = static_cast<unsigned char>(act ? g : g | SLOT_INACTIVE);
}

// ============================================================================================
// Morton keys and the adaptive hierarchy (inc/swarm/morton/morton_index.cuh:41-145)
// ============================================================================================
__device__ __forceinline__ uint64_t expand3(uint32_t v)
{
    uint64_t b = v & 0x1fffffu;
    b = (b | b << 32) & 0x001f00000000ffffULL;
    b = (b | b << 16) & 0x001f0000ff0000ffULL;
    b = (b | b << 8)  & 0x100f00f00f00f00fULL;
    b = (b | b << 4)  & 0x10c30c30c30c30c3ULL;
    b = (b | b << 2)  & 0x1249249249249249ULL;
    return b;
}

__global__ __launch_bounds__(256) void k_morton_keys(const float4 *pts, int n, float ox, float oy, float oz,
                                                    float width, int max_level, int dim, uint64_t *keys)
{
    long long i = (long long)blockIdx.x*blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4 p = pts[i];
    int cells = 1 << max_level;
    float scale = static_cast<float>(cells) / width;
    int ix = min(cells - 1, max(0, static_cast<int>((p.x - ox)*scale)));
    int iy = min(cells - 1, max(0, static_cast<int>((p.y - oy)*scale)));
    int iz = (dim == 2) ? 0 : min(cells - 1, max(0, static_cast<int>((p.z - oz)*scale)));
    keys[i] = expand3(uint32_t(ix)) | (expand3(uint32_t(iy)) << 1) | (expand3(uint32_t(iz)) << 2);
}

// sorted record m carries its code 3*i + image; the activity of physical particle i marks it. Every
// CHUNK consecutive records also get the tight box of their active ones (empty, lo > hi, without any):
// the search skips the chunks of a leaf that no query of the wavefront can use.
__global__ __launch_bounds__(256) void k_records(const int *sidx, const float4 *pts, const unsigned char *active,
                                                const int *codes, int n, float4 *rec, gdx_box *chunk)
{
    const long long m = (long long)blockIdx.x*blockDim.x + threadIdx.x;
    float lo[3], hi[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) { lo[a] = __builtin_inff(); hi[a] = -__builtin_inff(); }
    if (m < n)
    {
        int p = sidx[m];
        float4 q = pts[p];
        int code = codes ? codes[p] : 3*p;
        if (active && !active[code / 3])
        {
            // no coordinates: no distance to it passes a test
            rec[m] = make_float4(__builtin_nanf(""), __builtin_nanf(""), __builtin_nanf(""),
                                 __int_as_float(code | int(0x80000000u)));
        }
        else
        {
            rec[m] = make_float4(q.x, q.y, q.z, __int_as_float(code));
            lo[0] = hi[0] = q.x;
            lo[1] = hi[1] = q.y;
            lo[2] = hi[2] = q.z;
        }
    }
#pragma unroll
    for (int a = 0; a < 3; ++a)
    {
#pragma unroll
        for (int o = 1; o < CHUNK; o <<= 1)
        {
            lo[a] = fminf(lo[a], __shfl_xor(lo[a], o, WAVE));
            hi[a] = fmaxf(hi[a], __shfl_xor(hi[a], o, WAVE));
        }
    }
    if (m < n && threadIdx.x % CHUNK == 0)
        chunk[m / CHUNK] = gdx_box{lo[0], lo[1], lo[2], 0, hi[0], hi[1], hi[2], 0};
}

// ============================================================================================
// azimuthal wedge: periodic ghosts (inc/swarm/morton/morton_ghost.cuh:28-86)
// ============================================================================================
// Cartesian distance from a record to the radial half-plane at azimuth offset `off` from it
// (_get_morton_seam_dist, morton_ghost.cuh:28-35)
__device__ __forceinline__ float seam_dist(float px, float py, float off)
{
    float R = hypotf(px, py);
    return (cosf(off) >= 0.0f) ? R*fabsf(sinf(off)) : R;
}

// largest search cap of the epoch (the max_element of swarm_runtime.cu:413-414); caps are >= 0
__global__ __launch_bounds__(256) void k_cap_max(const float4 *pts, int n, unsigned int *out)
{
    long long i = (long long)blockIdx.x*blockDim.x + threadIdx.x;
    float w = i < n ? pts[i].w : 0.0f;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) w = fmaxf(w, __shfl_xor(w, o, WAVE));
    if (threadIdx.x % WAVE == 0) atomicMax(out, __float_as_uint(w));
}

// ghosts per particle: one for each seam whose distance is within the largest cap (morton_gcount)
__global__ __launch_bounds__(256) void k_ghost_count(bound_state u, const float4 *pts, int n, float q_max,
                                                    float x_min, float x_max, unsigned int *count)
{
    long long i = (long long)blockIdx.x*blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4 p = pts[i];
    float posx = static_cast<float>(ld(u.x, i));
    unsigned c = 0;
    if (seam_dist(p.x, p.y, posx - x_min) <= q_max) ++c;
    if (seam_dist(p.x, p.y, x_max - posx) <= q_max) ++c;
    count[i] = c;
}

// physical records first (code 3i), then each particle's ghosts at n + offset: image 2 rotated by
// +width near x_min, image 1 rotated by -width near x_max (morton_gwrite); the rotation's sine and
// cosine are computed once on the host
__global__ __launch_bounds__(256) void k_ghost_write(bound_state u, const float4 *pts, int n, const unsigned int *off,
                                                    float q_max, float x_min, float x_max, float cw, float sw,
                                                    float4 *rec, int *code)
{
    long long i = (long long)blockIdx.x*blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4 p = pts[i];
    rec[i] = p;
    code[i] = 3*int(i);
    float posx = static_cast<float>(ld(u.x, i));
    long long g = n + off[i];
    if (seam_dist(p.x, p.y, posx - x_min) <= q_max)
    {
        rec[g] = make_float4(cw*p.x - sw*p.y, sw*p.x + cw*p.y, p.z, 0.0f);
        code[g] = 3*int(i) + 2;
        ++g;
    }
    if (seam_dist(p.x, p.y, x_max - posx) <= q_max)
    {
        rec[g] = make_float4(cw*p.x + sw*p.y, -sw*p.x + cw*p.y, p.z, 0.0f);
        code[g] = 3*int(i) + 1;
    }
}

// The adaptive hierarchy straight from the sorted keys: a node of level L begins at a record whose key differs
// from the one before it above level L, and exists if its parent's cell holds more than the leaf target. So each
// record knows by itself at which levels it begins nodes, a scan of the counts (level by level, 256 records a
// count) numbers the nodes breadth first, and they are written in any order: five launches and no turn of the
// host, however many levels there are. 0.39 ms for 1e7 records and 66 us for 65536; level by level, with a count,
// a scan, the host's read of the frontier's size and an expansion for each, the kernels alone took 0.9 and 0.24 ms.
constexpr int NODE_ROUNDS = 4;
constexpr int NODE_UNIT = NODE_ROUNDS*WAVE;       // records per wavefront

// leading levels that two keys share
__device__ __forceinline__ int shared_levels(uint64_t a, uint64_t b, int max_level)
{
    const uint64_t x = a ^ b;
    return x ? max_level - 1 - (63 - __clzll(static_cast<long long>(x))) / 3 : max_level;
}

// record i begins the nodes of levels x + 1 ... y (none if y <= x)
__device__ __forceinline__ int2 begun_levels(const uint64_t *keys, int n, int i, int leaf_target, int max_level)
{
    const uint64_t key = keys[i];
    const bool ahead = (long long)i + leaf_target < n;
    int above = 0;                               // levels shared with the record before
    if (i > 0)
    {
        above = shared_levels(keys[i - 1], key, max_level);
        if (above == max_level) return make_int2(above, above);
        // whether the cell of that level, which record i - 1 is in, holds more than leaf_target records
        const int shift = 3*(max_level - above);
        const uint64_t cell = key >> shift;
        int lo = i > leaf_target ? i - leaf_target : 0, hi = i - 1;     // its first record, if not before lo
        if (keys[lo] >> shift != cell)
        {
            ++lo;
            while (lo < hi)
            {
                const int mid = lo + (hi - lo) / 2;
                if (keys[mid] >> shift == cell) hi = mid;
                else lo = mid + 1;
            }
        }
        if ((long long)lo + leaf_target >= n || keys[lo + leaf_target] >> shift != cell) return make_int2(above, above);
    }
    else if (!ahead) return make_int2(0, 0);
    const int deeper = ahead ? shared_levels(key, keys[i + leaf_target], max_level) : -1;
    return make_int2(above, min(max_level, max(above, deeper) + 1));
}

__global__ __launch_bounds__(256) void k_node_counts(const uint64_t *keys, int n, int leaf_target, int max_level,
                                                    int units, unsigned int *counts)
{
    const int unit = (blockIdx.x*256 + threadIdx.x) / WAVE, lane = threadIdx.x % WAVE;
    if (unit >= units) return;
    int2 v[NODE_ROUNDS];
#pragma unroll
    for (int r = 0; r < NODE_ROUNDS; ++r)
    {
        const long long i = (long long)unit*NODE_UNIT + r*WAVE + lane;
        v[r] = i < n ? begun_levels(keys, n, int(i), leaf_target, max_level) : make_int2(0, 0);
    }
    for (int L = 1; L <= max_level; ++L)
    {
        int c = 0;
#pragma unroll
        for (int r = 0; r < NODE_ROUNDS; ++r) c += __popcll(__ballot(v[r].x < L && L <= v[r].y));
        if (lane == 0) counts[(long long)(L - 1)*units + unit] = c;
    }
    if (unit == 0 && lane == 0) counts[(long long)max_level*units] = 0u;
}

// offsets: the exclusive scan of the counts, its last entry the number of nodes below the root. Nodes past `cap`
// are not written: the host compares the number with the capacity.
__global__ __launch_bounds__(256) void k_node_write(const uint64_t *keys, int n, int leaf_target, int max_level,
                                                   int dim, float ox, float oy, float oz, float width, int units,
                                                   const unsigned int *offsets, unsigned int cap, gdx_node *nodes,
                                                   unsigned int *masks, unsigned int *total)
{
    const int unit = (blockIdx.x*256 + threadIdx.x) / WAVE, lane = threadIdx.x % WAVE;
    if (unit >= units) return;
    if (unit == 0 && lane == 0)
    {
        nodes[0] = gdx_node{ox, oy, oz, width, 0, n, -1, 0};
        *total = offsets[(long long)max_level*units];
    }
    int2 v[NODE_ROUNDS];
    unsigned int in[NODE_ROUNDS];                // the node of the level above that holds the record
    bool any = false;
#pragma unroll
    for (int r = 0; r < NODE_ROUNDS; ++r)
    {
        const long long i = (long long)unit*NODE_UNIT + r*WAVE + lane;
        v[r] = i < n ? begun_levels(keys, n, int(i), leaf_target, max_level) : make_int2(0, 0);
        in[r] = 0u;
        any = any || v[r].y > v[r].x;
    }
    if (!__ballot(any)) return;
    for (int L = 1; L <= max_level; ++L)
    {
        unsigned int next = 1u + offsets[(long long)(L - 1)*units + unit];
#pragma unroll
        for (int r = 0; r < NODE_ROUNDS; ++r)
        {
            const bool begins = v[r].x < L && L <= v[r].y;
            const unsigned long long m = __ballot(begins);
            const unsigned int at = next + __popcll(m & lanemask_lt(lane));
            next += __popcll(m);
            const unsigned int parent = in[r];
            in[r] = begins ? at : at - 1u;
            if (!begins || at >= cap) continue;
            const int i = unit*NODE_UNIT + r*WAVE + lane;
            const uint64_t key = keys[i];
            const int shift = 3*(max_level - L);
            const uint64_t cell = key >> shift;
            // end of the cell: within leaf_target records, or beyond them
            int lo = i + 1, hi = int(min((long long)i + leaf_target, (long long)n));
            if (hi < n && keys[hi] >> shift == cell) { lo = hi + 1; hi = n; }
            while (lo < hi)
            {
                const int mid = lo + (hi - lo) / 2;
                if (keys[mid] >> shift == cell) lo = mid + 1;
                else hi = mid;
            }
            float w = width, lx = ox, ly = oy, lz = oz;
            for (int l = 1; l <= L; ++l)
            {
                const unsigned code = unsigned(key >> (3*(max_level - l)));
                w = 0.5f*w;
                if (code & 1u) lx += w;
                if (code & 2u) ly += w;
                if (dim == 3 && (code & 4u)) lz += w;
            }
            nodes[at] = gdx_node{lx, ly, lz, w, i, lo - i, -1, 0};
            if (L - 1 > v[r].x || i == 0) nodes[parent].first_child = int(at);
            atomicOr(masks + parent, 1u << (unsigned(cell) & 7u));
        }
    }
}

// ============================================================================================
// exact top-K: one lane per query, 64 Morton-consecutive queries per wavefront share one
// traversal of the hierarchy's boxes
// ============================================================================================
constexpr int TOPK_BLOCK = 256;
// a popped node of level l pushes at most its eight children: 20 levels hold at most 20*7 + 1 entries
constexpr int TOPK_STACK = 160;

__device__ __forceinline__ bool nb_less(float da, int ia, float db, int ib)   // morton_types.cuh:68-72
{ return da < db || (da == db && ia < ib); }

// box of a hierarchy node as the search reads it: its cube padded against the rounding of the keys
// (morton_index.cuh:296-314), open in z for a two-dimensional index, and where its children or its records
// are. Formed once per build: the pad alone is some fifteen instructions, and a node is tested by several
// wavefronts.
__global__ __launch_bounds__(256) void k_node_boxes(gdx_node *nodes, const unsigned int *masks,
                                                   const unsigned int *total, unsigned int cap, int dim,
                                                   int max_level, gdx_box *box)
{
    const unsigned int i = blockIdx.x*blockDim.x + threadIdx.x;
    if (i >= cap || i > *total) return;
    gdx_node nd = nodes[i];
    const unsigned int mask = masks[i];
    // child codes in bits 8..15 beside the child count (bits 0..3)
    nd.child_count = __popc(mask) | int(mask << 8);
    nodes[i].child_count = nd.child_count;
    const float ux = nd.lx + nd.width, uy = nd.ly + nd.width, uz = nd.lz + nd.width;
    const float scale = fmaxf(1.0f, fmaxf(fmaxf(fabsf(nd.lx), fabsf(ux)),
        fmaxf(fmaxf(fabsf(nd.ly), fabsf(uy)), fmaxf(fabsf(nd.lz), fabsf(uz)))));
    const float pad = 2.0f*static_cast<float>(max_level + 2)*FLT_EPSILON*scale;
    const int nch = nd.child_count & 15;
    gdx_box b{nd.lx - pad, nd.ly - pad, nd.lz - pad, nch ? nd.first_child : nd.begin,
              ux + pad, uy + pad, uz + pad, nch ? nch : -nd.count};
    if (dim == 2) { b.lz = -__builtin_inff(); b.hz = __builtin_inff(); }
    box[i] = b;
}

// two boxes, or four records, by one scalar load at a uniform address (field by field the compiler moves
// each to its use and waits there again)
typedef float f32x16 __attribute__((ext_vector_type(16), aligned(16)));
// boxes read together; the box arrays hold as many more than they have boxes
constexpr int BOX_GROUP = 4;

// squared distance of a point to a box, rounded differently from the records' distances: reach() widens
// the limit it is compared with, so that no record within the limit lies in a rejected box
__device__ __forceinline__ float box_d2(float qx, float qy, float qz, float lx, float ly, float lz, float hx, float hy,
                                        float hz)
{
    const float dx = fmaxf(fmaxf(lx - qx, qx - hx), 0.0f);
    const float dy = fmaxf(fmaxf(ly - qy, qy - hy), 0.0f);
    const float dz = fmaxf(fmaxf(lz - qz, qz - hz), 0.0f);
    return fmaf(dz, dz, fmaf(dy, dy, dx*dx));
}

// the first `count` of the boxes [p, p + BOX_GROUP) that some lane's point reaches within its limit, as a mask
__device__ __forceinline__ unsigned boxes_reached(const gdx_box *p, int count, float qx, float qy, float qz, float lim)
{
    const f32x16 *g = reinterpret_cast<const f32x16 *>(p);
    const f32x16 v[BOX_GROUP / 2] = {g[0], g[1]};
    unsigned mask = 0u;
#pragma unroll
    for (int u = 0; u < BOX_GROUP; ++u)
    {
        const f32x16 &w = v[u / 2];
        const int o = 8*(u % 2);
        const float d2 = box_d2(qx, qy, qz, w[o], w[o + 1], w[o + 2], w[o + 4], w[o + 5], w[o + 6]);
        if (__ballot(d2 <= lim)) mask |= 1u << u;
    }
    return __builtin_amdgcn_readfirstlane(mask & ((2u << min(count - 1, BOX_GROUP - 1)) - 1u));
}

// |rounding| of both sums is below 3 ulp of the larger, or 2^-148 where they are subnormal; a negative
// limit (a lane without a query) stays negative
__device__ __forceinline__ float reach(float lim) { return lim < 0.0f ? lim : fmaf(lim, 1.000001f, 1.0e-37f); }

// insert (nd, nc) into the ascending list; precondition: it precedes the current last entry
template <int K>
__device__ __forceinline__ void topk_insert(float (&d)[K], int (&c)[K], float nd, int nc)
{
    bool carry = true;
#pragma unroll
    for (int k = K - 1; k > 0; --k)
    {
        bool lt = nb_less(nd, nc, d[k - 1], c[k - 1]);
        float dk = lt ? d[k - 1] : (carry ? nd : d[k]);
        int ck = lt ? c[k - 1] : (carry ? nc : c[k]);
        d[k] = dk;
        c[k] = ck;
        carry = lt;
    }
    if (carry) { d[0] = nd; c[0] = nc; }
}

// insert (nd, nc) keeping one entry per physical particle (code / 3): an entry of the same particle is
// replaced when the candidate precedes it, else the candidate is dropped. The list stays the K first of
// the candidates seen so far with each particle collapsed to its nearest image, which is what the
// reference's 3K candidates with duplicate removal (morton_query.cuh:62-140) select: every record up
// to the K-th particle's distance belongs to one of those K particles, so at most 3K records precede
// it. Precondition as topk_insert.
template <int K>
__device__ __forceinline__ void topk_insert_dedup(float (&d)[K], int (&c)[K], float nd, int nc)
{
    const unsigned pn = static_cast<unsigned>(nc) / 3u;
    int e = -1;
    float de = 0.0f;
    int ce = 0;
#pragma unroll
    for (int k = 0; k < K; ++k)
    {
        const bool same = e < 0 && c[k] != INT_MAX && static_cast<unsigned>(c[k]) / 3u == pn;
        e = same ? k : e;
        de = same ? d[k] : de;
        ce = same ? c[k] : ce;
    }
    if (e >= 0)
    {
        if (!nb_less(nd, nc, de, ce)) return;
#pragma unroll
        for (int k = 0; k < K - 1; ++k)
        {
            d[k] = k >= e ? d[k + 1] : d[k];
            c[k] = k >= e ? c[k + 1] : c[k];
        }
        d[K - 1] = __builtin_inff();
        c[K - 1] = INT_MAX;
    }
    topk_insert<K>(d, c, nd, nc);
}

__device__ __forceinline__ float readlane_f(float v, int l)
{ return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); }

// Traversal shared by both selection schemes: the wavefront pops nodes from one LDS stack, children
// nearest-first from the wavefront's centre, and pushes only the nodes some lane needs; every popped leaf
// goes to leaf(begin, end). cut() is the lane's current pruning distance (the smaller of its cap and its
// K-th candidate so far, negative for a lane without a query). A stack entry holds the node's children or
// records itself, so that a pop reads no node: testing a popped node again would spare one pop in twenty.
// The children's boxes come through scalar loads, and once more as one box per lane for their distances
// from the centre.
template <class Cut, class Leaf>
__device__ __forceinline__ void traverse(const gdx_box *__restrict__ boxes, float qx, float qy, float qz, bool qactive,
                                         float cx, float cy, float cz, int2 *stack, unsigned int *overflow, Cut cut_of,
                                         Leaf leaf)
{
    const int lane = threadIdx.x % WAVE;
    if (__ballot(qactive) == 0ull) return;
    int sp = 0;
    int first = boxes[0].first, info = boxes[0].info;
    while (true)
    {
        if (info < 0)
        {
            leaf(first, first - info);
        }
        else
        {
            // children some lane needs, each child's distance from the wavefront's centre kept by the lane of
            // its index; the needed children go on the stack farthest first (nearest on top, equal distances
            // in child order), each lane writing its own child at its rank
            const int nch = info;
            const gdx_box mine = boxes[first + min(lane, nch - 1)];
            const float lim = reach(cut_of());
            unsigned needed = boxes_reached(boxes + first, nch, qx, qy, qz, lim);
            if (nch > BOX_GROUP)
                needed |= boxes_reached(boxes + first + BOX_GROUP, nch - BOX_GROUP, qx, qy, qz, lim) << BOX_GROUP;
            int nv = __popc(needed);
            if (sp + nv > TOPK_STACK)
            {
                if (lane == 0) atomicOr(overflow, 1u);
                nv = 0;
            }
            const float kd = box_d2(cx, cy, cz, mine.lx, mine.ly, mine.lz, mine.hx, mine.hy, mine.hz);
            int rank = 0;
            for (unsigned rest = needed; rest; rest &= rest - 1u)
            {
                const int m = __builtin_ctz(rest);
                const float km = readlane_f(kd, m);
                rank += km < kd || (km == kd && m < lane);
            }
            if (nv > 0 && lane < nch && ((needed >> lane) & 1u))
                stack[sp + nv - 1 - rank] = make_int2(mine.first, mine.info);
            sp += nv;
            __builtin_amdgcn_wave_barrier();
        }
        sp = __builtin_amdgcn_readfirstlane(sp);
        if (sp == 0) break;
        --sp;
        const int2 e = stack[sp];
        first = __builtin_amdgcn_readfirstlane(e.x);
        info = __builtin_amdgcn_readfirstlane(e.y);
        __builtin_amdgcn_wave_barrier();
    }
}

// insertion scheme: every eligible record goes through the lane's sorted K-entry register list
template <int K, bool DEDUP = false>
__device__ void topk_wave(const float4 *rec, const gdx_box *__restrict__ boxes, float qx, float qy, float qz, float q2,
                          bool qactive, float cx, float cy, float cz, float (&d)[K], int (&c)[K], int2 *stack,
                          unsigned int *overflow)
{
    const int lane = threadIdx.x % WAVE;
    const float cap = qactive ? q2 : -1.0f;
#pragma unroll
    for (int k = 0; k < K; ++k) { d[k] = __builtin_inff(); c[k] = INT_MAX; }
    traverse(boxes, qx, qy, qz, qactive, cx, cy, cz, stack, overflow,
             [&] { return fminf(cap, d[K - 1]); },
             [&](int begin, int end) {
                 for (int t0 = begin; t0 < end; t0 += WAVE)
                 {
                     int idx = t0 + lane;
                     float4 v = idx < end ? rec[idx] : make_float4(0.f, 0.f, 0.f, __int_as_float(-1));
                     int cnt = min(WAVE, end - t0);
                     for (int j = 0; j < cnt; ++j)
                     {
                         float px = readlane_f(v.x, j), py = readlane_f(v.y, j), pz = readlane_f(v.z, j);
                         int code = __builtin_amdgcn_readlane(__float_as_int(v.w), j);
                         float dx = qx - px, dy = qy - py, dz = qz - pz;
                         float d2 = dx*dx + dy*dy + dz*dz;
                         bool e = code >= 0 && d2 <= cap && nb_less(d2, code, d[K - 1], c[K - 1]);
                         if (e)
                         {
                             if constexpr (DEDUP) topk_insert_dedup<K>(d, c, d2, code);
                             else topk_insert<K>(d, c, d2, code);
                         }
                     }
                 }
             });
}

// ---- tiled scheme: candidates collected per lane in LDS, merged B at a time (gdx_topk.h) ----
// the lane's `cnt` buffered keys buf[r * WAVE] merged into L. A slot past the count becomes a key above
// TOPK_EMPTY by its upper word alone: no list entry is larger, so it never enters one.
constexpr uint32_t TOPK_NO_KEY = 0x7fe00000u;
constexpr unsigned TILE_ROW = WAVE*sizeof(uint64_t);      // bytes of one key per lane

template <int K, int B>
__device__ __forceinline__ void topk_flush(uint64_t (&L)[K], const char *col, int cnt)
{
    uint64_t S[B];
#pragma unroll
    for (int r = 0; r < B; ++r)
    {
        const uint64_t v = *reinterpret_cast<const uint64_t *>(col + r*TILE_ROW);
        const uint32_t hi = r < cnt ? uint32_t(v >> 32) : TOPK_NO_KEY;
        S[r] = (uint64_t(hi) << 32) | uint32_t(v);
    }
    odd_even_sort<B>(S);
    topk_merge_sorted<K, B>(L, S);
}

// tiled scheme: a record passes the lane's filter when it lies within the cap and precedes the lane's
// K-th key as of its last merge (a stale, hence larger, cutoff: the filter keeps a superset of the
// records the exact list would take); passing keys are appended to the lane's column of an LDS buffer
// and the wavefront merges every lane's buffer once some lane holds B. The K smallest keys of a union do
// not depend on the order of merging, so the result is the insertion scheme's, bit for bit.
// records per overflow check of the tiled scheme: a merge runs before a group when some lane could not
// take all of it
constexpr int TILE_GROUP = 4;             // one f32x16

template <int K, int B>
__device__ void topk_wave_tiled(const float4 *__restrict__ rec, const gdx_box *__restrict__ boxes,
                                const gdx_box *__restrict__ chunks, float qx, float qy, float qz, float q2,
                                bool qactive, float cx, float cy, float cz, float (&d)[K], int (&c)[K], int2 *stack,
                                uint64_t *buf, unsigned int *overflow)
{
    const int lane = threadIdx.x % WAVE;
    const float cap = qactive ? q2 : -1.0f;
    uint64_t L[K];
#pragma unroll
    for (int k = 0; k < K; ++k) L[k] = TOPK_EMPTY;
    char *tile = reinterpret_cast<char *>(buf);
    const unsigned col = lane*unsigned(sizeof(uint64_t));
    unsigned put = col;                       // byte offset of the lane's next free slot
    // the lane's cap and the distance of its K-th key as of its last merge; ties at that distance pass and
    // the merge decides them
    float lim = fminf(cap, __uint_as_float(uint32_t(L[K - 1] >> 32)));
    float far = reach(lim);
    auto merge = [&] {
        topk_flush<K, B>(L, tile + col, int((put - col)/TILE_ROW));
        put = col;
        lim = fminf(cap, __uint_as_float(uint32_t(L[K - 1] >> 32)));
        far = reach(lim);
    };
    // inactive records hold no coordinates (k_records): their distance is NaN and passes nothing
    auto test = [&](float x, float y, float z, float code) {
        const float dx = qx - x, dy = qy - y, dz = qz - z;
        const float d2 = dx*dx + dy*dy + dz*dz;
        if (d2 <= lim)
        {
            *reinterpret_cast<uint64_t *>(tile + put) = (uint64_t(__float_as_uint(d2)) << 32)
                | __float_as_uint(code);
            put += TILE_ROW;
        }
    };
    traverse(boxes, qx, qy, qz, qactive, cx, cy, cz, stack, overflow, [&] { return lim; },
             [&](int begin, int end) {
                 const int last = (end - 1) / CHUNK;
                 for (int c0 = begin / CHUNK; c0 <= last; c0 += BOX_GROUP)
                 {
                     unsigned needed = boxes_reached(chunks + c0, last - c0 + 1, qx, qy, qz, far);
                     for (; needed; needed &= needed - 1u)
                     {
                         // the chunk's records inside the leaf, at uniform addresses (scalar loads), four
                         // together where the leaf holds them
                         const int at = (c0 + __builtin_ctz(needed))*CHUNK;
                         const int t1 = min(end, at + CHUNK);
                         for (int t = max(begin, at); t < t1; t += TILE_GROUP)
                         {
                             if (__ballot(put > col + (B - TILE_GROUP)*TILE_ROW)) merge();
                             if (t + TILE_GROUP <= t1)
                             {
                                 const f32x16 v = *reinterpret_cast<const f32x16 *>(rec + t);
#pragma unroll
                                 for (int u = 0; u < TILE_GROUP; ++u)
                                     test(v[4*u], v[4*u + 1], v[4*u + 2], v[4*u + 3]);
                             }
                             else
                             {
                                 for (int r = t; r < t1; ++r)
                                 {
                                     const float4 v = rec[r];
                                     test(v.x, v.y, v.z, v.w);
                                 }
                             }
                         }
                     }
                 }
             });
    if (__ballot(put > col)) merge();
#pragma unroll
    for (int k = 0; k < K; ++k)
    {
        d[k] = __uint_as_float(uint32_t(L[k] >> 32));
        c[k] = int(uint32_t(L[k]));
    }
}

__device__ __forceinline__ void wave_centre(float qx, float qy, float qz, bool qactive, float &cx, float &cy, float &cz)
{
    float lo[3] = {qactive ? qx : __builtin_inff(), qactive ? qy : __builtin_inff(), qactive ? qz : __builtin_inff()};
    float hi[3] = {qactive ? qx : -__builtin_inff(), qactive ? qy : -__builtin_inff(), qactive ? qz : -__builtin_inff()};
#pragma unroll
    for (int a = 0; a < 3; ++a)
    {
#pragma unroll
        for (int m = 32; m > 0; m >>= 1)
        {
            lo[a] = fminf(lo[a], __shfl_xor(lo[a], m, WAVE));
            hi[a] = fmaxf(hi[a], __shfl_xor(hi[a], m, WAVE));
        }
    }
    cx = 0.5f*(lo[0] + hi[0]);
    cy = 0.5f*(lo[1] + hi[1]);
    cz = 0.5f*(lo[2] + hi[2]);
}

// col_cache_get (inc/swarm/_col_cache.cuh:73-159) over Morton-ordered queries
// one query per physical record; DEDUP when two images of one particle can share a search ball
// TILE = 0: the insertion scheme; TILE = B > 0: the tiled scheme with B-key merges (no image dedup);
// WPB wavefronts per block (the block shape: every wavefront runs its own queries with its own LDS
// stack and tile, so the shape changes only how the wavefronts are packed onto the CUs)
template <bool DEDUP, int TILE, int WPB>
__global__ __launch_bounds__(WPB*WAVE) void k_col_topk(const float4 *__restrict__ rec,
                                                        const gdx_box *__restrict__ boxes,
                                                        const gdx_box *__restrict__ chunks, int n,
                                                        const int *__restrict__ sidx,
                                                        const float4 *__restrict__ pts,
                                                        const int *__restrict__ pidx_slot,
                                                        const unsigned char *__restrict__ group,
                                                        bound_state u, int *__restrict__ nbr,
                                                        double *__restrict__ measure,
                                                        unsigned long long *__restrict__ graph,
                                                        unsigned int *__restrict__ overflow,
                                                        unsigned char *__restrict__ nbr_image,
                                                        unsigned long long *__restrict__ again, float image_d2)
{
    static_assert(!(DEDUP && TILE), "image dedup runs on the insertion scheme");
    static_assert(TILE == 0 || TILE >= TILE_GROUP, "a merge tile holds at least one record group");
    __shared__ int2 stacks[WPB][TOPK_STACK];
    __shared__ uint64_t tiles[WPB][TILE > 0 ? TILE : 1][WAVE];
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
    long long m = ((long long)xcd_block()*WPB + wave)*WAVE + lane;
    bool valid = m < n;
    float4 me = valid ? rec[m] : make_float4(0.f, 0.f, 0.f, __int_as_float(-1));
    int code = __float_as_int(me.w);
    bool qactive = valid && code >= 0 && (!X_WEDGE || code % 3 == 0);
    if constexpr (DEDUP)
    {
        // after a tiled pass: only the queries it left
        if (again) qactive = qactive && ((again[m / WAVE] >> lane) & 1ull);
        if (__ballot(qactive) == 0ull) return;
    }
    int p = valid ? sidx[m] : 0;
    float q = qactive ? pts[p].w : 0.0f;
    float q2 = q*q;
    float cx, cy, cz;
    wave_centre(me.x, me.y, me.z, qactive, cx, cy, cz);
    float d[N_K];
    int c[N_K];
    if constexpr (TILE > 0)
        topk_wave_tiled<N_K, TILE>(rec, boxes, chunks, me.x, me.y, me.z, q2, qactive, cx, cy, cz, d, c, stacks[wave],
                                   &tiles[wave][0][0], overflow);
    else
        topk_wave<N_K, DEDUP>(rec, boxes, me.x, me.y, me.z, q2, qactive, cx, cy, cz, d, c, stacks[wave], overflow);
    unsigned long long mask = 0ull;
    const int g = qactive ? int(group[p]) : -1;
    auto write = [&]() {
        int s = pidx_slot[p];
        float max_d2 = 0.0f;
        int row[N_K];
#pragma unroll
        for (int k = 0; k < N_K; ++k)
        {
            if (c[k] != INT_MAX)
            {
                max_d2 = fmaxf(max_d2, d[k]);
                int j = c[k] / 3;
                row[k] = pidx_slot[j];
                mask |= 1ull << group[j];
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
                const int k = bitrev_slot(t);
                nbr_image[(long long)s*N_K + t] = static_cast<unsigned char>(c[k] != INT_MAX ? c[k] % 3 : 0);
            }
        }
        double radius = sqrt(static_cast<double>(max_d2));
        measure[s] = ball_measure(ld(u.y, p), ld(u.z, p), radius);
    };
    if constexpr (X_WEDGE && !DEDUP)
    {
        // Two images of one particle both in a list lie within twice the list's radius of each other. A list
        // whose diameter is below the least distance of two images of any particle therefore holds every
        // particle once and is what the search with removal would give; the caps that make the removal
        // necessary are mostly far larger than the lists. The other queries (a list that is not full reaches
        // to the cap) are left to a second pass with removal, as a mask per wavefront. Wedge of 1e6
        // representatives, K = 32: 18.2 ms with removal for every query, 1.4 ms so.
        if (again)
        {
            const float far2 = c[N_K - 1] != INT_MAX ? d[N_K - 1] : q2;
            const bool left = qactive && !(4.001f*far2 < image_d2);
            const unsigned long long mine = __ballot(left);
            if (lane == 0 && valid) again[m / WAVE] = mine;
            qactive = qactive && !left;
        }
    }
    else
    {
        (void)image_d2;
    }
    if (qactive) write();
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

// runtime-K exact top-K for arbitrary query points (test access to the search contract)
template <int K>
__global__ __launch_bounds__(TOPK_BLOCK) void k_knn(const float4 *rec, const gdx_box *boxes, const float4 *queries,
                                                   int nq, int *codes, float *dist, unsigned int *overflow)
{
    __shared__ int2 stacks[TOPK_BLOCK / WAVE][TOPK_STACK];
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
    long long m = ((long long)blockIdx.x*(TOPK_BLOCK / WAVE) + wave)*WAVE + lane;
    bool valid = m < nq;
    float4 qp = valid ? queries[m] : make_float4(0.f, 0.f, 0.f, 0.f);
    float q2 = qp.w*qp.w;
    float cx, cy, cz;
    wave_centre(qp.x, qp.y, qp.z, valid, cx, cy, cz);
    float d[K];
    int c[K];
    topk_wave<K>(rec, boxes, qp.x, qp.y, qp.z, q2, valid, cx, cy, cz, d, c, stacks[wave], overflow);
    if (!valid) return;
#pragma unroll
    for (int k = 0; k < K; ++k)
    {
        codes[m*K + k] = c[k] == INT_MAX ? -1 : c[k];
        dist[m*K + k] = d[k];
    }
}

// ============================================================================================
// slot order and per-slot state
// ============================================================================================
// the state in slot order, published as it is (the operator's publish writes only slots changed since)
__global__ __launch_bounds__(256) void k_gather_state(bound_state u, const int *slot_pidx, int n_active,
                                                     const uint64_t *rng_p, double2 *st, double2 *res, float2 *res32,
                                                     uint64_t *rng, gdx_env *env, double *hgs)
{
    long long s = (long long)blockIdx.x*blockDim.x + threadIdx.x;
    if (s >= n_active) return;
    int p = slot_pidx[s];
    const double2 v = make_double2(ld(u.size, p), ld(u.numr, p));
    st[s] = v;
    res[s] = v;
    res32[s] = make_float2(static_cast<float>(v.x), static_cast<float>(v.y));
    rng[s] = rng_p[p];
    if constexpr (COAG_KERNEL == 3)
    {
        double y = ld(u.y, p), z = ld(u.z, p);
        env[s] = make_env(y, z);
        if constexpr (PARTNER_HG)
        {
            double R = cyl_R(y, z);
            hgs[s] = R*hg(R);
        }
    }
}

__global__ __launch_bounds__(256) void k_scatter_state(bound_state u, const int *slot_pidx, int n_active,
                                                      const double2 *st, const uint64_t *rng, uint64_t *rng_p)
{
    long long s = (long long)blockIdx.x*blockDim.x + threadIdx.x;
    if (s >= n_active) return;
    int p = slot_pidx[s];
    double2 v = st[s];
    *reinterpret_cast<double *>(const_cast<char *>(u.size.base) + (long long)p*u.size.stride) = v.x;
    *reinterpret_cast<double *>(const_cast<char *>(u.numr.base) + (long long)p*u.numr.stride) = v.y;
    rng_p[p] = rng[s];
}

// colstate_flag (src/swarm/colstate_flag.cu:13-29): the finiteness screen of a reused epoch
__global__ __launch_bounds__(256) void k_state_flag(bound_state u, int n, int *bad)
{
    long long i = (long long)blockIdx.x*blockDim.x + threadIdx.x;
    if (i >= n) return;
    bool finite = isfinite(ld(u.x, i)) && isfinite(ld(u.y, i)) && isfinite(ld(u.z, i)) && isfinite(ld(u.size, i))
        && isfinite(ld(u.numr, i));
    if (u.vx.base) finite = finite && isfinite(ld(u.vx, i)) && isfinite(ld(u.vy, i)) && isfinite(ld(u.vz, i));
    if (!finite) atomicMin(bad, int(i) + 1);
}

inline int blocks_for(long long n, int per) { return int((n + per - 1) / per); }

}  // namespace

// first non-finite particle + 1, or 0
int state_flag(context &c)
{
    c.bad.alloc(1);
    int big = INT_MAX;
    hip_check(hipMemcpyAsync(c.bad.p, &big, sizeof(int), hipMemcpyHostToDevice, c.stream), "reset bad");
    k_state_flag<<<blocks_for(c.n, 256), 256, 0, c.stream>>>(c.user, c.n, c.bad.p);
    hip_check(hipGetLastError(), "launch state flag");
    int bad = 0;
    hip_check(hipMemcpyAsync(&bad, c.bad.p, sizeof(int), hipMemcpyDeviceToHost, c.stream), "read bad");
    hip_check(hipStreamSynchronize(c.stream), "state flag");
    return bad == INT_MAX ? 0 : bad;
}

// ================================================================================================
// host side
// ================================================================================================
void scan_exclusive_u32(const unsigned int *in, unsigned int *out, int n, sort_scratch &s, hipStream_t st)
{
    if (n <= 0) return;
    int nb = blocks_for(n, SCAN_TILE);
    s.partial.alloc(size_t(nb));
    k_scan_reduce<<<nb, SCAN_BLOCK, 0, st>>>(in, n, s.partial.p);
    k_scan_partials<<<1, SCAN_BLOCK, 0, st>>>(s.partial.p, nb);
    k_scan_down<<<nb, SCAN_BLOCK, 0, st>>>(in, out, n, s.partial.p);
    hip_check(hipGetLastError(), "launch scan");
}

// keys sorted in place, idx becomes the stable permutation; `bits` bits in use, of which every third is zero in
// flat keys (two-dimensional Morton keys)
void sort_keys(dbuf<uint64_t> &keys, dbuf<int> &idx, int n, int bits, bool flat, sort_scratch &s, hipStream_t st)
{
    const int items = sort_items(n), nb = blocks_for(n, SORT_BLOCK*items);
    s.keys_alt.alloc(size_t(n));
    s.vals_alt.alloc(size_t(n));
    s.hist.alloc(size_t(RADIX)*nb + RADIX);
    unsigned int *const totals = s.hist.p + size_t(RADIX)*nb;
    bool first = true;
    for (int shift = 0; shift < bits; shift += flat ? 12 : 8)
    {
        const key_digit digit{shift, flat};
        const int *vals = first ? nullptr : idx.p;
        if (items == SORT_ITEMS) k_radix_hist<SORT_ITEMS><<<nb, SORT_BLOCK, 0, st>>>(keys.p, n, digit, s.hist.p, nb);
        else k_radix_hist<SORT_ITEMS_SMALL><<<nb, SORT_BLOCK, 0, st>>>(keys.p, n, digit, s.hist.p, nb);
        k_radix_rows<<<RADIX, SORT_BLOCK, 0, st>>>(s.hist.p, nb, totals);
        if (items == SORT_ITEMS)
            k_radix_scatter<SORT_ITEMS><<<nb, SORT_BLOCK, 0, st>>>(keys.p, vals, n, digit, s.hist.p, totals, nb,
                                                                  s.keys_alt.p, s.vals_alt.p);
        else
            k_radix_scatter<SORT_ITEMS_SMALL><<<nb, SORT_BLOCK, 0, st>>>(keys.p, vals, n, digit, s.hist.p, totals, nb,
                                                                        s.keys_alt.p, s.vals_alt.p);
        hip_check(hipGetLastError(), "launch radix pass");
        swap_buf(keys, s.keys_alt);
        swap_buf(idx, s.vals_alt);
        first = false;
    }
}

// slot order and both maps from the sorted records; totals: SLOT_DIGITS counts, active groups first
static void slot_order(context &c, int nr, unsigned int *totals)
{
    hipStream_t st = c.stream;
    const int items = sort_items(nr), nb = blocks_for(nr, SORT_BLOCK*items);
    unsigned int *const hist = c.scratch.hist.p;
    const int *sidx = c.index.idx.p;
    if (items == SORT_ITEMS) k_slot_hist<SORT_ITEMS><<<nb, SORT_BLOCK, 0, st>>>(sidx, c.bin.p, nr, c.n, hist, nb);
    else k_slot_hist<SORT_ITEMS_SMALL><<<nb, SORT_BLOCK, 0, st>>>(sidx, c.bin.p, nr, c.n, hist, nb);
    k_radix_rows<<<SLOT_DIGITS, SORT_BLOCK, 0, st>>>(hist, nb, totals);
    if (items == SORT_ITEMS)
        k_slot_maps<SORT_ITEMS><<<nb, SORT_BLOCK, 0, st>>>(sidx, c.bin.p, nr, c.n, hist, totals, nb, c.slot_pidx.p,
                                                          c.pidx_slot.p);
    else
        k_slot_maps<SORT_ITEMS_SMALL><<<nb, SORT_BLOCK, 0, st>>>(sidx, c.bin.p, nr, c.n, hist, totals, nb,
                                                                c.slot_pidx.p, c.pidx_slot.p);
    hip_check(hipGetLastError(), "launch slot order");
}

// morton_index::build (inc/swarm/morton/morton_index.cuh:168-229), enqueued: complete after morton_settle()
void morton_build(morton_index &ix, const float4 *points, const unsigned char *active, int n, float ox, float oy,
                  float oz, float width, int dim, int leaf_target, int max_level, sort_scratch &s, hipStream_t st,
                  const int *codes)
{
    if (n <= 0 || !(width > 0.0f)) throw status_error(12, "invalid adaptive Morton size");
    if (dim != 2 && dim != 3) throw status_error(12, "adaptive Morton dimension must be 2 or 3");
    if (leaf_target <= 0) throw status_error(12, "adaptive Morton leaf target must be positive");
    if (max_level <= 0 || max_level > 20) throw status_error(12, "adaptive Morton max level must be 1 through 20");
    ix.n = n; ix.dim = dim; ix.max_level = max_level; ix.leaf_target = leaf_target;
    ix.ox = ox; ix.oy = oy; ix.oz = oz; ix.width = width;
    ix.keys.alloc(size_t(n));
    ix.idx.alloc(size_t(n));
    ix.rec.alloc(size_t(n));
    ix.chunks.alloc(size_t(blocks_for(n, CHUNK) + BOX_GROUP));
    k_morton_keys<<<blocks_for(n, 256), 256, 0, st>>>(points, n, ox, oy, oz, width, max_level, dim, ix.keys.p);
    hip_check(hipGetLastError(), "launch morton keys");
    sort_keys(ix.keys, ix.idx, n, 3*max_level, dim == 2, s, st);
    k_records<<<blocks_for(n, 256), 256, 0, st>>>(ix.idx.p, points, active, codes, n, ix.rec.p,
                                                     ix.chunks.p);
    hip_check(hipGetLastError(), "launch morton records");

    const int units = blocks_for(n, NODE_UNIT), grid = blocks_for(units, 256 / WAVE);
    const long long entries = (long long)max_level*units + 1;
    if (entries > INT_MAX) throw status_error(12, "adaptive Morton size exceeds the index limit");
    ix.counts.alloc(size_t(entries) + 1);
    ix.nodes.alloc(std::max<size_t>(1024, size_t(n) / size_t(leaf_target)*5 + 64));
    k_node_counts<<<grid, 256, 0, st>>>(ix.keys.p, n, leaf_target, max_level, units, ix.counts.p);
    scan_exclusive_u32(ix.counts.p, ix.counts.p, int(entries), s, st);
    write_nodes(ix, st);
}

// the nodes and their boxes, as many as the node array holds
void write_nodes(morton_index &ix, hipStream_t st)
{
    const int units = blocks_for(ix.n, NODE_UNIT), grid = blocks_for(units, 256 / WAVE);
    const unsigned int cap = static_cast<unsigned int>(std::min<size_t>(ix.nodes.n, INT_MAX));
    ix.masks.alloc(ix.nodes.n);
    ix.boxes.alloc(ix.nodes.n + BOX_GROUP);
    hip_check(hipMemsetAsync(ix.masks.p, 0, sizeof(unsigned int)*cap, st), "zero child masks");
    unsigned int *const total = ix.counts.p + size_t(ix.max_level)*units + 1;
    k_node_write<<<grid, 256, 0, st>>>(ix.keys.p, ix.n, ix.leaf_target, ix.max_level, ix.dim, ix.ox, ix.oy, ix.oz,
                                       ix.width, units, ix.counts.p, cap, ix.nodes.p, ix.masks.p, total);
    k_node_boxes<<<blocks_for(cap, 256), 256, 0, st>>>(ix.nodes.p, ix.masks.p, total, cap, ix.dim, ix.max_level,
                                                       ix.boxes.p);
    hip_check(hipGetLastError(), "launch hierarchy");
}

// number of nodes below the root, in device memory
const unsigned int *morton_total(const morton_index &ix)
{
    return ix.counts.p + size_t(ix.max_level)*blocks_for(ix.n, NODE_UNIT) + 1;
}

// the host's part, once it has read that number: more nodes than the array held are written again
void morton_settle(morton_index &ix, unsigned int total, hipStream_t st)
{
    if (total >= static_cast<unsigned int>(INT_MAX)) throw status_error(11, "Morton node index overflow");
    ix.node_count = int(total) + 1;
    if (size_t(ix.node_count) <= ix.nodes.n) return;
    ix.nodes.alloc(size_t(ix.node_count) + size_t(ix.node_count) / 8);
    write_nodes(ix, st);
}

void knn_query(const morton_index &ix, const float4 *queries, int nq, int k, int *codes, float *d2,
               unsigned int *overflow, hipStream_t st)
{
    if (nq <= 0) return;
    int nb = blocks_for(nq, TOPK_BLOCK);
    switch (k)
    {
    case 1: k_knn<1><<<nb, TOPK_BLOCK, 0, st>>>(ix.rec.p, ix.boxes.p, queries, nq, codes, d2, overflow); break;
    case 2: k_knn<2><<<nb, TOPK_BLOCK, 0, st>>>(ix.rec.p, ix.boxes.p, queries, nq, codes, d2, overflow); break;
    case 4: k_knn<4><<<nb, TOPK_BLOCK, 0, st>>>(ix.rec.p, ix.boxes.p, queries, nq, codes, d2, overflow); break;
    case 8: k_knn<8><<<nb, TOPK_BLOCK, 0, st>>>(ix.rec.p, ix.boxes.p, queries, nq, codes, d2, overflow); break;
    case 16: k_knn<16><<<nb, TOPK_BLOCK, 0, st>>>(ix.rec.p, ix.boxes.p, queries, nq, codes, d2, overflow); break;
    case 32: k_knn<32><<<nb, TOPK_BLOCK, 0, st>>>(ix.rec.p, ix.boxes.p, queries, nq, codes, d2, overflow); break;
    case 64: k_knn<64><<<nb, TOPK_BLOCK, 0, st>>>(ix.rec.p, ix.boxes.p, queries, nq, codes, d2, overflow); break;
    default: throw status_error(15, "knn query K must be 1, 2, 4, 8, 16, 32 or 64");
    }
    hip_check(hipGetLastError(), "launch knn");
}

// the largest search cap and the unique-identifier test of swarm_runtime.cu:331-340, 413-415
static void wedge_cap(context &c)
{
    const int n = c.n;
    hipStream_t st = c.stream;
    const float x_min = static_cast<float>(X_MIN), x_max = static_cast<float>(X_MAX);
    unsigned int *const cap = c.slot_totals.p;      // free until the slot order
    hip_check(hipMemsetAsync(cap, 0, sizeof(unsigned int), st), "zero cap maximum");
    k_cap_max<<<blocks_for(n, 256), 256, 0, st>>>(c.pts.p, n, cap);
    unsigned int bits = 0;
    hip_check(hipMemcpyAsync(&bits, cap, sizeof bits, hipMemcpyDeviceToHost, st), "read cap maximum");
    hip_check(hipStreamSynchronize(st), "cap maximum");
    std::memcpy(&c.q_max, &bits, sizeof bits);
    // _get_image_dist_min (inc/swarm/param_grid.cuh:86-89): the closest any two images of one particle get
    // (each sine rounded once from double to float, as in the ghost rotation below)
    auto sinf1 = [](float a) { return static_cast<float>(std::sin(static_cast<double>(a))); };
    const float image_dist_min = 2.0f*static_cast<float>(Y_MIN)
        *std::fmin(sinf1(static_cast<float>(Z_MIN)), sinf1(static_cast<float>(Z_MAX)))
        *std::fabs(sinf1(0.5f*(x_max - x_min)));
    c.unique_ids = image_dist_min < 0.0f || image_dist_min > 2.0f*c.q_max;
}

// morton_ghost_index::build with ghosts (morton_ghost.cuh:96-168): count, scan, write physical records
// then ghosts
static void wedge_records(context &c)
{
    const int n = c.n;
    hipStream_t st = c.stream;
    const float x_min = static_cast<float>(X_MIN), x_max = static_cast<float>(X_MAX);
    c.ghost_count.alloc(size_t(n));
    c.ghost_off.alloc(size_t(n));
    k_ghost_count<<<blocks_for(n, 256), 256, 0, st>>>(c.user, c.pts.p, n, c.q_max, x_min, x_max, c.ghost_count.p);
    hip_check(hipGetLastError(), "launch ghost count");
    scan_exclusive_u32(c.ghost_count.p, c.ghost_off.p, n, c.scratch, st);
    unsigned int last[2] = {0u, 0u};
    hip_check(hipMemcpyAsync(&last[0], c.ghost_count.p + (n - 1), sizeof(unsigned int), hipMemcpyDeviceToHost, st),
              "read last ghost count");
    hip_check(hipMemcpyAsync(&last[1], c.ghost_off.p + (n - 1), sizeof(unsigned int), hipMemcpyDeviceToHost, st),
              "read last ghost offset");
    hip_check(hipStreamSynchronize(st), "ghost offsets");
    const long long total = (long long)n + last[0] + last[1];
    if (total > INT_MAX / 3) throw status_error(12, "wedge record count exceeds the index limit");
    c.n_records = int(total);
    c.wedge_rec.alloc(size_t(total));
    c.wedge_code.alloc(size_t(total));
    const float width = x_max - x_min;
    const float sw = static_cast<float>(std::sin(static_cast<double>(width)));
    const float cw = static_cast<float>(std::cos(static_cast<double>(width)));
    k_ghost_write<<<blocks_for(n, 256), 256, 0, st>>>(c.user, c.pts.p, n, c.ghost_off.p, c.q_max, x_min, x_max, cw,
                                                     sw, c.wedge_rec.p, c.wedge_code.p);
    hip_check(hipGetLastError(), "launch ghost write");
}

// the evolve_collisions geometry branch (src/swarm/swarm_runtime.cu:384-448) for bound particle state
void geometry_epoch(context &c)
{
    const int n = c.n;
    hipStream_t st = c.stream;
    c.geometry_valid = false;
    c.state_loaded = false;
    ++c.epochs;
    c.pts.alloc(n);
    c.active.alloc(n);
    c.group.alloc(n);
    c.bin.alloc(n);
    c.slot_totals.alloc(SLOT_DIGITS);
    c.bad.alloc(1);
    c.graph.alloc(LOCAL_GROUPS + 1);           // the word behind the graph is the traversals' overflow flag
    unsigned int *const overflow = reinterpret_cast<unsigned int *>(c.graph.p + LOCAL_GROUPS);
    c.epoch_host.resize(1);
    epoch_results &got = *c.epoch_host.p;
    c.pidx_slot.alloc(n);
    c.slot_pidx.alloc(n);
    int big = INT_MAX;
    hip_check(hipMemcpyAsync(c.bad.p, &big, sizeof(int), hipMemcpyHostToDevice, st), "reset bad");
    k_site_init<<<blocks_for(n, 256), 256, 0, st>>>(c.user, n, c.pts.p, c.active.p, c.group.p, c.bin.p, c.bad.p);
    hip_check(hipGetLastError(), "launch site init");
    hip_check(hipMemcpyAsync(&got.bad, c.bad.p, sizeof(int), hipMemcpyDeviceToHost, st), "read bad");

    // root cube of morton_ghost_index::build_index: width 2.0002*Y_MAX centred on the origin
    float root_width = 2.0002f*static_cast<float>(Y_MAX);
    float o = -0.5f*root_width;
    c.n_records = n;
    c.unique_ids = true;
    // the Morton search of a wedge indexes seam ghosts; the k-d search adds its own images (kd_build)
    if (X_WEDGE) wedge_cap(c);
    if (X_WEDGE && c.search == GDX_COL_SEARCH_MORTON)
    {
        wedge_records(c);
        morton_build(c.index, c.wedge_rec.p, c.active.p, c.n_records, o, o, o, root_width, DIM, c.leaf_target,
                     MORTON_MAX_LEVEL, c.scratch, st, c.wedge_code.p);
    }
    else
    {
        morton_build(c.index, c.pts.p, c.active.p, n, o, o, o, root_width, DIM, c.leaf_target, MORTON_MAX_LEVEL,
                     c.scratch, st);
    }
    const int nr = c.n_records;

    // slot order: active owners grouped by controller group, Morton order inside each group
    slot_order(c, nr, c.slot_totals.p);
    const unsigned int *counts = got.bins;
    hip_check(hipMemcpyAsync(got.bins, c.slot_totals.p, sizeof(unsigned int)*SLOT_DIGITS, hipMemcpyDeviceToHost, st),
              "group counts");
    hip_check(hipMemcpyAsync(&got.nodes, morton_total(c.index), sizeof(unsigned int), hipMemcpyDeviceToHost, st),
              "node count");
    // the epoch's one turn of the host before the search: particles that are not finite have been indexed as
    // inactive sites at the origin
    hip_check(hipStreamSynchronize(st), "slot order");
    if (got.bad != INT_MAX)
        throw status_error(14, "non-finite particle state before collision search at particle "
                           + std::to_string(got.bad - 1));
    morton_settle(c.index, got.nodes, st);
    c.group_beg.assign(LOCAL_GROUPS, 0);
    c.group_cnt.assign(counts, counts + LOCAL_GROUPS);
    c.group_all.assign(LOCAL_GROUPS, 0);
    for (int g = 0; g < LOCAL_GROUPS; ++g) c.group_all[g] = int(counts[g] + counts[SLOT_INACTIVE + g]);
    int acc = 0;
    for (int g = 0; g < LOCAL_GROUPS; ++g) { c.group_beg[g] = acc; acc += c.group_cnt[g]; }
    c.n_active = acc;

    // neighbour lists, measures and the group dependency graph
    const size_t na = size_t(std::max(1, c.n_active));
    c.nbr.alloc(na*N_K);
    c.measure.alloc(na);
    hip_check(hipMemsetAsync(c.graph.p, 0, sizeof(unsigned long long)*(LOCAL_GROUPS + 1), st), "zero graph");
    if (c.search == GDX_COL_SEARCH_KDTREE)
    {
        kd_build(c);
        kd_query(c);
    }
    else
    {
        int waves = blocks_for(nr, WAVE);
        if (X_WEDGE) c.nbr_image.alloc(na*N_K);
        const float image_dist = image_distance(X_MIN, X_MAX, Y_MIN, Z_MIN, Z_MAX), image_d2 = image_dist*image_dist;
#define GDX_TOPK_SHAPED(DEDUP, TILE, WPB)                                                                    \
    k_col_topk<DEDUP, TILE, WPB><<<xcd_grid(blocks_for(waves, WPB)), WPB*WAVE, 0, st>>>(                     \
        c.index.rec.p, c.index.boxes.p, c.index.chunks.p, nr, c.index.idx.p, c.pts.p, c.pidx_slot.p,         \
        c.group.p, c.user, c.nbr.p, c.measure.p, c.graph.p, overflow, c.nbr_image.p, again, image_d2)
#define GDX_TOPK_LAUNCH(DEDUP, TILE)                                                                         \
    do                                                                                                        \
    {                                                                                                         \
        if (c.topk_waves == 1) GDX_TOPK_SHAPED(DEDUP, TILE, 1);                                               \
        else if (c.topk_waves == 2) GDX_TOPK_SHAPED(DEDUP, TILE, 2);                                          \
        else GDX_TOPK_SHAPED(DEDUP, TILE, 4);                                                                 \
    } while (0)
        unsigned long long *again = nullptr;
        const bool removal = X_WEDGE && !c.unique_ids;
        if (removal && c.topk_tile)
        {
            c.again.alloc(size_t(waves));
            again = c.again.p;
        }
        if (!removal || c.topk_tile)
        {
            if (c.topk_tile == 8) GDX_TOPK_LAUNCH(false, 8);
            else if (c.topk_tile == 16) GDX_TOPK_LAUNCH(false, 16);
            else if (c.topk_tile == 32) GDX_TOPK_LAUNCH(false, 32);
            else GDX_TOPK_LAUNCH(false, 0);
        }
        if (removal) GDX_TOPK_LAUNCH(bool(X_WEDGE), 0);
#undef GDX_TOPK_LAUNCH
#undef GDX_TOPK_SHAPED
        hip_check(hipGetLastError(), "launch top-K");
    }
    const unsigned long long *graph = got.graph;
    hip_check(hipMemcpyAsync(got.graph, c.graph.p, sizeof(unsigned long long)*(LOCAL_GROUPS + 1), hipMemcpyDeviceToHost, st),
              "read graph");
    hip_check(hipStreamSynchronize(st), "top-K");
    if (static_cast<unsigned int>(graph[LOCAL_GROUPS])) throw status_error(11, "traversal stack overflow in col_cache_get");
    c.edges.assign(size_t(LOCAL_GROUPS)*LOCAL_WORDS, 0u);
    for (int g = 0; g < LOCAL_GROUPS; ++g)
        for (int d = 0; d < LOCAL_GROUPS; ++d)
            if (graph[g] >> d & 1ull) c.edges[size_t(g)*LOCAL_WORDS + d / 32] |= 1u << (d % 32);
    c.geometry_valid = true;
    c.rev_valid = false;
    load_state(c);
}

void load_state(context &c)
{
    if (!c.geometry_valid) throw status_error(16, "collision geometry has not been built");
    hipStream_t st = c.stream;
    const size_t na = size_t(std::max(1, c.n_active));
    c.st.alloc(na);
    c.res.alloc(na);
    c.res32.alloc(na);
    c.cached.alloc(na);
    c.rng.alloc(na);
    c.queue.alloc(na);
    c.qstart.alloc(na);
    c.cqueue.alloc(na);
    c.cstart.alloc(na);
    c.lam.alloc(na);
    c.lam_add.alloc(na);
    c.dirty.alloc(na);
    c.stale.alloc(na);
    c.qsum.alloc(na);
    if (c.diag) c.evw.alloc(na);
    c.qevents.alloc(na);
    if (COAG_KERNEL == 3) c.env.alloc(na);
    if (PARTNER_HG) c.hgs.alloc(na);
    if (c.n_active > 0)
    {
        k_gather_state<<<blocks_for(c.n_active, 256), 256, 0, st>>>(c.user, c.slot_pidx.p, c.n_active, c.rng_p.p, c.st.p,
                                                                    c.res.p, c.res32.p, c.rng.p, c.env.p, c.hgs.p);
        hip_check(hipGetLastError(), "launch gather state");
    }
    // a new state: no kept bound is valid, no publish is pending
    hip_check(hipMemsetAsync(c.dirty.p, 0, na, st), "reset dirty flags");
    hip_check(hipMemsetAsync(c.lam_add.p, 0, sizeof(double)*na, st), "reset bound increments");
    invalidate_bounds(c);
    c.state_loaded = true;
}

void invalidate_bounds(context &c)
{
    // on the context's stream, completed before any run (batches launch on the first handle's stream)
    if (c.stale.p)
    {
        hip_check(hipMemsetAsync(c.stale.p, 1, c.stale.n, c.stream), "mark bounds stale");
        hip_check(hipStreamSynchronize(c.stream), "mark bounds stale");
    }
    c.model_version = majorant_version(c.model);
}

// reverse neighbour lists of the geometry epoch: for every slot j the owners whose rows hold j, in any order.
// Bound by the atomics on the slots' counts and cursors, and by the scattered writes. A block's consecutive owners
// are close in space and share most of their neighbours, so it first counts its entries per slot in a hash table
// in LDS and then takes each slot's places by one global atomic: some 10,000 for 131,072 entries. An entry whose
// slot finds no room in the table takes its place by itself. 1e7 owners of 32 neighbours: counts 4.6 -> 1.5 ms,
// lists 7.4 -> 3.8 ms.
constexpr int REV_BLOCK = 1024;
constexpr int REV_SLOTS = 16384, REV_PROBES = 16;
constexpr int REV_OWNERS = 4096, REV_OWNERS_SMALL = 1024;      // per block; the smaller below one block per CU

// the table place of slot j, entering it if it is new; -1: no room within the probes
__device__ __forceinline__ int rev_place(unsigned *keys, unsigned j)
{
    const unsigned h = (j*2654435761u) >> 18;
    static_assert(REV_SLOTS == 1 << 14, "the hash keeps 14 bits");
    for (int p = 0; p < REV_PROBES; ++p)
    {
        const unsigned at = (h + p) & (REV_SLOTS - 1);
        unsigned k = keys[at];
        if (k == 0u) k = atomicCAS(keys + at, 0u, j + 1u);
        if (k == 0u || k == j + 1u) return int(at);
    }
    return -1;
}

template <bool FILL>
__global__ __launch_bounds__(REV_BLOCK) void k_reverse(const int *nbr, int n, int owners, unsigned *cursor, int *rev)
{
    __shared__ unsigned keys[REV_SLOTS], count[REV_SLOTS];
    for (int i = threadIdx.x; i < REV_SLOTS; i += REV_BLOCK) keys[i] = count[i] = 0u;
    __syncthreads();
    const long long first = (long long)blockIdx.x*owners;
    const int entries = int(min((long long)owners, n - first))*N_K;
    const int *const row = nbr + first*N_K;
    for (int i = threadIdx.x; i < entries; i += REV_BLOCK)
    {
        const int j = row[i];
        if (j < 0) continue;
        const int at = rev_place(keys, unsigned(j));
        if (at >= 0) atomicAdd(count + at, 1u);
        else if (!FILL) atomicAdd(cursor + j, 1u);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < REV_SLOTS; i += REV_BLOCK)
        if (count[i])
        {
            const unsigned from = atomicAdd(cursor + (keys[i] - 1u), count[i]);
            if (FILL) count[i] = from;
        }
    if (!FILL) return;
    __syncthreads();
    for (int i = threadIdx.x; i < entries; i += REV_BLOCK)
    {
        const int j = row[i];
        if (j < 0) continue;
        const int at = rev_place(keys, unsigned(j));      // every slot with room is in the table by now
        rev[atomicAdd(at >= 0 ? count + at : cursor + j, 1u)] = int(first) + i / N_K;
    }
}

// the lists of n > 0 owners' rows: slot j's owners are rev[beg[j] ... end[j])
static void reverse_lists(const int *nbr, int n, unsigned *beg, unsigned *end, int *rev, sort_scratch &s, hipStream_t st)
{
    const int owners = n >= 256*REV_OWNERS ? REV_OWNERS : REV_OWNERS_SMALL, blocks = blocks_for(n, owners);
    hip_check(hipMemsetAsync(end, 0, sizeof(unsigned)*size_t(n), st), "zero reverse counts");
    k_reverse<false><<<blocks, REV_BLOCK, 0, st>>>(nbr, n, owners, end, nullptr);
    hip_check(hipGetLastError(), "launch reverse count");
    scan_exclusive_u32(end, beg, n, s, st);
    hip_check(hipMemcpyAsync(end, beg, sizeof(unsigned)*size_t(n), hipMemcpyDeviceToDevice, st), "reverse cursors");
    // after the fill each cursor is the end of its slot's list
    k_reverse<true><<<blocks, REV_BLOCK, 0, st>>>(nbr, n, owners, end, rev);
    hip_check(hipGetLastError(), "launch reverse fill");
}

// the lists of given rows (host arrays, nbr and rev n x N_K; test access)
void check_reverse(const int *nbr, int n, unsigned *beg, unsigned *end, int *rev)
{
    dbuf<int> rows, lists;
    dbuf<unsigned> from, to;
    sort_scratch s;
    const size_t entries = size_t(n)*N_K;
    rows.alloc(entries);
    lists.alloc(entries);
    from.alloc(size_t(n));
    to.alloc(size_t(n));
    hip_check(hipMemcpy(rows.p, nbr, sizeof(int)*entries, hipMemcpyHostToDevice), "rows");
    reverse_lists(rows.p, n, from.p, to.p, lists.p, s, nullptr);
    hip_check(hipMemcpy(beg, from.p, sizeof(unsigned)*size_t(n), hipMemcpyDeviceToHost), "reverse lists");
    hip_check(hipMemcpy(end, to.p, sizeof(unsigned)*size_t(n), hipMemcpyDeviceToHost), "reverse lists");
    hip_check(hipMemcpy(rev, lists.p, sizeof(int)*entries, hipMemcpyDeviceToHost), "reverse lists");
}

void build_reverse(context &c)
{
    const int n = c.n_active;
    if ((long long)n > MAJORANT_MAX_OWNERS)
        throw status_error(GDX_COL_ERR_ARG, "a swarm with a majorant holds at most " + std::to_string(MAJORANT_MAX_OWNERS)
                                            + " active owners (32-bit reverse neighbour offsets)");
    const size_t na = size_t(std::max(1, n));
    c.rev_beg.alloc(na);
    c.rev_end.alloc(na);
    c.rev.alloc(na*N_K);
    if (n > 0) reverse_lists(c.nbr.p, n, c.rev_beg.p, c.rev_end.p, c.rev.p, c.scratch, c.stream);
    c.rev_valid = true;
    invalidate_bounds(c);
}

void store_state(context &c)
{
    if (!c.state_loaded) throw status_error(16, "collision state has not been loaded");
    if (c.n_active > 0)
    {
        k_scatter_state<<<blocks_for(c.n_active, 256), 256, 0, c.stream>>>(c.user, c.slot_pidx.p, c.n_active, c.st.p,
                                                                          c.rng.p, c.rng_p.p);
        hip_check(hipGetLastError(), "launch scatter state");
    }
}

}  // namespace gdx
