// Learned rate majorant: training and inference kernels of the 8-64-64-1 perceptron (gdx_mlp.h) and the
// C ABI of a majorant model (gdx_col_majorant_*). No counterpart in the reference.
//
//   k_mlp_infer   y = softplus(net(x)) for n feature rows, four 16-row tiles per wavefront step; few rows
//                 take k_mlp_infer_few, one tile per wavefront
//   k_mlp_grad    forward + backward of a minibatch: each block takes ROW_TILES tiles, one per wavefront,
//                 and writes one partial gradient row (deterministic, no atomics); weight gradients are
//                 MFMA products over the sample dimension, their operands transposed through LDS
//   k_mlp_reduce  sum of the partial rows in row order (gradient check)
//   k_mlp_adam    the same sum, then Adam (Kingma and Ba 2015, bias-corrected) on the FP32 master
//                 parameters and the BF16 fragments, one parameter per thread
// Loss of a sample: (ln softplus(z) - ln t)^2, the mean over the minibatch.
#include "gdx_internal.h"
#include "gdx_mlp.h"

#include <cmath>
#include <cstring>
#include <mutex>
#include <vector>

// Scratch of gdx_col_majorant_grad_noalloc: one partial gradient row per 128 samples for up to
// GDX_COL_MAJORANT_GRAD_NOALLOC_MAX samples, then the reduced row (gradient
// and loss sum). Every row the kernels read is written first by the same call, so nothing is cleared.
constexpr int GRAD_NOALLOC_ROWS = GDX_COL_MAJORANT_GRAD_NOALLOC_MAX / 128;
constexpr size_t GRAD_NOALLOC_FLOATS = size_t(GRAD_NOALLOC_ROWS + 1)*gdx::mlp::P_STRIDE;
static __device__ __align__(256) float scratch[GRAD_NOALLOC_FLOATS];

namespace gdx {
namespace mlp {
namespace {

constexpr int BLOCK = 256;
constexpr int WAVES = BLOCK / 64;
// tiles of 16 samples per partial gradient row, and the block that forms one: a wavefront per tile
constexpr int ROW_TILES = 8;
constexpr int ROW_BLOCK = 64*ROW_TILES;

__device__ void build_pack(const float *p, const float *mu, const float *inv_sigma, pack *P, int tid, int nthreads)
{
    for (int e = tid; e < 4*64; e += nthreads)
    {
        int c = e / 64, lane = e % 64, g = lane >> 4, i = lane & 15;
        v4s r;
        for (int v = 0; v < 4; ++v)
        {
            int k = 4*g + v;
            r[v] = k < F ? bf16_rn(p[P_W1 + k*H + 16*c + i]) : short(0);
        }
        P->w1a[c][lane] = r;
    }
    for (int e = tid; e < 16*64; e += nthreads)
    {
        int t = e / 64, lane = e % 64, g = lane >> 4, i = lane & 15;
        int hi = t / 4, lo = t % 4;
        v4s a, b;
        for (int v = 0; v < 4; ++v)
        {
            a[v] = bf16_rn(p[P_W2 + (16*lo + 4*g + v)*H + 16*hi + i]);   // m = hi, c = lo
            b[v] = bf16_rn(p[P_W2 + (16*hi + i)*H + 16*lo + 4*g + v]);   // a = hi, b = lo
        }
        P->w2a[t][lane] = a;
        P->w2b[t][lane] = b;
    }
    for (int e = tid; e < H; e += nthreads)
    {
        P->b1[e] = p[P_B1 + e];
        P->b2[e] = p[P_B2 + e];
        P->w3[e] = p[P_W3 + e];
    }
    if (tid == 0) P->b3 = p[P_B3];
    if (tid < F) { P->mu[tid] = mu[tid]; P->inv_sigma[tid] = inv_sigma[tid]; }
}

__global__ void k_mlp_pack(const float *p, const float *norm, pack *P)
{
    build_pack(p, norm, norm + F, P, threadIdx.x, blockDim.x);
}

// Up to INFER_FEW rows, one tile a wavefront: bound by the latency of one pass, so the row's own inputs are read
// first and each layer's weights where they are used. In a loop over tiles the compiler reads all weights ahead of
// the loop and the inputs behind them, which a single tile has to wait for: 4.4 us a launch of 10,000 rows, 3.7 so.
__global__ __launch_bounds__(BLOCK, 4) void k_mlp_infer_few(const pack *P, const float *X, int n, float *y)
{
    const int lane = threadIdx.x & 63, j = lane & 15;
    const int first = 16*(int(blockIdx.x)*WAVES + int(threadIdx.x)/64);
    if (first >= n) return;
    const bool valid = first + j < n;
    forward_state f;
    const float z = tile_forward(P, input_fragment(P, X + (long long)(valid ? first + j : 0)*F, valid), f);
    if (lane < 16 && valid) y[first + lane] = softplus(z);
}

// Many rows: bound by the vector units, 128 SiLU a row, an exponential and a reciprocal each at half the rate.
// The weights stay in registers (a wavefront keeps them for all its tiles: nothing the kernel writes can
// alias them), so the grid is what the GPU holds at once, four wavefronts per SIMD at 122 registers; the
// bound of four keeps the accumulators out of the accumulation registers, which cost a move for each value
// read. A tile leaves its results in 16 lanes, four times over: with four tiles a step every lane takes one
// row through the softplus, some 120 instructions that every tile paid before. A million rows: 58 -> 47.5 us.
constexpr int INFER_TILES = 4;
constexpr int INFER_BLOCKS = 1024;
// The most rows that go one tile a wavefront: their time grows with every tile a SIMD gets, 16,384 rows, the loop's
// with every step, 65,536 rows. 65,600 rows: 7.4 us against 7.9 with the loop, 81,920: 8.2 against 9.0, 90,112: 9.2
// against 9.1, 106,496: 10.3 against 9.0.
constexpr long long INFER_FEW = 5*16*1024;

__global__ __launch_bounds__(BLOCK, 4) void k_mlp_infer(const pack *__restrict__ P, const float *__restrict__ X,
                                                       long long n, float *__restrict__ y)
{
    static_assert(16*INFER_TILES == 64, "a lane holds the row of its own tile");
    const int lane = threadIdx.x & 63, g = lane >> 4, j = lane & 15;
    const long long steps = (n + 63) / 64;
    for (long long t = (long long)blockIdx.x*WAVES + threadIdx.x/64; t < steps; t += (long long)gridDim.x*WAVES)
    {
        const long long first = t*64;
        float z = 0.0f;
#pragma unroll
        for (int k = 0; k < INFER_TILES; ++k)
        {
            const long long r = first + 16*k + j;
            const bool valid = r < n;
            v4s x = input_fragment(P, X + (valid ? r : 0)*F, valid);
            forward_state f;
            const float v = tile_forward(P, x, f);
            z = g == k ? v : z;
        }
        const long long row = first + lane;
        if (row < n) y[row] = softplus(z);
    }
}

// sum over the 16 lanes of a row (lanes sharing lane / 16)
__device__ __forceinline__ float row_sum(float v)
{
    v += __shfl_xor(v, 1, 64);
    v += __shfl_xor(v, 2, 64);
    v += __shfl_xor(v, 4, 64);
    v += __shfl_xor(v, 8, 64);
    return v;
}

// forward + backward over the samples idx[start .. start + count) (idx null: identity); one partial row
// per ROW_TILES tiles, one block each. lt holds ln(target).
// A training step is a chain of latencies (the samples, the weights, two matrix layers each way), not
// work: a row's eight tiles ran one after the other on one wavefront. Here each of the block's
// wavefronts takes one tile through both passes and leaves its operands in LDS; then the wavefronts share
// out the row's gradient instead, each accumulating its part over the tiles in order. Every sum is formed
// by the same operations in the same order as by one wavefront, so the gradient is the same bit for bit.
// A batch of 8,192 samples (64 rows): 72 us with a wavefront per row, 10.1 us with a block per row.
__global__ __launch_bounds__(ROW_BLOCK) void k_mlp_grad(const pack *__restrict__ P, const float *__restrict__ X,
                                                       const float *__restrict__ lt, const int *__restrict__ idx,
                                                       long long start, int count, float *__restrict__ partial)
{
    // per tile: the operands of the weight gradients, contracted over the tile's samples (four samples of
    // one unit together, as a fragment takes them), and the lanes' terms of the vector gradients
    __shared__ short sH1[ROW_TILES][H][16], sDA2[ROW_TILES][H][16], sDA1[ROW_TILES][H][16], sX[ROW_TILES][16][16];
    __shared__ float term[3][ROW_TILES][16][64], sdz[ROW_TILES][64], sd[ROW_TILES][64];
    const int lane = threadIdx.x & 63, g = lane >> 4, j = lane & 15, wv = threadIdx.x / 64;
    const float inv_count = 1.0f / float(count);
    {
        const int tt = wv;
        const int row = (int(blockIdx.x)*ROW_TILES + tt)*16 + j;
        const bool valid = row < count;
        long long r = 0;
        if (valid) r = idx ? (long long)idx[start + row] : start + row;
        v4s x = input_fragment(P, X + r*F, valid);
        const float target = valid ? lt[r] : 0.0f;
        forward_state f;
        float z = tile_forward(P, x, f);
        float y = softplus(z);
        float d = valid ? logf(y) - target : 0.0f;
        float dz = valid ? 2.0f*d*sigmoid(z)/y*inv_count : 0.0f;
        sdz[tt][lane] = dz;
        sd[tt][lane] = d;

        // layer 3 and the layer-2 pre-activation gradient (C layout)
        v4s da2b[4];
#pragma unroll
        for (int m = 0; m < 4; ++m)
        {
            v4s q;
#pragma unroll
            for (int v = 0; v < 4; ++v)
            {
                float a2 = f.a2[m][v];
                term[0][tt][4*m + v][lane] = silu(a2);
                float da2 = dz*P->w3[16*m + 4*g + v]*silu_grad(a2);
                term[1][tt][4*m + v][lane] = da2;
                q[v] = bf16_rn(da2);
                sDA2[tt][16*m + 4*g + v][j] = q[v];
            }
            da2b[m] = q;
        }
        // dH1^T = W2 dA2^T, then the layer-1 pre-activation gradient
#pragma unroll
        for (int a = 0; a < 4; ++a)
        {
            v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int b = 0; b < 4; ++b) acc = mfma(P->w2b[4*a + b][lane], da2b[b], acc);
#pragma unroll
            for (int v = 0; v < 4; ++v)
            {
                float da1 = acc[v]*silu_grad(f.a1[a][v]);
                term[2][tt][4*a + v][lane] = da1;
                sDA1[tt][16*a + 4*g + v][j] = bf16_rn(da1);
                sH1[tt][16*a + 4*g + v][j] = f.h1[a][v];
            }
        }
        // inputs past F are zero
#pragma unroll
        for (int v = 0; v < 4; ++v) sX[tt][4*g + v][j] = x[v];
    }
    __syncthreads();

    float *out = partial + (long long)blockIdx.x*P_STRIDE;
    // weight gradients: wavefront wv takes the dW2 tiles (a, b) and (a, b + 1), a = wv / 2, b = 2 (wv % 2),
    // and with even wv the dW1 columns of a
    {
        const int a = wv / 2, b = 2*(wv % 2);
        v4f acc2[2], acc1 = {0.0f, 0.0f, 0.0f, 0.0f};
        acc2[0] = acc2[1] = acc1;
#pragma unroll
        for (int tt = 0; tt < ROW_TILES; ++tt)
        {
            const v4s ha = *reinterpret_cast<const v4s *>(&sH1[tt][16*a + j][4*g]);
#pragma unroll
            for (int k = 0; k < 2; ++k)
                acc2[k] = mfma(ha, *reinterpret_cast<const v4s *>(&sDA2[tt][16*(b + k) + j][4*g]), acc2[k]);
            if (b == 0)
                acc1 = mfma(*reinterpret_cast<const v4s *>(&sX[tt][j][4*g]),
                            *reinterpret_cast<const v4s *>(&sDA1[tt][16*a + j][4*g]), acc1);
        }
#pragma unroll
        for (int v = 0; v < 4; ++v)
        {
#pragma unroll
            for (int k = 0; k < 2; ++k) out[P_W2 + (16*a + 4*g + v)*H + 16*(b + k) + j] = acc2[k][v];
            if (b == 0 && g < F/4) out[P_W1 + (4*g + v)*H + 16*a + j] = acc1[v];
        }
    }
    // vector gradients: unit 16 m + 4 g + v in [4 m + v][lane], wavefront wv takes two of the sixteen
#pragma unroll
    for (int k = 0; k < 2; ++k)
    {
        const int mv = 2*wv + k;
        float gw3 = 0.0f, gb2 = 0.0f, gb1 = 0.0f;
#pragma unroll
        for (int tt = 0; tt < ROW_TILES; ++tt)
        {
            gw3 = fmaf(sdz[tt][lane], term[0][tt][mv][lane], gw3);
            gb2 += term[1][tt][mv][lane];
            gb1 += term[2][tt][mv][lane];
        }
        const int hrow = 16*(mv / 4) + 4*g + mv % 4;
        const float s3 = row_sum(gw3), s2 = row_sum(gb2), s1 = row_sum(gb1);
        if (j == 0)
        {
            out[P_W3 + hrow] = s3;
            out[P_B2 + hrow] = s2;
            out[P_B1 + hrow] = s1;
        }
    }
    if (wv == 0)
    {
        float gb3 = 0.0f, loss = 0.0f;
#pragma unroll
        for (int tt = 0; tt < ROW_TILES; ++tt)
        {
            loss = fmaf(sd[tt][lane], sd[tt][lane], loss);
            gb3 += sdz[tt][lane];
        }
        gb3 = row_sum(gb3);
        loss = row_sum(loss);
        if (lane == 0) { out[P_B3] = gb3; out[P_LOSS] = loss; }
    }
}

// gradient and loss sum of one minibatch: partial rows summed in row order
__global__ void k_mlp_reduce(const float *partial, int rows, float *grad)
{
    for (int p = blockIdx.x*blockDim.x + threadIdx.x; p <= P_LOSS; p += gridDim.x*blockDim.x)
    {
        float s = 0.0f;
        for (int w = 0; w < rows; ++w) s += partial[(long long)w*P_STRIDE + p];
        grad[p] = s;
    }
}

struct adam_args
{
    float lr, beta1, beta2, eps, bc1, bc2;
};

// the sum of the partial rows, one parameter per thread, rows in order (ROWS_AHEAD loads in flight), then
// Adam and the parameter's places in the packed fragments (build_pack's layout, inverted). Spread over the
// GPU: one block of 1024 threads took 85 us a step of 64 rows, this takes
// 3.6 us.
constexpr int ADAM_BLOCK = 64;
constexpr int ROWS_AHEAD = 32;

__global__ __launch_bounds__(ADAM_BLOCK) void k_mlp_adam(float *__restrict__ p, float *__restrict__ m1,
                                                        float *__restrict__ m2, const float *__restrict__ partial,
                                                        int rows, adam_args A, pack *__restrict__ P,
                                                        float *__restrict__ loss_out)
{
    const int e = int(blockIdx.x)*ADAM_BLOCK + int(threadIdx.x);
    if (e > P_LOSS) return;
    float g = 0.0f;
    int w = 0;
    for (; w + ROWS_AHEAD <= rows; w += ROWS_AHEAD)
    {
        float v[ROWS_AHEAD];
#pragma unroll
        for (int k = 0; k < ROWS_AHEAD; ++k) v[k] = partial[(long long)(w + k)*P_STRIDE + e];
#pragma unroll
        for (int k = 0; k < ROWS_AHEAD; ++k) g += v[k];
    }
    for (; w < rows; ++w) g += partial[(long long)w*P_STRIDE + e];
    if (e == P_LOSS)
    {
        if (loss_out) *loss_out = g;
        return;
    }
    float m = A.beta1*m1[e] + (1.0f - A.beta1)*g;
    float v = A.beta2*m2[e] + (1.0f - A.beta2)*(g*g);
    m1[e] = m;
    m2[e] = v;
    const float q = p[e] - A.lr*(m / A.bc1) / (sqrtf(v / A.bc2) + A.eps);
    p[e] = q;
    short *w1a = reinterpret_cast<short *>(P->w1a), *w2a = reinterpret_cast<short *>(P->w2a);
    short *w2b = reinterpret_cast<short *>(P->w2b);
    if (e < P_B1)
    {
        const int k = (e - P_W1) / H, h = (e - P_W1) % H;
        w1a[((h / 16)*64 + (k / 4)*16 + h % 16)*4 + k % 4] = bf16_rn(q);
    }
    else if (e < P_W2) P->b1[e - P_B1] = q;
    else if (e < P_B2)
    {
        const int r = (e - P_W2) / H, c = (e - P_W2) % H;
        // r in steps of 16 lo + 4 g + v, c = 16 hi + i; and the other way round
        w2a[((4*(c / 16) + r / 16)*64 + (r % 16 / 4)*16 + c % 16)*4 + r % 4] = bf16_rn(q);
        w2b[((4*(r / 16) + c / 16)*64 + (c % 16 / 4)*16 + r % 16)*4 + c % 4] = bf16_rn(q);
    }
    else if (e < P_W3) P->b2[e - P_B2] = q;
    else if (e < P_B3) P->w3[e - P_W3] = q;
    else P->b3 = q;
}

constexpr uint64_t SPLITMIX_STEP = 0x9e3779b97f4a7c15ull;
__host__ __device__ inline uint64_t splitmix_of(uint64_t z)
{
    z = (z ^ (z >> 30))*0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27))*0x94d049bb133111ebull;
    return z ^ (z >> 31);
}
uint64_t splitmix(uint64_t &s) { return splitmix_of(s += SPLITMIX_STEP); }
double unit(uint64_t &s) { return double(splitmix(s) >> 11)*0x1.0p-53; }

}  // namespace

// ---- mean and standard deviation of each feature over the rows, in FP64 and two passes ----
// Bound by the read of the rows, 32 bytes each; a block's threads take a column each, eight to a row, and leave one
// sum per column, which one block adds up in a fixed order. 262144 rows: 22 us, where the rows were copied to
// the host as FP64 and summed there in 11 ms.
constexpr int STATS_BLOCKS = 512, STATS_BLOCK = 256;

template <bool CENTRED>
__global__ __launch_bounds__(STATS_BLOCK) void k_feature_sums(const float *rows, long long n, const double *mean,
                                                             double *partial)
{
    static_assert(F == 8, "eight threads to a row");
    __shared__ double sums[STATS_BLOCK / 64][F];
    const int c = threadIdx.x % F, lane = threadIdx.x % 64;
    const double mu = CENTRED ? mean[c] : 0.0;
    double sum = 0.0;
    for (long long r = ((long long)blockIdx.x*STATS_BLOCK + threadIdx.x) / F; r < n; r += STATS_BLOCKS*STATS_BLOCK / F)
    {
        const double v = double(rows[r*F + c]) - mu;
        sum += CENTRED ? v*v : v;
    }
#pragma unroll
    for (int o = F; o < 64; o <<= 1) sum += __shfl_xor(sum, o, 64);
    if (lane < F) sums[threadIdx.x / 64][lane] = sum;
    __syncthreads();
    if (threadIdx.x < F)
    {
        double s = 0.0;
        for (int w = 0; w < STATS_BLOCK / 64; ++w) s += sums[w][threadIdx.x];
        partial[blockIdx.x*F + threadIdx.x] = s;
    }
}

// out[c]: the mean of the sums over n rows, or its root
__global__ __launch_bounds__(STATS_BLOCK) void k_feature_fold(const double *partial, long long n, bool root, double *out)
{
    __shared__ double sums[STATS_BLOCK / F][F];
    const int c = threadIdx.x % F, g = threadIdx.x / F;
    double sum = 0.0;
    for (int b = g; b < STATS_BLOCKS; b += STATS_BLOCK / F) sum += partial[b*F + c];
    sums[g][c] = sum;
    __syncthreads();
    if (threadIdx.x >= F) return;
    double s = 0.0;
    for (int k = 0; k < STATS_BLOCK / F; ++k) s += sums[k][threadIdx.x];
    s /= double(n);
    out[threadIdx.x] = root ? sqrt(s) : s;
}

// ---- the training order: the Fisher-Yates shuffle of one epoch, for i = n - 1 ... 1 a swap of positions i and
// k_i = draw mod (i + 1), without its n dependent steps ----
// Position x holds, just before step i, what the latest earlier step i' > i with k_i' = x moved there: what
// position i' held just before step i'. So position i ends with the value found from the successor of i among the
// steps with the same k, ascending, by following next(y), the first step after y with k = y, to its end (k_i itself
// where there is no successor). The steps are grouped by one stable sort; the walks end, since they ascend, after
// one link on average and ln n or so at most. 262144 samples: 1.7 ms on the host and 1 MB copied -> 65 us.
constexpr int SHUFFLE_BLOCK = 256;
// the host shuffles larger sets: the draws, links and the sort's second copies take 32 bytes a sample
constexpr long long SHUFFLE_MAX = 1ll << 26;

// first: state before the epoch's first draw, which step n - 1 takes
__global__ __launch_bounds__(SHUFFLE_BLOCK) void k_shuffle_draws(uint64_t first, int n, uint64_t *key, int *next)
{
    const int i = blockIdx.x*SHUFFLE_BLOCK + threadIdx.x;
    if (i >= n) return;
    key[i] = splitmix_of(first + uint64_t(n - i)*SPLITMIX_STEP) % uint64_t(i + 1);      // 0 for i = 0
    next[i] = -1;
}

// after the sort: link[i] = i's successor among the steps with its k, or -1 - k
__global__ __launch_bounds__(SHUFFLE_BLOCK) void k_shuffle_links(const uint64_t *key, const int *step, int n, int *link,
                                                                int *next)
{
    const int p = blockIdx.x*SHUFFLE_BLOCK + threadIdx.x;
    if (p >= n) return;
    const int i = step[p], k = int(key[p]);
    const int succ = p + 1 < n && int(key[p + 1]) == k ? step[p + 1] : -1;
    link[i] = succ >= 0 ? succ : -1 - k;
    if (p == 0 || int(key[p - 1]) != k) next[k] = i == k ? succ : i;
}

__global__ __launch_bounds__(SHUFFLE_BLOCK) void k_shuffle_order(const int *link, const int *next, int n, int *perm)
{
    const int i = blockIdx.x*SHUFFLE_BLOCK + threadIdx.x;
    if (i >= n) return;
    int y = link[i];
    if (y < 0) y = -1 - y;
    else
        for (int z = next[y]; z >= 0; z = next[y]) y = z;
    perm[i] = y;
}

// one majorant model: FP32 parameters and Adam moments, the packed fragments, the input normalization
struct model
{
    dbuf<float> p, m1, m2, norm, partial, grad, loss;
    dbuf<pack> P;
    dbuf<int> perm;
    dbuf<double> stats;                 // sums of the feature statistics, then their results
    // workspace of the shuffles
    dbuf<uint64_t> draw;
    dbuf<int> step_of, link, next;
    sort_scratch scratch;
    long long steps = 0;
    unsigned long long version = 0;     // advanced by every change of the parameters or normalization
    std::vector<float> h_norm = std::vector<float>(2*F);
    std::string last_error;
};

int grad_rows(int count) { return (count + 16*ROW_TILES - 1) / (16*ROW_TILES); }

void model_init(model &M, uint64_t seed)
{
    // uniform(-1/sqrt(fan_in), 1/sqrt(fan_in)) weights and biases; the output bias puts softplus at 1
    std::vector<float> h(P_COUNT);
    uint64_t s = seed;
    auto fill = [&](int off, int count, int fan_in) {
        double bound = 1.0 / std::sqrt(double(fan_in));
        for (int i = 0; i < count; ++i) h[off + i] = float((2.0*unit(s) - 1.0)*bound);
    };
    fill(P_W1, F*H, F);
    fill(P_B1, H, F);
    fill(P_W2, H*H, H);
    fill(P_B2, H, H);
    fill(P_W3, H, H);
    h[P_B3] = 0.54132485f;       // softplus^-1(1)
    M.p.alloc(P_COUNT);
    M.m1.alloc(P_COUNT);
    M.m2.alloc(P_COUNT);
    M.norm.alloc(2*F);
    M.P.alloc(1);
    M.grad.alloc(P_COUNT + 1);
    for (int k = 0; k < F; ++k) { M.h_norm[k] = 0.0f; M.h_norm[F + k] = 1.0f; }
    hip_check(hipMemcpy(M.p.p, h.data(), sizeof(float)*P_COUNT, hipMemcpyHostToDevice), "majorant init");
    hip_check(hipMemset(M.m1.p, 0, sizeof(float)*P_COUNT), "majorant init");
    hip_check(hipMemset(M.m2.p, 0, sizeof(float)*P_COUNT), "majorant init");
    hip_check(hipMemcpy(M.norm.p, M.h_norm.data(), sizeof(float)*2*F, hipMemcpyHostToDevice), "majorant init");
    k_mlp_pack<<<1, 256>>>(M.p.p, M.norm.p, M.P.p);
    hip_check(hipGetLastError(), "majorant pack");
    hip_check(hipDeviceSynchronize(), "majorant pack");
}

const pack *model_pack(const model &M) { return M.P.p; }

void launch_mlp_infer(const pack *P, const float *X, long long n, float *y, hipStream_t st)
{
    if (n <= 0) return;
    if (n <= INFER_FEW)
    {
        const long long tiles = (n + 15) / 16;
        k_mlp_infer_few<<<dim3(unsigned((tiles + WAVES - 1) / WAVES)), BLOCK, 0, st>>>(P, X, int(n), y);
    }
    else
    {
        const long long steps = (n + 63) / 64;
        const long long blocks = std::min<long long>((steps + WAVES - 1) / WAVES, INFER_BLOCKS);
        k_mlp_infer<<<dim3(unsigned(blocks)), BLOCK, 0, st>>>(P, X, n, y);
    }
    hip_check(hipGetLastError(), "majorant inference launch");
}

}  // namespace mlp
}  // namespace gdx

using gdx::mlp::model;

struct gdx_col_majorant_ctx
{
    model m;
};

namespace {

thread_local std::string g_majorant_error;

template <typename F>
int mguard(gdx_col_majorant_ctx *h, F &&f)
{
    try
    {
        f();
        return GDX_COL_OK;
    }
    catch (const gdx::status_error &e)
    {
        (h ? h->m.last_error : g_majorant_error) = e.what();
        return e.code;
    }
    catch (const std::bad_alloc &)
    {
        (h ? h->m.last_error : g_majorant_error) = "host allocation failure";
        return GDX_COL_ERR_ALLOC;
    }
    catch (const std::exception &e)
    {
        (h ? h->m.last_error : g_majorant_error) = e.what();
        return GDX_COL_ERR_HIP;
    }
}

void check_arg(bool ok, const char *what)
{
    if (!ok) throw gdx::status_error(GDX_COL_ERR_ARG, what);
}

// Device address of `scratch` on the current GPU. The array's name is a host-side stand-in in host code;
// every GPU holds its own copy at its own address, looked up once per device with that device current.
constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
float *g_scratch_ptr[MAX_DEVICES] = {};

float *scratch_on_current_device()
{
    int dev = -1;
    gdx::hip_check(hipGetDevice(&dev), "current device");
    if (dev < 0 || dev >= MAX_DEVICES) throw gdx::status_error(GDX_COL_ERR_ARG, "device ordinal out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev])
    {
        void *p = nullptr;
        gdx::hip_check(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "scratch address");
        g_scratch_ptr[dev] = static_cast<float *>(p);
    }
    return g_scratch_ptr[dev];
}

}  // namespace

extern "C" {

int gdx_col_majorant_create(unsigned long long seed, gdx_col_majorant *out)
{
    if (!out) return GDX_COL_ERR_ARG;
    *out = nullptr;
    gdx_col_majorant_ctx *h = nullptr;
    int rc = mguard(nullptr, [&] {
        h = new gdx_col_majorant_ctx();
        gdx::mlp::model_init(h->m, seed);
    });
    if (rc != GDX_COL_OK) { delete h; return rc; }
    *out = h;
    return GDX_COL_OK;
}

int gdx_col_majorant_destroy(gdx_col_majorant h)
{
    delete h;
    return GDX_COL_OK;
}

const char *gdx_col_majorant_last_error(gdx_col_majorant h)
{
    return h ? h->m.last_error.c_str() : g_majorant_error.c_str();
}

int gdx_col_majorant_get_params(gdx_col_majorant h, float *params, float *norm)
{
    if (!h) return GDX_COL_ERR_ARG;
    return mguard(h, [&] {
        if (params)
            gdx::hip_check(hipMemcpy(params, h->m.p.p, sizeof(float)*gdx::mlp::P_COUNT, hipMemcpyDeviceToHost),
                           "majorant parameters");
        if (norm) std::memcpy(norm, h->m.h_norm.data(), sizeof(float)*2*gdx::mlp::F);
    });
}

int gdx_col_majorant_set_params(gdx_col_majorant h, const float *params, const float *norm)
{
    if (!h) return GDX_COL_ERR_ARG;
    return mguard(h, [&] {
        using namespace gdx::mlp;
        model &M = h->m;
        if (params)
        {
            for (int i = 0; i < P_COUNT; ++i) check_arg(std::isfinite(params[i]), "majorant parameters must be finite");
            gdx::hip_check(hipMemcpy(M.p.p, params, sizeof(float)*P_COUNT, hipMemcpyHostToDevice), "majorant parameters");
            gdx::hip_check(hipMemset(M.m1.p, 0, sizeof(float)*P_COUNT), "majorant parameters");
            gdx::hip_check(hipMemset(M.m2.p, 0, sizeof(float)*P_COUNT), "majorant parameters");
            M.steps = 0;
        }
        if (norm)
        {
            for (int k = 0; k < F; ++k)
            {
                check_arg(std::isfinite(norm[k]), "normalization mean must be finite");
                check_arg(std::isfinite(norm[F + k]) && norm[F + k] > 0.0f, "normalization scale must be positive");
                M.h_norm[k] = norm[k];
                M.h_norm[F + k] = 1.0f / norm[F + k];
            }
            gdx::hip_check(hipMemcpy(M.norm.p, M.h_norm.data(), sizeof(float)*2*F, hipMemcpyHostToDevice),
                           "majorant normalization");
            for (int k = 0; k < F; ++k) M.h_norm[F + k] = norm[F + k];
        }
        k_mlp_pack<<<1, 256>>>(M.p.p, M.norm.p, M.P.p);
        gdx::hip_check(hipGetLastError(), "majorant pack");
        gdx::hip_check(hipDeviceSynchronize(), "majorant pack");
        ++M.version;
    });
}

int gdx_col_majorant_infer(gdx_col_majorant h, const float *features, long long n, float *out)
{
    if (!h) return GDX_COL_ERR_ARG;
    return mguard(h, [&] {
        check_arg(n >= 0 && (n == 0 || (features && out)), "invalid inference arguments");
        gdx::mlp::launch_mlp_infer(h->m.P.p, features, n, out, nullptr);
        gdx::hip_check(hipDeviceSynchronize(), "majorant inference");
    });
}

int gdx_col_majorant_grad(gdx_col_majorant h, const float *features, const float *log_target, int n, float *grad,
                          double *loss)
{
    if (!h) return GDX_COL_ERR_ARG;
    return mguard(h, [&] {
        using namespace gdx::mlp;
        check_arg(n > 0 && features && log_target && grad, "invalid gradient arguments");
        model &M = h->m;
        const int rows = grad_rows(n);
        M.partial.alloc(size_t(rows)*P_STRIDE);
        k_mlp_grad<<<rows, ROW_BLOCK>>>(M.P.p, features, log_target, nullptr, 0, n, M.partial.p);
        gdx::hip_check(hipGetLastError(), "majorant gradient launch");
        k_mlp_reduce<<<(P_LOSS + 256) / 256, 256>>>(M.partial.p, rows, M.grad.p);
        gdx::hip_check(hipGetLastError(), "majorant gradient launch");
        std::vector<float> h_grad(P_LOSS + 1);
        gdx::hip_check(hipMemcpy(h_grad.data(), M.grad.p, sizeof(float)*(P_LOSS + 1), hipMemcpyDeviceToHost),
                       "majorant gradient");
        std::memcpy(grad, h_grad.data(), sizeof(float)*P_COUNT);
        if (loss) *loss = double(h_grad[P_LOSS]) / n;
    });
}

int gdx_col_majorant_feature_stats(gdx_col_majorant h, const float *features, long long n, double *mean, double *deviation)
{
    if (!h) return GDX_COL_ERR_ARG;
    return mguard(h, [&] {
        using namespace gdx::mlp;
        check_arg(n > 0 && features && mean && deviation, "invalid feature statistics arguments");
        model &M = h->m;
        M.stats.alloc(size_t(STATS_BLOCKS + 2)*F);
        double *const out = M.stats.p + size_t(STATS_BLOCKS)*F;
        k_feature_sums<false><<<STATS_BLOCKS, STATS_BLOCK>>>(features, n, nullptr, M.stats.p);
        k_feature_fold<<<1, STATS_BLOCK>>>(M.stats.p, n, false, out);
        k_feature_sums<true><<<STATS_BLOCKS, STATS_BLOCK>>>(features, n, out, M.stats.p);
        k_feature_fold<<<1, STATS_BLOCK>>>(M.stats.p, n, true, out + F);
        gdx::hip_check(hipGetLastError(), "feature statistics launch");
        double both[2*F];
        gdx::hip_check(hipMemcpy(both, out, sizeof(both), hipMemcpyDeviceToHost), "feature statistics");
        std::memcpy(mean, both, sizeof(double)*F);
        std::memcpy(deviation, both + F, sizeof(double)*F);
    });
}

int gdx_col_majorant_grad_noalloc(gdx_col_majorant h, const float *features, const float *log_target, int n,
                                  float *grad, double *loss)
{
    if (!h) return GDX_COL_ERR_ARG;
    return mguard(h, [&] {
        using namespace gdx::mlp;
        static_assert(16*ROW_TILES == 128, "scratch rows hold 128 samples");
        check_arg(n > 0 && features && log_target && grad, "invalid gradient arguments");
        check_arg(n <= GDX_COL_MAJORANT_GRAD_NOALLOC_MAX,
                  "gradient without allocation: n exceeds GDX_COL_MAJORANT_GRAD_NOALLOC_MAX samples");
        const int rows = grad_rows(n);
        if (rows > GRAD_NOALLOC_ROWS) throw gdx::status_error(GDX_COL_ERR_ARG, "scratch rows exceeded");
        float *partial = scratch_on_current_device();
        float *sum = partial + size_t(GRAD_NOALLOC_ROWS)*P_STRIDE;
        k_mlp_grad<<<rows, ROW_BLOCK>>>(h->m.P.p, features, log_target, nullptr, 0, n, partial);
        gdx::hip_check(hipGetLastError(), "majorant gradient launch");
        k_mlp_reduce<<<(P_LOSS + 256) / 256, 256>>>(partial, rows, sum);
        gdx::hip_check(hipGetLastError(), "majorant gradient launch");
        float loss_sum = 0.0f;
        gdx::hip_check(hipMemcpy(grad, sum, sizeof(float)*P_COUNT, hipMemcpyDeviceToHost), "majorant gradient");
        gdx::hip_check(hipMemcpy(&loss_sum, sum + P_LOSS, sizeof(float), hipMemcpyDeviceToHost), "majorant gradient");
        if (loss) *loss = double(loss_sum) / n;
    });
}

int gdx_col_majorant_train(gdx_col_majorant h, const float *features, const float *log_target, long long n,
                           const gdx_col_train_config *cfg, float *epoch_loss)
{
    if (!h) return GDX_COL_ERR_ARG;
    return mguard(h, [&] {
        using namespace gdx::mlp;
        check_arg(cfg && features && log_target, "invalid training arguments");
        check_arg(cfg->batch > 0 && cfg->epochs >= 0 && n >= cfg->batch, "training needs at least one full minibatch");
        check_arg(n <= (1ll << 31) - 1, "training set too large");
        check_arg(std::isfinite(cfg->lr) && cfg->lr > 0.0, "learning rate must be positive");
        model &M = h->m;
        ++M.version;
        const int B = cfg->batch;
        const long long batches = n / B;               // the last partial minibatch is dropped
        const int rows = grad_rows(B);
        M.partial.alloc(size_t(rows)*P_STRIDE);
        M.perm.alloc(size_t(n));
        M.loss.alloc(size_t(std::max<long long>(1, batches)));
        std::vector<int> perm(n > SHUFFLE_MAX ? static_cast<size_t>(n) : 0);
        if (n <= SHUFFLE_MAX)
        {
            M.draw.alloc(size_t(n));
            M.step_of.alloc(size_t(n));
            M.link.alloc(size_t(n));
            M.next.alloc(size_t(n));
        }
        std::vector<float> losses(static_cast<size_t>(std::max<long long>(1, batches)));
        uint64_t s = cfg->seed;
        const double b1 = cfg->beta1 > 0 ? cfg->beta1 : 0.9, b2 = cfg->beta2 > 0 ? cfg->beta2 : 0.999;
        const double eps = cfg->eps > 0 ? cfg->eps : 1e-8;
        for (int ep = 0; ep < cfg->epochs; ++ep)
        {
            // Fisher-Yates shuffle of the sample order, one per epoch
            if (n <= SHUFFLE_MAX)
            {
                const int m = int(n);
                const dim3 grid(unsigned((m + SHUFFLE_BLOCK - 1) / SHUFFLE_BLOCK));
                int bits = 1;
                while (bits < 31 && (1 << bits) < m) ++bits;
                k_shuffle_draws<<<grid, SHUFFLE_BLOCK>>>(s, m, M.draw.p, M.next.p);
                gdx::sort_keys(M.draw, M.step_of, m, bits, false, M.scratch, nullptr);
                k_shuffle_links<<<grid, SHUFFLE_BLOCK>>>(M.draw.p, M.step_of.p, m, M.link.p, M.next.p);
                k_shuffle_order<<<grid, SHUFFLE_BLOCK>>>(M.link.p, M.next.p, m, M.perm.p);
                gdx::hip_check(hipGetLastError(), "training order");
                s += uint64_t(n - 1)*SPLITMIX_STEP;
            }
            else
            {
                for (long long i = 0; i < n; ++i) perm[size_t(i)] = int(i);
                for (long long i = n - 1; i > 0; --i)
                {
                    long long k = (long long)(splitmix(s) % uint64_t(i + 1));
                    std::swap(perm[size_t(i)], perm[size_t(k)]);
                }
                gdx::hip_check(hipMemcpy(M.perm.p, perm.data(), sizeof(int)*size_t(n), hipMemcpyHostToDevice),
                               "training order");
            }
            for (long long b = 0; b < batches; ++b)
            {
                ++M.steps;
                adam_args A{float(cfg->lr), float(b1), float(b2), float(eps),
                            float(1.0 - std::pow(b1, double(M.steps))), float(1.0 - std::pow(b2, double(M.steps)))};
                k_mlp_grad<<<rows, ROW_BLOCK>>>(M.P.p, features, log_target, M.perm.p, b*B, B, M.partial.p);
                k_mlp_adam<<<(P_LOSS + ADAM_BLOCK) / ADAM_BLOCK, ADAM_BLOCK>>>(M.p.p, M.m1.p, M.m2.p, M.partial.p, rows,
                                                                              A, M.P.p, M.loss.p + b);
            }
            gdx::hip_check(hipGetLastError(), "training launch");
            gdx::hip_check(hipMemcpy(losses.data(), M.loss.p, sizeof(float)*size_t(batches), hipMemcpyDeviceToHost),
                           "training loss");
            if (epoch_loss)
            {
                double sum = 0.0;
                for (long long b = 0; b < batches; ++b) sum += losses[size_t(b)];
                epoch_loss[ep] = float(sum / double(batches*B));
            }
        }
        gdx::hip_check(hipDeviceSynchronize(), "training");
    });
}

}  // extern "C"

namespace gdx {

const void *majorant_pack(gdx_col_majorant m) { return m ? static_cast<const void *>(m->m.P.p) : nullptr; }
unsigned long long majorant_version(gdx_col_majorant m) { return m ? m->m.version : 0ull; }

}  // namespace gdx
