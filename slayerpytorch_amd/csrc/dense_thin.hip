// Fully connected synapse with few outputs (up to 32): the output layers of the reference's networks
// (slayer._denseLayer, src/slayer.py:393-440), out[n][o][t] = sum_k W[o][k] x[n][k][t] and its two gradients.
//
// With O outputs a sample of x meets O multiply-adds: at O = 10 five operations a byte, far below what the vector ALUs
// do in the time the byte takes to arrive, and the small layers are one launch's latency.  So plain fp32 multiply-adds
// straight from memory, time on the lanes as everywhere (one 16-byte vector of samples each): no tiles of 16 outputs that
// are partly empty, no transposed copies, and enough work-groups whatever the batch is, since the inputs k are split over
// wavefronts and work-groups.  All sums are added in a fixed order.
//
// Rows that are not whole vectors: the last vector of a row starts at sample T - 4 and overlaps the one before; product and
// input gradient store the shared samples twice with the same values, the weight gradient counts them once.
#include "common.h"

namespace slayer {

constexpr int kDtWaves = 8;       // wavefronts of a work-group that share its sums or its gradients
constexpr int kDtMaxO = 32;

// 16-byte accesses at any multiple of four bytes
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));

template <int VEC> struct ThinVec;
template <> struct ThinVec<4> {
    typedef float4_ext V;
    static __device__ __forceinline__ V load(const float *p) { return *reinterpret_cast<const f4u *>(p); }
    static __device__ __forceinline__ void store(float *p, V v) { *reinterpret_cast<f4u *>(p) = v; }
};
template <> struct ThinVec<1> {
    typedef float V;
    static __device__ __forceinline__ V load(const float *p) { return *p; }
    static __device__ __forceinline__ void store(float *p, V v) { *p = v; }
};

struct ThinArgs {
    const float *w, *x;      // x: input (product, weight gradient) or output gradient (input gradient)
    const float *g;          // output gradient (weight gradient)
    float *out;              // result, or partial sums [split][...] of it
    int N, K, O, T, TV;
    int vectors;             // N * TV
    int perSplit;            // inputs k (product, input gradient) or blocks of 64 vectors (weight gradient) per split
    int splits;
    FastDiv byTV, byVecBlocks;
};

// first sample of vector tv of a row
template <int VEC>
__device__ __forceinline__ int thin_start(int tv, int T) { return VEC == 4 ? min(tv * 4, T - 4) : tv; }

// ---- product -----------------------------------------------------------------------------------------
// A work-group owns 64 vectors (of any items) and a range of inputs, whose weights it lays into LDS as [k][o] first.  Its
// wavefronts take eight inputs each in turn: a lane keeps its vector's OB sums, loads the next eight rows' vectors while it
// multiplies these, and reads the weights as broadcasts, without a barrier.  The wavefronts' sums meet in LDS in three steps.
constexpr int thin_rows(int VEC) { return VEC == 4 ? 8 : 16; }   // rows of x in each of a wavefront's two sets of registers
constexpr int kDtChunk = kDtWaves * 16;                // a work-group's range is a multiple of this
constexpr int kDtWeights = 16384;                      // floats of weights in LDS, at most

constexpr int thin_sums(int OB, int VEC) { return 4 * (OB < 16 ? OB : 16) * VEC * 64; }   // floats of the sums of four wavefronts

template <int OB, int VEC>
__global__ __launch_bounds__(64 * kDtWaves) void dense_thin_kernel(ThinArgs p)
{
    typedef typename ThinVec<VEC>::V V;
    constexpr int RB = OB < 16 ? OB : 16;              // outputs per round of the final sum
    constexpr int ROWS = thin_rows(VEC), TRIP = kDtWaves * ROWS;
    extern __shared__ __align__(16) float lds[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int split = static_cast<int>(fastdiv(blockIdx.x, p.byVecBlocks));
    const int v = (static_cast<int>(blockIdx.x) - split * static_cast<int>(p.byVecBlocks.d)) * 64 + lane;
    const bool live = v < p.vectors;
    const int n = static_cast<int>(fastdiv(static_cast<uint32_t>(live ? v : 0), p.byTV));
    const int t = thin_start<VEC>((live ? v : 0) - n * p.TV, p.T);
    const int k0 = split * p.perSplit, k1 = min(p.K, k0 + p.perSplit);
    const float *x = p.x + static_cast<int64_t>(n) * p.K * p.T + t;

    V acc[OB];
#pragma unroll
    for (int o = 0; o < OB; ++o) acc[o] = V(0.0f);
    V a[ROWS], b[ROWS];
    auto fetch = [&](V (&r)[ROWS], int k) {         // (rows behind the range: the last one again)
#pragma unroll
        for (int i = 0; i < ROWS; ++i) r[i] = ThinVec<VEC>::load(x + static_cast<int64_t>(min(k + i, k1 - 1)) * p.T);
    };
    auto multiply = [&](V (&r)[ROWS], int k) {
        if (k + ROWS <= k1) {
#pragma unroll
            for (int i = 0; i < ROWS; ++i) {
                const float *w = lds + (k - k0 + i) * OB;
#pragma unroll
                for (int o = 0; o < OB; ++o) acc[o] = __builtin_elementwise_fma(V(w[o]), r[i], acc[o]);
            }
        } else {
#pragma unroll
            for (int i = 0; i < ROWS; ++i)
                if (k + i < k1) {
                    const float *w = lds + (k - k0 + i) * OB;
#pragma unroll
                    for (int o = 0; o < OB; ++o) acc[o] = __builtin_elementwise_fma(V(w[o]), r[i], acc[o]);
                }
        }
    };
    int k = k0 + wave * ROWS;
    fetch(a, k);
    fetch(b, k + TRIP);
    {   // lanes along k: contiguous loads, four of them in flight
        const int inputs = k1 - k0, cells = inputs * OB;
        const float inverse = 1.0f / static_cast<float>(inputs);
        for (int e0 = threadIdx.x; e0 < cells; e0 += 4 * 64 * kDtWaves) {
            float w[4];
            int at[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int e = e0 + j * 64 * kDtWaves;
                int o, i;
                divmod_small(e, inputs, inverse, o, i);
                at[j] = e < cells ? i * OB + o : -1;
                w[j] = (e < cells && o < p.O) ? p.w[static_cast<int64_t>(o) * p.K + k0 + i] : 0.0f;
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (at[j] >= 0) lds[at[j]] = w[j];
        }
    }
    __syncthreads();
    for (; k < k1; k += 2 * TRIP) {
        multiply(a, k);
        fetch(a, k + 2 * TRIP);
        if (k + TRIP < k1) multiply(b, k + TRIP);
        fetch(b, k + 3 * TRIP);
    }

    float *out = p.out + static_cast<int64_t>(split) * p.N * p.O * p.T;
#pragma unroll
    for (int o0 = 0; o0 < OB; o0 += RB) {
        auto meet = [&](int half) {                    // wavefronts half .. 2 half - 1 to 0 .. half - 1
            __syncthreads();
            if (wave >= half && wave < 2 * half) {
#pragma unroll
                for (int o = 0; o < RB; ++o) reinterpret_cast<V *>(lds)[((wave - half) * RB + o) * 64 + lane] = acc[o0 + o];
            }
            __syncthreads();
            if (wave < half) {
#pragma unroll
                for (int o = 0; o < RB; ++o) acc[o0 + o] += reinterpret_cast<const V *>(lds)[(wave * RB + o) * 64 + lane];
            }
        };
        static_assert(kDtWaves == 8, "three steps");
        meet(4);
        meet(2);
        meet(1);
    }
    if (wave == 0 && live) {
#pragma unroll
        for (int o = 0; o < OB; ++o)
            if (o < p.O) ThinVec<VEC>::store(out + (static_cast<int64_t>(n) * p.O + o) * p.T + t, acc[o]);
    }
}

// ---- input gradient ----------------------------------------------------------------------------------
// gradIn[n][k][t] = sum_o W[o][k] gradOut[n][o][t]: a lane keeps its vector's OB gradients and writes one vector per input.
// A work-group's lanes cover whole rows (of several items, or a piece of a long row), and take its inputs one after the
// other: the memory line that two rows share is then written by one work-group in quick succession and leaves L2 whole.
template <int OB, int VEC>
__global__ __launch_bounds__(512) void dense_thin_grad_input_kernel(ThinArgs p, int vecsPerBlock)
{
    typedef typename ThinVec<VEC>::V V;
    constexpr int KC = 64;
    __shared__ __align__(16) float lds[KC * OB];
    const int split = static_cast<int>(fastdiv(blockIdx.x, p.byVecBlocks));
    const int first = (static_cast<int>(blockIdx.x) - split * static_cast<int>(p.byVecBlocks.d)) * vecsPerBlock;
    const int v = first + static_cast<int>(threadIdx.x);
    const bool live = static_cast<int>(threadIdx.x) < vecsPerBlock && v < p.vectors;
    const int n = static_cast<int>(fastdiv(static_cast<uint32_t>(live ? v : 0), p.byTV));
    const int t = thin_start<VEC>((live ? v : 0) - n * p.TV, p.T);
    const int k0 = split * p.perSplit, k1 = min(p.K, k0 + p.perSplit);
    V g[OB];
#pragma unroll
    for (int o = 0; o < OB; ++o)
        g[o] = (live && o < p.O) ? ThinVec<VEC>::load(p.x + (static_cast<int64_t>(n) * p.O + o) * p.T + t) : V(0.0f);
    float *out = p.out + (static_cast<int64_t>(n) * p.K) * p.T + t;
    for (int k = k0; k < k1; k += KC) {
        const int kc = min(KC, k1 - k);
        __syncthreads();
        for (int e = threadIdx.x; e < KC * OB; e += blockDim.x) {
            const int o = e / KC, i = e - o * KC;
            lds[i * OB + o] = (o < p.O && i < kc) ? p.w[static_cast<int64_t>(o) * p.K + k + i] : 0.0f;
        }
        __syncthreads();
#pragma unroll 4
        for (int i = 0; i < kc; ++i) {
            V acc = V(0.0f);
#pragma unroll
            for (int o = 0; o < OB; ++o) acc = __builtin_elementwise_fma(V(lds[i * OB + o]), g[o], acc);
            if (live) ThinVec<VEC>::store(out + static_cast<int64_t>(k + i) * p.T, acc);
        }
    }
}

// The lanes' sums, M each: at step D the lanes of a pair keep half of the sums each (an odd one out is kept by the lower lane),
// until one is left, whose pairs add up.  store(e, sum) for every sum e < end, from one lane.
template <int M, int D, typename Store>
__device__ __forceinline__ void thin_butterfly(float (&acc)[M], int base, int end, int lane, Store store)
{
    if constexpr (D == 0) {
#pragma unroll
        for (int i = 0; i < M; ++i)
            if (base + i < end) store(base + i, acc[i]);
    } else if constexpr (M == 1) {
        float one[1] = {acc[0] + __shfl_xor(acc[0], D, 64)};
        if ((lane & D) != 0) end = 0;                  // (the lower lane stores)
        thin_butterfly<1, D / 2>(one, base, end, lane, store);
    } else {
        constexpr int H = (M + 1) / 2;
        const bool upper = (lane & D) != 0;
        float half[H];
#pragma unroll
        for (int i = 0; i < H; ++i) {
            const float low = acc[i], high = H + i < M ? acc[H + i < M ? H + i : 0] : 0.0f;
            half[i] = (upper ? high : low) + __shfl_xor(upper ? low : high, D, 64);
        }
        thin_butterfly<H, D / 2>(half, base + (upper ? H : 0), upper ? min(end, base + M) : min(end, base + H), lane, store);
    }
}

// ---- weight gradient ---------------------------------------------------------------------------------
// gradW[o][k] = sum_{n,t} gradOut[n][o][t] x[n][k][t]: time and items on the lanes, 64 vectors at a time.  The work-group's
// wavefronts take KB inputs each and share the OB gradients of those vectors in LDS, two sets in turn.  The lanes' OB x KB
// sums meet in a butterfly that halves their number at every step; a work-group's range of vectors is one row of the
// workspace, and a second launch adds the rows in order, in double precision.
template <int OB, int KB, int VEC>
__global__ __launch_bounds__(64 * kDtWaves) void dense_thin_wgrad_kernel(ThinArgs p)
{
    typedef typename ThinVec<VEC>::V V;
    __shared__ __align__(16) float lds[2][OB * 64 * VEC];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int split = static_cast<int>(fastdiv(blockIdx.x, p.byVecBlocks));      // (byVecBlocks: blocks of inputs here)
    const int k0 = (static_cast<int>(blockIdx.x) - split * static_cast<int>(p.byVecBlocks.d)) * (kDtWaves * KB) + wave * KB;
    const int blocks = (p.vectors + 63) >> 6;
    const int b0 = split * p.perSplit, b1 = min(blocks, b0 + p.perSplit);
    constexpr int GW = (OB + kDtWaves - 1) / kDtWaves; // gradient vectors that a lane stages

    float acc[KB * OB];
#pragma unroll
    for (int i = 0; i < KB * OB; ++i) acc[i] = 0.0f;
    V xa[KB], ga[GW];
    int skip = 0;                                      // samples of this lane's vector that the one before holds already
    auto fetch = [&](int b) {
        const int v = b * 64 + lane;
        const bool live = v < p.vectors;
        const int n = static_cast<int>(fastdiv(static_cast<uint32_t>(live ? v : 0), p.byTV));
        const int tv = (live ? v : 0) - n * p.TV;
        const int t = thin_start<VEC>(tv, p.T);
        skip = live ? tv * VEC - t : VEC;
        const float *x = p.x + static_cast<int64_t>(n) * p.K * p.T + t;
        const float *g = p.g + static_cast<int64_t>(n) * p.O * p.T + t;
#pragma unroll
        for (int i = 0; i < KB; ++i) xa[i] = ThinVec<VEC>::load(x + static_cast<int64_t>(min(k0 + i, p.K - 1)) * p.T);
#pragma unroll
        for (int i = 0; i < GW; ++i) ga[i] = ThinVec<VEC>::load(g + static_cast<int64_t>(min(wave + i * kDtWaves, p.O - 1)) * p.T);
    };
    auto drop = [&](V v) {                             // (both factors: an infinity must not meet a zero that stands for nothing)
        if constexpr (VEC == 4) {
            v.x = skip > 0 ? 0.0f : v.x;
            v.y = skip > 1 ? 0.0f : v.y;
            v.z = skip > 2 ? 0.0f : v.z;
            v.w = skip > 3 ? 0.0f : v.w;
        } else {
            v = skip > 0 ? 0.0f : v;
        }
        return v;
    };
    fetch(b0);
    int buf = 0;
    for (int b = b0; b < b1; ++b, buf ^= 1) {
        V *gl = reinterpret_cast<V *>(lds[buf]);
        V xs[KB];
#pragma unroll
        for (int i = 0; i < KB; ++i) xs[i] = drop(xa[i]);
#pragma unroll
        for (int i = 0; i < GW; ++i)
            if (wave + i * kDtWaves < OB) gl[(wave + i * kDtWaves) * 64 + lane] = drop(ga[i]);
        __syncthreads();                               // (one barrier per trip: the other set is written before the next)
        if (b + 1 < b1) fetch(b + 1);
#pragma unroll
        for (int o = 0; o < OB; ++o) {
            const V g = gl[o * 64 + lane];
#pragma unroll
            for (int i = 0; i < KB; ++i) {
                if constexpr (VEC == 4) {
                    float s = acc[i * OB + o];
                    s = __builtin_fmaf(g.x, xs[i].x, s);
                    s = __builtin_fmaf(g.y, xs[i].y, s);
                    s = __builtin_fmaf(g.z, xs[i].z, s);
                    acc[i * OB + o] = __builtin_fmaf(g.w, xs[i].w, s);
                } else {
                    acc[i * OB + o] = __builtin_fmaf(g, xs[i], acc[i * OB + o]);
                }
            }
        }
    }
    float *out = p.out + static_cast<int64_t>(split) * p.O * p.K;
    thin_butterfly<KB * OB, 32>(acc, 0, KB * OB, lane, [&](int e, float sum) {
        const int k = k0 + e / OB, o = e % OB;
        if (o < p.O && k < p.K) out[static_cast<int64_t>(o) * p.K + k] = sum;
    });
}

// out[i] = the splits' sums, in double precision: four groups of splits beside each other, each in order, eight loads in flight
__global__ __launch_bounds__(256) void dense_thin_sum_kernel(float *__restrict__ out, const float *__restrict__ part, int64_t n, int splits)
{
    __shared__ double sums[4][64];
    const int lane = threadIdx.x & 63, group = threadIdx.x >> 6;
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 64 + lane;
    const int s0 = group * splits / 4, s1 = (group + 1) * splits / 4;
    double s = 0.0;
    if (i < n) {
#pragma unroll 8
        for (int k = s0; k < s1; ++k) s += static_cast<double>(part[static_cast<int64_t>(k) * n + i]);
    }
    sums[group][lane] = s;
    __syncthreads();
    if (group == 0 && i < n) out[i] = static_cast<float>(((sums[0][lane] + sums[1][lane]) + sums[2][lane]) + sums[3][lane]);
}

// ---- host side ---------------------------------------------------------------------------------------
struct ThinPlan {
    int vectors, TV, vecBlocks;
    int fwdVec, fwdTV, fwdBlocks;      // product: samples per lane, the vectors of that and blocks of 64 of them
    int splits, perSplit;              // ... and ranges of inputs
    int wSplits, wPerSplit, kBlocks;   // weight gradient, over the blocks of 64 vectors; blocks of inputs
};

constexpr int kDtKB = 4;
constexpr int kDtOneLaunch = 512;

static int thin_outputs(int64_t O) { return O <= 2 ? static_cast<int>(O) : O <= 4 ? 4 : O <= 8 ? 8 : O <= 12 ? 12 : O <= 16 ? 16 : 32; }

static bool thin_plan(int64_t N, int64_t K, int64_t O, int64_t T, ThinPlan &p)
{
    if (N < 1 || K < 1 || O < 1 || T < 1 || O > kDtMaxO || K >= (1 << 24) || T >= (1 << 24)) return false;
    const int VEC = T >= 4 ? 4 : 1;
    const int64_t TV = ceil_div(T, VEC);
    if (N * TV >= (1LL << 30)) return false;
    p.TV = static_cast<int>(TV);
    p.vectors = static_cast<int>(N * TV);
    p.vecBlocks = (p.vectors + 63) / 64;
    // The product: vectors of four samples unless there are so few that most compute units would stand by.  One work-group of
    // eight wavefronts per 64 vectors while the inputs are few (a second launch costs more than a longer one), then as many
    // ranges of inputs as give two work-groups per compute unit; their weights fit LDS.
    p.fwdVec = VEC == 4 && p.vecBlocks >= 64 ? 4 : 1;
    p.fwdTV = p.fwdVec == 4 ? p.TV : static_cast<int>(T);
    p.fwdBlocks = static_cast<int>(ceil_div(N * p.fwdTV, 64));
    const int64_t mostPer = kDtWeights / thin_outputs(O) / kDtChunk * kDtChunk;
    int64_t splits = K <= kDtOneLaunch ? 1 : 512 / p.fwdBlocks;
    if (splits < 1) splits = 1;
    int64_t per = ceil_div(ceil_div(K, splits), kDtChunk) * kDtChunk;
    if (per > mostPer) per = mostPer;
    p.perSplit = static_cast<int>(per);
    p.splits = static_cast<int>(ceil_div(K, per));
    // The weight gradient: 32 inputs per work-group; as many ranges of vectors as give about 1024 work-groups, at least
    // two blocks of 64 vectors in each
    p.kBlocks = static_cast<int>(ceil_div(K, kDtWaves * kDtKB));
    splits = ceil_div(1024, p.kBlocks);
    const int64_t mostW = ceil_div(p.vecBlocks, 2);
    splits = splits < 1 ? 1 : splits > mostW ? mostW : splits;
    p.wPerSplit = static_cast<int>(ceil_div(p.vecBlocks, splits));
    p.wSplits = static_cast<int>(ceil_div(p.vecBlocks, p.wPerSplit));
    return static_cast<int64_t>(p.fwdBlocks) * p.splits < (1LL << 23) && static_cast<int64_t>(p.kBlocks) * p.wSplits < (1LL << 23);
}

static ThinArgs thin_args(const ThinPlan &p, int64_t N, int64_t K, int64_t O, int64_t T)
{
    ThinArgs a{};
    a.N = static_cast<int>(N); a.K = static_cast<int>(K); a.O = static_cast<int>(O); a.T = static_cast<int>(T);
    a.TV = p.TV; a.vectors = p.vectors;
    a.byTV = make_fastdiv(static_cast<uint32_t>(p.TV));
    return a;
}

static int thin_sum(float *out, const float *part, int64_t n, int splits, hipStream_t st)
{
    hipLaunchKernelGGL(dense_thin_sum_kernel, dim3(static_cast<unsigned>(ceil_div(n, 64))), dim3(256), 0, st, out, part, n, splits);
    return launch_status();
}

}  // namespace slayer

// outputs per lane: as thin_outputs()
#define SLAYER_THIN(KERNEL, GRID, BLOCK, ...)                                                                                  \
    do {                                                                                                                       \
        if (O <= 1) { if (vec) KERNEL(1, 4, GRID, BLOCK, __VA_ARGS__); else KERNEL(1, 1, GRID, BLOCK, __VA_ARGS__); }            \
        else if (O <= 2) { if (vec) KERNEL(2, 4, GRID, BLOCK, __VA_ARGS__); else KERNEL(2, 1, GRID, BLOCK, __VA_ARGS__); }       \
        else if (O <= 4) { if (vec) KERNEL(4, 4, GRID, BLOCK, __VA_ARGS__); else KERNEL(4, 1, GRID, BLOCK, __VA_ARGS__); }       \
        else if (O <= 8) { if (vec) KERNEL(8, 4, GRID, BLOCK, __VA_ARGS__); else KERNEL(8, 1, GRID, BLOCK, __VA_ARGS__); }       \
        else if (O <= 12) { if (vec) KERNEL(12, 4, GRID, BLOCK, __VA_ARGS__); else KERNEL(12, 1, GRID, BLOCK, __VA_ARGS__); }    \
        else if (O <= 16) { if (vec) KERNEL(16, 4, GRID, BLOCK, __VA_ARGS__); else KERNEL(16, 1, GRID, BLOCK, __VA_ARGS__); }    \
        else { if (vec) KERNEL(32, 4, GRID, BLOCK, __VA_ARGS__); else KERNEL(32, 1, GRID, BLOCK, __VA_ARGS__); }                 \
    } while (0)

extern "C" int slayer_dense_thin_supported(int64_t N, int64_t K, int64_t O, int64_t T)
{
    slayer::ThinPlan p;
    return slayer::thin_plan(N, K, O, T, p) ? 1 : 0;
}

extern "C" int64_t slayer_dense_thin_workspace_bytes(int64_t N, int64_t K, int64_t O, int64_t T, int32_t gradWeight)
{
    slayer::ThinPlan p;
    if (!slayer::thin_plan(N, K, O, T, p)) return 0;
    if (gradWeight) return p.wSplits > 1 ? 4LL * p.wSplits * O * K : 0;
    return p.splits > 1 ? 4LL * p.splits * N * O * T : 0;
}

extern "C" int slayer_dense_thin_f32(float *out, const float *weight, const float *x, float *workspace, int64_t N, int64_t K,
                                     int64_t O, int64_t T, void *stream)
{
    using namespace slayer;
    ThinPlan p;
    if (N < 0 || K < 0 || O < 0 || T < 0) return SLAYER_EINVAL;
    if (!thin_plan(N, K, O, T, p)) return SLAYER_EUNSUPPORTED;
    if (!out || !weight || !x || (p.splits > 1 && !workspace)) return SLAYER_EINVAL;
    hipStream_t st = static_cast<hipStream_t>(stream);
    ThinArgs a = thin_args(p, N, K, O, T);
    a.w = weight; a.x = x; a.out = p.splits > 1 ? workspace : out;
    a.perSplit = p.perSplit; a.splits = p.splits;
    a.TV = p.fwdTV; a.vectors = static_cast<int>(N * p.fwdTV);
    a.byTV = make_fastdiv(static_cast<uint32_t>(p.fwdTV));
    a.byVecBlocks = make_fastdiv(static_cast<uint32_t>(p.fwdBlocks));
    const dim3 grid(static_cast<unsigned>(p.fwdBlocks * p.splits)), block(64 * kDtWaves);
    const bool vec = p.fwdVec == 4;
    const int weights = p.perSplit < a.K ? p.perSplit : a.K;
#define SLAYER_THIN_FWD(OB, VEC, G, B, A)                                                                                     \
    hipLaunchKernelGGL((dense_thin_kernel<OB, VEC>), G, B,                                                                     \
                       4 * (thin_sums(OB, VEC) > weights * OB ? thin_sums(OB, VEC) : weights * OB), st, A)
    SLAYER_THIN(SLAYER_THIN_FWD, grid, block, a);
#undef SLAYER_THIN_FWD
    const int status = launch_status();
    if (status != SLAYER_OK || p.splits == 1) return status;
    return thin_sum(out, workspace, N * O * T, p.splits, st);
}

extern "C" int slayer_dense_thin_grad_input_f32(float *gradIn, const float *weight, const float *gradOut, int64_t N, int64_t K,
                                                int64_t O, int64_t T, void *stream)
{
    using namespace slayer;
    ThinPlan p;
    if (N < 0 || K < 0 || O < 0 || T < 0) return SLAYER_EINVAL;
    if (!thin_plan(N, K, O, T, p)) return SLAYER_EUNSUPPORTED;
    if (!gradIn || !weight || !gradOut) return SLAYER_EINVAL;
    hipStream_t st = static_cast<hipStream_t>(stream);
    ThinArgs a = thin_args(p, N, K, O, T);
    a.w = weight; a.x = gradOut; a.out = gradIn;
    // whole rows per work-group (as many items as 512 lanes hold, no more than give 256 work-groups their inputs), or pieces
    // of 512 vectors of long ones; the inputs of a batch of few vectors are cut until there are about 1024 work-groups
    int vecs = 512;
    if (p.TV <= 512) vecs = static_cast<int>(p.TV * (512 / p.TV < N ? 512 / p.TV : N));
    const int vecBlocks = (p.vectors + vecs - 1) / vecs;
    int64_t splits = ceil_div(1024, vecBlocks);
    const int64_t most = ceil_div(K, 8);
    splits = splits < 1 ? 1 : splits > most ? most : splits;
    a.perSplit = static_cast<int>(ceil_div(K, splits));
    a.splits = static_cast<int>(ceil_div(K, a.perSplit));
    a.byVecBlocks = make_fastdiv(static_cast<uint32_t>(vecBlocks));
    const dim3 grid(static_cast<unsigned>(vecBlocks * a.splits)), block(static_cast<unsigned>((vecs + 63) / 64 * 64));
    const bool vec = T >= 4;
#define SLAYER_THIN_GI(OB, VEC, G, B, A) hipLaunchKernelGGL((dense_thin_grad_input_kernel<OB, VEC>), G, B, 0, st, A, vecs)
    SLAYER_THIN(SLAYER_THIN_GI, grid, block, a);
#undef SLAYER_THIN_GI
    return launch_status();
}

extern "C" int slayer_dense_thin_grad_weight_f32(float *gradW, const float *gradOut, const float *x, float *workspace, int64_t N,
                                                 int64_t K, int64_t O, int64_t T, void *stream)
{
    using namespace slayer;
    ThinPlan p;
    if (N < 0 || K < 0 || O < 0 || T < 0) return SLAYER_EINVAL;
    if (!thin_plan(N, K, O, T, p)) return SLAYER_EUNSUPPORTED;
    if (!gradW || !gradOut || !x || (p.wSplits > 1 && !workspace)) return SLAYER_EINVAL;
    hipStream_t st = static_cast<hipStream_t>(stream);
    ThinArgs a = thin_args(p, N, K, O, T);
    a.x = x; a.g = gradOut; a.out = p.wSplits > 1 ? workspace : gradW;
    a.perSplit = p.wPerSplit; a.splits = p.wSplits;
    a.byVecBlocks = make_fastdiv(static_cast<uint32_t>(p.kBlocks));
    const dim3 grid(static_cast<unsigned>(p.kBlocks * p.wSplits)), block(64 * kDtWaves);
    const bool vec = T >= 4;
#define SLAYER_THIN_GW(OB, VEC, G, B, A) hipLaunchKernelGGL((dense_thin_wgrad_kernel<OB, kDtKB, VEC>), G, B, 0, st, A)
    SLAYER_THIN(SLAYER_THIN_GW, grid, block, a);
#undef SLAYER_THIN_GW
    const int status = launch_status();
    if (status != SLAYER_OK || p.wSplits == 1) return status;
    return thin_sum(gradW, workspace, O * K, p.wSplits, st);
}
