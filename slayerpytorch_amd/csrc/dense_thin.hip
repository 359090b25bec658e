// Fully connected synapse with few outputs (up to 32): the output layers of the reference's networks
// (slayer._denseLayer, src/slayer.py:393-440), out[n][o][t] = sum_k W[o][k] x[n][k][t] and its two gradients.
//
// With O outputs a sample of x meets O multiply-adds: at O = 10 five operations a byte, far below what the chip does in the
// time the byte takes to arrive, and the small layers are one launch's latency.  So fp32 arithmetic straight from memory, time
// on the lanes as everywhere (one 16-byte vector of samples each), no transposed copies, and enough work-groups whatever the
// batch is, since the inputs k are split over wavefronts and work-groups: the product on fp32 matrix instructions (tiles of 16
// outputs; those that are not there cost no memory), the gradients as multiply-adds of the vector ALUs.  All sums are added
// in a fixed order.
//
// Rows that are not whole vectors: the last vector of a row starts at sample T - 4 and overlaps the one before; product and
// input gradient store the shared samples twice with the same values, the weight gradient counts them once.
#include "common.h"
#include "fir_core.h"   // f32x4

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
// On fp32 matrix instructions, v_mfma_f32_16x16x4_f32, straight from memory: lane (r, h) holds four weights W[r][k + 4 h ..]
// with one 16-byte load, and the vector r of rows k + 4 h .. + 3 with four, which is 4 VEC instructions' worth of operands (a
// vector's four samples are columns of four products).  Neither needs LDS, and two steps of loads are in flight while a
// wavefront multiplies (four times as many: no faster, (64, 256, 2000) -> 8 27 -> 40 us).  A work-group owns 16 vectors (of any items) and a range of inputs, 16 at a time per
// wavefront; the wavefronts' sums meet in LDS in three steps.  Its pieces of the rows end within memory lines that the next
// work-group reads too, so neighbours run on one die: in the order of their numbers 4096 -> 10 on (12, 300) 19 us, this 16;
// 30000 -> 10 on (4, 300) 62, 32; 4096 -> 10 on (64, 300) 73, 66.  Vector instructions with the weights as broadcasts from LDS
// or the scalar cache: 512 -> 11 on (8, 300) 10.2 us, 4096 -> 10 on (64, 300) 76.
constexpr int kDtSteps = 1;                            // steps of 16 inputs in each of a wavefront's two sets of registers
constexpr int kDtChunk = kDtWaves * kDtSteps * 16;     // inputs of a work-group's trip

template <int OT, int VEC>
__global__ __launch_bounds__(64 * kDtWaves) void dense_thin_kernel(ThinArgs p)
{
    typedef typename ThinVec<VEC>::V V;
    __shared__ __align__(16) f32x4 lds[kDtWaves / 2 * OT * VEC * 64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, h = lane >> 4;
    const uint32_t block = xcd_contiguous(blockIdx.x, gridDim.x);   // neighbours share memory lines
    const int split = static_cast<int>(fastdiv(block, p.byVecBlocks));
    const int v = (static_cast<int>(block) - split * static_cast<int>(p.byVecBlocks.d)) * 16 + r;
    const bool live = v < p.vectors;
    const int n = static_cast<int>(fastdiv(static_cast<uint32_t>(live ? v : 0), p.byTV));
    const int t = thin_start<VEC>((live ? v : 0) - n * p.TV, p.T);
    const int k0 = split * p.perSplit, k1 = min(p.K, k0 + p.perSplit);
    const float *x = p.x + static_cast<int64_t>(n) * p.K * p.T + t;
    // (outputs that are not there: the last one again, into sums that nobody stores)
    const float *w[OT];
#pragma unroll
    for (int ot = 0; ot < OT; ++ot) w[ot] = p.w + static_cast<int64_t>(min(ot * 16 + r, p.O - 1)) * p.K;

    f32x4 acc[OT][VEC];
#pragma unroll
    for (int ot = 0; ot < OT; ++ot)
#pragma unroll
        for (int e = 0; e < VEC; ++e) acc[ot][e] = f32x4{0.f, 0.f, 0.f, 0.f};
    struct Set {
        V x[kDtSteps][4];
        float4_ext w[kDtSteps][OT];
    } a, b;
    // inputs k .. k + 16 kDtSteps; those behind the range as zeros, both factors (nothing may meet an infinity)
    auto fetch = [&](Set &s, int k) {
#pragma unroll
        for (int i = 0; i < kDtSteps; ++i) {
            const int kk = k + i * 16 + 4 * h;
            if (k + i * 16 + 16 <= k1) {
#pragma unroll
                for (int ot = 0; ot < OT; ++ot) s.w[i][ot] = ThinVec<4>::load(w[ot] + kk);
#pragma unroll
                for (int j = 0; j < 4; ++j) s.x[i][j] = ThinVec<VEC>::load(x + static_cast<int64_t>(kk + j) * p.T);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
#pragma unroll
                    for (int ot = 0; ot < OT; ++ot) s.w[i][ot][j] = kk + j < k1 ? w[ot][kk + j] : 0.f;
                    s.x[i][j] = kk + j < k1 ? ThinVec<VEC>::load(x + static_cast<int64_t>(kk + j) * p.T) : V(0.f);
                }
            }
        }
    };
    auto multiply = [&](const Set &s) {
#pragma unroll
        for (int i = 0; i < kDtSteps; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int ot = 0; ot < OT; ++ot)
#pragma unroll
                    for (int e = 0; e < VEC; ++e) {
                        float xe;
                        if constexpr (VEC == 4) xe = s.x[i][j][e];
                        else xe = s.x[i][j];
                        acc[ot][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(s.w[i][ot][j], xe, acc[ot][e], 0, 0, 0);
                    }
    };
    int k = k0 + wave * kDtSteps * 16;
    fetch(a, k);
    for (;;) {
        if (k >= k1) break;
        if (k + kDtChunk < k1) fetch(b, k + kDtChunk);
        multiply(a);
        k += kDtChunk;
        if (k >= k1) break;
        if (k + kDtChunk < k1) fetch(a, k + kDtChunk);
        multiply(b);
        k += kDtChunk;
    }

    auto meet = [&](int half) {                        // wavefronts half .. 2 half - 1 to 0 .. half - 1
        __syncthreads();
        if (wave >= half && wave < 2 * half) {
#pragma unroll
            for (int c = 0; c < OT * VEC; ++c) lds[((wave - half) * OT * VEC + c) * 64 + lane] = acc[c / VEC][c % VEC];
        }
        __syncthreads();
        if (wave < half) {
#pragma unroll
            for (int c = 0; c < OT * VEC; ++c) acc[c / VEC][c % VEC] += lds[(wave * OT * VEC + c) * 64 + lane];
        }
    };
    static_assert(kDtWaves == 8, "three steps");
    meet(4);
    meet(2);
    meet(1);
    // element q of a sum is output 4 h + q of its tile, for vector r
    if (wave == 0 && live) {
        float *out = p.out + static_cast<int64_t>(split) * p.N * p.O * p.T + static_cast<int64_t>(n) * p.O * p.T + t;
#pragma unroll
        for (int ot = 0; ot < OT; ++ot)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int o = ot * 16 + 4 * h + q;
                if (o >= p.O) continue;
                if constexpr (VEC == 4)
                    ThinVec<4>::store(out + static_cast<int64_t>(o) * p.T,
                                      float4_ext{acc[ot][0][q], acc[ot][1][q], acc[ot][2][q], acc[ot][3][q]});
                else
                    ThinVec<1>::store(out + static_cast<int64_t>(o) * p.T, acc[ot][0][q]);
            }
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
        const int shift = kc <= 8 ? 3 : kc <= 16 ? 4 : 6;   // (a few inputs: a few weights)
        for (int e = threadIdx.x; e < OB << shift; e += blockDim.x) {
            const int o = e >> shift, i = e & ((1 << shift) - 1);
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

constexpr int thin_inputs(int O) { return O <= 16 ? 4 : 1; }   // of a wavefront of the weight gradient
constexpr int kDtOneLaunch = 1024, kDtBlocks = 2048;

static bool thin_plan(int64_t N, int64_t K, int64_t O, int64_t T, ThinPlan &p)
{
    if (N < 1 || K < 1 || O < 1 || T < 1 || O > kDtMaxO || K >= (1 << 24) || T >= (1 << 24)) return false;
    const int VEC = T >= 4 ? 4 : 1;
    const int64_t TV = ceil_div(T, VEC);
    if (N * TV >= (1LL << 30)) return false;
    p.TV = static_cast<int>(TV);
    p.vectors = static_cast<int>(N * TV);
    p.vecBlocks = (p.vectors + 63) / 64;
    // The product: vectors of four samples unless there are so few that most compute units would stand by (one / four samples:
    // 512 -> 11 on (8, 300), 600 vectors, 4.0 / 6.2 us; 512 -> 10 on (12, 350), 1056, 5.6 / 6.2; 4096 -> 10 on (12, 300), 900,
    // 29 / 20 (before neighbours shared a die); 512 -> 16 on (32, 350) 12.7 / 7.6).  One work-group of eight wavefronts per 16 vectors while the inputs are few
    // (a second launch costs more than a longer one), then as many ranges of inputs as give eight work-groups per compute unit.
    p.fwdVec = VEC == 4 && p.vectors >= 800 ? 4 : 1;
    p.fwdTV = p.fwdVec == 4 ? p.TV : static_cast<int>(T);
    p.fwdBlocks = static_cast<int>(ceil_div(N * p.fwdTV, 16));
    int64_t splits = K <= kDtOneLaunch ? 1 : kDtBlocks / p.fwdBlocks;
    if (splits < 1) splits = 1;
    const int64_t per = ceil_div(ceil_div(K, splits), kDtChunk) * kDtChunk;
    p.perSplit = static_cast<int>(per);
    p.splits = static_cast<int>(ceil_div(K, per));
    // The weight gradient: 32 inputs per work-group, 8 where there are more than 16 outputs (a wavefront's sums, 32 per input,
    // meet in one butterfly: 250 -> 25 at (1, 500) 9.8 -> 5.4 us, 512 -> 32 at (4, 500) 12.0 -> 7.9); as many ranges of vectors as give about 1024 work-groups, at least
    // two blocks of 64 vectors in each
    p.kBlocks = static_cast<int>(ceil_div(K, kDtWaves * thin_inputs(static_cast<int>(O))));
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

// outputs per lane
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
    if (O <= 16 && p.fwdVec == 4) hipLaunchKernelGGL((dense_thin_kernel<1, 4>), grid, block, 0, st, a);
    else if (O <= 16) hipLaunchKernelGGL((dense_thin_kernel<1, 1>), grid, block, 0, st, a);
    else if (p.fwdVec == 4) hipLaunchKernelGGL((dense_thin_kernel<2, 4>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((dense_thin_kernel<2, 1>), grid, block, 0, st, a);
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
    // Whole rows per work-group (as many items as 512 lanes hold), or pieces of 512 vectors of long ones; the inputs of a
    // batch of few vectors are cut until there are about 1024 work-groups or eight inputs in each, four where a lane has up to
    // 32 outputs to multiply for each (250 -> 25 at (1, 500): 7.2 -> 4.5 us, with the weights read for those inputs alone).
    int vecs = 512;
    if (p.TV <= 512) vecs = static_cast<int>(p.TV * (512 / p.TV < N ? 512 / p.TV : N));
    const int vecBlocks = (p.vectors + vecs - 1) / vecs;
    int64_t splits = ceil_div(1024, vecBlocks);
    const int64_t most = ceil_div(K, O <= 16 ? 8 : 4);
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
#define SLAYER_THIN_GW(OB, VEC, G, B, A) hipLaunchKernelGGL((dense_thin_wgrad_kernel<OB, thin_inputs(OB), VEC>), G, B, 0, st, A)
    SLAYER_THIN(SLAYER_THIN_GW, grid, block, a);
#undef SLAYER_THIN_GW
    const int status = launch_status();
    if (status != SLAYER_OK || p.wSplits == 1) return status;
    return thin_sum(gradW, workspace, O * K, p.wSplits, st);
}
