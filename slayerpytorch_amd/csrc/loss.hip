// Spike-train loss of the output layer in two launches: the error signal
// error = psp(out - desired) [+ addend] and loss = 1/2 * sum(error^2) * Ts, which the reference
// evaluates as a chain of tensor expressions (src/spikeLoss.py:56-58 and :100-104).  The output layer
// is tiny (classes x batch rows), so the cost of that chain is its launches, not its bytes.
#include "common.h"

namespace slayer {

// One work-group per row, which sits in LDS between zeros.  A lane makes four consecutive outputs: per four taps it reads the
// next four samples and the taps with one 16-byte access each for 16 multiply-adds, where one output per lane took one access
// per sample and tap.  Small tensors are one launch's latency ((120, 300), 77 taps: 6 us either way), large ones bound by memory
// ((12800, 2000), 8 taps: 59 -> 56 us).

// The filter, then `before` zeros (a multiple of four), the row and zeros up to `end` floats behind its start.
struct RowInLds {
    float *filt, *row;
    __device__ __forceinline__ RowInLds(float *lds, int F, int before) : filt(lds), row(lds + ((F + 3) & ~3) + before) {}
    template <typename Sample>
    __device__ __forceinline__ void fill(const float *srm, int T, int F, int before, int end, Sample sample) const
    {
        for (int k = threadIdx.x; k < ((F + 3) & ~3); k += 256) filt[k] = k < F ? srm[k] : 0.0f;
        for (int t = static_cast<int>(threadIdx.x) - before; t < end; t += 256) row[t] = t >= 0 && t < T ? sample(t) : 0.0f;
    }
};

// outputs t .. t + 3 of a row; vec: rows are whole 16-byte vectors
__device__ __forceinline__ void store4(float *__restrict__ row, int t, int T, const float (&y)[4], bool vec)
{
    if (vec) {
        *reinterpret_cast<float4 *>(row + t) = make_float4(y[0], y[1], y[2], y[3]);
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (t + j < T) row[t + j] = y[j];
    }
}

// error[t] = Ts * sum_k diff[t - k] srm[k] [+ addend]: every output is the full tap chain acc = fma(d[t-k], srm[k], acc),
// k = 0 .. F-1, then * Ts - the arithmetic of the temporal convolution kernels, bit for bit (taps that reach before
// the row multiply a zero).
//
// COUNT: the spike-count loss.  Inside [start, stop) the output's own spikes are what is desired, and the addend is
// (spikes of the row in the region * Ts - count wanted) / length * scale, in double precision, rounded at the end; outside
// nothing is desired and the addend is that times zero.  The work-group counts its row while it stages it: one launch for
// what takes sixteen small ones as tensor expressions ((64, 10) rows of 300 samples, with the sum: 93 -> 11 us of launches).
struct CountTarget {
    const uint8_t *wanted;      // one per row: whether the first of the two counts is wanted, or the second
    int start, stop;
    double counts[2], length, scale;
};

template <bool COUNT>
__global__ __launch_bounds__(256) void spike_loss_rows_kernel(float *__restrict__ error, float *__restrict__ partial,
                                                              const float *__restrict__ out,
                                                              const float *__restrict__ desired,
                                                              const float *__restrict__ addend,
                                                              const float *__restrict__ srm, int T, int F, float Ts, bool vec,
                                                              CountTarget target)
{
    extern __shared__ __align__(16) float lds[];
    __shared__ float wsum[4];
    __shared__ double counted[4];
    const int64_t base = static_cast<int64_t>(blockIdx.x) * T;
    const int before = (F + 3) & ~3, end = (T + 3) & ~3;
    const RowInLds x(lds, F, before);
    double mine = 0.0;
    auto inside = [&](int t) { return t >= target.start && t < target.stop; };
    if constexpr (COUNT) {
        x.fill(srm, T, F, before, end, [&](int t) {
            const float s = out[base + t];
            if (inside(t)) mine += static_cast<double>(s);
            return s - s * (inside(t) ? 1.0f : 0.0f);
        });
#pragma unroll
        for (int off = kWave / 2; off > 0; off >>= 1) mine += __shfl_down(mine, off, kWave);
        if ((threadIdx.x & (kWave - 1)) == 0) counted[threadIdx.x / kWave] = mine;
    } else {
        x.fill(srm, T, F, before, end, [&](int t) { return out[base + t] - desired[base + t]; });
    }
    __syncthreads();
    float addIn = 0.0f, addOut = 0.0f;
    if constexpr (COUNT) {
        const float actual = static_cast<float>(((counted[0] + counted[1]) + counted[2]) + counted[3]) * Ts;
        const double e = (static_cast<double>(actual) - (target.wanted[blockIdx.x] ? target.counts[0] : target.counts[1])) /
                         target.length * target.scale;
        addIn = static_cast<float>(e);
        addOut = static_cast<float>(e * 0.0);
    }
    float sq = 0.0f;
    for (int t = 4 * threadIdx.x; t < T; t += 1024) {
        float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        float4 late = *reinterpret_cast<const float4 *>(x.row + t);
        auto block = [&](int k, int taps) {     // (a tap that is not there must not meet an infinite sample)
            const float4 early = *reinterpret_cast<const float4 *>(x.row + t - k - 4);
            const float4 f = *reinterpret_cast<const float4 *>(x.filt + k);
            const float w[8] = {early.x, early.y, early.z, early.w, late.x, late.y, late.z, late.w};
            const float tap[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (i < taps) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[j] = fmaf(w[4 + j - i], tap[i], acc[j]);
                }
            late = early;
        };
        for (int k = 0; k + 4 <= F; k += 4) block(k, 4);
        if ((F & 3) != 0) block(F & ~3, F & 3);
        float e[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            e[j] = t + j < T ? acc[j] * Ts : 0.0f;
            if constexpr (COUNT) {
                if (t + j < T) e[j] += inside(t + j) ? addIn : addOut;
            } else if (addend && t + j < T) {
                e[j] += addend[base + t + j];
            }
            sq = fmaf(e[j], e[j], sq);
        }
        store4(error + base, t, T, e, vec);
    }
    // fixed-shape reduction: lanes of a wavefront, then the four wavefronts in order
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) sq += __shfl_down(sq, off, kWave);
    if ((threadIdx.x & (kWave - 1)) == 0) wsum[threadIdx.x / kWave] = sq;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = ((wsum[0] + wsum[1]) + wsum[2]) + wsum[3];
}

// grad[t] = Ts * sum_k x[t + k] srm[k] with x = error * (gradLoss * Ts), gradLoss one float on the device: the scaling and
// the correlation in one launch (three, and the scaled tensor in memory, when torch scales): (120, 300), 77 taps 17.3 -> 8 us,
// (12800, 2000), 8 taps 66 -> 45 us.  The sums are in double precision, which the vector ALUs add at the rate of single:
// closer to the exact sum (2.5e-8 of its 2-norm) than the matrix cores' (7.9e-8) and the chain's (1.9e-7) that they take the place of.
__global__ __launch_bounds__(256) void spike_loss_grad_kernel(float *__restrict__ grad, const float *__restrict__ error,
                                                              const float *__restrict__ gradLoss,
                                                              const float *__restrict__ srm, int T, int F, float Ts, bool vec)
{
    extern __shared__ __align__(16) float lds[];
    const int64_t base = static_cast<int64_t>(blockIdx.x) * T;
    const int end = ((T + 3) & ~3) + ((F + 3) & ~3) + 4;
    const RowInLds x(lds, F, 0);
    const float scale = gradLoss[0] * Ts;
    x.fill(srm, T, F, 0, end, [&](int t) { return error[base + t] * scale; });
    __syncthreads();
    for (int t = 4 * threadIdx.x; t < T; t += 1024) {
        double acc[4] = {0.0, 0.0, 0.0, 0.0};
        float4 early = *reinterpret_cast<const float4 *>(x.row + t);
        auto block = [&](int k, int taps) {
            const float4 late = *reinterpret_cast<const float4 *>(x.row + t + k + 4);
            const float4 f = *reinterpret_cast<const float4 *>(x.filt + k);
            const float w[8] = {early.x, early.y, early.z, early.w, late.x, late.y, late.z, late.w};
            const float tap[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (i < taps) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[j] = fma(static_cast<double>(w[j + i]), static_cast<double>(tap[i]), acc[j]);
                }
            early = late;
        };
        for (int k = 0; k + 4 <= F; k += 4) block(k, 4);
        if ((F & 3) != 0) block(F & ~3, F & 3);
        if (((acc[0] + acc[1]) + (acc[2] + acc[3])) * 0.0 != 0.0) {   // a tap that is not finite has met the zeros behind the row
            for (int j = 0; j < 4; ++j) {
                double sum = 0.0;
                for (int k = 0; k < min(T - t - j, F); ++k) sum = fma(static_cast<double>(x.row[t + j + k]), static_cast<double>(x.filt[k]), sum);
                acc[j] = sum;
            }
        }
        const float y[4] = {static_cast<float>(acc[0]) * Ts, static_cast<float>(acc[1]) * Ts, static_cast<float>(acc[2]) * Ts,
                            static_cast<float>(acc[3]) * Ts};
        store4(grad + base, t, T, y, vec);
    }
}

// loss = scale * sum of the row sums, in an order that the number of rows alone determines.
__global__ __launch_bounds__(1024) void spike_loss_sum_kernel(float *__restrict__ loss, const float *__restrict__ partial,
                                                              int64_t rows, float scale)
{
    // one work-group: 1024 lanes with four sums each, so that the loads of a trip do not wait for one another (12800 rows:
    // 256 lanes with one sum 14.2 us, this 4.7)
    __shared__ float wsum[16];
    float part[4] = {0.f, 0.f, 0.f, 0.f};
    int64_t r = threadIdx.x;
    for (; r + 3 * 1024 < rows; r += 4 * 1024) {
#pragma unroll
        for (int k = 0; k < 4; ++k) part[k] += partial[r + k * 1024];
    }
    for (; r < rows; r += 1024) part[0] += partial[r];
    float acc = (part[0] + part[1]) + (part[2] + part[3]);
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) acc += __shfl_down(acc, off, kWave);
    if ((threadIdx.x & (kWave - 1)) == 0) wsum[threadIdx.x / kWave] = acc;
    __syncthreads();
    if (threadIdx.x < kWave) {
        acc = threadIdx.x < 16 ? wsum[threadIdx.x] : 0.f;
#pragma unroll
        for (int off = 8; off > 0; off >>= 1) acc += __shfl_down(acc, off, kWave);
        if (threadIdx.x == 0) loss[0] = acc * scale;
    }
}

// A row and the filter must fit the LDS of one work-group (60 KB without what rounds them up), and the work-groups, one per
// row, a launch (lanes beyond the 2^32 of a launch would be left out without an error).
static bool rows_fit(int64_t rows, int64_t T, int64_t F)
{
    return (2 * F + T) * static_cast<int64_t>(sizeof(float)) <= 60 * 1024 && rows < (1LL << 24);
}
static int64_t row_lds_bytes(int64_t T, int64_t F) { return (2 * ((F + 3) & ~3LL) + ((T + 3) & ~3LL) + 8) * static_cast<int64_t>(sizeof(float)); }

}  // namespace slayer

extern "C" int64_t slayer_spike_loss_workspace_bytes(int64_t rows)
{
    return rows > 0 ? rows * static_cast<int64_t>(sizeof(float)) : 0;
}

// Both losses: target is null for the one with desired spike trains.
static int launch_loss(float *loss, float *error, const float *out, const float *desired, const float *addend,
                       const slayer::CountTarget *target, const float *srm, float *workspace, int64_t rows, int64_t T, int64_t F,
                       float Ts, void *stream)
{
    using namespace slayer;
    if (rows < 0 || T < 0 || F < 0) return SLAYER_EINVAL;
    if (!loss) return SLAYER_EINVAL;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int64_t live = (rows > 0 && T > 0) ? rows : 0;
    if (live > 0) {
        if (!error || !out || !(target ? static_cast<const void *>(target->wanted) : desired) || !workspace || (F > 0 && !srm))
            return SLAYER_EINVAL;
        if (!rows_fit(live, T, F)) return SLAYER_EUNSUPPORTED;
        const int64_t ldsBytes = row_lds_bytes(T, F);
        const dim3 grid(static_cast<unsigned>(live));
        const bool vec = T % 4 == 0 && aligned16(error);
        if (target)
            hipLaunchKernelGGL(spike_loss_rows_kernel<true>, grid, dim3(256), static_cast<size_t>(ldsBytes), st, error, workspace, out,
                               desired, addend, srm, static_cast<int>(T), static_cast<int>(F), Ts, vec, *target);
        else
            hipLaunchKernelGGL(spike_loss_rows_kernel<false>, grid, dim3(256), static_cast<size_t>(ldsBytes), st, error, workspace, out,
                               desired, addend, srm, static_cast<int>(T), static_cast<int>(F), Ts, vec, CountTarget{});
        const int status = launch_status();
        if (status != SLAYER_OK) return status;
    }
    hipLaunchKernelGGL(spike_loss_sum_kernel, dim3(1), dim3(1024), 0, st, loss, workspace, live, 0.5f * Ts);
    return launch_status();
}

extern "C" int slayer_spike_loss_f32(float *loss, float *error, const float *out, const float *desired,
                                     const float *addend, const float *srm, float *workspace, int64_t rows,
                                     int64_t T, int64_t F, float Ts, void *stream)
{
    return launch_loss(loss, error, out, desired, addend, nullptr, srm, workspace, rows, T, F, Ts, stream);
}

extern "C" int slayer_count_loss_f32(float *loss, float *error, const float *out, const uint8_t *wanted, const float *srm,
                                     float *workspace, int64_t rows, int64_t T, int64_t F, float Ts, int64_t start, int64_t stop,
                                     double countTrue, double countFalse, double length, double scale, void *stream)
{
    using namespace slayer;
    if (start < 0 || stop < 0 || start > T || stop > T) return SLAYER_EINVAL;
    const CountTarget target{wanted, static_cast<int>(start), static_cast<int>(stop), {countTrue, countFalse}, length, scale};
    return launch_loss(loss, error, out, nullptr, nullptr, &target, srm, workspace, rows, T, F, Ts, stream);
}

extern "C" int slayer_spike_loss_grad_f32(float *grad, const float *error, const float *gradLoss, const float *srm,
                                          int64_t rows, int64_t T, int64_t F, float Ts, void *stream)
{
    using namespace slayer;
    if (rows < 0 || T < 0 || F < 0) return SLAYER_EINVAL;
    if (rows == 0 || T == 0) return SLAYER_OK;
    if (!grad || !error || !gradLoss || (F > 0 && !srm)) return SLAYER_EINVAL;
    if (!rows_fit(rows, T, F)) return SLAYER_EUNSUPPORTED;
    hipLaunchKernelGGL(spike_loss_grad_kernel, dim3(static_cast<unsigned>(rows)), dim3(256),
                       static_cast<size_t>(row_lds_bytes(T, F)), static_cast<hipStream_t>(stream), grad, error, gradLoss, srm,
                       static_cast<int>(T), static_cast<int>(F), Ts, T % 4 == 0 && aligned16(grad));
    return launch_status();
}
