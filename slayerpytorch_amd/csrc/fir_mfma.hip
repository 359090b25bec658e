// Temporal FIR of neuron rows on the matrix cores, for dense input and filters of 34 to 129 taps, where the
// register-window kernels of fir.hip are bound by FMA issue (an FIR of 77 taps needs 154 flop per 8 bytes).
// Correlation only (plain, or with the spike function's surrogate gradient applied to the samples on their way
// into LDS): the convolution's input is mostly spike trains, which the tiled kernel of fir.hip serves through
// its event-driven path.
//
// For Y[m] = sum_t X[m+t] * filt[t], the 16 outputs of block b (16 samples) of 16 rows are the 16x16 product
//
//     Y[16b + i][row c] = sum_k  filt[k - i] * X[16b + k][row c]        (k over the 15 + F samples from 16b on)
//
// of a banded Toeplitz matrix made of the filter (zero where k - i is not a tap) and the rows' samples.
//
// A work-group is ONE wavefront that walks over the chunks of 16 consecutive rows; the window of samples lives in
// registers and moves on by what one step consumes, so each step reads only new samples (the walk is unrolled by the
// window size).  No barriers: the wavefronts of a compute unit overlap each other's memory and matrix work.
//
// Two kernels.  fir_mfma_split_kernel: tiles of 16 whole rows kept in LDS exactly as they lie in memory, copied with
// 16-byte accesses that run through the rows' memory front to back, for short aligned rows whose length spreads them over
// the LDS banks as it is (T / 4 odd).  fir_walk_kernel: rows of any length and alignment, straight from and to memory.
//
// The matrix instructions sum their products in their own order, so results agree with the sequential chain to
// rounding (a few 1e-7 of sum |x| |filt|), not bit for bit.  A structural zero times a non-finite sample would
// be NaN where the chain has no such term: a wavefront that meets a non-finite sample computes its outputs with the
// sequential chain over the valid taps instead.
#include "common.h"
#include "fir_core.h"

namespace slayer {

constexpr int kMfmaMaxBlocks = 19;   // blocks of 16 samples per row of a tile: 8 tiles in a compute unit's 160 KB of LDS

struct MfmaFirArgs {
    float *out;
    const float *in, *filt;
    int64_t rows;
    int T, F;
    int nv;         // 16-byte vectors per lane and tile that are in use (<= NV; nv KiB of LDS)
    uint32_t nItems;
    float Ts;
    FirGate gate;  // GATED: the samples are in * gain * exp(-|u - theta| / tau), applied on the way into LDS
};

// ---- bf16 instructions on a three-way split of both operands ------------------------------------------------------
// v_mfma_f32_16x16x32_bf16 multiplies 8 pairs in the time the fp32 instruction takes for one.  An fp32 number is the sum of
// three bf16 numbers: the nearest one, the one nearest to the remainder, and what is left then (8 significant bits each and
// the signs of the remainders: all 24 bits).  A product of two split numbers is then the sum of nine bf16 products, each
// exact in the instruction's fp32 accumulator.  The three smallest (mid x low, low x mid, low x low: below 2^-24 of the
// product together, of either sign) are left out; the six others take 6 / 8 of an fp32 instruction's time.  (Cut instead
// of rounded parts leave out up to 2^-21, always towards zero: sums of one term were 5.8e-8 off, root mean square, where the
// chain is 2.5e-8 off.  Rounded: 2.6e-8, and full windows 5.5e-8 instead of 7.6e-8 of their 2-norm, the chain 1.6e-7.)
// The instruction reads a bf16 operand below 2^-126 as zero, which drops parts of samples and taps
// below 2^-102 of size: at most 2^-124 * (sum |filt| + sum |x| over an output's window) in absolute terms.
// A tap that is not finite has no split, so then all tiles take the chains (as a tile with such a sample does).
//
// The rows are cut into chunks of 32 samples.  A lane (c = lane % 16, h = lane / 16) holds samples 8h .. 8h + 7 of
// each chunk of row c in the window - split once per sample, three register quadruples per chunk - and, for either
// 16-output block of a chunk, filt[32 s + 8h + e - c (- 16 for the second block)] for the window's chunks s, split the
// same way when the kernel starts.  One step makes both blocks of a chunk from the NC chunks from it on.
//
// The tile: vector e of the 16 rows' memory is vector e of LDS, no index arithmetic; the range check of the buffers
// masks what lies behind the last row of the tensor.  The last chunk of a row ends in the first samples of the next
// row, which the walk masks.
// NC: chunks in the window (the second block of a chunk reaches 31 + F samples from the chunk's start); NCE: chunks
// that the first block reaches.  NV: 16-byte vectors per lane and tile.
template <int NCE, int NC, int NV, bool GATED>
__global__ __launch_bounds__(64, 2) void fir_mfma_split_kernel(MfmaFirArgs p)
{
    extern __shared__ __align__(16) float X[];
    const int lane = threadIdx.x;
    const int c = lane & 15, h = lane >> 4;
    const int T = p.T, F = p.F;
    const int nCh = (T + 31) >> 5;

    const BufferRsrc bufF = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p.filt), 0, F * 4, 0x00020000);
    SplitPlanes aE[NCE], aO[NC];
    bool badTap = false;
#pragma unroll
    for (int s = 0; s < NC; ++s) {
        float fe[8], fo[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int tap = 32 * s + 8 * h + e - c;
            fe[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(bufF, masked_offset(tap >= 0 && tap < F, tap * 4), 0, 0));
            fo[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(bufF, masked_offset(tap >= 16 && tap - 16 < F, (tap - 16) * 4), 0, 0));
            badTap |= fe[e] * 0.0f != 0.0f || fo[e] * 0.0f != 0.0f;
        }
        if (s < NCE) aE[s] = split_bf16(fe);
        aO[s] = split_bf16(fo);
    }
    // (a tap that is not finite has no split: every tile as chains)
    const bool chainsAlways = __builtin_amdgcn_ballot_w64(badTap) != 0;

    struct Tile {
        int64_t row0;
        int nRows;
    };
    auto tile_of = [&](uint32_t i) {
        Tile q;
        q.row0 = static_cast<int64_t>(xcd_contiguous(i, p.nItems)) * 16;
        q.nRows = static_cast<int>(min(static_cast<int64_t>(16), p.rows - q.row0));
        return q;
    };
    // A tile's vectors (and, GATED, those of its potentials) come in three parts.  The first travels while the tile
    // before is walked: as many vectors as the registers hold beside the walk's operands (12 registers per chunk of
    // either filter operand and of the window; about 50 others).  The second is fetched when that walk has ended and
    // its window is free, ahead of the stores.  What does not fit beside the filter operands even then is fetched by
    // stage(), one vector for each one that it has put into LDS.
    constexpr int kRoom = (242 - 50 - 12 * (NCE + 2 * NC)) / 4;
    constexpr int kStageRoom = (242 - 50 - 12 * (NCE + NC)) / 4;
    constexpr int kAhead = (GATED ? kStageRoom / 2 : kStageRoom) < NV ? (GATED ? kStageRoom / 2 : kStageRoom) : NV;
    constexpr int kEarly = (GATED ? (kRoom + 1) / 2 : kRoom) < kAhead ? (GATED ? (kRoom + 1) / 2 : kRoom) : kAhead;
    constexpr int kEarlyU = kRoom / 2 < kAhead ? kRoom / 2 : kAhead;
    static_assert(kRoom >= 2 && kAhead >= 1, "no registers left for the tile");
    float4 pre[NV], preU[GATED ? NV : 1];
    auto fetch_one = [&](const Tile &q, int k) {
        const BufferRsrc bufIn = make_buffer(p.in + q.row0 * T, q.nRows * T * 4);
        pre[k] = buffer_load4(bufIn, lane * 16, kWave * 16 * k);
        if (GATED) {
            const BufferRsrc bufU = make_buffer(p.gate.u + q.row0 * T, q.nRows * T * 4);
            preU[k] = buffer_load4(bufU, lane * 16, kWave * 16 * k);
        }
    };
    auto fetch = [&](const Tile &q, bool second) {
        const BufferRsrc bufIn = make_buffer(p.in + q.row0 * T, q.nRows * T * 4);
        const BufferRsrc bufU = make_buffer(GATED ? p.gate.u + q.row0 * T : p.in, q.nRows * T * 4);
#pragma unroll
        for (int k = 0; k < kAhead; ++k) {
            if ((k >= kEarly) == second) pre[k] = buffer_load4(bufIn, lane * 16, kWave * 16 * k);
            if (GATED && (k >= kEarlyU) == second) preU[k] = buffer_load4(bufU, lane * 16, kWave * 16 * k);
        }
    };
    auto stage = [&](const Tile &q) {
        bool bad = false;
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            float4 x = pre[k];
            if (GATED)
                x = make_float4(x.x * spike_pdf(preU[k].x, p.gate.theta, p.gate.tau, p.gate.gain),
                                x.y * spike_pdf(preU[k].y, p.gate.theta, p.gate.tau, p.gate.gain),
                                x.z * spike_pdf(preU[k].z, p.gate.theta, p.gate.tau, p.gate.gain),
                                x.w * spike_pdf(preU[k].w, p.gate.theta, p.gate.tau, p.gate.gain));
            if (k + kAhead < NV) fetch_one(q, k + kAhead);
            if (k >= p.nv) continue;
            bad |= ((x.x + x.y) + (x.z + x.w)) * 0.0f != 0.0f;
            *reinterpret_cast<float4 *>(X + 4 * (lane + kWave * k)) = x;
        }
        return __builtin_amdgcn_ballot_w64(bad) != 0;
    };

    uint32_t i = blockIdx.x;
    if (i >= p.nItems) return;
    Tile cur = tile_of(i);
    fetch(cur, false);
    fetch(cur, true);
    {
        const BufferRsrc none = make_buffer(p.out, 0);
#pragma unroll
        for (int k = 0; k < NV; ++k) buffer_store4(none, (lane + kWave * k) * 16, 0, make_float4(static_cast<float>(k), 0.0f, 0.0f, 0.0f));
    }
    for (;;) {
        const bool chains = stage(cur) || chainsAlways;
        wave_sync();
        const uint32_t iNext = i + gridDim.x;
        const bool more = iNext < p.nItems;
        Tile next = tile_of(more ? iNext : i);
        if (!more) next.nRows = 0;
        fetch(next, false);
        if (chains) {
            for (int e = lane; e < cur.nRows * T; e += kWave) {
                const int r = e / T, t = e - r * T;
                const float *x = p.in + (cur.row0 + r) * T;
                const float *gu = GATED ? p.gate.u + (cur.row0 + r) * T : nullptr;
                const int taps = min(T - t, F);
                float acc = 0.0f;
                for (int k = 0; k < taps; ++k) {
                    acc = __builtin_fmaf(GATED ? x[t + k] * spike_pdf(gu[t + k], p.gate.theta, p.gate.tau, p.gate.gain) : x[t + k],
                                         p.filt[k], acc);
                }
                p.out[(cur.row0 + r) * T + t] = acc * p.Ts;
            }
        } else {
            // step m makes outputs 32 m .. 32 m + 31 from chunks m .. m + NC - 1 and writes them over chunk m
            float *col = X + c * T + 8 * h;
            const float *zeros = X + 16 * T;
            // chunk s of the lane's row; behind the row (where the next row lies), zeros
            auto raw = [&](int s, float4 &v0, float4 &v1) {
                const int t = 32 * s + 8 * h;
                v0 = *reinterpret_cast<const float4 *>(t < T ? col + 32 * s : zeros);
                v1 = *reinterpret_cast<const float4 *>(t + 4 < T ? col + 32 * s + 4 : zeros);
            };
            auto split = [&](const float4 &v0, const float4 &v1) {
                const float x[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
                return split_bf16(x);
            };
            SplitPlanes w[NC];
#pragma unroll
            for (int s = 0; s < NC; ++s) {
                float4 v0, v1;
                raw(s, v0, v1);
                w[s] = split(v0, v1);
            }
            for (int m0 = 0; m0 < nCh; m0 += NC) {
#pragma unroll
                for (int u = 0; u < NC; ++u) {
                    const int m = m0 + u;
                    if (m < nCh) {
                        float4 v0, v1;
                        raw(m + NC, v0, v1);  // the chunk that the next step adds
                        __builtin_amdgcn_sched_barrier(0);
                        // four sums: the leading products and the five smaller ones, of either block
                        f32x4 e0 = {0.0f, 0.0f, 0.0f, 0.0f}, e1 = e0, o0 = e0, o1 = e0;
#pragma unroll
                        for (int s = 0; s < NC; ++s) {
                            const SplitPlanes &x = w[(u + s) % NC];
                            if (s < NCE) e1 = mfma_bf16(aE[s].lo, x.hi, e1);
                            o1 = mfma_bf16(aO[s].lo, x.hi, o1);
                            if (s < NCE) e1 = mfma_bf16(aE[s].hi, x.lo, e1);
                            o1 = mfma_bf16(aO[s].hi, x.lo, o1);
                            if (s < NCE) e1 = mfma_bf16(aE[s].mid, x.mid, e1);
                            o1 = mfma_bf16(aO[s].mid, x.mid, o1);
                            if (s < NCE) e1 = mfma_bf16(aE[s].mid, x.hi, e1);
                            o1 = mfma_bf16(aO[s].mid, x.hi, o1);
                            if (s < NCE) e1 = mfma_bf16(aE[s].hi, x.mid, e1);
                            o1 = mfma_bf16(aO[s].hi, x.mid, o1);
                            if (s < NCE) e0 = mfma_bf16(aE[s].hi, x.hi, e0);
                            o0 = mfma_bf16(aO[s].hi, x.hi, o0);
                        }
                        const int t = 32 * m + 4 * h;
                        if (t < T)
                            *reinterpret_cast<float4 *>(col + 32 * m - 4 * h) =
                                make_float4((e0.x + e1.x) * p.Ts, (e0.y + e1.y) * p.Ts, (e0.z + e1.z) * p.Ts, (e0.w + e1.w) * p.Ts);
                        if (t + 16 < T)
                            *reinterpret_cast<float4 *>(col + 32 * m + 16 - 4 * h) =
                                make_float4((o0.x + o1.x) * p.Ts, (o0.y + o1.y) * p.Ts, (o0.z + o1.z) * p.Ts, (o0.w + o1.w) * p.Ts);
                        w[u] = split(v0, v1);
                    }
                }
            }
        }
        wave_sync();
        fetch(next, true);
        const BufferRsrc bufOut = make_buffer(p.out + cur.row0 * T, chains ? 0 : cur.nRows * T * 4);
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            buffer_store4(bufOut, lane * 16, kWave * 16 * k, *reinterpret_cast<const float4 *>(X + (k < p.nv ? 4 * (lane + kWave * k) : 0)));
            if (k % 8 == 7) __builtin_amdgcn_sched_barrier(0);
        }
        if (!more) break;
        wave_sync();
        i = iNext;
        cur = next;
    }
}

// ---- the same product for rows of any length and alignment, gated or not -------------------------------------------
// One wavefront walks over 16 rows chunk by chunk (32 samples), as above, but the samples come straight from memory
// into the lane that multiplies them, two chunks ahead, and the outputs leave straight from the accumulators, either way 64
// contiguous bytes per row and instruction (a lane holds samples 4h .. 4h + 3 and 16 + 4h .. of a chunk): no LDS, so a row may have any length, and
// 16-byte accesses at any multiple of four bytes, so it may start anywhere.  Chunks that reach past the end of the row are
// loaded (and the last outputs stored) sample by sample.  A long row is cut into segments where there are few rows;
// a segment reads the NC - 1 chunks behind its own.  GATED: `shift` delays the gate against the samples, i.e. the samples
// are in[t + shift] (zero from T on): the adjoint of a delay that follows the spike function.
// An item (16 rows, one segment) in which a sample is not finite is noted and computed again as chains after the walk.
// Measured, against the kernels that these rows took before (chains on the vector ALUs for rows that are not whole
// vectors, fp32 matrix instructions for the others): gated, 110 taps, rows of 1450 samples: 65536 rows 580 -> 340 us, 8192
// rows 79 -> 40, 44 rows 13.4 -> 9.5; plain, 77 taps: (16384, 2000) 92 -> 46 us, (60000, 512) 84 -> 48, (25, 500) 11.2 ->
// 7.6.  Error against double precision (2-norm): 1.6e-7 -> 5.5e-8, sums of one term 2.5e-8 -> 2.6e-8.  Bound by the pieces of many rows that it reads and writes
// (3.4 TB/s; 4.1 where rows start on memory lines, 5.6 on tensors in the last-level cache): 77 taps take as long as 110, and
// a gate with half the instructions changed nothing.
struct WalkArgs {
    float *out;
    const float *in, *filt;
    int64_t rows;
    int T, F, shift;
    int segChunks, segs;    // chunks per segment, segments per row
    uint32_t nItems;
    FastDiv bySegs;
    float Ts;
    FirGate gate;
    const float *poolW;     // POOL: FirPool, and the divisors of its extents
    int poolOH, poolOW;
    FastDiv byHW, byW, byKH, byKW;
};

// POOL: the samples come from the rows of the pooled tensor whose windows the rows lie in, times the weight of the row's place
// there - the gradient of a pooling layer, spread on the way in instead of through memory (a quarter of the rows is read, and
// most of them from L2).  Training the gesture network on (4, 128, 128, 1450): 2778 -> 2580 us.
template <int NCE, int NC, bool GATED, bool POOL>
__global__ __launch_bounds__(64, 2) void fir_walk_kernel(WalkArgs p)
{
    const int lane = threadIdx.x;
    const int c = lane & 15, h = lane >> 4;
    const int T = p.T, F = p.F, nCh = (T + 31) >> 5;

    const BufferRsrc bufF = make_buffer(p.filt, F * 4);
    SplitPlanes aE[NCE], aO[NC];
    bool badTap = false;
#pragma unroll
    for (int s = 0; s < NC; ++s) {
        float fe[8], fo[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int tap = 32 * s + 4 * h + e + (e < 4 ? 0 : 12) - c;
            fe[e] = buffer_load<kCached>(bufF, masked_offset(tap >= 0 && tap < F, tap * 4), 0);
            fo[e] = buffer_load<kCached>(bufF, masked_offset(tap >= 16 && tap - 16 < F, (tap - 16) * 4), 0);
            badTap |= fe[e] * 0.0f != 0.0f || fo[e] * 0.0f != 0.0f;
        }
        if (s < NCE) aE[s] = split_bf16(fe);
        aO[s] = split_bf16(fo);
    }
    const bool chainsAlways = __builtin_amdgcn_ballot_w64(badTap) != 0;

    for (uint32_t i = blockIdx.x; i < p.nItems; i += gridDim.x) {
        const uint32_t item = xcd_contiguous(i, p.nItems);
        const uint32_t rowGroup = fastdiv(item, p.bySegs);
        const int seg = static_cast<int>(item - rowGroup * p.bySegs.d);
        const int64_t row0 = static_cast<int64_t>(rowGroup) * 16;
        const int nRows = static_cast<int>(min(static_cast<int64_t>(16), p.rows - row0));
        const int mBegin = seg * p.segChunks, mEnd = min(nCh, mBegin + p.segChunks);
        const BufferRsrc bufOut = make_buffer(p.out + row0 * T);
        const BufferRsrc bufU = make_buffer((GATED ? p.gate.u : p.in) + row0 * T);
        const int laneOff = masked_offset(c < nRows, (c * T + 4 * h) * 4);   // sample 4 h of the lane's row
        // POOL: the row of the pooled tensor behind row n of this one, counted from the first pooled plane of the item, and
        // the weight; a row behind the last whole window has none
        const uint32_t plane0 = POOL ? fastdiv(static_cast<uint32_t>(row0), p.byHW) : 0u;
        auto pooled = [&](uint32_t n, bool &inside, float &weight) {
            const uint32_t plane = fastdiv(n, p.byHW), pix = n - plane * p.byHW.d;
            const uint32_t y = fastdiv(pix, p.byW), x = pix - y * p.byW.d, a = fastdiv(y, p.byKH), b = fastdiv(x, p.byKW);
            inside = a < static_cast<uint32_t>(p.poolOH) && b < static_cast<uint32_t>(p.poolOW);
            weight = inside ? p.poolW[(y - a * p.byKH.d) * p.byKW.d + (x - b * p.byKW.d)] : 0.0f;
            return static_cast<int>(((plane - plane0) * p.poolOH + a) * p.poolOW + b);
        };
        const float *const in0 = POOL ? p.in + static_cast<int64_t>(plane0) * p.poolOH * p.poolOW * T : p.in + row0 * T;
        const BufferRsrc bufIn = make_buffer(in0);
        int laneIn = laneOff;
        float laneW = 1.0f;
        if (POOL) {
            bool inside;
            const int row = pooled(static_cast<uint32_t>(row0) + min(c, nRows - 1), inside, laneW);
            laneIn = masked_offset(inside && c < nRows, (row * T + 4 * h) * 4);
        }

        struct Raw {
            float4 x0, x1, u0, u1;
        };
        auto load = [&](Raw &r, int s) {
            const int t0 = 32 * s;
            if (t0 + 32 + p.shift <= T) {
                r.x0 = buffer_load4<kCached>(bufIn, laneIn, (t0 + p.shift) * 4);
                r.x1 = buffer_load4<kCached>(bufIn, laneIn, (t0 + p.shift) * 4 + 64);
                if (GATED) {
                    r.u0 = buffer_load4<kCached>(bufU, laneOff, t0 * 4);
                    r.u1 = buffer_load4<kCached>(bufU, laneOff, t0 * 4 + 64);
                }
            } else if (t0 >= T) {
                r.x0 = r.x1 = r.u0 = r.u1 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            } else {
                float x[8], u[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int k = t0 + e + (e < 4 ? 0 : 12), t = k + 4 * h;
                    const bool row = laneOff != kOutOfRange, inRow = laneIn != kOutOfRange;
                    x[e] = buffer_load<kCached>(bufIn, masked_offset(inRow && t + p.shift < T, laneIn + (k + p.shift) * 4), 0);
                    u[e] = GATED ? buffer_load<kCached>(bufU, masked_offset(row && t < T, laneOff + k * 4), 0) : 0.0f;
                }
                r.x0 = make_float4(x[0], x[1], x[2], x[3]);
                r.x1 = make_float4(x[4], x[5], x[6], x[7]);
                r.u0 = make_float4(u[0], u[1], u[2], u[3]);
                r.u1 = make_float4(u[4], u[5], u[6], u[7]);
            }
        };
        bool bad = false;
        auto enter = [&](const Raw &r) {
            float x[8] = {r.x0.x, r.x0.y, r.x0.z, r.x0.w, r.x1.x, r.x1.y, r.x1.z, r.x1.w};
            if (POOL) {
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] *= laneW;
            }
            if (GATED) {
                const float u[8] = {r.u0.x, r.u0.y, r.u0.z, r.u0.w, r.u1.x, r.u1.y, r.u1.z, r.u1.w};
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] *= spike_pdf(u[e], p.gate.theta, p.gate.tau, p.gate.gain);
            }
            bad |= (((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]))) * 0.0f != 0.0f;
            return split_bf16(x);
        };
        auto store = [&](int t0, const f32x4 &a, const f32x4 &b) {   // outputs t0 + 4 h .. + 3 of the lane's row
            const float y[4] = {(a.x + b.x) * p.Ts, (a.y + b.y) * p.Ts, (a.z + b.z) * p.Ts, (a.w + b.w) * p.Ts};
            // (cached: the two blocks of a chunk, and neighbouring chunks, complete each other's memory lines)
            if (t0 + 16 <= T) {
                buffer_store4<kCached>(bufOut, laneOff, t0 * 4, make_float4(y[0], y[1], y[2], y[3]));
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    buffer_store<kCached>(bufOut, masked_offset(laneOff != kOutOfRange && t0 + 4 * h + e < T, laneOff + (t0 + e) * 4), 0, y[e]);
            }
        };

        SplitPlanes w[NC];
        Raw raw[2];
        {
            Raw r[NC];
#pragma unroll
            for (int s = 0; s < NC; ++s) load(r[s], mBegin + s);
            load(raw[0], mBegin + NC);
#pragma unroll
            for (int s = 0; s < NC; ++s) w[s] = enter(r[s]);
        }
        for (int m0 = mBegin; m0 < mEnd; m0 += 2 * NC) {
#pragma unroll
            for (int v = 0; v < 2 * NC; ++v) {
                const int m = m0 + v, u = v % NC;
                if (m < mEnd) {
                    load(raw[(v + 1) & 1], m + NC + 1);   // (enters the window one step after the next)
                    __builtin_amdgcn_sched_barrier(0);
                    f32x4 e0 = {0.0f, 0.0f, 0.0f, 0.0f}, e1 = e0, o0 = e0, o1 = e0;
#pragma unroll
                    for (int s = 0; s < NC; ++s) {
                        const SplitPlanes &x = w[(u + s) % NC];
                        if (s < NCE) e1 = mfma_bf16(aE[s].lo, x.hi, e1);
                        o1 = mfma_bf16(aO[s].lo, x.hi, o1);
                        if (s < NCE) e1 = mfma_bf16(aE[s].hi, x.lo, e1);
                        o1 = mfma_bf16(aO[s].hi, x.lo, o1);
                        if (s < NCE) e1 = mfma_bf16(aE[s].mid, x.mid, e1);
                        o1 = mfma_bf16(aO[s].mid, x.mid, o1);
                        if (s < NCE) e1 = mfma_bf16(aE[s].mid, x.hi, e1);
                        o1 = mfma_bf16(aO[s].mid, x.hi, o1);
                        if (s < NCE) e1 = mfma_bf16(aE[s].hi, x.mid, e1);
                        o1 = mfma_bf16(aO[s].hi, x.mid, o1);
                        if (s < NCE) e0 = mfma_bf16(aE[s].hi, x.hi, e0);
                        o0 = mfma_bf16(aO[s].hi, x.hi, o0);
                    }
                    store(32 * m, e0, e1);
                    store(32 * m + 16, o0, o1);
                    w[u] = enter(raw[v & 1]);
                }
            }
        }
        if (chainsAlways || __builtin_amdgcn_ballot_w64(bad) != 0) {
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "agent");   // the walk's stores are done before the same samples are written again
            const int tA = 32 * mBegin, n = min(T, 32 * mEnd) - tA;
            for (int e = lane; e < nRows * n; e += kWave) {
                const int r = e / n, t = tA + e - r * n;
                bool inside = true;
                float weight = 1.0f;
                const float *x = POOL ? in0 + static_cast<int64_t>(pooled(static_cast<uint32_t>(row0) + r, inside, weight)) * T : p.in + (row0 + r) * T;
                const float *gu = GATED ? p.gate.u + (row0 + r) * T : nullptr;
                const int taps = min(T - t, F);
                float acc = 0.0f;
                for (int k = 0; k < taps; ++k) {
                    float v = inside && t + k + p.shift < T ? x[t + k + p.shift] : 0.0f;
                    if (POOL) v *= weight;
                    acc = __builtin_fmaf(GATED ? v * spike_pdf(gu[t + k], p.gate.theta, p.gate.tau, p.gate.gain) : v, p.filt[k], acc);
                }
                p.out[(row0 + r) * T + t] = acc * p.Ts;
            }
        }
    }
}

template <bool GATED>
static void launch_split(int nce, int nc, int nv, dim3 grid, size_t lds, hipStream_t st, const MfmaFirArgs &args)
{
#define SLAYER_SPLIT_NV(E, C)                                                                                          \
    if (nv <= 12) hipLaunchKernelGGL((fir_mfma_split_kernel<E, C, 12, GATED>), grid, dim3(64), lds, st, args);        \
    else if (nv <= 16) hipLaunchKernelGGL((fir_mfma_split_kernel<E, C, 16, GATED>), grid, dim3(64), lds, st, args);   \
    else hipLaunchKernelGGL((fir_mfma_split_kernel<E, C, 20, GATED>), grid, dim3(64), lds, st, args)
    if (nc == 3 && nce == 2) { SLAYER_SPLIT_NV(2, 3); }
    else if (nc == 3) { SLAYER_SPLIT_NV(3, 3); }
    else if (nc == 4 && nce == 3) { SLAYER_SPLIT_NV(3, 4); }
    else if (nc == 4) { SLAYER_SPLIT_NV(4, 4); }
    else if (nce == 4) { SLAYER_SPLIT_NV(4, 5); }
    else { SLAYER_SPLIT_NV(5, 5); }
#undef SLAYER_SPLIT_NV
}

// Segments of a row so that the walks of the wavefronts resident at once end together: the fewest chunks that any of
// them passes, counting what a segment reads beyond its own and about eight chunks' time for its start.
static int walk_segments(int64_t rowGroups, int nCh, int nc, int64_t resident)
{
    int best = 1;
    int64_t bestCost = -1;
    for (int segs = 1; segs <= nCh && segs <= 64; ++segs) {
        const int64_t cost = ceil_div(rowGroups * segs, resident) * (ceil_div(nCh, segs) + nc + 8);
        if (bestCost < 0 || cost < bestCost) {
            best = segs;
            bestCost = cost;
        }
    }
    return best;
}

template <bool GATED, bool POOL>
static void launch_walk(int nce, int nc, dim3 grid, hipStream_t st, const WalkArgs &a)
{
    if (nc == 3 && nce == 2) hipLaunchKernelGGL((fir_walk_kernel<2, 3, GATED, POOL>), grid, dim3(64), 0, st, a);
    else if (nc == 3) hipLaunchKernelGGL((fir_walk_kernel<3, 3, GATED, POOL>), grid, dim3(64), 0, st, a);
    else if (nc == 4 && nce == 3) hipLaunchKernelGGL((fir_walk_kernel<3, 4, GATED, POOL>), grid, dim3(64), 0, st, a);
    else if (nc == 4) hipLaunchKernelGGL((fir_walk_kernel<4, 4, GATED, POOL>), grid, dim3(64), 0, st, a);
    else if (nce == 4) hipLaunchKernelGGL((fir_walk_kernel<4, 5, GATED, POOL>), grid, dim3(64), 0, st, a);
    else hipLaunchKernelGGL((fir_walk_kernel<5, 5, GATED, POOL>), grid, dim3(64), 0, st, a);
}

// Aligned rows of at most 304 samples whose length spreads 16 of them over the LDS banks as it is (T / 4 odd): tiles.
static bool fits_tiles(int64_t T, const void *out, const void *in, const void *u)
{
    return T % 8 == 4 && T <= 16 * kMfmaMaxBlocks && aligned16(out) && aligned16(in) && aligned16(u);
}

bool launch_fir_corr_walk(float *out, const float *in, const float *filt, int64_t rows, int64_t T, int64_t F, int64_t shift,
                          float Ts, const FirGate &gate, hipStream_t stream, const FirPool &pool)
{
    // rows of a pooled tensor: counted in 32 bits, and 16 rows' windows within 2 GiB of the first one's plane
    if (pool.w && (!gate.u || rows >= (1LL << 31) || (static_cast<int64_t>(pool.OH) * pool.OW * 17 + 1) * T * 4 >= (1LL << 31))) return false;
    // (rows that the tiles take without a shift are shifted apart, so that a delay's gradient has the same bits either way)
    if ((shift > 0 || pool.w) && fits_tiles(T, out, in, gate.u)) return false;
    if (F < kFirMfmaMinTaps || F > kFirMfmaMaxTaps || T < 16 || T > kBufferMaxT || shift < 0 || shift > T) return false;
    const int nCh = static_cast<int>(ceil_div(T, 32));
    const int nce = static_cast<int>((15 + F + 31) / 32), nc = static_cast<int>((31 + F + 31) / 32);
    const int64_t rowGroups = ceil_div(rows, 16), resident = static_cast<int64_t>(compute_units()) * 8;
    if (rowGroups >= (1LL << 31)) return false;
    int segs = rowGroups < (1LL << 24) ? walk_segments(rowGroups, nCh, nc, resident) : 1;   // (items are counted in 32 bits)
    const int segChunks = static_cast<int>(ceil_div(nCh, segs));
    segs = static_cast<int>(ceil_div(nCh, segChunks));
    const int64_t items = rowGroups * segs;
    const int64_t waves = items < resident ? items : resident;   // (resident: a multiple of 8, one range of items per die)
    const FirPool m = pool.w ? pool : FirPool{nullptr, 1, 1, 1, 1, 1, 1};
    const WalkArgs a{out, in, filt, rows, static_cast<int>(T), static_cast<int>(F), static_cast<int>(shift), segChunks, segs,
                     static_cast<uint32_t>(items), make_fastdiv(static_cast<uint32_t>(segs)), Ts, gate, m.w, m.OH, m.OW,
                     make_fastdiv(static_cast<uint32_t>(m.H) * static_cast<uint32_t>(m.W)), make_fastdiv(static_cast<uint32_t>(m.W)),
                     make_fastdiv(static_cast<uint32_t>(m.KH)), make_fastdiv(static_cast<uint32_t>(m.KW))};
    const dim3 grid(static_cast<unsigned>(waves));
    if (pool.w) launch_walk<true, true>(nce, nc, grid, stream, a);
    else if (gate.u) launch_walk<true, false>(nce, nc, grid, stream, a);
    else launch_walk<false, false>(nce, nc, grid, stream, a);
    return true;
}

bool launch_fir_corr_mfma(float *out, const float *in, const float *filt, int64_t rows, int64_t T, int64_t F, float Ts,
                          const FirGate &gate, bool chainBits, hipStream_t stream)
{
    // Tiles of whole rows in LDS as they lie in memory, for aligned rows whose length spreads the 16 rows over the banks
    // as it is and that are short enough for eight tiles on a compute unit: the walk over rows in memory reads its first
    // chunks and its ragged last ones again, which counts on short rows (rows of 300 samples: 110 taps gated 111 us here,
    // 153 us there; 77 taps 112 and 157 us).  Everything else walks, but for rows that are not whole aligned vectors where
    // the caller has been promised the bits of the chain for them (chainBits).
    if (chainBits && !(T % 4 == 0 && aligned16(out) && aligned16(in) && aligned16(gate.u))) return false;
    const bool tiles = F >= kFirMfmaMinTaps && F <= kFirMfmaMaxTaps && T >= 16 && fits_tiles(T, out, in, gate.u) &&
                       ceil_div(rows, 16) < (1LL << 31);
    if (!tiles) return launch_fir_corr_walk(out, in, filt, rows, T, F, 0, Ts, gate, stream);
    const int nv = static_cast<int>(ceil_div(T, 16));
    const int64_t items = ceil_div(rows, 16);
    // wavefronts resident at once (8 per compute unit); each walks over its share of the tiles
    const int64_t resident = static_cast<int64_t>(compute_units()) * 8;
    const int64_t trips = ceil_div(items, resident);
    const int64_t waves = ceil_div(ceil_div(items, trips), 8) * 8;  // a multiple of 8: one range of tiles per die
    MfmaFirArgs args{out, in, filt, rows, static_cast<int>(T), static_cast<int>(F), nv, static_cast<uint32_t>(items), Ts, gate};
    const dim3 grid(static_cast<unsigned>(waves));
    const size_t lds = static_cast<size_t>(nv) * 1024;
    const int nce = static_cast<int>((15 + F + 31) / 32), nc = static_cast<int>((31 + F + 31) / 32);
    if (gate.u) launch_split<true>(nce, nc, nv, grid, lds, stream, args);
    else launch_split<false>(nce, nc, nv, grid, lds, stream, args);
    return true;
}

}  // namespace slayer
