// The 3x3, stride-1 gather (forward pass and input gradient of a convolution synapse) with the source rows in a ring.
//
// As in synapse_gather_planes_kernel the taps and 16 source channels are the reduction axis of v_mfma_f32_16x16x32_bf16 over
// operands split into three bf16 parts, and every sample is split once, when it is staged, into three planes in LDS.  There a
// work-group reloads and resplits the three rows under every row of destination pixels, between two barriers, which is more
// than half of its time.  Here it walks a strip of columns (eight pixels wide, four where there are two passes of 16 source
// channels) down the image, one step of 32 samples at a time: LDS holds four source rows of the strip as a ring, three that
// are read and the one below that is staged meanwhile, so that a sample is loaded 1.25 (1.5) times instead of 3.75 and a row
// costs one barrier.  The weights sit in registers, 60 per pass and tile of 16 channels: that makes the room in LDS and
// halves its reads.  Four wavefronts stage and four multiply, one of each on a SIMD, so that splitting runs beside the matrix
// instructions (all eight doing both, in phase or in opposite phases: 425 to 475 us where this takes 370).
//
// Measured, planes kernel -> this: 16 -> 32 channels on 16x16 pixels, (64, 300): forward 484 -> 370 us, input gradient 609 ->
// 345; (12, 300): 87 -> 76, 109 -> 74; (4, 1450): 150 -> 111, 187 -> 98; 32 -> 64 on 8x8, (64, 300), forward: 336 -> 280.
// Bound, in the forward pass of 16 -> 32 channels on large tensors, by its stores (rows of 300 samples start 16 bytes into a
// memory line and on: 286 us without the products, 179 with rows of 288 samples) and by the products (190 us without the
// stores, 130 of them matrix instructions), which overlap in part: a multiplying wavefront waits where its stores do.
#include <atomic>
#include <type_traits>

#include "fir_core.h"
#include "synapse_ring.h"

namespace slayer {

constexpr int kRgPos = 3 * 1024;     // bytes of a patch position: 3 planes x 32 samples x 16 channels
constexpr int kRgGroups = 5;         // groups of two taps (the tenth tap is not there: zeros)
constexpr int kRgSlots = 4;
constexpr int kRgMul = 4, kRgStage = 4;   // multiplying and staging wavefronts: one of each per SIMD

constexpr int ring_pixels(int P) { return P == 1 ? 8 : 4; }
constexpr int ring_slot(int P) { return (ring_pixels(P) + 2) * P * kRgPos; }
constexpr int ring_lds(int P) { return kRgSlots * ring_slot(P) + kRgPos + 128; }

struct RingArgs {
    RingGeom s;
    int oGroups, workers, units, steps, tLast, strips, segs, segRows;
    FastDiv byOGroups, byGroups, bySteps, byStrips, bySegs;
};

// Sums that are not finite, made again as chains from memory (a matrix instruction multiplies the parts of an infinity with
// the zeros of taps that are not there): lane (r, h) has channel m, samples t .. t + 3 of pixel (a, b).
template <bool BACKWARD>
__device__ __forceinline__ f32x4 ring_again(const RingGeom &s, f32x4 acc, int n, int grp, int m, int a, int b, int t, bool live)
{
    asm volatile("" : "+v"(t));   // (nothing of this is worked out ahead and kept in registers)
    const int64_t plane = static_cast<int64_t>(s.SH) * s.SW * s.T;
    const BufferRsrc src = make_buffer(s.src + (static_cast<int64_t>(n) * s.SC + static_cast<int64_t>(grp) * s.Qg) * plane);
    f32x4 again = {0.f, 0.f, 0.f, 0.f};
#pragma nounroll
    for (int k = 0; k < s.Qg * 9; ++k) {
        const int q = k / 9, ij = k - q * 9, i = ij / 3, j = ij - i * 3;
        const int y = BACKWARD ? a + s.padH - i : a - s.padH + i, x = BACKWARD ? b + s.padW - j : b - s.padW + j;
        const bool ok = live && static_cast<unsigned>(y) < static_cast<unsigned>(s.SH) && static_cast<unsigned>(x) < static_cast<unsigned>(s.SW);
        const float4 v = buffer_load4<0>(src, masked_offset(ok, q * static_cast<int>(plane) * 4 + ((y * s.SW + x) * s.T + t) * 4), 0);
        const float w = m >= s.Mg ? 0.f
                        : BACKWARD ? s.w[(static_cast<int64_t>(grp * s.Og + q) * s.Cg + m) * 9 + ij]
                                   : s.w[(static_cast<int64_t>(grp * s.Og + m) * s.Cg + q) * 9 + ij];
        again[0] = fmaf(w, v.x, again[0]);
        again[1] = fmaf(w, v.y, again[1]);
        again[2] = fmaf(w, v.z, again[2]);
        again[3] = fmaf(w, v.w, again[3]);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] = fabsf(acc[e]) < __builtin_inff() ? acc[e] : again[e];
    return acc;
}

// P: passes of 16 source channels.  TW: tiles of 16 destination channels of a wavefront.  NT: groups of TW tiles of the
// work-group; the multiplying wavefronts of a group share out the strip's pixels.
template <int P, int TW, int NT, bool BACKWARD>
__global__ __launch_bounds__(512) void synapse_gather_ring_kernel(RingArgs g)
{
    constexpr int PX = ring_pixels(P), WX = PX + 2, SLOT = ring_slot(P), NG = kRgGroups;
    constexpr int PIXELS = PX * NT / kRgMul;           // pixels of a multiplying wavefront
    constexpr int CELLS = WX * P, TASKS = (CELLS + kRgStage - 1) / kRgStage;   // positions of a row, and those of a staging wavefront
    static_assert(PIXELS >= 1, "every multiplying wavefront has products to make");
    extern __shared__ __align__(16) float lds[];
    char *const ldsBytes = reinterpret_cast<char *>(lds);
    typedef const uint4_ext __attribute__((address_space(3))) *LdsUint4;
    const uint32_t ldsBase = static_cast<uint32_t>(reinterpret_cast<size_t>((__attribute__((address_space(3))) char *)ldsBytes));
    const RingGeom &s = g.s;

    uint32_t rest = xcd_contiguous(blockIdx.x, gridDim.x), qq = fastdiv(rest, g.byOGroups);
    const int og = static_cast<int>(rest - qq * g.byOGroups.d);
    rest = qq; qq = fastdiv(rest, g.byGroups);
    const int grp = static_cast<int>(rest - qq * g.byGroups.d), worker = static_cast<int>(qq);

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, h = lane >> 4;
    const int64_t srcPlane = static_cast<int64_t>(s.SH) * s.SW * s.T, dstPlane = static_cast<int64_t>(s.DH) * s.DW * s.T;
    const int planeBytes = static_cast<int>(srcPlane) * 4, rowBytes = s.SW * s.T * 4, pixBytes = s.T * 4;

    if (tid < kRgPos / 16) reinterpret_cast<uint4_ext *>(ldsBytes + kRgSlots * SLOT)[tid] = uint4_ext{0u, 0u, 0u, 0u};
    uint32_t *const flags = reinterpret_cast<uint32_t *>(ldsBytes + kRgSlots * SLOT + kRgPos);   // [slot][staging wavefront]

    // ---- the walk: unit after unit, the rows of a unit (two more than it has destination rows) one after the other
    struct Place {
        int unit, row, n, t0, x0, a0, rows;            // rows: source rows of the unit; row: which of them
    };
    auto decode = [&](Place &p) {
        const uint32_t v = static_cast<uint32_t>(min(p.unit, g.units - 1));
        const uint32_t q = fastdiv(v, g.bySteps), q2 = fastdiv(q, g.byStrips), q3 = fastdiv(q2, g.bySegs);
        p.t0 = min(static_cast<int>(v - q * g.bySteps.d) << 5, g.tLast);
        p.x0 = static_cast<int>(q - q2 * g.byStrips.d) * PX;
        p.a0 = static_cast<int>(q2 - q3 * g.bySegs.d) * g.segRows;
        p.n = static_cast<int>(q3);
        p.rows = min(g.segRows, s.DH - p.a0) + 2;
    };
    auto advance = [&](Place &p) {
        if (++p.row == p.rows) {
            p.row = 0;
            p.unit += g.workers;
            decode(p);
        }
    };
    Place at{worker, 0, 0, 0, 0, 0, 0};
    decode(at);
    int trips = 0;                                     // rows of all units of this worker
    for (Place p = at; p.unit < g.units;) {
        trips += p.rows;
        p.unit += g.workers;
        decode(p);
    }

    if (wave >= kRgMul) {
        // ---- staging wavefronts: a row from memory, two rows ahead in two sets of registers, into the planes of the slot that
        // nobody reads.  Wavefront w takes positions w, w + kRgStage .. of the row (pass by pass), a lane sample `sample` of
        // channels 8 oct .. + 7.  No branches: the compiler then counts the loads in flight exactly.
        const int stager = wave - kRgMul, sample = lane & 31, oct = lane >> 5;
        const int stageAddr = (sample & 3) * 256 + (((oct * 8 + (sample >> 2)) ^ (4 * (sample & 3))) << 4);
        int cell[TASKS], cellX[TASKS], cellBytes[TASKS];
#pragma unroll
        for (int i = 0; i < TASKS; ++i) {
            cell[i] = stager + kRgStage * i < CELLS ? stager + kRgStage * i : stager;   // (those that are not there: the first one again)
            const int pass = cell[i] / WX;
            cellX[i] = cell[i] - pass * WX;
            cellBytes[i] = (pass * 16 + oct * 8) * planeBytes + sample * 4;
        }
        typedef float Row[TASKS][8];
        auto issue = [&](Row &R, const Place &p) {     // the place's row into registers (behind the last unit: nothing)
            const BufferRsrc src = make_buffer(s.src + (static_cast<int64_t>(p.n) * s.SC + static_cast<int64_t>(grp) * s.Qg) * srcPlane);
            const int y = p.a0 + p.row + (BACKWARD ? s.padH - 2 : -s.padH), x = p.x0 + (BACKWARD ? s.padW - 2 : -s.padW);
            const bool row = p.unit < g.units && static_cast<unsigned>(y) < static_cast<unsigned>(s.SH) && p.t0 + sample < s.T;
#pragma unroll
            for (int i = 0; i < TASKS; ++i) {
                const bool ok = row && static_cast<unsigned>(x + cellX[i]) < static_cast<unsigned>(s.SW);
                const int from = masked_offset(ok, cellBytes[i] + y * rowBytes + (x + cellX[i]) * pixBytes + p.t0 * 4);
#pragma unroll
                for (int c = 0; c < 8; ++c) R[i][c] = buffer_load<0>(src, from, c * planeBytes);
            }
        };
        int slot = 0;
        auto stage = [&](const Row &R) {               // registers to the planes of the slot
            uint32_t low = 0;
#pragma unroll
            for (int i = 0; i < TASKS; ++i) {
#pragma unroll
                for (int c = 0; c < 8; ++c) low |= __builtin_bit_cast(uint32_t, R[i][c]);
                const SplitPlanes sp = split_bf16<false>(R[i]);
                uint4_ext *to = reinterpret_cast<uint4_ext *>(ldsBytes + slot * SLOT + cell[i] * kRgPos + stageAddr);
                to[0] = sp.hi;
                to[64] = sp.mid;
                to[128] = sp.lo;
            }
            const bool any = __builtin_amdgcn_ballot_w64((low & 0xffffu) != 0u) != 0;
            if (lane == 0) flags[slot * kRgStage + stager] = any ? 1u : 0u;
            slot = (slot + 1) & (kRgSlots - 1);
        };
        Row RA, RB;
        issue(RB, at);
        advance(at);
        issue(RA, at);
        stage(RB);                                     // the first row
        advance(at);
        issue(RB, at);
        __syncthreads();
#pragma nounroll
        for (int k = 0; k < trips; k += 2) {           // (behind the last row: zeros that nobody reads)
            stage(RA);
            advance(at);
            issue(RA, at);
            __syncthreads();
            stage(RB);
            advance(at);
            issue(RB, at);
            __syncthreads();
        }
        return;
    }

    // ---- multiplying wavefronts
    const int tileGroup = wave % NT, share = wave / NT;
    // weights of this wavefront's tiles: lane (r, h): channels 8 (h % 2) .. + 7 of the pass at tap 2 G + h / 2, for
    // destination channel 16 tile + r
    int mFirst[TW], oOff[TW];                          // first channel that this lane stores
    uint4_ext wr[P][NG][TW][3];
#pragma unroll
    for (int ot = 0; ot < TW; ++ot) {
        const int m = ((og * NT + tileGroup) * TW + ot) * 16 + r;
        mFirst[ot] = m - (r & 8);
        oOff[ot] = mFirst[ot] * static_cast<int>(dstPlane) * 4;
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
            for (int G = 0; G < NG; ++G) {
                const int ij = 2 * G + (h >> 1), q0 = p * 16 + (h & 1) * 8;
                float v[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    v[j] = 0.f;
                    if (ij < 9 && m < s.Mg)
                        v[j] = s.w[BACKWARD ? (static_cast<int64_t>(grp * s.Og + q0 + j) * s.Cg + m) * 9 + ij
                                            : (static_cast<int64_t>(grp * s.Og + m) * s.Cg + q0 + j) * 9 + ij];
                }
                const SplitPlanes sp = split_bf16<false>(v);
                wr[p][G][ot][0] = sp.hi;
                wr[p][G][ot][1] = sp.mid;
                wr[p][G][ot][2] = sp.lo;
            }
    }
    // Operand of group G for sample r of pixel 0: offset in its slot (the zeros': from the first slot), by the lane's tap.  A
    // half step 16 samples on lies 64 bytes off, before or behind.
    const int halfStep = (r & 1) != 0 ? -64 : 64;
    uint32_t off[NG];
#pragma unroll
    for (int G = 0; G < NG; ++G) {
        const int ij = 2 * G + (h >> 1), j = ij % 3;
        const uint32_t cell = (r & 3) * 256 + ((((h & 1) * 8 + (r >> 2)) ^ (4 * (r & 3))) << 4);
        off[G] = ldsBase + cell + (ij < 9 ? static_cast<uint32_t>((BACKWARD ? 2 - j : j) * kRgPos) : static_cast<uint32_t>(kRgSlots * SLOT));
    }
    __syncthreads();
    int slot = 0;                                      // of the row `at`
#pragma nounroll
    for (int k = 0; k < ((trips + 1) & ~1); ++k) {
        const int a = at.a0 + at.row - 2;
        const bool row = at.row >= 2 && at.unit < g.units;   // a destination row has its window
        const int s0 = ((slot + 2) & (kRgSlots - 1)) * SLOT, s1 = ((slot + 3) & (kRgSlots - 1)) * SLOT, s2 = slot * SLOT;
        // slot of filter row i: the oldest of the three is source row 0 of the window
        const int i0 = BACKWARD ? s2 : s0, i1 = s1, i2 = BACKWARD ? s0 : s2;
        const uint32_t base[NG] = {static_cast<uint32_t>(i0), static_cast<uint32_t>(h < 2 ? i0 : i1), static_cast<uint32_t>(i1),
                                   static_cast<uint32_t>(i2), static_cast<uint32_t>(h < 2 ? i2 : 0)};
        const bool all = __builtin_amdgcn_ballot_w64(lane < kRgSlots * kRgStage && lane / kRgStage != ((slot + 1) & (kRgSlots - 1)) &&
                                                     flags[lane & (kRgSlots * kRgStage - 1)] != 0u) != 0;
        const BufferRsrc dst = make_buffer(s.dst + (static_cast<int64_t>(at.n) * s.DC + static_cast<int64_t>(grp) * s.Mg) * dstPlane);
        if (row) {
#pragma nounroll
            for (int c = 0; c < PIXELS; ++c) {
                const int pixel = share * PIXELS + c, b = at.x0 + pixel;
                if (b >= s.DW) break;
                f32x4 sums[2][TW];
                auto multiply = [&](auto partsTag, int half) {
                    constexpr int PARTS = decltype(partsTag)::value;
                    const int shift = pixel * kRgPos + (half ? halfStep : 0);
                    f32x4 (&acc)[TW] = sums[half];
                    f32x4 small[TW];
#pragma unroll
                    for (int ot = 0; ot < TW; ++ot) acc[ot] = small[ot] = f32x4{0.f, 0.f, 0.f, 0.f};
                    constexpr int AHEAD = 1;           // groups whose operands are on their way (two: no faster)
                    uint4_ext x[AHEAD + 1][PARTS];
                    auto fetch = [&](int set, int p, int G) {
                        // (the zeros lie at one place whatever the pixel and the pass)
                        const uint32_t from = off[G] + base[G] + (G == NG - 1 && h >= 2 ? 0 : shift + p * WX * kRgPos);
#pragma unroll
                        for (int part = 0; part < PARTS; ++part)
                            x[set][part] = *reinterpret_cast<LdsUint4>(static_cast<size_t>(from + part * 1024));
                    };
#pragma unroll
                    for (int pg = 0; pg < AHEAD; ++pg) fetch(pg, pg / NG, pg % NG);
#pragma unroll
                    for (int pg = 0; pg < P * NG; ++pg) {
                        const int set = pg % (AHEAD + 1), p = pg / NG, G = pg % NG;
                        if (pg + AHEAD < P * NG) fetch((pg + AHEAD) % (AHEAD + 1), (pg + AHEAD) / NG, (pg + AHEAD) % NG);
                        __builtin_amdgcn_sched_barrier(0);
#define SLAYER_RING_MUL(SUM, XP, WP) \
    _Pragma("unroll") for (int ot = 0; ot < TW; ++ot) SUM[ot] = mfma_bf16(x[set][XP], wr[p][G][ot][WP], SUM[ot]);
                        SLAYER_RING_MUL(small, 0, 2)
                        if constexpr (PARTS == 3) {
                            SLAYER_RING_MUL(small, 2, 0)
                            SLAYER_RING_MUL(small, 1, 1)
                        }
                        SLAYER_RING_MUL(small, 0, 1)
                        if constexpr (PARTS == 3) {
                            SLAYER_RING_MUL(small, 1, 0)
                        }
                        SLAYER_RING_MUL(acc, 0, 0)
#undef SLAYER_RING_MUL
                        __builtin_amdgcn_sched_barrier(0);
                    }
#pragma unroll
                    for (int ot = 0; ot < TW; ++ot) acc[ot] += small[ot];
                };
                // (a step's second half beyond the row's end: nothing to do)
                const bool two = at.t0 + 16 < s.T;
                if (all) {
                    multiply(std::integral_constant<int, 3>{}, 0);
                    if (two) multiply(std::integral_constant<int, 3>{}, 1);
                } else {
                    multiply(std::integral_constant<int, 1>{}, 0);
                    if (two) multiply(std::integral_constant<int, 1>{}, 1);
                }
                if (!two) {
#pragma unroll
                    for (int ot = 0; ot < TW; ++ot) sums[1][ot] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
                float z = 0.f;
#pragma unroll
                for (int hf = 0; hf < 2; ++hf)
#pragma unroll
                    for (int ot = 0; ot < TW; ++ot)
                        z = fmaf((sums[hf][ot][0] + sums[hf][ot][1]) + (sums[hf][ot][2] + sums[hf][ot][3]), 0.f, z);
                if (__builtin_amdgcn_ballot_w64(z != 0.f) != 0u) {
#pragma unroll
                    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
                        for (int ot = 0; ot < TW; ++ot) {
                            const int t = at.t0 + hf * 16 + h * 4;
                            sums[hf][ot] = ring_again<BACKWARD>(s, sums[hf][ot], at.n, grp, ((og * NT + tileGroup) * TW + ot) * 16 + r, a, b,
                                                                t, t < s.T);
                        }
                }
                // lanes r and r + 8 exchange a half step, so that a store writes 128 bytes in a row of eight channels instead of
                // 64 of sixteen
                const int t = at.t0 + (r >> 3) * 16 + h * 4, to = (a * s.DW + b) * pixBytes + t * 4;
#pragma unroll
                for (int ot = 0; ot < TW; ++ot) {
                    float first[4], second[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float give = r < 8 ? sums[1][ot][e] : sums[0][ot][e];
                        const float got = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, give), 0x128, 0xf, 0xf, false));
                        first[e] = r < 8 ? sums[0][ot][e] : got;
                        second[e] = r < 8 ? got : sums[1][ot][e];
                    }
                    buffer_store4<0>(dst, masked_offset(t < s.T && mFirst[ot] < s.Mg, oOff[ot] + to), 0,
                                     make_float4(first[0], first[1], first[2], first[3]));
                    buffer_store4<0>(dst, masked_offset(t < s.T && mFirst[ot] + 8 < s.Mg, oOff[ot] + 8 * static_cast<int>(dstPlane) * 4 + to), 0,
                                     make_float4(second[0], second[1], second[2], second[3]));
                }
            }
        }
        advance(at);
        slot = (slot + 1) & (kRgSlots - 1);
        __syncthreads();                               // the next row is staged, and everyone is through with the oldest
    }
}

template <int P, int TW, int NT, bool BACKWARD>
static int launch_ring_one(const RingArgs &g, unsigned blocks, hipStream_t st)
{
    // more LDS than a kernel may use without asking; asked once per device (a host-side setting, no allocation)
    static std::atomic<bool> raised[64];
    int device = 0;
    hipError_t err = hipGetDevice(&device);
    if (err == hipSuccess && (device < 0 || device >= 64)) err = hipErrorInvalidDevice;
    if (err == hipSuccess && !raised[device].load(std::memory_order_acquire)) {
        err = hipFuncSetAttribute(reinterpret_cast<const void *>(&synapse_gather_ring_kernel<P, TW, NT, BACKWARD>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, ring_lds(P));
        if (err == hipSuccess) raised[device].store(true, std::memory_order_release);
    }
    if (err != hipSuccess) return note_hip_error(err);
    hipLaunchKernelGGL((synapse_gather_ring_kernel<P, TW, NT, BACKWARD>), dim3(blocks), dim3(512), ring_lds(P), st, g);
    return launch_status();
}

// What this kernel and the planes kernel take, in hundredths of a microsecond: a launch whose busiest work-group walks so many
// rows and multiplies under all but two of a unit's, a wavefront as many pixels of each as the strip has for it; and one whose
// busiest work-group makes so many pairs of a block of pixels and a step.  A walk has the longer start - the weights into
// registers, three rows before the first product - and where a call is small or an image so narrow that strips are mostly
// empty, the planes kernel wins: planes / this, us, (1, 300), 32 -> 64 channels of 8 x 8, forward, 14 / 19, 16 -> 16 of 16 x 5,
// input gradient, 7 / 11; (8, 300), 16 -> 32 of 64 x 1, forward, 39 / 45; but 16 -> 32 of 16 x 16, (12, 300), forward, 87 / 76.
// Fitted to 260 sizes (1 to 32 items, 1 to 24 pixels, 20 to 1450 samples, spikes and full samples, each instance by itself);
// none of those sizes is more than 8 % slower this way than by the planes kernel, and none more than 15 % slower than by the
// better of the two.
struct RingCost {
    int planes, pair, walk, row, pixel;
};

static RingCost ring_gather_cost(int P, int TW, int NT, bool two, bool backward)   // two: tiles of the planes kernel's work-group
{
    RingCost c{};
    if (P == 1) {
        c.planes = backward ? (two ? 385 : 421) : (two ? 581 : 466);
        c.pair = backward ? (two ? 457 : 295) : (two ? 355 : 272);
        if (TW == 1) { c.walk = backward ? 710 : 841; c.row = backward ? 52 : 65; c.pixel = backward ? 80 : 59; }
        else { c.walk = backward ? 729 : 1281; c.row = backward ? 101 : 69; c.pixel = backward ? 129 : 104; }
    } else {
        c.planes = backward ? (two ? 565 : 449) : (two ? 752 : 491);
        c.pair = backward ? (two ? 728 : 541) : (two ? 645 : 523);
        if (NT == 1) { c.walk = backward ? 783 : 1139; c.row = 121; c.pixel = backward ? 36 : 33; }
        else if (NT == 2) { c.walk = backward ? 892 : 1196; c.row = backward ? 75 : 81; c.pixel = backward ? 122 : 92; }
        else { c.walk = backward ? 1000 : 1273; c.row = 64; c.pixel = backward ? 139 : 112; }
    }
    return c;
}

// Pairs of eight pixels of a row and a step that the planes kernel's busiest work-group makes (launch_gather_mfma).
static int64_t planes_pairs(const RingGeom &s)
{
    const int64_t pairs = static_cast<int64_t>(s.N) * s.DH * ceil_div(s.DW, 8) * ((s.T + 31) / 32);
    int64_t slices = 252 / (static_cast<int64_t>(s.groups) * ceil_div(s.Mg, s.Mg >= 32 ? 32 : 16));
    if (slices < 1) slices = 1;
    return ceil_div(pairs, slices < pairs ? slices : pairs);
}

// What the busiest work-group of a walk takes; `most`: pixels of a whole strip that a multiplying wavefront has
static int64_t walk_cost(const RingArgs &g, const RingCost &c, int most)
{
    const int64_t units = ceil_div(g.units, g.workers), last = g.s.DW - static_cast<int64_t>(g.strips - 1) * ring_pixels(g.s.Qg / 16);
    const int64_t pixels = static_cast<int64_t>(g.strips - 1) * most + (last < most ? last : most);   // of a row of the image
    return c.walk + units * (g.segRows + 2) * c.row + units * g.segRows * c.pixel * pixels / g.strips;
}

static bool ring_pays(const RingArgs &g, const RingCost &c, int most, int64_t pairs)
{
    return walk_cost(g, c, most) < c.planes + pairs * c.pair;
}

template <bool BACKWARD>
int launch_gather_ring(const RingGeom &s, hipStream_t st)
{
    if ((s.Qg != 16 && s.Qg != 32) || s.Mg < 16 || (s.T % 4 != 0 && s.T < 32)) return SLAYER_EUNSUPPORTED;
    const int P = s.Qg / 16, PX = ring_pixels(P);
    const int TW = P == 1 && s.Mg > 16 ? 2 : 1;
    const int NT = P == 1 ? 1 : s.Mg <= 16 ? 1 : s.Mg <= 32 ? 2 : 4;
    RingArgs g{};
    g.s = s;
    g.oGroups = static_cast<int>(ceil_div(s.Mg, 16 * TW * NT));
    g.steps = (s.T + 31) / 32;
    g.tLast = s.T % 4 == 0 ? (g.steps - 1) * 32 : s.T - 32;
    g.strips = static_cast<int>(ceil_div(s.DW, PX));
    const int64_t base = static_cast<int64_t>(s.groups) * g.oGroups;
    const int64_t columns = static_cast<int64_t>(s.N) * g.steps * g.strips;
    int64_t workers = compute_units() / base;
    if (workers < 1) workers = 1;
    // The units are columns of the image, cut into the number of segments with the fewest rows to walk for the work-group with
    // most of them: a segment's two first rows are only staged, which counts as one.
    int64_t best = 0, segs = 1;
    for (int64_t k = 1; k <= s.DH && k <= 16; ++k) {
        const int64_t rows = ceil_div(s.DH, k), used = ceil_div(s.DH, rows);
        const int64_t cost = ceil_div(columns * used, workers) * (rows + 1);
        if (best == 0 || cost < best) { best = cost; segs = k; }
    }
    g.segRows = static_cast<int>(ceil_div(s.DH, segs));
    g.segs = static_cast<int>(ceil_div(s.DH, g.segRows));
    const int64_t units = columns * g.segs;
    if (units < 1 || units >= (1LL << 30)) return SLAYER_EUNSUPPORTED;
    g.units = static_cast<int>(units);
    if (workers > units) workers = units;
    g.workers = static_cast<int>(workers);
    if (!rings_forced() && !ring_pays(g, ring_gather_cost(P, TW, NT, s.Mg >= 32, BACKWARD), PX * NT / kRgMul, planes_pairs(s))) return SLAYER_EUNSUPPORTED;
    const int64_t blocks = base * workers;
    if (blocks >= (1LL << 22)) return SLAYER_EUNSUPPORTED;
    g.byOGroups = make_fastdiv(static_cast<uint32_t>(g.oGroups));
    g.byGroups = make_fastdiv(static_cast<uint32_t>(s.groups));
    g.bySteps = make_fastdiv(static_cast<uint32_t>(g.steps));
    g.byStrips = make_fastdiv(static_cast<uint32_t>(g.strips));
    g.bySegs = make_fastdiv(static_cast<uint32_t>(g.segs));
    const unsigned nb = static_cast<unsigned>(blocks);
    if (P == 1) return TW == 2 ? launch_ring_one<1, 2, 1, BACKWARD>(g, nb, st) : launch_ring_one<1, 1, 1, BACKWARD>(g, nb, st);
    if (NT == 1) return launch_ring_one<2, 1, 1, BACKWARD>(g, nb, st);
    if (NT == 2) return launch_ring_one<2, 1, 2, BACKWARD>(g, nb, st);
    return launch_ring_one<2, 1, 4, BACKWARD>(g, nb, st);
}

// ---- weight gradient ---------------------------------------------------------------------------------
// gradW[o][c][i][j] = sum over n, a, b, t of gradOut[n][o][a][b][t] in[n][c][a - padH + i][b - padW + j][t]: the same walk with
// time as the reduction axis.  A position in LDS is three planes of 16 channels x 32 samples, time innermost: an operand of tap
// (i, j) is the position that the tap reads under a pixel, 16 channels at once, one 16-byte read per plane and lane.  A
// multiplying wavefront has 16 source channels and two pixels of the strip; it takes a pixel's gradients straight from memory,
// a row ahead, splits them once and multiplies them with the nine positions.  The wavefronts' sums meet in LDS at the end.
// The kernel with the patch of four pixels in LDS splits a sample once per tap and tile of columns, and loads it up to nine
// times.  Full samples, spikes: 16 -> 32 channels of 16 x 16, (64, 300): 592, 442 -> 368, 256 us, (12, 300): 118, 81 -> 74, 60;
// 32 -> 64 channels of 8 x 8, (64, 300): 432, 289 -> 318, 240; 16 -> 16 of 16 x 16, (32, 300): 168, 125 -> 110, 88.  Spikes are
// near the memory (4 TB/s); full samples are held by the products (148 us at 2.1 GHz) and, in the same wavefronts, the splits
// of the gradients.  Splitting beside the products of the pixel before needs 24 registers more than there are: 634 us.
template <int P, int OT>
__global__ __launch_bounds__(512) void synapse_wgrad_ring_kernel(RingArgs g, float *__restrict__ partial, int nW)
{
    constexpr int PX = ring_pixels(P), WX = PX + 2, SLOT = ring_slot(P);
    constexpr int PIXELS = PX * P / kRgMul;            // of a multiplying wavefront
    constexpr int CELLS = WX * P, TASKS = (CELLS + kRgStage - 1) / kRgStage;
    extern __shared__ __align__(16) float lds[];
    char *const ldsBytes = reinterpret_cast<char *>(lds);
    typedef const uint4_ext __attribute__((address_space(3))) *LdsUint4;
    const uint32_t ldsBase = static_cast<uint32_t>(reinterpret_cast<size_t>((__attribute__((address_space(3))) char *)ldsBytes));
    const RingGeom &s = g.s;

    uint32_t rest = xcd_contiguous(blockIdx.x, gridDim.x), qq = fastdiv(rest, g.byOGroups);
    const int og = static_cast<int>(rest - qq * g.byOGroups.d);
    rest = qq; qq = fastdiv(rest, g.byGroups);
    const int grp = static_cast<int>(rest - qq * g.byGroups.d), worker = static_cast<int>(qq);

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, h = lane >> 4;
    const int64_t srcPlane = static_cast<int64_t>(s.SH) * s.SW * s.T, dstPlane = static_cast<int64_t>(s.DH) * s.DW * s.T;
    const int planeBytes = static_cast<int>(srcPlane) * 4, rowBytes = s.SW * s.T * 4, pixBytes = s.T * 4;
    uint32_t *const flags = reinterpret_cast<uint32_t *>(ldsBytes + kRgSlots * SLOT);   // [slot][staging wavefront]

    struct Place {
        int unit, row, n, t0, skip, x0, a0, rows;      // skip: samples of the step that the one before has, too
    };
    auto decode = [&](Place &p) {
        const uint32_t v = static_cast<uint32_t>(min(p.unit, g.units - 1));
        const uint32_t q = fastdiv(v, g.bySteps), q2 = fastdiv(q, g.byStrips), q3 = fastdiv(q2, g.bySegs);
        const int t = static_cast<int>(v - q * g.bySteps.d) << 5;
        p.t0 = min(t, g.tLast);
        p.skip = t - p.t0;
        p.x0 = static_cast<int>(q - q2 * g.byStrips.d) * PX;
        p.a0 = static_cast<int>(q2 - q3 * g.bySegs.d) * g.segRows;
        p.n = static_cast<int>(q3);
        p.rows = min(g.segRows, s.DH - p.a0) + 2;
    };
    auto advance = [&](Place &p) {
        if (++p.row == p.rows) {
            p.row = 0;
            p.unit += g.workers;
            decode(p);
        }
    };
    Place at{worker, 0, 0, 0, 0, 0, 0, 0};
    decode(at);
    int trips = 0;
    for (Place p = at; p.unit < g.units;) {
        trips += p.rows;
        p.unit += g.workers;
        decode(p);
    }

    f32x4 acc[OT][9];
#pragma unroll
    for (int ot = 0; ot < OT; ++ot)
#pragma unroll
        for (int ij = 0; ij < 9; ++ij) acc[ot][ij] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int pass = wave % P, pixel0 = (wave % kRgMul) / P * PIXELS;   // of a multiplying wavefront

    if (wave >= kRgMul) {
        // ---- staging, as in the gather; a lane samples 8 oct .. + 7 of channel `channel`
        const int stager = wave - kRgMul, channel = lane >> 2, oct = lane & 3;
        int cell[TASKS], cellX[TASKS], cellBytes[TASKS];
#pragma unroll
        for (int i = 0; i < TASKS; ++i) {
            cell[i] = stager + kRgStage * i < CELLS ? stager + kRgStage * i : stager;
            const int of = cell[i] / WX;
            cellX[i] = cell[i] - of * WX;
            cellBytes[i] = (of * 16 + channel) * planeBytes + oct * 32;
        }
        typedef float4 Row[TASKS][2];
        auto issue = [&](Row &R, const Place &p) {
            const BufferRsrc src = make_buffer(s.src + (static_cast<int64_t>(p.n) * s.SC + static_cast<int64_t>(grp) * s.Qg) * srcPlane);
            const int y = p.a0 + p.row - s.padH, x = p.x0 - s.padW;
            const bool row = p.unit < g.units && static_cast<unsigned>(y) < static_cast<unsigned>(s.SH);
#pragma unroll
            for (int i = 0; i < TASKS; ++i) {
                const bool ok = row && static_cast<unsigned>(x + cellX[i]) < static_cast<unsigned>(s.SW);
                const int from = cellBytes[i] + y * rowBytes + (x + cellX[i]) * pixBytes + p.t0 * 4;
#pragma unroll
                for (int q = 0; q < 2; ++q)
                    R[i][q] = buffer_load4<0>(src, masked_offset(ok && p.t0 + oct * 8 + q * 4 < s.T, from + q * 16), 0);
            }
        };
        int slot = 0;
        auto stage = [&](const Row &R) {
            uint32_t low = 0;
#pragma unroll
            for (int i = 0; i < TASKS; ++i) {
                const float v[8] = {R[i][0].x, R[i][0].y, R[i][0].z, R[i][0].w, R[i][1].x, R[i][1].y, R[i][1].z, R[i][1].w};
#pragma unroll
                for (int e = 0; e < 8; ++e) low |= __builtin_bit_cast(uint32_t, v[e]);
                const SplitPlanes sp = split_bf16<false>(v);
                uint4_ext *to = reinterpret_cast<uint4_ext *>(ldsBytes + slot * SLOT + cell[i] * kRgPos) + lane;
                to[0] = sp.hi;
                to[64] = sp.mid;
                to[128] = sp.lo;
            }
            const bool any = __builtin_amdgcn_ballot_w64((low & 0xffffu) != 0u) != 0;
            if (lane == 0) flags[slot * kRgStage + stager] = any ? 1u : 0u;
            slot = (slot + 1) & (kRgSlots - 1);
        };
        Row RA, RB;
        issue(RB, at);
        advance(at);
        issue(RA, at);
        stage(RB);
        advance(at);
        issue(RB, at);
        __syncthreads();
#pragma nounroll
        for (int k = 0; k < trips; k += 2) {
            stage(RA);
            advance(at);
            issue(RA, at);
            __syncthreads();
            stage(RB);
            advance(at);
            issue(RB, at);
            __syncthreads();
        }
    } else {
        // ---- multiplying: lane (r, h) has channel r of a position and output channel r of a tile, samples 8 h .. + 7
        int oOff[OT];
#pragma unroll
        for (int ot = 0; ot < OT; ++ot) {
            const int o = (og * OT + ot) * 16 + r;
            oOff[ot] = masked_offset(o < s.Mg, o * static_cast<int>(dstPlane) * 4 + h * 32);
        }
        float4 G[PIXELS][OT][2];
        auto issue = [&](float4 (&to)[OT][2], int c, const Place &p) {   // the gradients under the place's window
            const BufferRsrc src = make_buffer(s.dst + (static_cast<int64_t>(p.n) * s.DC + static_cast<int64_t>(grp) * s.Mg) * dstPlane);
            const int a = p.a0 + p.row - 2, b = p.x0 + pixel0 + c, from = (a * s.DW + b) * pixBytes + p.t0 * 4;
            const bool row = p.row >= 2 && p.unit < g.units && b < s.DW;
#pragma unroll
            for (int ot = 0; ot < OT; ++ot)
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const bool ok = row && oOff[ot] != kOutOfRange && p.t0 + h * 8 + q * 4 < s.T;
                    int off = ok ? oOff[ot] + from + q * 16 : kOutOfRange;
                    asm volatile("" : "+v"(off));      // (no branch around a load)
                    to[ot][q] = buffer_load4<0>(src, off, 0);
                }
        };
        const uint32_t base = ldsBase + r * 64 + h * 16 + (pass * WX + pixel0) * kRgPos;
        int slot = 0;
        // the nine taps of one pixel.  The products of a step start from zero, the leading ones apart from the small ones, and
        // the vector ALU, which rounds, adds them to the sums - those of the tap before, beside the products of this one.
        auto multiply = [&](const SplitPlanes (&gp)[OT], const uint32_t (&from)[3], auto partsTag) {
            constexpr int PARTS = decltype(partsTag)::value;
            uint4_ext x[2][PARTS];
            f32x4 lead[2][OT], rest[2][OT];
            const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
            auto fetch = [&](int set, int k) {
#pragma unroll
                for (int part = 0; part < PARTS; ++part)
                    x[set][part] = *reinterpret_cast<LdsUint4>(static_cast<size_t>(from[k / 3] + k % 3 * kRgPos + part * 1024));
            };
            fetch(0, 0);
#pragma unroll
            for (int k = 0; k <= 9; ++k) {
                const int set = k & 1;
                if (k + 1 < 9) fetch(set ^ 1, k + 1);
                if (k < 9) {
#define SLAYER_RING_MUL(TO, GP, XP, FROM) \
    _Pragma("unroll") for (int ot = 0; ot < OT; ++ot) TO[set][ot] = mfma_bf16(gp[ot].GP, x[set][XP], FROM);
                    SLAYER_RING_MUL(rest, lo, 0, zero)
                    SLAYER_RING_MUL(lead, hi, 0, zero)
                    if constexpr (PARTS == 3) {
                        SLAYER_RING_MUL(rest, hi, 2, rest[set][ot])
                        SLAYER_RING_MUL(rest, mid, 1, rest[set][ot])
                    }
                    SLAYER_RING_MUL(rest, mid, 0, rest[set][ot])
                    if constexpr (PARTS == 3) {
                        SLAYER_RING_MUL(rest, hi, 1, rest[set][ot])
                    }
#undef SLAYER_RING_MUL
                }
                if (k > 0) {
#pragma unroll
                    for (int ot = 0; ot < OT; ++ot) acc[ot][k - 1] += lead[set ^ 1][ot] + rest[set ^ 1][ot];
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        Place ahead = at;
#pragma unroll
        for (int c = 0; c < PIXELS; ++c) issue(G[c], c, ahead);
        advance(ahead);
        __syncthreads();
#pragma nounroll
        for (int k = 0; k < ((trips + 1) & ~1); ++k) {   // (the staging wavefronts take two at a time)
            const uint32_t from[3] = {base + ((slot + 2) & (kRgSlots - 1)) * SLOT, base + ((slot + 3) & (kRgSlots - 1)) * SLOT, base + slot * SLOT};
            const bool all = __builtin_amdgcn_ballot_w64(lane < kRgSlots * kRgStage && lane / kRgStage != ((slot + 1) & (kRgSlots - 1)) &&
                                                         flags[lane & (kRgSlots * kRgStage - 1)] != 0u) != 0;
            const bool work = at.row >= 2 && at.unit < g.units;
#pragma unroll
            for (int c = 0; c < PIXELS; ++c) {
                SplitPlanes gp[OT];
#pragma unroll
                for (int ot = 0; ot < OT; ++ot) {
                    float v[8] = {G[c][ot][0].x, G[c][ot][0].y, G[c][ot][0].z, G[c][ot][0].w,
                                  G[c][ot][1].x, G[c][ot][1].y, G[c][ot][1].z, G[c][ot][1].w};
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[e] = h * 8 + e >= at.skip ? v[e] : 0.f;
                    gp[ot] = split_bf16<false>(v);
                    // (here, before the registers are loaded again, and not in the branch)
                    asm volatile("" : "+v"(gp[ot].hi), "+v"(gp[ot].mid), "+v"(gp[ot].lo));
                }
                __builtin_amdgcn_sched_barrier(0);
                issue(G[c], c, ahead);
                __builtin_amdgcn_sched_barrier(0);
                if (work && at.x0 + pixel0 + c < s.DW) {
                    const uint32_t under[3] = {from[0] + c * kRgPos, from[1] + c * kRgPos, from[2] + c * kRgPos};
                    if (all) multiply(gp, under, std::integral_constant<int, 3>{});
                    else multiply(gp, under, std::integral_constant<int, 1>{});
                }
            }
            advance(ahead);
            advance(at);
            slot = (slot + 1) & (kRgSlots - 1);
            __syncthreads();
        }
    }

    // ---- the wavefronts' sums, in order; element q of a tile is output channel 4 h + q, input channel r
    __syncthreads();
    f32x4 *const red = reinterpret_cast<f32x4 *>(lds);
    constexpr int TILES = OT * 9;
    if (wave >= P && wave < kRgMul) {
#pragma unroll
        for (int k = 0; k < TILES; ++k) red[((wave - P) * TILES + k) * 64 + lane] = acc[k / 9][k % 9];
    }
    __syncthreads();
    if (wave < P) {
        float *row = partial + static_cast<int64_t>(worker) * nW;
#pragma unroll
        for (int k = 0; k < TILES; ++k) {
            f32x4 v = acc[k / 9][k % 9];
#pragma unroll
            for (int w = 1; w < kRgMul / P; ++w) v += red[((w * P + wave - P) * TILES + k) * 64 + lane];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int o = (og * OT + k / 9) * 16 + 4 * h + q, c = pass * 16 + r;
                if (o < s.Mg) row[static_cast<int64_t>(grp * s.Mg + o) * (s.Qg * 9) + c * 9 + k % 9] = v[q];
            }
        }
    }
}

// The walk against the kernel with the patch of four pixels (plan_wgrad_lds), from 60 steps of a pixel per compute unit on, as in
// the gather: full samples, spikes, patch against this, us: 15 steps, 32 -> 64 channels of 7 x 9, (5, 173), 38, 29 against 38,
// 33; 17 x 17, 16 -> 32, (32, 64), 75, 72 against 66, 53; 16 x 16, 32 -> 96, (8, 100), 139, 97 against 124, 95; narrow images,
// under which wavefronts stand by: 32 x 3, 16 -> 32, (4, 1450), 76, 51 against 77, 72; 64 x 2, 16 -> 16, (32, 100), 67, 53 against
// 62, 58.  Both leave rows of sums, `add` the time of adding up a million of them.  A twentieth in favour of the patch.  It
// does not take rows of less than 16 samples; the vector kernel against this, us: 16 -> 32 channels of 16 x 16, (64, 8), 97, 97
// against 41, 35; of 32 x 32, (16, 4), 35, 35 against 41, 35.
static bool ring_wgrad_pays(const RingArgs &g, int P, int OT)
{
    const RingGeom &s = g.s;
    const int64_t base = static_cast<int64_t>(s.groups) * g.oGroups;
    if (s.T < 8 || static_cast<int64_t>(s.N) * g.steps * s.DH * s.DW * base < 60 * 256) return false;
    if (s.T < 16) return true;
    struct Cost {
        RingCost c;
        int addPatch, addWalk;
    };
    const Cost c = P == 1 ? OT == 1 ? Cost{{545, 290, 790, 73, 45}, 1110, 880} : Cost{{585, 225, 935, 92, 82}, 620, 470}
                          : OT == 1 ? Cost{{590, 330, 612, 119, 22}, 475, 543} : Cost{{730, 266, 962, 86, 85}, 405, 442};
    // the patch kernel's column groups: at most nine tiles of 16 columns beside one tile of output channels, six beside two
    const int64_t colGroups = P == 1 ? OT : OT + 1;
    const int64_t pairs = static_cast<int64_t>(s.N) * s.DH * ceil_div(s.DW, 4) * g.steps, nW = static_cast<int64_t>(s.groups) * s.Mg * s.Qg * 9;
    int64_t slices = 504 / (base * colGroups);
    if (slices < 1) slices = 1;
    if (slices > pairs) slices = pairs;
    const int64_t patch = c.c.planes + ceil_div(pairs, slices) * c.c.pair + slices * nW * c.addPatch / 1000000;
    const int64_t walk = walk_cost(g, c.c, ring_pixels(P) * P / kRgMul) + g.workers * nW * c.addWalk / 1000000;
    return walk * 21 < patch * 20;
}

// Tiles and walk of the weight gradient; false where the kernel does not take the geometry.
static bool plan_wgrad_ring(const RingGeom &s, RingArgs &g, int &P, int &OT)
{
    if ((s.Qg != 16 && s.Qg != 32) || s.Mg < 16 || (s.T % 4 != 0 && s.T < 32) || s.T < 1) return false;
    P = s.Qg / 16;
    OT = s.Mg <= 16 ? 1 : 2;
    g = RingArgs{};
    g.s = s;
    g.oGroups = static_cast<int>(ceil_div(s.Mg, 16 * OT));
    g.steps = (s.T + 31) / 32;
    g.tLast = s.T % 4 == 0 ? (g.steps - 1) * 32 : s.T - 32;
    g.strips = static_cast<int>(ceil_div(s.DW, ring_pixels(P)));
    const int64_t base = static_cast<int64_t>(s.groups) * g.oGroups, columns = static_cast<int64_t>(s.N) * g.steps * g.strips;
    int64_t workers = 256 / base;                      // (one work-group per compute unit; a number that sizes alone determine)
    if (workers < 1) workers = 1;
    int64_t best = 0, segs = 1;                        // as in the gather
    for (int64_t k = 1; k <= s.DH && k <= 16; ++k) {
        const int64_t rows = ceil_div(s.DH, k), used = ceil_div(s.DH, rows);
        const int64_t cost = ceil_div(columns * used, workers) * (rows + 1);
        if (best == 0 || cost < best) { best = cost; segs = k; }
    }
    if (s.DH < 1 || s.DW < 1 || columns < 1) return false;
    g.segRows = static_cast<int>(ceil_div(s.DH, segs));
    g.segs = static_cast<int>(ceil_div(s.DH, g.segRows));
    const int64_t units = columns * g.segs;
    if (units < 1 || units >= (1LL << 30) || base >= (1LL << 20)) return false;
    g.units = static_cast<int>(units);
    if (workers > units) workers = units;
    g.workers = static_cast<int>(workers);
    if (!ring_wgrad_pays(g, P, OT)) return false;
    g.byOGroups = make_fastdiv(static_cast<uint32_t>(g.oGroups));
    g.byGroups = make_fastdiv(static_cast<uint32_t>(s.groups));
    g.bySteps = make_fastdiv(static_cast<uint32_t>(g.steps));
    g.byStrips = make_fastdiv(static_cast<uint32_t>(g.strips));
    g.bySegs = make_fastdiv(static_cast<uint32_t>(g.segs));
    return true;
}

int ring_wgrad_rows(const RingGeom &s)
{
    RingArgs g;
    int P, OT;
    return plan_wgrad_ring(s, g, P, OT) ? g.workers : 0;
}

template <int P, int OT>
static int launch_wgrad_ring_one(const RingArgs &g, float *workspace, hipStream_t st)
{
    static_assert(kRgSlots * ring_slot(P) >= (kRgMul - P) * OT * 9 * 1024, "the sums of three wavefronts fit the ring");
    static std::atomic<bool> raised[64];
    int device = 0;
    hipError_t err = hipGetDevice(&device);
    if (err == hipSuccess && (device < 0 || device >= 64)) err = hipErrorInvalidDevice;
    if (err == hipSuccess && !raised[device].load(std::memory_order_acquire)) {
        err = hipFuncSetAttribute(reinterpret_cast<const void *>(&synapse_wgrad_ring_kernel<P, OT>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, ring_lds(P));
        if (err == hipSuccess) raised[device].store(true, std::memory_order_release);
    }
    if (err != hipSuccess) return note_hip_error(err);
    const unsigned blocks = static_cast<unsigned>(g.s.groups) * g.oGroups * g.workers;
    hipLaunchKernelGGL((synapse_wgrad_ring_kernel<P, OT>), dim3(blocks), dim3(512), ring_lds(P), st, g, workspace,
                       g.s.groups * g.s.Mg * g.s.Qg * 9);
    return launch_status();
}

int launch_wgrad_ring(const RingGeom &s, float *workspace, hipStream_t st)
{
    RingArgs g;
    int P, OT;
    if (!plan_wgrad_ring(s, g, P, OT)) return SLAYER_EUNSUPPORTED;
    if (P == 1) return OT == 1 ? launch_wgrad_ring_one<1, 1>(g, workspace, st) : launch_wgrad_ring_one<1, 2>(g, workspace, st);
    return OT == 1 ? launch_wgrad_ring_one<2, 1>(g, workspace, st) : launch_wgrad_ring_one<2, 2>(g, workspace, st);
}

template int launch_gather_ring<false>(const RingGeom &, hipStream_t);
template int launch_gather_ring<true>(const RingGeom &, hipStream_t);

}  // namespace slayer
