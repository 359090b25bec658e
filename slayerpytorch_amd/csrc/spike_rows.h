// Where the whole-row spike kernel (spike.hip) keeps a tile in LDS.  Plain C++: the kernel, its launch and a host test that
// walks over every shape share it.
#ifndef SLAYER_SPIKE_ROWS_H
#define SLAYER_SPIKE_ROWS_H

#include <cstddef>
#include <cstdint>

namespace slayer {

struct SpikeRowsLayout {
    bool served;
    int parts;      // lanes per row
    int rounds;     // blocks of `parts` samples that a response reaches
    int blocks;     // blocks of a row
    int pitch;      // samples from one row of the tile to the next, a multiple of `parts`
    size_t ldsBytes;
};

// Rows whose blocks fit the bit registers (not served: rows beyond 4032 samples, refractory kernels beyond 60 blocks).
// Lanes per row: 8 for short refractory kernels, 16 for long ones (fewer trips per spike); 16 too where a tile of 8 rows
// would take over 11 KB of LDS (fewer than 14 tiles per compute unit: (12,16,34,34,496) takes 228 us with 8 lanes and
// 194 us with 16); more where a tile of 4 or 2 rows would take over 20 KB (8000 rows of 1000 samples: 37 us with 17 KB tiles of
// 16 lanes per row, 58 us with 32 lanes; tiles of 12 KB the other way cost rows of 640 samples half as much again) or
// the tensor has too few rows for four wavefronts per compute unit.
constexpr SpikeRowsLayout spike_rows_layout(int64_t T, int64_t nuSize, int64_t nNeurons, int64_t computeUnits)
{
    SpikeRowsLayout l{false, nuSize <= 24 ? 8 : 16, 0, 0, 0, 0};
    if (T > 4096 || nuSize > 4096) return l;
    for (;; l.parts *= 2) {
        l.rounds = static_cast<int>((nuSize + 2 * l.parts - 2) / l.parts);
        if (l.rounds < 2) l.rounds = 2;
        if (l.rounds > 3) l.rounds = (l.rounds + 3) & ~3;
        l.blocks = static_cast<int>((T + l.parts - 1) / l.parts);
        l.pitch = (l.blocks + l.rounds) * l.parts;
        while (l.pitch % 64 != l.parts % 64) l.pitch += l.parts;   // (the rows of a tile start in different banks)
        const int R = 64 / l.parts;
        l.ldsBytes = (static_cast<size_t>(R) * l.pitch + 2 * 64 + 3 * R + (l.rounds + 1) * l.parts) * sizeof(float);
        l.served = l.blocks <= 63 && l.rounds <= 60;
        if (l.parts == 64 || (l.served && l.ldsBytes <= (l.parts == 8 ? 11 : 20) * 1024 && (nNeurons + R - 1) / R >= 4 * computeUnits)) return l;
    }
}

// The walk over every sample takes a row in blocks of as many samples as lanes serve it, 16 at most, and in steps of 32
// samples; block m of the step that starts with block b0, of `walkRounds` blocks that a response reaches.  The last step may
// look past the row's pitch, where the next row (or the spike bits) lies.  All its blocks from the end of the row on are
// padding, whose samples never change, so what lies beyond the pitch is taken from the last block before it.  (Only blocks
// beyond the first `walkRounds` + 1 of a step can: one of the step's blocks at least belongs to the row, and the pitch holds
// as many more.)
constexpr int spike_walk_block(int b0, int m, int walkRounds, int pitchBlocks)
{
    return m <= walkRounds || b0 + m < pitchBlocks ? b0 + m : pitchBlocks - 1;
}

// Whether that walk exists for a layout, and its lanes per row and blocks.
struct SpikeWalk {
    bool exists;
    int lanes, rounds;
};

constexpr SpikeWalk spike_walk(int parts, int rounds)
{
    return {parts == 8 ? rounds <= 4 : parts == 16 ? rounds <= 3 : rounds == 2, parts < 16 ? parts : 16, parts <= 16 ? rounds : 3};
}

// Whether all tiles of a layout are on the GPU at once (160 KB of LDS per compute unit, in granules of 1280 bytes).
constexpr bool spike_rows_at_once(const SpikeRowsLayout &l, int64_t nNeurons, int64_t computeUnits)
{
    const int64_t perUnit = 160 * 1024 / static_cast<int64_t>((l.ldsBytes + 1279) / 1280 * 1280);
    return (nNeurons + 64 / l.parts - 1) / (64 / l.parts) <= perUnit * computeUnits;
}

// Rows of whole vectors of more than 600 samples, with a short kernel, go in pieces where the tiles of the whole-row
// kernel are more than the GPU holds at once - but for rows of at most 700 samples that would leave the pieces' second
// round of eight-row tiles about half empty.  Whole / in pieces, potentials that fire 7 % of the time (22 %): 14000 rows of 600
// samples 34 / 42 us (39 / 42), 40000: 79 / 94 (95 / 88); of 640, 12000 rows 31 / 41 (36 / 40), 14000 41 / 42 (50 / 41),
// 20000 53 / 68 (63 / 63), 40000 87 / 88 (105 / 78); of 1000, 8000 rows 36 / 49 (42 / 50), 10000 58 / 52 (73 / 55),
// 16000 78 / 58 (98 / 62); of 1200, 6000 rows 47 / 58 (58 / 54), 8000 68 / 60 (90 / 57).
constexpr bool spike_rows_better_in_pieces(const SpikeRowsLayout &whole, int64_t T, int64_t nNeurons, int64_t computeUnits)
{
    const bool halfRound = T <= 700 && nNeurons > 64 * computeUnits && nNeurons <= 104 * computeUnits;
    return T > 600 && !(whole.served && (halfRound || spike_rows_at_once(whole, nNeurons, computeUnits)));
}

}  // namespace slayer

#endif
