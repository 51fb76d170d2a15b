// Where the staged operand loads of the thin-tile and bf16 GEMMs (k_thin.hip, k_dense.hip) read:
// plain C++, so that a host program can walk every load of a tile.
//
// A load names a buffer descriptor of `records` bytes, a byte offset of its lane and one of its wave
// (a scalar register). The range check is not relied on for the scalar offset, counted or not:
//   - a load that has to read lies inside the buffer with both offsets added, on its own;
//   - one that must not read (rows past a tile's pairs, stages past the last) is refused by its lane
//     offset: that is `records` or more, and the scalar offset is no more than `records`, so
//     records - scalar does not wrap.
#pragma once

#include <cstdint>

namespace brx {

constexpr int kTWaves = 4;        // waves of a thin-tile block

struct StageSrc {
    uint32_t records, soffset;
};

// Descriptor bytes and scalar offset of the loads of stage (or step) s of n; those past the last read
// nothing, through a descriptor of no bytes at no scalar offset.
constexpr StageSrc stage_src(int s, int n, uint32_t bytes, uint32_t offset) {
    return s < n ? StageSrc{bytes, offset} : StageSrc{0u, 0u};
}

// Lane offset of a 16-byte A copy: chunk c of the stage at row offset `row`; rows past the tile's
// pairs take the buffer's size.
constexpr uint32_t a_lane_offset(int r, int rows, uint32_t row, int c, uint32_t bytes) {
    return r >= rows ? bytes : row + 16u * (uint32_t)c;
}

// A copies (1 KB, 8 rows of 128 bytes) of a thin step: SG stages of 16 MQ rows. NA a wave, the waves
// past the last copy of a small step repeat it; all of a wave's belong to one stage of the step.
template <int SG, int MQ>
constexpr int kTACopies = SG * 2 * MQ;
template <int SG, int MQ>
constexpr int kTAWave = (kTACopies<SG, MQ> + kTWaves - 1) / kTWaves;
template <int SG, int MQ>
constexpr int thin_a_copy(int wv, int i) {
    const int c = wv * kTAWave<SG, MQ> + i;
    return c < kTACopies<SG, MQ> ? c : kTACopies<SG, MQ> - 1;
}
template <int SG, int MQ>
constexpr int thin_a_row(int wv, int i, int lane) {
    return (thin_a_copy<SG, MQ>(wv, i) * 8 + (lane >> 3)) % (16 * MQ);
}
template <int SG, int MQ>
constexpr int thin_a_stage(int wv) {
    return thin_a_copy<SG, MQ>(wv, 0) / (2 * MQ);
}

// B loads of a thin step of `bits`-bit weights (16: bf16): lane group g's first load of weight row
// `row` (K inputs; bf16 groups 0 to 3 start at chunks 0, 2, 1 and 3), and the scalar offset of step p
// in the matrix.
constexpr uint32_t thin_b_lane(int bits, int K, uint32_t row, int g) {
    return row * (uint32_t)(K * bits / 8) + (uint32_t)(bits == 16 ? 16 * (2 * (g & 1) + (g >> 1)) : 4 * bits * g);
}
constexpr uint32_t thin_b_step(int bits, int SG, int p) { return (uint32_t)p * (uint32_t)(8 * bits * SG); }

}  // namespace brx
