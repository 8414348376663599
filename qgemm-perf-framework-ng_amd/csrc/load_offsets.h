// Byte offsets of the bounded loads and copies, as constexpr functions: the
// kernels call them, and tests/test_load_offsets.py compiles them for the host
// and walks every lane's accesses.
#pragma once

#include <cstdint>

namespace pfng {

// A buffer load's per-lane and uniform offsets. Whether the uniform one takes
// part in the range check is not relied on: the edge of the matrix has to show
// in `lane` alone, and `uniform` stays below the resource's size.
struct BufferOffset {
    uint32_t lane, uniform;
};

// Lane offset that lies past every resource of the q4_0 tiles (the largest, 128
// rows of 2^24 elements, ends below it, and or-ing it into an offset below that
// cannot wrap).
constexpr uint32_t kPastEnd = 0xf0000000u;

// q4_0 staging pieces (gemm_mfma.hip): first of the five dwords that cover half
// `piece & 1` of block `piece >> 1` of an activation row, or block `j` of a
// weight row, `row` rows into the tile.
constexpr uint32_t q4_0_act_piece(uint32_t row, uint32_t piece, uint32_t nb) {
    return row * nb * 34u + ((34u * (piece >> 1) + 16u * (piece & 1u)) & ~3u);
}
constexpr uint32_t q4_0_weight_piece(uint32_t row, uint32_t j, uint32_t nb) {
    return row * nb * 18u + ((18u * j) & ~3u);
}

// The piece `step` bytes (whole rows) below the one at `piece`, in the stage
// that starts `stage` bytes into the rows. past: kPastEnd to send the load out
// of the resource, else 0.
constexpr BufferOffset q4_0_stage_piece(uint32_t piece, uint32_t step, uint32_t stage, uint32_t past) {
    return {(piece + step) | past, stage};
}

// iq2_xxs weight blocks (66 bytes, at any even address) in the tile GEMV at every
// k: their copies of 80 bytes start on a dword, 2 bytes before the block where its
// index in the matrix is odd, and 12 more behind a row's first block, so that they
// end at most 2 bytes past the block and only where the index is even.
constexpr int iq2_copy_back(int super_block) { return super_block > 0 ? 12 : 0; }
constexpr int iq2_copy_odd(int block) { return 2 * (block & 1); }

// q8_K activation blocks (292 bytes) in the q4_K tile GEMV: byte at which the
// second half's 176-byte copy starts, from the first half's start. Where rows
// share one alignment that is 0..12 bytes before the block, and the halves are
// 16-byte chunks; else it is the block, and the second half its last 176 bytes.
constexpr int kQ4kHalf1Chunk = 128, kQ4kHalf1Block = 116;

}  // namespace pfng
