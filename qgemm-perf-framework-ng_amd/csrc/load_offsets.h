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

}  // namespace pfng
