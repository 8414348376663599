// int8-MFMA GEMM path for gfx950 (prefill-sized m).
//
// q4_0 x q8_0: C[m][n] = sum_b S_b[m][n] * da[m][b] * dw[n][b], with S_b the
// exact int32 dot of block b (llama_reference.cpp:134-146).
//
// Workgroup tile BM x BN, K stages of KB blocks (32*KB elements):
//   * global -> registers: every thread loads 16-byte pieces (half a q8_0
//     block, one q4_0 block, as the five dwords that cover it), consecutive
//     lanes consecutive pieces of a row, several pieces ahead of their use.
//   * registers -> LDS: activation int8 realigned; weight nibbles expanded to
//     16*(q-8) int8; fp16 scales kept per row. Rows are padded so the 16-byte
//     MFMA operand reads are free of bank conflicts. The pieces of stage s+1
//     are stored between the items of stage s.
//   * per block and 32x32 tile: S16 = v_mfma_i32_32x32x32_i8(act, w16) (= 16*S_b),
//     P = v_mfma_f32_32x32x8_f16(da, dw) (the exact outer product da*dw on the
//     matrix core), acc = fma(S16 as fp32, P, acc); C = acc / 16 at the end.
// What bounds it: MFMA results and VALU results share the vector registers'
// write port, so an item's two MFMAs (64 cycles) and its 32 VALU operations
// (2 cycles each: a subtraction that turns S16 into fp32, see based_sum, and
// the FMA) add up instead of overlapping. Measured in a 128x128-tile workgroup pair per
// CU at 2.0 GHz: 163 cycles an item, 126 with the staging left out. The pieces and
// the subtraction against block pairs (68 / 36 bytes) staged in a phase of their
// own after each stage and the conversion v_cvt_f32_i32 (about 5 cycles), tile
// choice included, us in one process: 2048x11008x4096 260.3 -> 250.3 (738 TOPS),
// 2048x4096x11008 236.0 -> 230.3, 1024x4096x4096 60.6 -> 57.2, 480x11008x4096 86.0 ->
// 77.9, 480x1536x4096 19.8 -> 16.8, 333x4096x4096 30.7 -> 26.6, 200x4096x11008 51.0 ->
// 39.4. Loading the pieces from their own byte address (two past a dword for every
// other block), which needs no realignment, is slower (2048x11008x4096 269.5 against
// 261.0 us, 333x4096x4096 35.9 against 29.0).
// Smaller problems use smaller tiles whose stage blocks are shared by several
// K-waves (their partial sums are added through LDS at the end), so that one
// workgroup keeps eight waves on its CU.
//
// A diagnostic instantiation writes S_b instead of accumulating (block isums).
#include <type_traits>

#include "device_common.h"
#include "kernels.h"
#include "load_offsets.h"

namespace pfng {

namespace {

constexpr uint32_t kBufferWord3 = 0x00020000;  // raw buffer resource

// BM x BN workgroup tile, WM x WN waves over it, each wave's stage blocks
// divided among WK waves (WK > 1: the WK partial accumulators are added
// through LDS at the end, in wave order), KB q4_0 blocks per K stage.
// AHEAD staging pieces per thread are in flight (a stage has kPieces of them:
// a deep prefetch for the small tiles, whose stages are too short to cover a
// memory round trip).
// FOLD: the accumulators are added into a second set after every FOLD stages (1 or
// 2; 0: never), so that no fp32 sum runs over more than a few dozen terms, as in
// the 16-wave tile GEMV. Relative error from 64 bits on random layers:
// 100x11008x4096 1.47e-7 without, 9.3e-8 with (9.4e-8 in the tile GEMV),
// 333x4096x4096 2.0e-7 -> 9.3e-8.
template <int BM, int BN, int WM, int WN, int KB, int WK = 1, int AHEAD = 6, int FOLD = 0, int MINW = 2>
struct Q40Config {
    static constexpr int kBM = BM, kBN = BN, kWM = WM, kWN = WN, kKB = KB, kWK = WK, kAhead = AHEAD;
    // waves per SIMD the register budget must allow: the fp32 epilogue needs two
    // resident waves per SIMD to keep the VALU issuing while the other waits
    static constexpr int kMinWavesPerEU = MINW;
    static constexpr int kFold = FOLD;
    using Isums = Q40Config<BM, BN, WM, WN, KB, WK, AHEAD, 0, MINW>;  // of the diagnostic, which folds nothing
    static constexpr int kThreads = 64 * WM * WN * WK;
    static constexpr int kWaveBlocks = KB / WK;  // blocks per stage of one wave
    static constexpr bool kTails = KB > 4;       // k % 128 == 0: stages of 4 blocks are always full
    static constexpr int TM = BM / WM / 32;  // 32x32 tiles per wave along m
    static constexpr int TN = BN / WN / 32;  // along n
    // whether the last two stages run behind the K loop too, without its loads of
    // further stages, which the last stage of an even number would wait for (the
    // copies of two larger stages cost the 128x128 tile 200 bytes of spills). us in
    // the loop and apart, q4_0 100x400x512 4.97 / 4.42, 512x4096x2048 16.7 / 15.9,
    // 64x16640x1024 10.5 / 9.9; long or odd rows within 1 %.
    static constexpr bool kLastApart = TM * TN == 1;
    // staging pieces of 16 bytes: half an activation block, one weight block
    static constexpr int kActPerRow = 2 * KB, kWPerRow = KB;
    static constexpr int kActPT = BM * kActPerRow / kThreads;  // pieces per thread
    static constexpr int kWPT = BN * kWPerRow / kThreads;
    static constexpr int kPieces = kActPT + kWPT;
    static constexpr int kActRows = kThreads / kActPerRow, kWRows = kThreads / kWPerRow;  // rows per piece index
    static constexpr int kRowStride = KB * 32 + 16;  // LDS bytes per tile row (int8 + pad)
    // LDS layout
    static constexpr int kAq = 0;
    static constexpr int kAd = kAq + BM * kRowStride;       // fp16 da[row][KB]
    static constexpr int kWq = kAd + BM * KB * 2;
    // dw[row][KB] as 32-bit words: block t's fp16 scale in the low half for
    // even t, in the high half for odd t, zeros in the other half
    static constexpr int kWd = kWq + BN * kRowStride;
    static constexpr int kBufBytes = kWd + BN * KB * 4;  // one stage
    // zeros that the upper K-half lanes read as their weight scale words
    static constexpr int kZero = 2 * kBufBytes;
    static constexpr int kZeroBytes = TN * 32 * KB * 4;
    static constexpr int kLdsBytes = kZero + kZeroBytes;  // double-buffered stages + zeros
    static_assert(TM >= 1 && TN >= 1, "tile too small");
    static_assert(KB % 4 == 0, "KB must be a multiple of 4 (scale vectors are read four at a time)");
    static_assert(2 * kPieces % kAhead == 0, "a round of two stages uses each register set equally often");
    static_assert(kActPT * kActRows == BM && kWPT * kWRows == BN, "pieces must split evenly over threads");
    static_assert(kActRows * kActPerRow == kThreads && kWRows * kWPerRow == kThreads, "whole rows per piece index");
    static_assert(kAd % 16 == 0 && kWq % 16 == 0 && kWd % 16 == 0, "LDS regions 16-byte aligned");
    static_assert(kWaveBlocks * WK == KB && kWaveBlocks % 4 == 0, "each wave takes a multiple of 4 blocks");
    static_assert((WK - 1) * WM * WN * TM * TN * 16 * 64 * 4 <= 2 * kBufBytes, "K-wave reduction fits in LDS");
    static_assert(kZeroBytes % 16 == 0 && kZeroBytes >= 16, "zero strip of whole 16-byte words");
};

// A piece as loaded: the five dwords that cover its 16 bytes and (of an odd
// block, and of an even block's first half) its fp16 scale.
struct PieceRegs {
    uint32_t v[5];
};

// What a thread needs of its pieces. Piece p of an operand lies p * kActRows
// (kWRows) rows below piece 0 in memory and in LDS, so one offset serves all,
// plus the row step (one addition per piece). Rows past the matrix edge read
// zeros (the buffer resources end at the edge, and the row is part of the lane
// offset, so they are out of range whether or not the check counts the uniform
// offset, which only carries the stage); their results are not stored.
// BM * nb * 34 < 2^32 for every k up to kMaxTiledK (mfma_supported declines
// longer rows).
// Consecutive lanes take consecutive pieces of a row, so a wave's load covers
// whole runs of a few rows (a lane per block pair would touch 32 rows per load,
// and the address coalescer, not the VALU, would set the staging's cost).
// Block j starts 34 j (18 j) bytes into the row: two bytes before a dword for
// odd j, whose values are then dword-aligned, and on a dword for even j, whose
// values sit two bytes off. Either way the piece is bytes [2, 18) or [4, 20) of
// the five dwords from the one at or before its block (half), none of which
// lies past the block pair's end.
// Where nb is not a multiple of KB, the last stage's loads of blocks past the
// row's end are sent out of the resource (to kPastEnd) and read zeros: a zero
// scale on both sides, so such a block adds S * 0.
struct StageSlots {
    uint32_t a, w;               // load offsets of piece 0
    uint32_t a_past, w_past;     // kPastEnd where its block lies past the row in the last stage, else 0
    uint32_t sel_a, sel_w;       // v_perm selectors: bytes [2, 6) or [4, 8) of a dword pair
    uint32_t ad_shift, wd_mask;  // the scale's place in dword 0
    int aq, ad, ad_step, wq, wd; // LDS places of piece 0, within a stage buffer
};

template <class C>
__device__ __forceinline__ StageSlots stage_slots(int nb) {
    constexpr uint32_t kEven = 0x05040302u, kOdd = 0x07060504u;
    StageSlots o;
    const int ra = threadIdx.x / C::kActPerRow, pa = threadIdx.x % C::kActPerRow;
    const int ja = pa >> 1, ha = pa & 1;
    o.a = q4_0_act_piece(ra, pa, nb);
    const int rw = threadIdx.x / C::kWPerRow, jw = threadIdx.x % C::kWPerRow;
    o.w = q4_0_weight_piece(rw, jw, nb);
    const int tail = C::kTails ? nb % C::kKB : 0;
    o.a_past = tail && ja >= tail ? kPastEnd : 0u;
    o.w_past = tail && jw >= tail ? kPastEnd : 0u;
    o.sel_a = ja & 1 ? kOdd : kEven;
    o.sel_w = jw & 1 ? kOdd : kEven;
    o.ad_shift = ja & 1 ? 16 : 0;
    o.wd_mask = jw & 1 ? 0xffff0000u : 0x0000ffffu;
    o.aq = C::kAq + ra * C::kRowStride + ja * 32 + ha * 16;
    // a second half carries no scale: its lane's store goes to the row's pad
    o.ad = ha ? C::kAq + ra * C::kRowStride + C::kKB * 32 + 2 * (ja & 7) : C::kAd + (ra * C::kKB + ja) * 2;
    o.ad_step = C::kActRows * (ha ? C::kRowStride : C::kKB * 2);
    o.wq = C::kWq + rw * C::kRowStride + jw * 32;
    o.wd = C::kWd + (rw * C::kKB + jw) * 4;
    return o;
}

__device__ __forceinline__ void load5(__amdgpu_buffer_rsrc_t r, BufferOffset o, uint32_t (&v)[5]) {
    const i32x4 x = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(r, o.lane, o.uniform, 0));
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = (uint32_t)x[i];
    v[4] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, o.lane + 16u, o.uniform, 0);
}

// Load / store of piece p (activation pieces first). kb: the stage's first
// block; last: whether it is the last stage; buf: the stage's LDS buffer.
template <class C>
__device__ __forceinline__ void load_piece(__amdgpu_buffer_rsrc_t ra, __amdgpu_buffer_rsrc_t rw, const StageSlots &o,
                                           int nb, int kb, bool last, int p, PieceRegs &r) {
    const uint32_t mask = last ? kPastEnd : 0u;
    const bool act = p < C::kActPT;
    // opaque, so that the sums with the lane offsets are not kept in a register per piece
    uint32_t step = act ? (uint32_t)(p * C::kActRows) * (uint32_t)nb * 34u
                        : (uint32_t)((p - C::kActPT) * C::kWRows) * (uint32_t)nb * 18u;
    asm volatile("" : "+s"(step));
    if (act)
        load5(ra, q4_0_stage_piece(o.a, step, kb * 34, o.a_past & mask), r.v);
    else
        load5(rw, q4_0_stage_piece(o.w, step, kb * 18, o.w_past & mask), r.v);
}

template <class C>
__device__ __forceinline__ void store_piece(uint8_t *buf, const StageSlots &o, int p, const PieceRegs &r) {
    const uint32_t(&v)[5] = r.v;
    if (p < C::kActPT) {
        uint32_t x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = __builtin_amdgcn_perm(v[i + 1], v[i], o.sel_a);
        *reinterpret_cast<uint4 *>(buf + o.aq + p * C::kActRows * C::kRowStride) = make_uint4(x[0], x[1], x[2], x[3]);
        *reinterpret_cast<uint16_t *>(buf + o.ad + p * o.ad_step) = (uint16_t)(v[0] >> o.ad_shift);
    } else {
        const int q = p - C::kActPT;
        uint32_t lo[4], hi[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) q4_0_unpack16(__builtin_amdgcn_perm(v[i + 1], v[i], o.sel_w), lo[i], hi[i]);
        uint4 *dst = reinterpret_cast<uint4 *>(buf + o.wq + q * C::kWRows * C::kRowStride);
        dst[0] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
        dst[1] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
        *reinterpret_cast<uint32_t *>(buf + o.wd + q * C::kWRows * C::kKB * 4) = v[0] & o.wd_mask;
    }
}

// Operand fragments of one block t for the wave's TM x TN tiles. ad holds the
// da of blocks t4..t4+3 (t4 = t rounded down to a multiple of 4) in its four
// fp16 slots; wd holds dw of block t in slot t % 4 and zeros elsewhere, and
// the K-half 1 lanes read theirs from the zero strip, so the f16 MFMA of ad
// and wd is the exact outer product da * dw of block t.
template <class C>
struct Frags {
    i32x4 av[C::TM];
    i32x4 wv[C::TN];
    f16x4 ad[C::TM];
    f16x4 wd[C::TN];
};

// Per-lane LDS base addresses of one stage buffer; every fragment read is a
// base plus a compile-time offset (within the 16-bit ds_read immediate range).
struct FragBases {
    const uint8_t *aq, *ad, *wq, *wd;
};

template <class C>
__device__ __forceinline__ FragBases frag_bases(uint8_t *lds, int buf, int lane, int wave_m, int wave_n) {
    const int li = lane & 31, lh = lane >> 5;
    const int ra = wave_m * C::TM * 32 + li, rw = wave_n * C::TN * 32 + li;
    const uint8_t *b0 = lds + buf * C::kBufBytes;
    FragBases b;
    b.aq = b0 + C::kAq + ra * C::kRowStride + lh * 16;
    b.ad = b0 + C::kAd + ra * C::kKB * 2;
    b.wq = b0 + C::kWq + rw * C::kRowStride + lh * 16;
    b.wd = lh ? lds + C::kZero : b0 + C::kWd + rw * C::kKB * 4;
    return b;
}

// The activation fragment tm / weight fragment tn of block tb + j (tb a
// multiple of 4, j known at compile time).
template <class C>
__device__ __forceinline__ void load_frag_a(const FragBases &b, int tb, int j, int tm, Frags<C> &f) {
    f.av[tm] = *reinterpret_cast<const i32x4 *>(b.aq + tm * 32 * C::kRowStride + (tb + j) * 32);
    f.ad[tm] = *reinterpret_cast<const f16x4 *>(b.ad + tm * 32 * C::kKB * 2 + (tb + (j & ~3)) * 2);
}
template <class C>
__device__ __forceinline__ void load_frag_w(const FragBases &b, int tb, int j, int tn, Frags<C> &f) {
    f.wv[tn] = *reinterpret_cast<const i32x4 *>(b.wq + tn * 32 * C::kRowStride + (tb + j) * 32);
    const uint32_t word = *reinterpret_cast<const uint32_t *>(b.wd + tn * 32 * C::kKB * 4 + (tb + j) * 4);
    f.wd[tn] = __builtin_bit_cast(f16x4, (j & 2) ? make_uint2(0u, word) : make_uint2(word, 0u));
}

struct ItemRegs {
    i32x16 s16;
    f32x16 p;
};

// One K stage of one wave: its kWaveBlocks blocks (from tb) x TM x TN tiles
// = a flat list of items, software-pipelined so the MFMAs of item i+1 are in
// flight while the VALU epilogue of item i runs, and the LDS fragments of
// later blocks load meanwhile. With 2 x 2 tiles a block walks them in a snake
// (a0 w0, a0 w1, a1 w1, a1 w0; the next block a0 w1, a0 w0, a1 w0, a1 w1), and
// each fragment of block t+1 is read right after the last MFMA that uses block
// t's, two items or more before its first use: one set of fragment registers
// serves both blocks. piece(p), p = 0 .. kPieces - 1, is called at
// even distances along the list, behind the MFMAs of the next item: the next
// stage's pieces go to the other LDS buffer and the loads after them go out
// while the matrix cores work, instead of in a phase of their own.
// fresh: the accumulators start over with the stage's first block.
template <class C, bool kIsums, bool kFresh, class Piece>
__device__ __forceinline__ void compute_stage(uint8_t *lds, int buf, f32x16 (&acc)[C::TM][C::TN], int32_t *isums,
                                              int m, int n, int nb, int m0, int n0, int s, int tb, int lane,
                                              int wave_m, int wave_n, Piece piece) {
    constexpr int kTiles = C::TM * C::TN;
    constexpr int kItems = C::kWaveBlocks * kTiles;
    constexpr bool kSnake = C::TM == 2 && C::TN == 2;
    // blocks whose fragments are in registers or on their way: two (one tile
    // per block leaves less time per block: three or four)
    constexpr int kSets = kTiles == 1 ? (C::kWaveBlocks == 4 ? 4 : 3) : 2;
    static_assert(C::kWaveBlocks >= kSets && (kTiles == 1 || kSnake || kTiles == 2), "fragment sets");
    const FragBases bases = frag_bases<C>(lds, buf, lane, wave_m, wave_n);
    Frags<C> fr[kSets];
    ItemRegs it[2];
    auto tile_of = [](int item) {
        const int x = item % kTiles;
        if (!kSnake) return x;
        const int t = item / kTiles, tm = x >> 1;
        return 2 * tm + ((x ^ tm ^ t) & 1);
    };
    auto load_block = [&](int t) {
#pragma unroll
        for (int tm = 0; tm < C::TM; ++tm) load_frag_a<C>(bases, tb, t, tm, fr[t % kSets]);
#pragma unroll
        for (int tn = 0; tn < C::TN; ++tn) load_frag_w<C>(bases, tb, t, tn, fr[t % kSets]);
    };
    // the fragment reads that may follow the MFMAs of `item`
    auto load_after = [&](int item) {
        const int t = item / kTiles, x = item % kTiles;
        if constexpr (kSnake) {
            if (t + 1 >= C::kWaveBlocks) return;
            Frags<C> &f = fr[(t + 1) % kSets];
            const int freed = 1 ^ (t & 1);  // the weight fragment this block is done with first
            if (x == 1) load_frag_a<C>(bases, tb, t + 1, 0, f);
            if (x == 2) load_frag_w<C>(bases, tb, t + 1, freed, f);
            if (x == 3) {
                load_frag_w<C>(bases, tb, t + 1, freed ^ 1, f);
                load_frag_a<C>(bases, tb, t + 1, 1, f);
            }
        } else if (x == kTiles - 1 && t + kSets < C::kWaveBlocks) {
            load_block(t + kSets);
        }
    };
    auto issue = [&](int item) {
        const int t = item / kTiles, tile = tile_of(item);
        const int tm = tile / C::TN, tn = tile % C::TN;
        const Frags<C> &f = fr[t % kSets];
        ItemRegs &r = it[item & 1];
        r.s16 = mfma_i8_32x32x32(f.av[tm], f.wv[tn], kIsums ? (i32x16){} : sum_base16());
        if constexpr (!kIsums) r.p = mfma_f16_32x32x8(f.ad[tm], f.wd[tn], (f32x16){});
        load_after(item);
    };
#pragma unroll
    for (int t = 0; t < (kSnake ? 1 : kSets); ++t) load_block(t);
    issue(0);
#pragma unroll
    for (int item = 0; item < kItems; ++item) {
        const int t = item / kTiles, tile = tile_of(item);
        const int tm = tile / C::TN, tn = tile % C::TN;
        if (item + 1 < kItems) issue(item + 1);
        // keep the order: without the fences the scheduler sinks the MFMAs of
        // item+1 below this epilogue and reuses their result registers, which
        // exposes every MFMA's latency
        __builtin_amdgcn_sched_barrier(0);
        const ItemRegs &r = it[item & 1];
        if constexpr (kIsums) {
            const int col = n0 + wave_n * C::TN * 32 + tn * 32 + (lane & 31);
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int row = m0 + wave_m * C::TM * 32 + tm * 32 + mfma_row(lane, q);
                const int blk = s * C::kKB + tb + t;
                if (row < m && col < n && blk < nb) isums[((size_t)row * n + col) * nb + blk] = r.s16[q] / 16;
            }
        } else {
#pragma unroll
            for (int q = 0; q < 16; ++q)
                acc[tm][tn][q] = kFresh && t == 0 ? based_sum(r.s16[q]) * r.p[q]
                                                  : fmaf(based_sum(r.s16[q]), r.p[q], acc[tm][tn][q]);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int p = (item * C::kPieces + kItems - 1) / kItems; p < ((item + 1) * C::kPieces + kItems - 1) / kItems; ++p) {
            piece(p);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// kIsums == false: fp32 C. kIsums == true: int32 block sums (diagnostic).
template <class C, bool kIsums>
__global__ __launch_bounds__(C::kThreads, C::kMinWavesPerEU) void gemm_q4_0_kernel(const uint8_t *__restrict__ w,
                                                                                  const uint8_t *__restrict__ a,
                                                                                  float *__restrict__ c,
                                                                                  int32_t *__restrict__ isums, int m,
                                                                                  int n, int nb) {
    extern __shared__ __align__(16) uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int wk = wave / (C::kWM * C::kWN);   // which share of each stage's blocks
    const int wmn = wave % (C::kWM * C::kWN);  // which TM x TN sub-tile
    const int wave_m = wmn / C::kWN;
    const int wave_n = wmn % C::kWN;
    const TileOrigin to = xcd_tile(blockIdx.x, (m + C::kBM - 1) / C::kBM, (n + C::kBN - 1) / C::kBN);
    const int m0 = to.mi * C::kBM, n0 = to.ni * C::kBN;
    const int li = lane & 31;  // operand row / result column within a 32x32 tile

    f32x16 acc[C::TM][C::TN];
#pragma unroll
    for (int i = 0; i < C::TM; ++i)
#pragma unroll
        for (int j = 0; j < C::TN; ++j) acc[i][j] = (f32x16){};
    f32x16 total[C::TM][C::TN];  // kFold
    auto fold = [&]() __attribute__((always_inline)) {
        if constexpr (C::kFold > 0 && !kIsums) {
#pragma unroll
            for (int i = 0; i < C::TM; ++i)
#pragma unroll
                for (int j = 0; j < C::TN; ++j)
#pragma unroll
                    for (int q = 0; q < 16; ++q) total[i][j][q] += acc[i][j][q];
        }
    };
    if constexpr (C::kFold > 0 && !kIsums) {
#pragma unroll
        for (int i = 0; i < C::TM; ++i)
#pragma unroll
            for (int j = 0; j < C::TN; ++j) total[i][j] = (f32x16){};
    }

    // Double-buffered LDS with one barrier per stage: while stage s is computed
    // from one buffer, the pieces of stage s+1 go from registers into the
    // other one by one between the items, each register set being refilled at
    // once with the piece kAhead pieces on (so kAhead pieces are in flight).
    // Past the end the stage index is clamped, so the loop body has no
    // divergent control flow; rounds of two stages make register set and
    // buffer compile-time constants, and an odd last stage (kLastApart: the last
    // one or two) is computed after the loop.
    const int stages = (nb + C::kKB - 1) / C::kKB;
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(a + (size_t)m0 * nb * 34), 0,
        (int)((uint32_t)(m - m0 < C::kBM ? m - m0 : C::kBM) * (uint32_t)nb * 34u), kBufferWord3);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(w + (size_t)n0 * nb * 18), 0,
        (int)((uint32_t)(n - n0 < C::kBN ? n - n0 : C::kBN) * (uint32_t)nb * 18u), kBufferWord3);
    const StageSlots slots = stage_slots<C>(nb);
    for (int i = threadIdx.x; i < C::kZeroBytes / 16; i += C::kThreads)
        reinterpret_cast<uint4 *>(lds + C::kZero)[i] = make_uint4(0u, 0u, 0u, 0u);
    PieceRegs regs[C::kAhead];
    // piece x of the sequence over all stages
    auto load = [&](int st, int p, PieceRegs &r) __attribute__((always_inline)) {
        const int last = stages - 1;
        load_piece<C>(ra, rw, slots, nb, (st < last ? st : last) * C::kKB, st >= last, p, r);
    };
    {
        PieceRegs first[C::kPieces];
#pragma unroll
        for (int p = 0; p < C::kPieces; ++p) load(0, p, first[p]);
#pragma unroll
        for (int x = 0; x < C::kAhead; ++x) load(1 + x / C::kPieces, x % C::kPieces, regs[x]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int p = 0; p < C::kPieces; ++p) store_piece<C>(lds, slots, p, first[p]);
    }
    __syncthreads();
    const int tb = wk * C::kWaveBlocks;
    int s = 0;
    // one stage of a round (R = 0 or 1), from buffer R; More: the pieces of stages
    // after the next are loaded
    auto stage = [&](auto R, auto More) __attribute__((always_inline)) {
        constexpr int rr = decltype(R)::value;
        __builtin_amdgcn_sched_barrier(0);
        compute_stage<C, kIsums, C::kFold == 1 || (C::kFold == 2 && rr == 0)>(
            lds, rr, acc, isums, m, n, nb, m0, n0, s + rr, tb, lane, wave_m, wave_n,
            [&](int p) __attribute__((always_inline)) {
                PieceRegs &r = regs[(rr * C::kPieces + p) % C::kAhead];
                store_piece<C>(lds + (rr ^ 1) * C::kBufBytes, slots, p, r);
                const int x = p + C::kAhead;
                if (decltype(More)::value || x < C::kPieces) load(s + rr + 1 + x / C::kPieces, x % C::kPieces, r);
            });
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
    };
    // the last stage, from buffer R
    auto last_stage = [&](auto R) __attribute__((always_inline)) {
        constexpr int rr = decltype(R)::value;
        compute_stage<C, kIsums, C::kFold == 1 || (C::kFold == 2 && rr == 0)>(
            lds, rr, acc, isums, m, n, nb, m0, n0, s + rr, tb, lane, wave_m, wave_n, [](int) {});
        fold();
    };
    using First = std::integral_constant<int, 0>;
    using Second = std::integral_constant<int, 1>;
    for (; s + 1 + C::kLastApart < stages; s += 2) {
        stage(First{}, std::true_type{});
        if constexpr (C::kFold == 1) fold();
        stage(Second{}, std::true_type{});
        fold();
    }
    if (!C::kLastApart) {
        if (s < stages) last_stage(First{});
    } else if (s + 1 < stages) {
        stage(First{}, std::false_type{});
        if constexpr (C::kFold == 1) fold();
        last_stage(Second{});
    } else {
        last_stage(First{});
    }
    if constexpr (C::kFold > 0 && !kIsums) {
#pragma unroll
        for (int i = 0; i < C::TM; ++i)
#pragma unroll
            for (int j = 0; j < C::TN; ++j) acc[i][j] = total[i][j];
    }

    if constexpr (!kIsums) {
        if constexpr (C::kWK > 1) {
            // add the other K-waves' partials to wave wk == 0's, in wave order;
            // the stage buffers are free once every wave has left the loop
            constexpr int kRegs = C::TM * C::TN * 16;
            float *red = reinterpret_cast<float *>(lds);
            __syncthreads();
            if (wk > 0) {
                float *dst = red + ((wk - 1) * C::kWM * C::kWN + wmn) * kRegs * 64 + lane;
#pragma unroll
                for (int tm = 0; tm < C::TM; ++tm)
#pragma unroll
                    for (int tn = 0; tn < C::TN; ++tn)
#pragma unroll
                        for (int r = 0; r < 16; ++r) dst[((tm * C::TN + tn) * 16 + r) * 64] = acc[tm][tn][r];
            }
            __syncthreads();
            if (wk > 0) return;
#pragma unroll
            for (int w2 = 1; w2 < C::kWK; ++w2) {
                const float *src = red + ((w2 - 1) * C::kWM * C::kWN + wmn) * kRegs * 64 + lane;
#pragma unroll
                for (int tm = 0; tm < C::TM; ++tm)
#pragma unroll
                    for (int tn = 0; tn < C::TN; ++tn)
#pragma unroll
                        for (int r = 0; r < 16; ++r) acc[tm][tn][r] += src[((tm * C::TN + tn) * 16 + r) * 64];
            }
        }
#pragma unroll
        for (int tm = 0; tm < C::TM; ++tm)
#pragma unroll
            for (int tn = 0; tn < C::TN; ++tn) {
                const int col = n0 + wave_n * C::TN * 32 + tn * 32 + li;
                if (col < n) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int row = m0 + wave_m * C::TM * 32 + tm * 32 + mfma_row(lane, r);
                        if (row < m) store_through(&c[(size_t)row * n + col], acc[tm][tn][r] * kBasedSumScale);
                    }
                }
            }
    }
}

template <class C, bool kIsums>
hipError_t launch_q4_0(const void *w, const void *a, float *c, int32_t *isums, int64_t m, int64_t n, int64_t k,
                       hipStream_t stream) {
    const dim3 grid((unsigned)(((n + C::kBN - 1) / C::kBN) * ((m + C::kBM - 1) / C::kBM)));
    hipLaunchKernelGGL((gemm_q4_0_kernel<C, kIsums>), grid, dim3(C::kThreads), C::kLdsBytes, stream,
                       static_cast<const uint8_t *>(w), static_cast<const uint8_t *>(a), c, isums, (int)m, (int)n,
                       (int)(k / 32));
    return hipGetLastError();
}

// The tiles, from large to small problems; every one takes any k % 128 == 0 (a
// last stage that the row does not fill reads zeros).
// 128x128, 4 waves of 64x64, 4 blocks per stage, two workgroups per CU; half a
// stage's pieces in flight (all six would spill: the accumulators, two items'
// results and the fragments leave no room)
using Q40Big = Q40Config<128, 128, 2, 2, 4, 1, 3>;
// 128x64, 8 waves of 32x32, 8 blocks per stage (as 4 waves of 64x32 in 2 K-waves
// it is no faster, and has no registers left to fold into)
using Q40Mid = Q40Config<128, 64, 4, 2, 8, 1, 5, 2>;
// 64x64, 4 waves of 32x32 in 2 K-waves each taking 8 of a 16-block stage
using Q40SmallK2 = Q40Config<64, 64, 2, 2, 16, 2, 6, 2>;
// 32x64, 2 waves of 32x32 in 4 K-waves each taking 4 of a 16-block stage
using Q40WideK4 = Q40Config<32, 64, 1, 2, 16, 4, 8, 2>;
// 64x64, 4 waves of 32x32, 8 blocks per stage, two workgroups per CU (short k)
using Q40Small = Q40Config<64, 64, 2, 2, 8, 1, 6, 2>;
// 64x64, 2 waves of 64x32, 4 blocks per stage, four workgroups per CU (no
// registers left to fold into)
using Q40Small4 = Q40Config<64, 64, 1, 2, 4>;
// 32x32, 2 K-waves each taking 4 of an 8-block stage, several workgroups per CU
// (short k)
using Q40Tiny = Q40Config<32, 32, 1, 1, 8, 2, 6, 2>;
// 32x32, one wave in 8 K-waves each taking 4 of a 32-block stage, two stages'
// pieces in flight
using Q40TinyK8 = Q40Config<32, 32, 1, 1, 32, 8, 12, 2>;
// The tiles whose wave takes 8 blocks of a stage, folded after every stage: sums
// of 8 terms, as the tile GEMV has up to k = 4096 (one group per wave and round).
// us folded every two stages and every one: 126x12859x3584 (128x64) 24.8 / 25.2,
// 42x15892x2304 (64x64) 12.1 / 12.3. Folding at all costs the 64x64 and 32x32 tiles
// as much: 906x5111x2816 50.6 / 51.2 (error 1.7e-7 / 8.9e-8), 50x373x1152 6.8 / 6.9
// (8.4e-8 / 6.7e-8).
using Q40MidS = Q40Config<128, 64, 4, 2, 8, 1, 5, 1>;
using Q40SmallK2S = Q40Config<64, 64, 2, 2, 16, 2, 6, 1>;
using Q40SmallS = Q40Config<64, 64, 2, 2, 8, 1, 6, 1>;

enum {
    kCfgBig = 0,
    kCfgMid = 1,
    kCfgMidS = 2,
    kCfgSmallK2 = 3,
    kCfgSmallK2S = 4,
    kCfgWideK4 = 5,
    kCfgTinyK8 = 6,
    kCfgSmall = 7,
    kCfgSmallS = 8,
    kCfgTiny = 9,
    kCfgSmall4 = 10,
    kCfgTiles = 11,  // the first that is no tile of this file
    kCfgWhole = 11
};

// f called with the configuration type of a tile of this file
template <class F>
auto with_tile(int config, F f) {
    switch (config) {
    case kCfgBig: return f(Q40Big{});
    case kCfgMid: return f(Q40Mid{});
    case kCfgMidS: return f(Q40MidS{});
    case kCfgSmallK2: return f(Q40SmallK2{});
    case kCfgSmallK2S: return f(Q40SmallK2S{});
    case kCfgWideK4: return f(Q40WideK4{});
    case kCfgSmall: return f(Q40Small{});
    case kCfgSmallS: return f(Q40SmallS{});
    case kCfgTiny: return f(Q40Tiny{});
    case kCfgSmall4: return f(Q40Small4{});
    default: return f(Q40TinyK8{});
    }
}

int64_t tiles_of(int64_t m, int64_t n, int64_t bm, int64_t bn) { return ((m + bm - 1) / bm) * ((n + bn - 1) / bn); }

// Tile choice: the least predicted time. A workgroup of the K-split tiles has a
// CU to itself, so they take rounds of one tile per CU; the 128x128 and the plain
// 64x64 tile run two, the 2-wave tiles four workgroups per CU. Nanoseconds per
// round beyond the launch, fixed and per element of k (padded to whole stages),
// fitted to 47 shapes with each tile forced (m 32..2048, n 100..14336, k 128..11008;
// mostly within 8 %), us there: k = 4096, one tile per CU 32x32 11, 32x64 12.7,
// 64x64 17.5, 128x64 27.5, 128x128 60, two 88, four of the 2-wave 64x64 55; two
// rounds 64x64 33.6, 128x64 53.6. Against a choice by tile counts among the plain
// 64x64, the 2-K-wave 32x32 and 64x64, and the 128x128 tiles (with the staging of
// that time): 333x4096x4096 30.7 -> 26.6 us, 100x11008x4096 34.2 -> 26.6, 333x1536x4096
// 19.2 -> 17.0, 200x4096x11008 51.0 -> 39.4, 480x4096x11008 76.1 -> 69.0, 130x8000x1664
// 20.7 -> 14.1, 480x4096x1536 14.0 -> 13.1.
int64_t q4_0_tile_ns(int config, int64_t m, int64_t n, int64_t k, int cus) {
    auto rounds = [&](int64_t bm, int64_t bn) { return (tiles_of(m, n, bm, bn) + cus - 1) / cus; };
    auto padded = [&](int64_t unit) { return (k + unit - 1) / unit * unit; };
    switch (config) {
    case kCfgBig: {
        const int64_t r = rounds(128, 128);
        return r / 2 * (5000 + 198 * k / 10) + r % 2 * (3400 + 135 * k / 10);
    }
    case kCfgMid:
    case kCfgMidS: return rounds(128, 64) * (2900 + 575 * padded(256) / 100);
    case kCfgSmallK2:
    case kCfgSmallK2S: return rounds(64, 64) * (1700 + 335 * padded(512) / 100);
    case kCfgSmall:
    case kCfgSmallS: {
        const int64_t r = rounds(64, 64), p = padded(256);
        return r / 2 * (1600 + 665 * p / 100) + r % 2 * (2200 + 465 * p / 100) * (r > 1 ? 4 : 5) / 5;
    }
    case kCfgSmall4: {
        const int64_t r = rounds(64, 64), rest = r % 4;
        // short rows beyond four rounds wait for the outputs of the rounds before: us
        // here and on the 128x128 tile 1335x4488x128 10.8 / 9.3, 1531x7108x512 30.0 /
        // 27.9, 2048x14336x128 31.6 / 27.9 (1945x4367x640 29.2 / 31.4 stays)
        const int64_t late = r > 4 && k <= 1024 ? 800 + (rest ? 400 : 0) : 0;
        return late + r / 4 * (2200 + 125 * k / 10) + (rest ? 1800 + (rest > 1 ? 105 : 83) * k / 10 : 0);
    }
    case kCfgWideK4: return rounds(32, 64) * (1800 + 22 * padded(512) / 10);
    case kCfgTiny: {
        const int64_t r = rounds(32, 32), p = padded(256), rest = r % 4;
        return r / 4 * (1700 + 475 * p / 100) + (rest ? 800 + 310 * p / 100 + (rest - 1) * (300 + 55 * p / 100) : 0);
    }
    default: return rounds(32, 32) * (1900 + 175 * padded(1024) / 100);
    }
}

// Rounding (see chain_rounding) of an output's nb block terms in a tile's order:
// a K-wave adds its blocks one after another, over kFold stages before they go
// into the total; the K-waves' partials are added in order.
template <class C>
int64_t tile_rounding(int64_t nb) {
    int64_t sum = 0, joined = 0;
    for (int v = 0; v < C::kWK; ++v) {
        const int64_t full = nb / C::kKB, rest = nb % C::kKB - v * C::kWaveBlocks;
        const int64_t terms = full * C::kWaveBlocks + (rest < 0 ? 0 : rest < C::kWaveBlocks ? rest : C::kWaveBlocks);
        if constexpr (C::kFold > 0) {
            const int64_t run = C::kFold * C::kWaveBlocks, runs = terms / run, last = terms % run;
            sum += runs * chain_rounding(run) + chain_rounding(last);
            if (runs > 0) sum += run * (chain_rounding(runs) - 1) + (last ? terms : 0);
        } else {
            sum += chain_rounding(terms);
        }
        joined += terms;
        if (v > 0 && terms > 0) sum += joined;
    }
    return sum;
}

int64_t q4_0_tile_rounding(int config, int64_t nb) {
    if (config == kCfgWhole) return 4 * chain_rounding(nb / 4) + 9 * (nb / 4);  // four K slices
    return with_tile(config, [&](auto c) { return tile_rounding<decltype(c)>(nb); });
}

// The limit of a shape: where the automatic path could run the tile GEMV, that
// of its 16 waves (8-block groups dealt out in turn); else eight K-waves up to one
// 32x32 tile per CU, two while there are fewer than two 128x128 and 1.25 64x64 tiles
// per CU, one sum per output above that and at the k of 4-block stages.
int64_t q4_0_rounding_limit(int64_t m, int64_t n, int64_t k, int cus, bool automatic) {
    const int64_t nb = k / 32;
    if (automatic && m > 16 && gemv_supported(PFNG_WEIGHT_Q4_0_ACTIVATION_Q8_0, m, k)) {
        int64_t sum = 0, joined = 0;
        for (int v = 0; v < 16 && v < nb / 8; ++v) {
            const int64_t terms = 8 * ((nb / 8 - v + 15) / 16);
            sum += chain_rounding(terms);
            joined += terms;
            if (v > 0) sum += joined;
        }
        return sum;
    }
    if (k % 1024 == 0 && tiles_of(m, n, 32, 32) <= cus) return 8 * chain_rounding(nb / 8) + 35 * (nb / 8);
    if (k % 256 == 0 && tiles_of(m, n, 128, 128) < 2 * (int64_t)cus && 4 * tiles_of(m, n, 64, 64) < 5 * (int64_t)cus)
        return 2 * chain_rounding(nb / 2) + nb;
    return chain_rounding(nb);
}

// The q4_0 tile with the least predicted time (a later one, mostly smaller,
// only if it is 3 % less) among those within the shape's rounding limit. Without
// the limit, errors from 64 bits against the tile GEMV's: 100x20480x4096
// (2-wave 64x64) 2.2 times, 48x28672x8192 (64x64) 2.6, 74x10537x3072 (32x32) 1.7.
int64_t best_q4_0_tile(int64_t m, int64_t n, int64_t k, int cus, bool automatic, int &config) {
    const int64_t limit = q4_0_rounding_limit(m, n, k, cus, automatic);
    int64_t best = kNoTile;
    config = kCfgBig;
    for (int c = kCfgBig; c < kCfgTiles; ++c) {
        const int64_t ns = q4_0_tile_ns(c, m, n, k, cus);
        if (ns + ns * 3 / 100 < best && within_rounding(q4_0_tile_rounding(c, k / 32), limit)) {
            best = ns;
            config = c;
        }
    }
    return best;
}

// Whole-K 32x96 tiles, one per CU and one round (480x1536x1536: 7.0 us against
// 8.9 us for the 64x64 tile), where their four K slices are within the limit
bool q4_0_takes_whole(int64_t m, int64_t n, int64_t k, int cus, bool automatic) {
    const int64_t tiles = tiles_of(m, n, 32, 96);
    return q4_0_small_supported(k) && 2 * tiles >= cus && tiles <= cus &&
           within_rounding(q4_0_tile_rounding(kCfgWhole, k / 32), q4_0_rounding_limit(m, n, k, cus, automatic));
}

}  // namespace

bool mfma_supported(int type, int64_t m, int64_t k) {
    (void)m;
    if (k > kMaxTiledK) return false;  // 32-bit load offsets
    if (type == PFNG_WEIGHT_Q4_0_ACTIVATION_Q8_0) return k % (32 * 4) == 0;  // whole dwords per block pair, stages of 4 blocks
    // the super-block formats take any k % 256 == 0 (gemm_kquant.hip)
    return (type == PFNG_WEIGHT_Q4_K_ACTIVATION_Q8_K || type == PFNG_WEIGHT_IQ2_XXS_ACTIVATION_Q8_K) && k % 256 == 0;
}

// Rounds of 16-row tiles, one per CU, each repeating its activation chunks C =
// m / 16: measured at n = 4096 (one round) and m = 16, 37, 64, 100, 128, k = 4096 and
// 11008, us q4_0 5.2, 8.3, 9.9, 13.7, 15.6, q4_K 5.1, 7.7, 9.6, 13.2, 15.2, iq2_xxs 4.8,
// 6.6, 7.4, 11.2, 12.6 at k = 4096.
int64_t tile_gemv_ns(int type, int64_t m, int64_t n, int64_t k, int cus) {
    const int64_t rounds = (n + 16 * (int64_t)cus - 1) / (16 * (int64_t)cus), chunks = (m + 15) / 16;
    const int64_t round = type == PFNG_WEIGHT_Q4_0_ACTIVATION_Q8_0   ? 2000 + 1500 * chunks
                          : type == PFNG_WEIGHT_Q4_K_ACTIVATION_Q8_K ? 1900 + 1430 * chunks
                                                                     : 1800 + 1120 * chunks;
    return 1700 + rounds * round * (1024 + 3 * k / 4) / 4096;
}

int64_t gemm_ns(int type, int64_t m, int64_t n, int64_t k, int cus, bool automatic) {
    if (type != PFNG_WEIGHT_Q4_0_ACTIVATION_Q8_0) return kquant_gemm_ns(type, m, n, k, cus, automatic);
    if (q4_0_takes_whole(m, n, k, cus, automatic)) return 3000 + 26 * k / 10;  // 5.7 us at k = 1024, 7.0 at 1536
    int config;
    return 2000 + best_q4_0_tile(m, n, k, cus, automatic, config);
}

// The tile GEMV repeats its activation chunks in every round, so on wide outputs
// the GEMM tiles overtake it from m = 17. At k = 4096, us GEMV / GEMM: q4_0 n = 11008
// m = 16 12.0 / 12.8, m = 37 20.4 / 17.2, m = 64 24.2 / 17.3, m = 100 35.6 / 27.8; n =
// 14336 m = 37 29.1 / 17.7, m = 64 33.7 / 18.4; q4_K n = 11008 m = 100 33.9 / 31.3, n =
// 14336 m = 64 32.6 / 25.5; iq2_xxs n = 11008 m = 128 35.2 / 27.9, n = 14336 m = 64 27.3 /
// 21.5. A single round (n <= 4096) keeps the GEMV: q4_0 m = 64 9.9 / 11.1. The
// K-quant GEMM tiles add a slice's super-blocks in one sum, which from about 16
// of them (k = 8192) is less exact than the GEMV's 16 waves (k = 14336: 1.18e-7
// against 1.08e-7 from 64 bits), so longer rows stay there. A partly filled last
// round of the GEMV takes less than a whole one, so near a tie the GEMV is the
// faster one (q4_K 38x13594x8192, predicted 45.0 / 42.6, takes 41.1 / 44.1): the
// GEMM has to be predicted 7 % faster (100x11008x4096, 37.4 / 34.7, takes 33.9 / 31.3).
bool mfma_preferred(int type, int64_t m, int64_t n, int64_t k) {
    if (type != PFNG_WEIGHT_Q4_0_ACTIVATION_Q8_0 && k > 8192) return false;
    return m > 16 && n > 16 * kMi355xCus &&
           gemm_ns(type, m, n, k, kMi355xCus, true) * 107 / 100 < tile_gemv_ns(type, m, n, k, kMi355xCus);
}

MfmaPlan plan_mfma(int type, int64_t m, int64_t n, int64_t k, int cus, bool automatic) {
    if (type != PFNG_WEIGHT_Q4_0_ACTIVATION_Q8_0) return plan_kquant(type, m, n, k, cus, automatic);
    MfmaPlan p;
    if (q4_0_takes_whole(m, n, k, cus, automatic)) {
        p.config = kCfgWhole;
        return p;
    }
    best_q4_0_tile(m, n, k, cus, automatic, p.config);
    return p;
}

hipError_t launch_mfma_mul_mat(int type, const void *w, const void *a, float *c, int64_t m, int64_t n, int64_t k,
                               const MfmaPlan &plan, hipStream_t stream) {
    if (type != PFNG_WEIGHT_Q4_0_ACTIVATION_Q8_0) return launch_kquant_mul_mat(type, w, a, c, m, n, k, plan, stream);
    if (plan.config == kCfgWhole) return launch_q4_0_small(w, a, c, nullptr, m, n, k, stream);
    return with_tile(plan.config, [&](auto t) {
        return launch_q4_0<decltype(t), false>(w, a, c, nullptr, m, n, k, stream);
    });
}

hipError_t launch_mfma_block_isums(int type, const void *w, const void *a, int32_t *out, int64_t m, int64_t n,
                                   int64_t k, const MfmaPlan &plan, hipStream_t stream) {
    if (type != PFNG_WEIGHT_Q4_0_ACTIVATION_Q8_0)
        return launch_kquant_block_isums(type, w, a, out, m, n, k, plan, stream);
    if (plan.config == kCfgWhole) return launch_q4_0_small(w, a, nullptr, out, m, n, k, stream);
    return with_tile(plan.config, [&](auto t) {
        return launch_q4_0<typename decltype(t)::Isums, true>(w, a, nullptr, out, m, n, k, stream);
    });
}

}  // namespace pfng
