// Prefill GEMM (rows >= 9) on CDNA4 int8 MFMA, activation-quantized route
// (ops/native_compute.zig:13304-13478 for Q8_0, :23427-23775 for Q4_0):
//   dot[m][n][b] = sum_i qx[m][32b+i] * qw[n][32b+i]            (int32, exact)
//   y[m][n]      = sum_b (sx[m][b] * sw[n][b]) * f32(dot[m][n][b])
//
// Per 32x32 output tile and per pair of blocks (b, b+1) a wavefront issues
//   2 x v_mfma_i32_32x32x32_i8     the int32 dots of block b and of block b+1
//   1 x v_mfma_f32_32x32x1_2b_f32  the scale products sx[m][b]*sw[n][b] of both
//                                  blocks (two rank-1 outer products; each entry
//                                  is the correctly rounded f32 product)
// and then one int->float conversion and one fused multiply-add per element and
// block on the vector ALU.  All three results share the 32x32 MFMA register
// layout, so the epilogue is element-wise.  On this chip the vector ALU and the
// matrix pipe of a SIMD do not run these two halves side by side, so a pair costs
// their sum; everything else (global loads, LDS traffic, barriers) is arranged to
// hide behind that.
//
// Workgroup = kWavesM x kWavesN output tiles of 32x32, times kSplit wavefronts per
// tile that share the K loop: a stage holds 2*kSplit blocks and wavefront ks of a
// tile takes pair ks of every stage.  The kSplit partial sums of a tile are added
// in LDS at the end, in ks order (so y is a fixed-order sum of kSplit block-ascending
// partial sums).  Four wavefronts on every SIMD, where LDS allows as two workgroups of
// eight: they wait at barriers of their own, so one computes while the other meets (a
// workgroup of sixteen spent a quarter of its K loop at barriers).  A wavefront with two
// tiles (kPerM = 2) reads one weight fragment for both.  Bound by the vector ALU beside the
// MFMA: about 230 SIMD cycles per 32 x 32 outputs and block (300 before, Q4_0), of which
// the arithmetic alone takes 140.  2048 rows, K = 4096, N = 14336: Q4_0 513 -> 393 us
// (612 TOP/s), Q8_0 434 -> 400 us.
//
// Operands reach LDS without passing through registers: activations and Q8_0 weight
// bytes are fetched with global_load_lds_dwordx4 into a ring of kRing stages (4, or
// 3 for the widest stages), kRing - 1 stages ahead of the one being consumed.  One
// such load moves 64 x 16 bytes: whole 128-byte lines of kRowsPerLoad rows, with
// consecutive lanes on the chunks of one line (one cache-line lookup per eight
// lanes).  LDS holds a stage row-major with the 16-byte chunk index XOR-swizzled by
// the row, so that the MFMA fragment reads (one row per lane, same chunk column) of 16
// consecutive lanes hit 16 different bank groups.  Block scales arrive the same way
// (f32 activation scales as they are, fp16 weight scales zero-extended to 32 bits
// and converted when read).  Q4_0 nibble chunks stay packed in LDS: a lane half of an
// MFMA operand is one nibble of every byte, shifted to the top of its byte and so
// sixteen times its value (two instructions a word), and the scale is a sixteenth.
//
// MFMA operands: A = activations (row = lane % 32 -> m), B = weights (column =
// lane % 32 -> n); lane / 32 selects bytes [16*(lane/32), +16) of the block.
// Result register v of a lane is row 8*(v/4) + 4*(lane/32) + v%4, column
// lane % 32, so stores are 128 bytes contiguous along n.
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <type_traits>

#include "device_common.h"
#include "gemv_common.h"
#include "qmatmul_launch.h"

namespace afhip {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v32f __attribute__((ext_vector_type(32)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// A wavefront owns kPerM x kPerN tiles of 32 x 32.
template <int kWavesM, int kWavesN, int kSplit, bool kQ4, int kPerM = 1, int kPerN = 1>
struct GemmShape {
    static constexpr int kTiles = kWavesM * kWavesN;
    static constexpr int kWaves = kTiles * kSplit;
    static constexpr int kThreads = 64 * kWaves;
    static constexpr int kTM = 32 * kWavesM * kPerM, kTN = 32 * kWavesN * kPerN;
    static constexpr int kStageBlocks = 2 * kSplit;              // one pair per wavefront and stage
    static constexpr int kChunksPerRow = 2 * kStageBlocks;       // 16-byte chunks of int8 per row and stage
    static constexpr int kRowsPerLoad = 64 / kChunksPerRow;      // rows one 64-lane LDS load covers
    static constexpr int kGroupsA = kTM / kRowsPerLoad, kGroupsB = kTN / kRowsPerLoad;
    static constexpr int kABytes = kTM * kChunksPerRow * 16, kBBytes = kTN * kStageBlocks * (kQ4 ? 16 : 32);
    // LDS keeps a stage of an operand row-major, [row][chunk], with the chunk index
    // XOR-swizzled by the row so that 16 consecutive rows reading the same chunk
    // column hit 16 different 16-byte bank groups (a row is 16 * kChunksPerRow bytes,
    // the banks wrap every 256 bytes).
    static constexpr int kRowsPerWrap = 16 / kChunksPerRow > 0 ? 16 / kChunksPerRow : 1;
    __device__ static constexpr int chunk_pos(int row, int chunk) {
        return row * kChunksPerRow + (chunk ^ ((row / kRowsPerWrap) % kChunksPerRow));
    }
    static_assert(kChunksPerRow == 4 || kChunksPerRow == 8 || kChunksPerRow == 16, "swizzle covers rows of 64..256 bytes");
    static constexpr int kSxBytes = kTM * kStageBlocks * 4, kSwBytes = kTN * kStageBlocks * 4;
    static constexpr int kStageBytes = kABytes + kBBytes + kSxBytes + kSwBytes;
    static constexpr int kReduceBytes = kSplit > 1 ? kSplit * kTM * kTN * 4 : 0;
    // LDS stages: loads run kRing - 1 stages ahead of the consumer
    static constexpr int kRing = 4 * kStageBytes <= 160 * 1024 ? 4 : 3;
    static constexpr int kLdsBytes = kRing * kStageBytes > kReduceBytes ? kRing * kStageBytes : kReduceBytes;
    static_assert(kSplit == 1 || kSplit == 2 || kSplit == 4 || kSplit == 8, "kSplit");
    static_assert(kThreads <= 1024, "workgroup size");
    static_assert(kTM % kRowsPerLoad == 0 && kTN % kRowsPerLoad == 0, "tile rows per load");
    static_assert(kLdsBytes <= 160 * 1024, "LDS");
};

// s_waitcnt for "at most kLeft vector memory operations outstanding" (nothing else waited for).
template <int kLeft>
__device__ __forceinline__ void wait_vm_outstanding() {
    static_assert(kLeft >= 0 && kLeft < 64, "six bits");
    // simm16: vmcnt[3:0] | expcnt << 4 | lgkmcnt << 8 | vmcnt[5:4] << 14
    __builtin_amdgcn_s_waitcnt((kLeft & 15) | (7 << 4) | (15 << 8) | ((kLeft >> 4) << 14));
}

// One 64-lane load from global memory straight into LDS: lane l's `bytes` at
// base + voff land at lds_addr + l * max(bytes, 4) (a 2-byte element is zero-extended
// to 4).  Issued as inline assembly on purpose: the compiler would otherwise make
// every later LDS read wait for all such loads in flight, which defeats the ring.
// Completion is tracked with wait_vm_outstanding; base and lds_addr are wave-uniform.
// M0 is declared as clobbered, so the compiler keeps nothing of its own in it across these statements.
__device__ __forceinline__ void lds_load16(const void* base, uint32_t voff, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds_addr), "v"(voff), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void lds_load4(const void* base, uint32_t voff, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" : : "s"(lds_addr), "v"(voff), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void lds_load2(const void* base, uint32_t voff, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_ushort %1, %2" : : "s"(lds_addr), "v"(voff), "s"(base) : "memory", "m0");
}

extern __shared__ __align__(16) unsigned char gemm_lds[];

// kShareK: this launch walks only a share of K per workgroup (see below); a template parameter
// so that the ordinary kernel carries none of it.
// kStamps (diagnostic): the kernel computes as usual but, instead of results, every wavefront stores eight
// 32-bit counts over the start of dst, [8 * (workgroup * wavefronts + wavefront)]: shader-clock cycles before
// the K loop, in it, waiting for its own loads, waiting at the workgroup barrier, 100 MHz reference ticks
// spent in the loop (cycles / ticks = the clock the chip held), cycles after the loop, 0, and the HW_ID register.
template <int kType, int kWavesM, int kWavesN, int kSplit, bool kWriteDots, bool kShareK = false, bool kStamps = false, int kPerM = 1,
          int kPerN = 1>
__device__ __forceinline__ void gemm_i8_body(
    float* __restrict__ dst, int* __restrict__ dots, const int8_t* __restrict__ qx, const float* __restrict__ sx,
    const uint8_t* __restrict__ weight, int rows, int in_dim, int out_dim, int m_tiles, int n_tiles,
    int share_blocks, float* __restrict__ partial, const Epilogue& ep) {
    using S = GemmShape<kWavesM, kWavesN, kSplit, kType == 2, kPerM, kPerN>;
    static_assert(kPerM * kPerN == 1 || (!kWriteDots && !kStamps), "block dots and clock readings: one tile a wavefront");
    constexpr int kWaves = S::kWaves, kSB = S::kStageBlocks, kRPL = S::kRowsPerLoad, kCPR = S::kChunksPerRow;
    constexpr int kTM = S::kTM, kTN = S::kTN, kRing = S::kRing;
    constexpr int kQuantBytes = kType == 2 ? 16 : 32;
    constexpr bool kQ4 = kType == 2;
    // units of 64 lanes per stage, by kind
    constexpr int kUnitsA = S::kGroupsA;                          // LDS loads of activation bytes
    constexpr int kUnitsB = kQ4 ? kTN * kSB / 64 : S::kGroupsB;   // Q4_0: of 16-byte nibble chunks
    constexpr int kUnitsSx = kTM * kSB / 64, kUnitsSw = kTN * kSB / 64;
    constexpr int kPerA = (kUnitsA + kWaves - 1) / kWaves, kPerB = (kUnitsB + kWaves - 1) / kWaves;
    constexpr int kPerSx = (kUnitsSx + kWaves - 1) / kWaves, kPerSw = (kUnitsSw + kWaves - 1) / kWaves;
    // each kind starts its round-robin over the wavefronts where the previous one stopped
    constexpr int kStartB = kUnitsA % kWaves, kStartSx = (kStartB + kUnitsB) % kWaves, kStartSw = (kStartSx + kUnitsSx) % kWaves;

    // K range of this workgroup: all of it, or (a small grid spread over more compute units)
    // share blockIdx.y of share_blocks blocks, whose sums go to partial[share][rows][out_dim] for splitk_reduce_kernel, or, of two
    // shares without an epilogue, are added to a dst that the quantizer's launch has cleared (partial is null then;
    // 0 + a + b = 0 + b + a to the bit, whoever comes first).  kb_full is the row pitch, kb the blocks walked here.
    const int kb_full = in_dim >> 5;
    const int blk_begin = kShareK ? static_cast<int>(blockIdx.y) * share_blocks : 0;
    const int kb = kShareK ? min(share_blocks, kb_full - blk_begin) : kb_full;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ks = wave / S::kTiles, tile = wave % S::kTiles;
    const int wm = tile / kWavesN, wn = tile % kWavesN;
    const int lj = lane & 31, lh = lane >> 5;

    // Workgroups that share a weight tile (same n tile, different m tiles) sit on the same XCD (consecutive workgroup ids go
    // round-robin over the eight), so each L2 reads every weight byte once.  The tiles of the columns that eight do not divide
    // go to all XCDs in equal parts (whole columns to each: 5632 columns of 128 put six on four of them and five on the others).
    const int xcd = blockIdx.x & 7, slot_id = blockIdx.x >> 3, whole = (n_tiles >> 3) * m_tiles;
    int m_tile, n_tile;
    if (slot_id < whole) {
        m_tile = slot_id % m_tiles;
        n_tile = (slot_id / m_tiles) * 8 + xcd;
    } else {
        const int rest = (n_tiles & 7) * m_tiles, part = (rest + 7) >> 3, index = xcd * part + slot_id - whole;
        if (slot_id - whole >= part || index >= rest) return;
        m_tile = index % m_tiles;
        n_tile = (n_tiles & ~7) + index / m_tiles;
    }
    const int m0 = m_tile * kTM, n0 = n_tile * kTN;

    const size_t blocks = static_cast<size_t>(out_dim) * kb_full;
    const uint8_t* a_base = reinterpret_cast<const uint8_t*>(qx) + static_cast<size_t>(m0) * in_dim + static_cast<size_t>(blk_begin) * 32;
    const uint8_t* b_base = weight + (static_cast<size_t>(n0) * kb_full + blk_begin) * kQuantBytes;
    const uint8_t* sx_base = reinterpret_cast<const uint8_t*>(sx + static_cast<size_t>(m0) * kb_full + blk_begin);
    const uint8_t* sw_base = weight + blocks * kQuantBytes + (static_cast<size_t>(n0) * kb_full + blk_begin) * 2;

    const int stages = (kb + kSB - 1) / kSB;
    const int last_blocks = kb - (stages - 1) * kSB;  // blocks in the last stage, 1..kSB

    // first unit of each kind this wavefront handles (then every kWaves-th)
    const int ua0 = wave;
    const int ub0 = (wave + kWaves - kStartB) % kWaves;
    const int usx0 = (wave + kWaves - kStartSx) % kWaves;
    const int usw0 = (wave + kWaves - kStartSw) % kWaves;
    // the round-robin leaves every wavefront kLoads loads a stage, or one more to some
    constexpr int kUnits = kUnitsA + kUnitsB + kUnitsSx + kUnitsSw, kLoads = kUnits / kWaves, kOneMore = kUnits % kWaves;
    const bool one_more = kOneMore != 0 && wave < kOneMore;
    auto wait_for_stage = [&]() {  // all but the last stage issued
        if (kOneMore != 0 && one_more) wait_vm_outstanding<kLoads + 1>();
        else wait_vm_outstanding<kLoads>();
    };

    // Per-lane byte offsets of the loads of a stage whose blocks from `blocks_here` on are clamped to the one before (the last
    // stage: nothing is read past a row's end; the scales of the clamped blocks are taken as zero).
    // LDS position p = lane of a 64-lane load is chunk slot p % kCPR of row p / kCPR: eight (or more) consecutive lanes
    // read one 128-byte line, in swizzled order.
    auto chunk_offset = [&](int unit, int l, int tile_rows, int first_row, int last_row, int blocks_here) {
        const int r = min(unit * kRPL + l / kCPR, tile_rows - 1);
        const int c = (l % kCPR) ^ ((r / S::kRowsPerWrap) % kCPR);
        return static_cast<uint32_t>(min(first_row + r, last_row) - first_row) * static_cast<uint32_t>(kb_full) * 32u +
               (min(c >> 1, blocks_here - 1) * 2 + (c & 1)) * 16;
    };
    auto offset_a = [&](int i, int l, int blocks_here) { return chunk_offset(ua0 + i * kWaves, l, kTM, m0, rows - 1, blocks_here); };
    // Q4_0: LDS position of a row's nibble chunk, [row][block] with the block XOR-swizzled by the row like the chunks
    auto nibble_slot = [](int r, int blk) { return blk ^ ((r / (16 / kSB)) % kSB); };
    auto offset_b = [&](int i, int l, int blocks_here) {
        if (!kQ4) return chunk_offset(ub0 + i * kWaves, l, kTN, n0, out_dim - 1, blocks_here);
        const int q = min((ub0 + i * kWaves) * 64 + l, kTN * kSB - 1), r = q / kSB;
        return static_cast<uint32_t>(min(n0 + r, out_dim - 1) - n0) * static_cast<uint32_t>(kb_full) * 16u +
               min(nibble_slot(r, q % kSB), blocks_here - 1) * 16;
    };
    auto scale_offset = [&](int unit, int l, int values, int first_row, int last_row, int blocks_here) {
        const int q = min(unit * 64 + l, values - 1);
        return static_cast<uint32_t>(min(first_row + q / kSB, last_row) - first_row) * static_cast<uint32_t>(kb_full) +
               min(q % kSB, blocks_here - 1);
    };
    auto offset_sx = [&](int i, int l, int blocks_here) { return 4 * scale_offset(usx0 + i * kWaves, l, kTM * kSB, m0, rows - 1, blocks_here); };
    auto offset_sw = [&](int i, int l, int blocks_here) { return 2 * scale_offset(usw0 + i * kWaves, l, kTN * kSB, n0, out_dim - 1, blocks_here); };
    uint32_t off_a[kPerA], off_b[kPerB], off_sx[kPerSx], off_sw[kPerSw];  // of a full stage
#pragma unroll
    for (int i = 0; i < kPerA; ++i) off_a[i] = offset_a(i, lane, kSB);
#pragma unroll
    for (int i = 0; i < kPerB; ++i) off_b[i] = offset_b(i, lane, kSB);
#pragma unroll
    for (int i = 0; i < kPerSx; ++i) off_sx[i] = offset_sx(i, lane, kSB);
#pragma unroll
    for (int i = 0; i < kPerSw; ++i) off_sw[i] = offset_sw(i, lane, kSB);
    // ... and of the last stage, kept where registers allow: the three issues past the end repeat it, and on a short share of K
    // that is most of them
    constexpr bool kKeepLast = kPerM * kPerN == 1;
    uint32_t last_a[kPerA], last_b[kPerB], last_sx[kPerSx], last_sw[kPerSw];
    if constexpr (kKeepLast) {
#pragma unroll
        for (int i = 0; i < kPerA; ++i) last_a[i] = offset_a(i, lane, last_blocks);
#pragma unroll
        for (int i = 0; i < kPerB; ++i) last_b[i] = offset_b(i, lane, last_blocks);
#pragma unroll
        for (int i = 0; i < kPerSx; ++i) last_sx[i] = offset_sx(i, lane, last_blocks);
#pragma unroll
        for (int i = 0; i < kPerSw; ++i) last_sw[i] = offset_sw(i, lane, last_blocks);
    }

    const uint32_t lds_base = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(gemm_lds)));
    constexpr int kOffB = S::kABytes, kOffSx = kOffB + S::kBBytes, kOffSw = kOffSx + S::kSxBytes;
    auto stage_ptr = [&](int slot) { return gemm_lds + slot * S::kStageBytes; };

    // Issues every load of stage `st` (clamped to the last stage) towards ring slot `slot`.
    auto issue_loads = [&](int slot, int st) {
        const int se = min(st, stages - 1);
        const uint32_t sp = lds_base + slot * S::kStageBytes;
        auto issue = [&](auto&& at_a, auto&& at_b, auto&& at_sx, auto&& at_sw) {
#pragma unroll
            for (int i = 0; i < kPerA; ++i) {
                const int u = ua0 + i * kWaves;
                if (u < kUnitsA) lds_load16(a_base + static_cast<size_t>(se) * (kSB * 32), at_a(i), sp + u * 1024);
            }
#pragma unroll
            for (int i = 0; i < kPerB; ++i) {
                const int u = ub0 + i * kWaves;
                if (u < kUnitsB) lds_load16(b_base + static_cast<size_t>(se) * (kSB * kQuantBytes), at_b(i), sp + kOffB + u * 1024);
            }
#pragma unroll
            for (int i = 0; i < kPerSx; ++i) {
                const int u = usx0 + i * kWaves;
                if (u < kUnitsSx) lds_load4(sx_base + static_cast<size_t>(se) * (kSB * 4), at_sx(i), sp + kOffSx + u * 256);
            }
#pragma unroll
            for (int i = 0; i < kPerSw; ++i) {
                const int u = usw0 + i * kWaves;
                if (u < kUnitsSw) lds_load2(sw_base + static_cast<size_t>(se) * (kSB * 2), at_sw(i), sp + kOffSw + u * 256);
            }
        };
        if (se == stages - 1 && last_blocks < kSB) {
            if constexpr (kKeepLast) {
                issue([&](int i) { return last_a[i]; }, [&](int i) { return last_b[i]; }, [&](int i) { return last_sx[i]; },
                      [&](int i) { return last_sw[i]; });
            } else {
                int l = lane;
                asm volatile("" : "+v"(l));
                issue([&](int i) { return offset_a(i, l, last_blocks); }, [&](int i) { return offset_b(i, l, last_blocks); },
                      [&](int i) { return offset_sx(i, l, last_blocks); }, [&](int i) { return offset_sw(i, l, last_blocks); });
            }
        } else {
            issue([&](int i) { return off_a[i]; }, [&](int i) { return off_b[i]; }, [&](int i) { return off_sx[i]; },
                  [&](int i) { return off_sw[i]; });
        }
    };

    // this lane's fragment positions (loop-invariant; only the ring slot changes).  Tile (i, j) of the wavefront lies 32 i rows
    // and 32 j columns on, a whole number of swizzle periods.
    const int row = wm * (32 * kPerM) + lj;  // activation row (A operand) inside the tile
    const int col = wn * (32 * kPerN) + lj;  // weight column (B operand) inside the tile
    const int b0 = 2 * ks;                   // first block of this wavefront's pair inside a stage
    const int frag_a0 = S::chunk_pos(row, 2 * b0 + lh), frag_a1 = S::chunk_pos(row, 2 * b0 + 2 + lh);
    const int frag_b0 = kQ4 ? col * kSB + nibble_slot(col, b0) : S::chunk_pos(col, 2 * b0 + lh);
    const int frag_b1 = kQ4 ? col * kSB + nibble_slot(col, b0 + 1) : S::chunk_pos(col, 2 * b0 + 2 + lh);
    const int frag_sx = row * kSB + b0 + lh;  // lanes 0-31 carry block b0, lanes 32-63 block b0 + 1
    const int frag_sw = col * kSB + b0 + lh;
    const int nibble_shift = lh ? 0 : 4;  // Q4_0: values 0..15 of a block are the low nibbles

    v16f acc[kPerM][kPerN] = {};

    // MFMA operands of one stage as read from LDS (scales still raw)
    struct Frag {
        int4 a0[kPerM], a1[kPerM], w0[kPerN], w1[kPerN];
        float ta[kPerM];
        uint32_t tb[kPerN];  // fp16 bits
    };
    auto read_frag = [&](int slot, Frag& f) {
        const unsigned char* sp = stage_ptr(slot);
        const int4* as = reinterpret_cast<const int4*>(sp);
        const int4* bs = reinterpret_cast<const int4*>(sp + kOffB);
        constexpr int kStepA = 32 * kCPR, kStepB = 32 * (kQ4 ? kSB : kCPR);
#pragma unroll
        for (int i = 0; i < kPerM; ++i) {
            f.a0[i] = as[frag_a0 + i * kStepA];
            f.a1[i] = as[frag_a1 + i * kStepA];
            f.ta[i] = reinterpret_cast<const float*>(sp + kOffSx)[frag_sx + i * 32 * kSB];
        }
#pragma unroll
        for (int j = 0; j < kPerN; ++j) {
            f.w0[j] = bs[frag_b0 + j * kStepB];
            f.w1[j] = bs[frag_b1 + j * kStepB];
            f.tb[j] = reinterpret_cast<const uint32_t*>(sp + kOffSw)[frag_sw + j * 32 * kSB];
        }
    };
    // Q4_0: sixteen times the value, nibble n as the byte 16 (n - 8); the scale takes the sixteenth back, so that every
    // product with the scale is the one of the plain value
    auto weight_bytes = [&](const int4& w) {
        if (!kQ4) return v4i{w.x, w.y, w.z, w.w};
        v4i v = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int i = 0; i < 4; ++i)
            v[i] = static_cast<int>(((static_cast<uint32_t>(v[i]) << nibble_shift) & 0xF0F0F0F0u) ^ 0x80808080u);
        return v;
    };
    // One pair of blocks, first block `blk` (absolute index): MFMAs of block blk and of
    // the scale products, vector-ALU work of block blk, then the same for block blk + 1 in
    // the registers block blk's dots have left (the two halves of a wavefront's work do
    // not overlap anyway, and 16 registers fewer are live).  `between` runs after the
    // last MFMA has been issued: the operand registers are free from there on.
    // `sixteenth`: the scale takes back the sixteen times of a Q4_0 weight; else the dot does.
    auto pair_step = [&](const Frag& f, int blk, auto sixteenth, auto&& between) {
        constexpr bool kSixteenth = kQ4 && decltype(sixteenth)::value;
        // blocks past the end of K (clamped re-reads of the last block) get scale 0
        const bool live = blk + lh < kb;
        const v16i zi = {};
        const v32f zf = {};
        v4i w0[kPerN], w1[kPerN], a0[kPerM], a1[kPerM];
        float tb[kPerN], ta[kPerM];
#pragma unroll
        for (int j = 0; j < kPerN; ++j) {
            w0[j] = weight_bytes(f.w0[j]);
            w1[j] = weight_bytes(f.w1[j]);
            tb[j] = live ? half_bits_to_f32(static_cast<uint16_t>(f.tb[j])) * (kSixteenth ? 0.0625f : 1.0f) : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < kPerM; ++i) {
            if (i == 0) {
#pragma unroll
                for (int i2 = 0; i2 < kPerM; ++i2) {
                    ta[i2] = live ? f.ta[i2] : 0.0f;
                    a0[i2] = v4i{f.a0[i2].x, f.a0[i2].y, f.a0[i2].z, f.a0[i2].w};
                    a1[i2] = v4i{f.a1[i2].x, f.a1[i2].y, f.a1[i2].z, f.a1[i2].w};
                }
            }
#pragma unroll
            for (int j = 0; j < kPerN; ++j) {
                const int n = n0 + col + 32 * j;
                v16f& sum = acc[i][j];
                v16i c = __builtin_amdgcn_mfma_i32_32x32x32_i8(a0[i], w0[j], zi, 0, 0, 0);
                v32f t = __builtin_amdgcn_mfma_f32_32x32x1f32(ta[i], tb[j], zf, 0, 0, 0);
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    if (kWriteDots && blk + h < kb) {
#pragma unroll
                        for (int v = 0; v < 16; ++v) {
                            const int m = m0 + row - lj + 32 * i + 8 * (v >> 2) + 4 * lh + (v & 3);
                            if (m < rows && n < out_dim) dots[(static_cast<size_t>(m) * out_dim + n) * kb_full + blk_begin + blk + h] = kQ4 ? c[v] >> 4 : c[v];
                        }
                    }
#pragma unroll
                    for (int v = 0; v < 16; ++v) sum[v] = __builtin_fmaf(t[16 * h + v], static_cast<float>(kQ4 && !kSixteenth ? c[v] >> 4 : c[v]), sum[v]);
                    if (h == 0) {
                        // compiler fence (no instruction): block blk is finished before block blk + 1 starts
                        asm volatile("" : "+v"(sum), "+v"(t) : : "memory");
                        c = __builtin_amdgcn_mfma_i32_32x32x32_i8(a1[i], w1[j], zi, 0, 0, 0);
                        if (i == kPerM - 1 && j == kPerN - 1) between();
                    }
                }
                asm volatile("" : "+v"(sum) : : "memory");
            }
        }
    };
    uint64_t stamp_begin = 0, stamp_loop = 0, stamp_tail = 0, ref_loop = 0, ref_tail = 0, stamp_wait = 0, stamp_barrier = 0;
    if (kStamps) stamp_begin = __builtin_readcyclecounter();
    // ---- prologue: stages 0 .. kRing-2 in flight, stages 0 and 1 landed, stage 0 in registers
    static_assert(kRing == 4, "the loop reads stage st + 1 while stage st + 2 lands and stage st + 3 is issued");
#pragma unroll
    for (int d = 0; d < kRing - 1; ++d) issue_loads(d, d);
    // Loads complete in order: a stage has landed for this wavefront once at most the
    // loads of the stages issued after it are outstanding.
    wait_for_stage();
    __syncthreads();
    {
        // The next stage's operands are read from LDS while this stage's arithmetic runs.
        Frag frag[2];
        read_frag(0, frag[0]);
        if (kStamps) {
            stamp_loop = __builtin_readcyclecounter();
            ref_loop = __builtin_amdgcn_s_memrealtime();
        }
        for (int st0 = 0; st0 < stages; st0 += kRing) {
#pragma unroll
            for (int d = 0; d < kRing; ++d) {
                const int st = st0 + d;  // may run past `stages` in the last round: zero scales, no effect
                // the slot of stage st - 1 is free (its fragments were read a stage ago): refill it, kRing - 1 stages ahead
                issue_loads((d + kRing - 1) % kRing, st + kRing - 1);
                // the next stage's operands landed before the last barrier
                pair_step(frag[d & 1], st * kSB + b0, std::true_type{}, [&]() { read_frag((d + 1) % kRing, frag[(d + 1) & 1]); });
                // stage st + 2 (issued two stages ago) has to be complete before the barrier:
                // the next stage reads its operands
                uint64_t s0 = 0, s1 = 0;
                if (kStamps) s0 = __builtin_readcyclecounter();
                wait_for_stage();
                if (kStamps) s1 = __builtin_readcyclecounter();
                __syncthreads();
                if (kStamps) {
                    stamp_wait += s1 - s0;
                    stamp_barrier += __builtin_readcyclecounter() - s1;
                }
            }
        }
    }
    if (kStamps) {
        stamp_tail = __builtin_readcyclecounter();
        ref_tail = __builtin_amdgcn_s_memrealtime();
    }

    // Loads still in flight target ring slots nobody reads again; they must land before
    // the ring is reused for the reduction (and before the workgroup ends).
    wait_vm_outstanding<0>();
    constexpr int kPerWave = kPerM * kPerN;
    if (kSplit > 1) {
        // ---- the kSplit partial sums of a tile meet in LDS
        __syncthreads();
        float* red = reinterpret_cast<float*>(gemm_lds);  // [ks][tile][tile of the wavefront][v][lane]
        auto store_sums = [&]() {
#pragma unroll
            for (int p = 0; p < kPerWave; ++p)
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    red[(((ks * S::kTiles + tile) * kPerWave + p) * 16 + v) * 64 + lane] = acc[p / kPerN][p % kPerN][v];
        };
        store_sums();
        // A sixteenth of a product of scales below 2^-122 is subnormal where the product may not be, and loses up to four of its
        // bits: 2^-150 times a dot of up to 2^19 a block, 2^-122 over 512 blocks, which no sum from 2^-96 on feels (2^-26 of it).
        // A wavefront with a smaller sum -- a zero is one -- looks its activation scales over and, if one is below 2^-98 (the
        // smallest fp16 scale is 2^-24; activations below 4e-28), forms its sums again from plain products, operands straight from
        // memory.  Error at 2^-116, 333 x 512 x 8200: 1.5e-5 without, 8.7e-7 with, as Q4_0 had unpacked.  Looking for such scales in
        // the K loop cost 1.1 % of all prefills, a branch there 4.5 %; this 0.1 %.
        if constexpr (kQ4 && !kWriteDots) {
            float least = __builtin_huge_valf();
#pragma unroll
            for (int p = 0; p < kPerWave; ++p)
#pragma unroll
                for (int v = 0; v < 16; ++v) least = __builtin_fminf(least, __builtin_fabsf(acc[p / kPerN][p % kPerN][v]));
            bool again = __ballot(least < 0x1p-96f) != 0;
            int l = lane;
            asm volatile("" : "+v"(l));  // addresses are formed anew: nothing of this takes registers in the loop above
            const int half = l >> 5;
            if (again) {
                bool small = false;
#pragma unroll 1
                for (int blk = b0; blk < kb; blk += kSB)
#pragma unroll
                    for (int i = 0; i < kPerM; ++i) {
                        const size_t r = min(m0 + wm * (32 * kPerM) + 32 * i + (l & 31), rows - 1) - m0;
                        small |= reinterpret_cast<const float*>(sx_base)[r * kb_full + min(blk + half, kb - 1)] < 0x1p-98f;
                    }
                again = __ballot(small) != 0;
            }
            if (again) {
#pragma unroll
                for (int p = 0; p < kPerWave; ++p) acc[p / kPerN][p % kPerN] = v16f{};
#pragma unroll 1
                for (int blk = b0; blk < kb; blk += kSB) {
                    const int blk1 = min(blk + 1, kb - 1), blk_h = half ? blk1 : blk;
                    Frag f;
#pragma unroll
                    for (int i = 0; i < kPerM; ++i) {
                        const size_t r = min(m0 + wm * (32 * kPerM) + 32 * i + (l & 31), rows - 1) - m0;
                        f.a0[i] = *reinterpret_cast<const int4*>(a_base + r * in_dim + blk * 32 + 16 * half);
                        f.a1[i] = *reinterpret_cast<const int4*>(a_base + r * in_dim + blk1 * 32 + 16 * half);
                        f.ta[i] = reinterpret_cast<const float*>(sx_base)[r * kb_full + blk_h];
                    }
#pragma unroll
                    for (int j = 0; j < kPerN; ++j) {
                        const size_t r = min(n0 + wn * (32 * kPerN) + 32 * j + (l & 31), out_dim - 1) - n0;
                        f.w0[j] = *reinterpret_cast<const int4*>(b_base + (r * kb_full + blk) * kQuantBytes);
                        f.w1[j] = *reinterpret_cast<const int4*>(b_base + (r * kb_full + blk1) * kQuantBytes);
                        f.tb[j] = reinterpret_cast<const uint16_t*>(sw_base)[r * kb_full + blk_h];
                    }
                    pair_step(f, blk, std::false_type{}, []() {});
                }
                store_sums();
            }
        }
        __syncthreads();
        if (dst == nullptr) return;
        constexpr int kPer = 16 / kSplit;
#pragma unroll
        for (int j = 0; j < kPer * kPerWave; ++j) {
            const int p = j / kPer, v = ks * kPer + j % kPer;
            float sum = red[((tile * kPerWave + p) * 16 + v) * 64 + lane];
#pragma unroll
            for (int k2 = 1; k2 < kSplit; ++k2) sum += red[(((k2 * S::kTiles + tile) * kPerWave + p) * 16 + v) * 64 + lane];
            const int m = m0 + row - lj + 32 * (p / kPerN) + 8 * (v >> 2) + 4 * lh + (v & 3), n = n0 + col + 32 * (p % kPerN);
            if (kStamps) {
                asm volatile("" : : "v"(sum));  // the sum is formed, not stored
            } else if (m < rows && n < out_dim) {
                const size_t at = static_cast<size_t>(m) * out_dim + n;
                if (kShareK && partial == nullptr) unsafeAtomicAdd(dst + at, sum);
                else if (kShareK) partial[static_cast<size_t>(blockIdx.y) * rows * out_dim + at] = sum;
                else dst[at] = finish_output(ep, n, at, sum);
            }
        }
        if (kStamps && lane == 0) {
            const uint64_t stamp_end = __builtin_readcyclecounter();
            int* out = reinterpret_cast<int*>(dst) + 8 * (static_cast<size_t>(blockIdx.x) * kWaves + wave);
            out[0] = static_cast<int>(stamp_loop - stamp_begin);
            out[1] = static_cast<int>(stamp_tail - stamp_loop);
            out[2] = static_cast<int>(stamp_wait);
            out[3] = static_cast<int>(stamp_barrier);
            out[4] = static_cast<int>(ref_tail - ref_loop);
            out[5] = static_cast<int>(stamp_end - stamp_tail);
            out[6] = 0;
            out[7] = static_cast<int>(__builtin_amdgcn_s_getreg((31 << 11) | 4));
        }
    } else {
        if (dst == nullptr) return;
#pragma unroll
        for (int j = 0; j < 16 * kPerWave; ++j) {
            const int p = j / 16, v = j % 16;
            const int m = m0 + row - lj + 32 * (p / kPerN) + 8 * (v >> 2) + 4 * lh + (v & 3), n = n0 + col + 32 * (p % kPerN);
            if (m < rows && n < out_dim) {
                const size_t at = static_cast<size_t>(m) * out_dim + n;
                const float sum = acc[p / kPerN][p % kPerN][v];
                if (kShareK && partial == nullptr) unsafeAtomicAdd(dst + at, sum);
                else if (kShareK) partial[static_cast<size_t>(blockIdx.y) * rows * out_dim + at] = sum;
                else dst[at] = finish_output(ep, n, at, sum);
            }
        }
    }
}

// A second matrix of the same shape on the same activations (gate and up; blockIdx.z = 1).
struct GemmSecond {
    float* dst = nullptr;
    const uint8_t* weight = nullptr;
    Epilogue ep;
};

template <int kType, int kWavesM, int kWavesN, int kSplit, bool kWriteDots, bool kShareK = false, bool kStamps = false, int kPerM = 1,
          int kPerN = 1>
__global__ __launch_bounds__(64 * kWavesM * kWavesN * kSplit) void gemm_i8_kernel(
    float* __restrict__ dst, int* __restrict__ dots, const int8_t* __restrict__ qx, const float* __restrict__ sx,
    const uint8_t* __restrict__ weight, int rows, int in_dim, int out_dim, int m_tiles, int n_tiles,
    int share_blocks, float* __restrict__ partial, Epilogue ep, GemmSecond second) {
    if (!kWriteDots && !kStamps && blockIdx.z != 0) {
        dst = second.dst;
        weight = second.weight;
        ep = second.ep;
    }
    gemm_i8_body<kType, kWavesM, kWavesN, kSplit, kWriteDots, kShareK, kStamps, kPerM, kPerN>(
        dst, dots, qx, sx, weight, rows, in_dim, out_dim, m_tiles, n_tiles, share_blocks, partial, ep);
}

namespace {

// Workgroups of a launch: an eighth of them for each XCD, whole columns of tiles and its part of the others.
long long gemm_grid(int m_tiles, int n_tiles) {
    return 8 * (static_cast<long long>(n_tiles >> 3) * m_tiles + ((n_tiles & 7) * static_cast<long long>(m_tiles) + 7) / 8);
}

// Grids that fill the compute units: f32 results of whole K only (no shares, no block dots).
template <int kType, int kWavesM, int kWavesN, int kSplit, int kPerM, int kPerN>
hipError_t launch_wide_tile(hipStream_t stream, float* dst, const int8_t* qx, const float* sx, const uint8_t* weight, int rows,
                            int in_dim, int out_dim, const Epilogue& ep, const GemmSecond& second) {
    using S = GemmShape<kWavesM, kWavesN, kSplit, kType == 2, kPerM, kPerN>;
    const int m_tiles = (rows + S::kTM - 1) / S::kTM, n_tiles = (out_dim + S::kTN - 1) / S::kTN;
    const long long grid = gemm_grid(m_tiles, n_tiles);
    if (grid > 0x7fffffffLL) return hipErrorInvalidValue;
    // per-lane load offsets are 32-bit, relative to the workgroup's first row
    if (static_cast<long long>(S::kTM > S::kTN ? S::kTM : S::kTN) * in_dim > 0x7fffffffLL) return hipErrorInvalidValue;
    auto kernel = gemm_i8_kernel<kType, kWavesM, kWavesN, kSplit, false, false, false, kPerM, kPerN>;
    static LdsLimit lds_limit;
    if (hipError_t e = allow_lds(kernel, S::kLdsBytes, &lds_limit); e != hipSuccess) return e;
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid), 1, second.dst ? 2 : 1), dim3(S::kThreads), S::kLdsBytes, stream, dst,
                       nullptr, qx, sx, weight, rows, in_dim, out_dim, m_tiles, n_tiles, in_dim / 32, nullptr, ep, second);
    return hipGetLastError();
}

template <int kType, int kWavesM, int kWavesN, int kSplit>
hipError_t launch_tile(hipStream_t stream, float* dst, int* dots, const int8_t* qx, const float* sx, const uint8_t* weight, int rows,
                       int in_dim, int out_dim, const Epilogue& ep, float* partial, const GemmSecond& second, bool cleared) {
    using S = GemmShape<kWavesM, kWavesN, kSplit, kType == 2>;
    const int m_tiles = (rows + S::kTM - 1) / S::kTM;
    const int n_tiles = (out_dim + S::kTN - 1) / S::kTN;
    const long long grid = gemm_grid(m_tiles, n_tiles);
    if (grid > 0x7fffffffLL) return hipErrorInvalidValue;
    // per-lane load offsets are 32-bit, relative to the workgroup's first row
    if (static_cast<long long>(S::kTM > S::kTN ? S::kTM : S::kTN) * in_dim > 0x7fffffffLL) return hipErrorInvalidValue;
    // K shares: only with room for their partial sums, never for the block-dot output
    const int kb = in_dim / 32;
    const int splits = partial != nullptr && dots == nullptr ? gemm_i8_splits(rows, in_dim, out_dim) : 1;
    const int share_blocks = (kb + splits - 1) / splits;
    const int shares = (kb + share_blocks - 1) / share_blocks;  // no empty share
    const bool add = cleared && shares == 2;
    float* sums = shares > 1 && !add ? partial : nullptr;
    dim3 g(static_cast<unsigned>(grid), static_cast<unsigned>(shares), second.dst && (shares == 1 || add) ? 2 : 1), b(S::kThreads);
    auto kernel_f32 = gemm_i8_kernel<kType, kWavesM, kWavesN, kSplit, false>;
    auto kernel_shares = gemm_i8_kernel<kType, kWavesM, kWavesN, kSplit, false, true>;
    auto kernel_dots = gemm_i8_kernel<kType, kWavesM, kWavesN, kSplit, true>;
    static LdsLimit lds_limit[3];
    if (hipError_t e = allow_lds(kernel_f32, S::kLdsBytes, &lds_limit[0]); e != hipSuccess) return e;
    if (hipError_t e = allow_lds(kernel_shares, S::kLdsBytes, &lds_limit[1]); e != hipSuccess) return e;
    if (hipError_t e = allow_lds(kernel_dots, S::kLdsBytes, &lds_limit[2]); e != hipSuccess) return e;
    if (dots)
        hipLaunchKernelGGL(kernel_dots, g, b, S::kLdsBytes, stream, dst, dots, qx, sx, weight, rows, in_dim, out_dim,
                           m_tiles, n_tiles, share_blocks, sums, ep, second);
    else if (shares > 1)
        hipLaunchKernelGGL(kernel_shares, g, b, S::kLdsBytes, stream, dst, dots, qx, sx, weight, rows, in_dim, out_dim,
                           m_tiles, n_tiles, share_blocks, sums, ep, second);
    else
        hipLaunchKernelGGL(kernel_f32, g, b, S::kLdsBytes, stream, dst, dots, qx, sx, weight, rows, in_dim, out_dim,
                           m_tiles, n_tiles, share_blocks, sums, ep, second);
    if (hipError_t e = hipGetLastError(); e != hipSuccess || shares == 1 || add) return e;
    if (hipError_t e = launch_splitk_reduce(stream, dst, sums, static_cast<size_t>(rows) * out_dim, out_dim, shares, ep);
        e != hipSuccess || second.dst == nullptr)
        return e;
    // (the partial sums have room for one matrix: the second follows)
    return launch_tile<kType, kWavesM, kWavesN, kSplit>(stream, second.dst, dots, qx, sx, second.weight, rows, in_dim, out_dim, second.ep,
                                                        partial, GemmSecond{}, false);
}

template <int kType>
hipError_t launch_type(hipStream_t stream, float* dst, int* dots, const int8_t* qx, const float* sx,
                       const uint8_t* weight, int rows, int in_dim, int out_dim, const Epilogue& ep, float* partial,
                       const GemmSecond& second, bool cleared) {
    // us of the whole op, M x K x N; "before" is the 64 x 128 tile by sixteen wavefronts that served these grids.
    static const char* env_tile = std::getenv("AFHIP_GEMM_TILE");  // tuning: "S", "X", "Y", "V" or "L", see below
    const char force = dots == nullptr && env_tile ? env_tile[0] : '\0';
    const long long units = gemv_compute_units();
    const long long grid = static_cast<long long>((rows + 63) / 64) * ((out_dim + 127) / 128);
    char tile = 'S';  // 32 x 64 outputs, K in four
    if (kType == 2) {
        // Q4_0.  "S" and "X" (64 x 128 outputs, two tiles a wavefront) both leave room for a second workgroup on a compute
        // unit.  "X" moves less per output but its few workgroups leave units idle on a small grid: 333 x 2048 x 5632
        // 26.9 / 35.0 (44.4 before), 333 x 4096 x 6144 51.5 / 60.4 (77.7), even at 11/8 of the units (512 x 2048 x 5632 37.4 / 37.0,
        // 45.7), 777 x 4096 x 4096 74 / 67 (84), 2048 x 4096 x 14336 498 / 398 (513).
        if (grid * 8 >= units * 11) tile = 'X';
    } else if (grid >= units) {
        // Q8_0, whose 64 x 128 stage does not fit twice: "Y" (64 x 64 outputs, two workgroups a unit) or "V" (128 x 128, two tiles
        // a wavefront, one workgroup a unit), whichever the rounds of an XCD's units make shorter (the two sum alike, so a pair, which
        // is one launch of twice the tiles, may choose for itself).  K = 4096: a round of "V" takes about 50 us, one workgroup more on
        // every unit about 15 of "Y".  Y / V: 333 x 4096 x 6144 47 / 52, 512 x 4096 x 4096 36 / 53, 512 x 4096 x 14336 103 / 103, 777 x
        // 4096 x 14336 168 / 192, 1024 x 4096 x 14336 210 / 201 (twice 406 / 361), 2048 x 4096 x 14336 445 / 366; over 110 single
        // calls and pairs (96 .. 2048 rows, K 1024 .. 14336, N 4096 .. 14336) at most 2 % above the better of the two but for
        // 2048 x 5120 x 5120 (202 / 184).
        constexpr long long kXcds = 8;
        auto rounds = [&](long long tile_rows, long long tile_cols) {
            const long long tiles = ((out_dim + tile_cols - 1) / tile_cols) * ((rows + tile_rows - 1) / tile_rows) * (second.dst ? 2 : 1);
            const long long units_of_xcd = units >= kXcds ? units / kXcds : 1;
            return ((tiles + kXcds - 1) / kXcds + units_of_xcd - 1) / units_of_xcd;
        };
        // 33 .. 64 rows have one row of tiles and fetch every weight once, so nothing is gained by a second workgroup that shares
        // them: "L" (64 x 128, one tile for each of sixteen wavefronts), Y / L: 64 x 4096 x 65536 85.4 / 77.9, 64 x 8192 x 32768
        // 79.5 / 71.3, a pair 180 / 160, 64 x 4096 x 128256 173 / 169, 40 x 4096 x 32768 34.4 / 35.0 (V, half empty, 105 at 8192).
        if (rows > 32 && rows <= 64) tile = 'L';
        else tile = 7 * rounds(128, 128) <= 2 * rounds(64, 64) ? 'V' : 'Y';
    }
    // Block dots, bound by writing them, take "S" on every grid: 512 x 4096 x 4096 Q4_0 4183 -> 3925, Q8_0 4273 -> 3447 from the tile
    // before, 300 x 2048 x 14336 4461 -> 2465 and 4671 -> 2229.
    if (force != '\0') tile = force;
    if (dots == nullptr) {
        if constexpr (kType == 2) {
            if (tile == 'X') return launch_wide_tile<2, 1, 4, 2, 2, 1>(stream, dst, qx, sx, weight, rows, in_dim, out_dim, ep, second);
        } else {
            if (tile == 'L') return launch_wide_tile<8, 2, 4, 2, 1, 1>(stream, dst, qx, sx, weight, rows, in_dim, out_dim, ep, second);
            if (tile == 'V') return launch_wide_tile<8, 2, 4, 2, 2, 1>(stream, dst, qx, sx, weight, rows, in_dim, out_dim, ep, second);
            if (tile == 'Y') return launch_wide_tile<8, 2, 2, 2, 1, 1>(stream, dst, qx, sx, weight, rows, in_dim, out_dim, ep, second);
        }
    }
    return launch_tile<kType, 1, 2, 4>(stream, dst, dots, qx, sx, weight, rows, in_dim, out_dim, ep, partial, second, cleared);
}

}  // namespace

// K shares of a GEMM launch: one when its 32 x 64 tiles fill the compute units anyway, else as
// many (a power of two, at most eight, at least 16 blocks = two stages each) as spread it over them.
int gemm_i8_splits(int rows, int in_dim, int out_dim) {
    const long workgroups = static_cast<long>((rows + 31) / 32) * ((out_dim + 63) / 64);
    const int kb = in_dim / 32;
    const int units = gemv_compute_units();
    int splits = 1;
    while (splits < 8 && workgroups * splits * 2 <= units && kb / (splits * 2) >= 16) splits *= 2;
    return splits;
}

bool gemm_i8_adds_to_result(int rows, int in_dim, int out_dim, const Epilogue& ep) {
    if (ep.bias != nullptr || ep.residual != nullptr || ep.activation != kActNone) return false;
    const int splits = gemm_i8_splits(rows, in_dim, out_dim), kb = in_dim / 32, share_blocks = (kb + splits - 1) / splits;
    return (kb + share_blocks - 1) / share_blocks == 2;
}

size_t gemm_i8_partial_bytes(size_t rows, size_t in_dim, size_t out_dim) {
    if (rows == 0 || rows > 0x7fffffff || in_dim > 0x7fffffff || out_dim > 0x7fffffff) return 0;
    const int splits = gemm_i8_splits(static_cast<int>(rows), static_cast<int>(in_dim), static_cast<int>(out_dim));
    return splits > 1 ? static_cast<size_t>(splits) * rows * out_dim * 4 : 0;
}

// dst = epilogue(sum over the K shares, in order): second kernel of a split-K launch.  first_in_dst: the first share's sums are in dst.  Four shares' values on their way at a
// time; a column is only worked out where an epilogue asks for it.  (us a call, against a serial loop over the shares with a
// remainder for every value: Q8_0 100 x 4096 x 1024 12.3 -> 11.7, Q4_0 32 x 14336 x 4096 19.4 -> 18.9.  Four values a thread did
// no better there and lost where the shares are large: Q4_K 32 x 4096 x 14336 22.2 -> 24.4, 64 x 4096 x 4096 17.0 -> 19.8.)
__global__ __launch_bounds__(256) void splitk_reduce_kernel(float* __restrict__ dst, const float* __restrict__ partial,
                                                            size_t count, int out_dim, int splits, Epilogue ep, int first_in_dst) {
    const bool plain = ep.bias == nullptr && ep.residual == nullptr && ep.activation == kActNone;
    for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < count;
         i += static_cast<size_t>(gridDim.x) * blockDim.x) {
        float total = 0.0f;
        if (first_in_dst) total += dst[i];
        for (int z0 = 0; z0 < splits; z0 += 4) {
            float part[4];
#pragma unroll
            for (int z = 0; z < 4; ++z) part[z] = partial[static_cast<size_t>(min(z0 + z, splits - 1)) * count + i];
#pragma unroll
            for (int z = 0; z < 4; ++z)
                if (z0 + z < splits) total += part[z];
        }
        dst[i] = plain ? total : finish_output(ep, static_cast<int>(i % out_dim), i, total);
    }
}

hipError_t launch_splitk_reduce(hipStream_t stream, float* dst, const float* partial, size_t count, int out_dim, int shares,
                                const Epilogue& ep, bool first_in_dst) {
    size_t grid = (count + 255) / 256;
    if (grid > 4096) grid = 4096;
    hipLaunchKernelGGL(splitk_reduce_kernel, dim3(static_cast<unsigned>(grid)), dim3(256), 0, stream, dst, partial, count, out_dim,
                       first_in_dst ? shares - 1 : shares, ep, first_in_dst ? 1 : 0);
    return hipGetLastError();
}

// Diagnostic: the Q8_0 64 x 64 tile kernel with its clock readings in place of results (see kStamps); dst has to
// hold 8 ints per wavefront of the grid, which it does whenever it holds the rows x out_dim results.
hipError_t launch_gemm_i8_stamps(hipStream_t stream, float* dst, const int8_t* qx, const float* sx, const uint8_t* weight,
                                 int rows, int in_dim, int out_dim) {
    using S = GemmShape<2, 2, 2, false>;
    const int m_tiles = (rows + S::kTM - 1) / S::kTM, n_tiles = (out_dim + S::kTN - 1) / S::kTN;
    const long long grid = gemm_grid(m_tiles, n_tiles);
    if (grid > 0x7fffffffLL || static_cast<long long>(S::kTN) * in_dim > 0x7fffffffLL) return hipErrorInvalidValue;
    if (static_cast<long long>(rows) * out_dim < grid * S::kWaves * 8) return hipErrorInvalidValue;
    auto kernel = gemm_i8_kernel<8, 2, 2, 2, false, false, true>;
    if (hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                           S::kLdsBytes);
        e != hipSuccess)
        return e;
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(S::kThreads), S::kLdsBytes, stream, dst, nullptr, qx, sx,
                       weight, rows, in_dim, out_dim, m_tiles, n_tiles, in_dim / 32, nullptr, Epilogue{}, GemmSecond{});
    return hipGetLastError();
}

hipError_t launch_gemm_i8(hipStream_t stream, int tensor_type, float* dst, int* dots, const int8_t* qx, const float* sx,
                          const uint8_t* weight_prepared, int rows, int in_dim, int out_dim, const Epilogue& ep, float* partial,
                          float* dst_b, const uint8_t* weight_b, const Epilogue& ep_b, bool cleared) {
    const GemmSecond second{dst_b, weight_b, ep_b};
    if (tensor_type == 2) return launch_type<2>(stream, dst, dots, qx, sx, weight_prepared, rows, in_dim, out_dim, ep, partial, second, cleared);
    return launch_type<8>(stream, dst, dots, qx, sx, weight_prepared, rows, in_dim, out_dim, ep, partial, second, cleared);
}

}  // namespace afhip
