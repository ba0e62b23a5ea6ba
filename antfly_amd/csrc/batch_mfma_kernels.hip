// Batched decode (a few to 64 rows, some Q4_0 matrices to 96) on CDNA4 int8 MFMA, activation-quantized route
// (ops/native_compute.zig:13304-13478 for Q8_0, :23427-23775 for Q4_0):
//   dot[m][n][b] = sum_i qx[m][32b+i] * qw[n][32b+i]            (int32, exact)
//   y[m][n]      = sum_b (sx[m][b] * sw[n][b]) * f32(dot[m][n][b])
//
// With so few rows the weights are read once and nothing is reused across workgroups, so the
// kernel is built like the decode GEMV, not like the prefill GEMM: single shot, no ring, no
// barrier inside the K loop.
//   * A workgroup of eight wavefronts owns 32 output columns and one share of K of at most
//     8 * kWaveBlocks blocks; wavefront w owns kWaveBlocks consecutive blocks of it (16 Q4_0 /
//     8 Q8_0: 8 KB of quant bytes).  It requests ALL its weight bytes at once with eight
//     global_load_lds_dwordx4 into its own 8 KB of LDS -- whole 128-byte lines, eight lanes per
//     line, chunk slots XOR-swizzled by the column so that the later fragment reads of 16
//     consecutive columns hit 16 different bank groups.  The LDS region is private to the
//     wavefront: no barrier before it is read.
//   * The activations were quantized beforehand into MFMA operand order
//     (quantize_fragments_kernel): the A fragment of 32 rows and one block is 1 KB contiguous,
//     lane l holding bytes [16 * (l / 32), +16) of row l % 32, so a wavefront takes it with one
//     coalesced 16-byte load per lane, straight into registers.  Rows past `rows` are zeros.
//   * Per block: v_mfma_i32_32x32x32_i8 gives the 32 x 32 int32 dots.  Q4_0 nibbles never become
//     separate bytes: with bit 3 flipped and placed in the high half of a byte a nibble n reads as
//     the int8 16 * (n - 8) (three operations per dword), so the MFMA yields 16 * dot exactly and
//     the weight scale is taken times 1/16 (a power of two: exact).  The scale products
//     sx[m][b] * sw[n][b] of two blocks come from one v_mfma_f32_32x32x1_2b_f32 (two rank-1
//     products, each entry the correctly rounded f32 product), then one convert and one fused
//     multiply-add per live result register and block.  Only the registers of rows that exist
//     are touched (kLive of 16: 4 for up to 8 rows, 8 for up to 16, ...).
//   * The eight wavefronts' sums meet in LDS in wavefront order (y is a fixed-order sum of eight
//     block-ascending partial sums); K shares of a long K go to partial[share][rows][out_dim]
//     and splitk_reduce_kernel adds them in share order.
//   * Up to eight rows (Q8_0: sixteen, as two groups of eight) on a K of whole 256-value runs take
//     batch8_mfma_kernel (further down): the 16x16x64 MFMA on two blocks at once, tiles of 8 .. 64
//     columns, weights requested two stages ahead instead of all at once, a long K in at most two
//     shares where that is possible.
//   * Nine to 64 rows take batch_groups_mfma_kernel (further down) on most shapes: this kernel's
//     arithmetic, 32 rows a workgroup whose operands stay in registers while it walks over groups
//     of columns, one workgroup per compute unit.
//   * Those that do not, and whose 64-column tiles times K shares make a grid of five eighths to
//     all of the compute units, take batch32_mfma_kernel (further down): this kernel's arithmetic,
//     staged weight requests, one workgroup per compute unit.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <type_traits>

#include "device_common.h"
#include "gemv_common.h"
#include "qmatmul_launch.h"

namespace afhip {

namespace {

typedef int bm_v4i __attribute__((ext_vector_type(4)));
typedef int bm_v16i __attribute__((ext_vector_type(16)));
typedef float bm_v16f __attribute__((ext_vector_type(16)));
typedef float bm_v32f __attribute__((ext_vector_type(32)));

constexpr int kBmWaves = 8;
constexpr int kBmThreads = 64 * kBmWaves;
constexpr int kBmWaveBytes = 8192;  // quant bytes one wavefront owns: 32 columns x kWaveBlocks blocks
constexpr int kBmLdsBytes = kBmWaves * kBmWaveBytes;

template <int kType>
struct BmFormat {
    static constexpr int kQuantBytes = kType == 2 ? 16 : 32;
    static constexpr int kWaveBlocks = kBmWaveBytes / (32 * kQuantBytes);  // 16 (Q4_0) / 8 (Q8_0)
    static constexpr int kShareBlocks = kBmWaves * kWaveBlocks;            // 128 / 64
};

// Column-group kernel.  A stage is the weights and scales of 32 columns and kStageBlocks blocks, 5 KB; kHalves stages are a wavefront's part of
// the workgroup's share of K, which kParts wavefronts share out (the others take other columns).  LDS: a ring of stages for each
// wavefront, the room where the sums meet, and two counters.
template <int kType, int kLive, int kHalves, int kParts>
struct BatchGroups {
    static constexpr int kStageBlocks = kType == 2 ? 8 : 4;
    static constexpr int kRun = kParts * kStageBlocks;  // consecutive blocks that the wavefronts' stages share out
    static constexpr int kSlots = 3, kSlotBytes = 5120;
    static constexpr int kGroupCols = 32 * (kBmWaves / kParts);  // columns the workgroup works on at a time
    static constexpr int kSumsAt = kBmWaves * kSlots * kSlotBytes, kCountersAt = kSumsAt + kBmWaves * kLive * 256;
    static constexpr int kLdsBytes = kCountersAt + 16;
    static constexpr int kSets = kHalves == 4 ? 1 : 2;  // register sets of MFMA results
    static_assert(kLdsBytes <= 160 * 1024, "LDS");
};

// One 64-lane load from global memory straight into LDS: lane l's 16 bytes at base + voff land
// at lds_addr + 16 * l.  Inline assembly: the compiler does not track these loads, which is why
// the kernel waits for them by hand before anything reads the LDS region.
__device__ __forceinline__ void bm_lds_load16(const void* base, uint32_t voff, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" : : "s"(lds_addr), "v"(voff), "s"(base) : "memory", "m0");
}

// the same where other workgroups are about to read the bytes too (no streaming hint)
__device__ __forceinline__ void bm_lds_load16_kept(const void* base, uint32_t voff, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds_addr), "v"(voff), "s"(base) : "memory", "m0");
}

extern __shared__ __align__(1024) unsigned char bm_lds[];  // (operand addresses inside rows of 128 bytes are formed by XOR)

// the second matrix of a pair launch (grid.z == 2)
struct BmSecond {
    float* dst;
    const uint8_t* weight;
    Epilogue ep;
};

// Program-order fence for the compiler (no instruction): what was computed into `a` so far is
// finished before anything behind the fence starts.  Keeps the scheduler from running the MFMAs of
// several blocks ahead and holding all their results in registers.
__device__ __forceinline__ void fence_registers(float (&a)[4]) {
    asm volatile("" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]));
}
__device__ __forceinline__ void fence_registers(float (&a)[8]) {
    asm volatile("" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4]), "+v"(a[5]), "+v"(a[6]), "+v"(a[7]));
}
__device__ __forceinline__ void fence_registers(float (&a)[12]) {
    asm volatile("" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4]), "+v"(a[5]), "+v"(a[6]), "+v"(a[7]), "+v"(a[8]),
                 "+v"(a[9]), "+v"(a[10]), "+v"(a[11]));
}
__device__ __forceinline__ void fence_registers(float (&a)[16]) {
    asm volatile("" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4]), "+v"(a[5]), "+v"(a[6]), "+v"(a[7]), "+v"(a[8]),
                 "+v"(a[9]), "+v"(a[10]), "+v"(a[11]), "+v"(a[12]), "+v"(a[13]), "+v"(a[14]), "+v"(a[15]));
}

}  // namespace

// X f32 [rows][in_dim] -> qa: [row tile][block][64 lanes][16 bytes] (lane = 32 * half + row % 32:
// bytes [16 * half, +16) of the block's 32 int8), sa: f32 [block][32 * row_tiles].  Rows past
// `rows` get zeros and scale 0.  Eight lanes per block as in quantize_activations_kernel
// (ops/native_compute.zig:11998-12028): same scale, reciprocal and rounding, bit for bit.
// kByteOrder (Q4_0 operands of batch32_mfma_kernel): within a block the lane half h holds the dwords
// x[8h..8h+3], x[16+8h..+3], x[8h+4..8h+7], x[16+8h+4..+7] instead of x[16h..16h+15] -- the values whose
// nibbles share the bytes [8 h, 8 h + 8) of the weight block, so that a lane unpacks whole bytes.
// zero_a (and zero_b): result arrays of zero_count floats that the matmul launch behind this one adds its two K shares'
// sums to; cleared here, by the launch that has to run first anyway.
template <bool kByteOrder>
__global__ __launch_bounds__(256) void quantize_fragments_kernel(const float* __restrict__ x, int rows, int in_dim, int row_tiles,
                                                                  uint32_t* __restrict__ qa, float* __restrict__ sa,
                                                                  float* __restrict__ zero_a, float* __restrict__ zero_b, size_t zero_count) {
    // blockIdx.y is the (padded) row, a thread four values of it: nothing is divided (64-bit quotients of a flat index
    // stood before the load), and the load leaves before the results are cleared.  What is left is the launch and one trip to
    // memory: 32 x 4096 4.0 us as kernel time, a pass of 32 rows through four matrices' calls 566.7 -> 557.8 us.
    const int units_per_row = in_dim >> 2, kb = in_dim >> 5, padded = row_tiles * 32;
    const int r = blockIdx.y, c4 = blockIdx.x * blockDim.x + threadIdx.x;
    const bool mine = c4 < units_per_row;
    float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (mine && r < rows) v = reinterpret_cast<const float4*>(x)[static_cast<size_t>(r) * units_per_row + c4];
    if (zero_a != nullptr) {
        const size_t first = (static_cast<size_t>(r) * gridDim.x + blockIdx.x) * blockDim.x + threadIdx.x;
        for (size_t i = first; i < zero_count; i += static_cast<size_t>(gridDim.x) * gridDim.y * blockDim.x) {
            zero_a[i] = 0.0f;
            if (zero_b != nullptr) zero_b[i] = 0.0f;
        }
    }
    if (!mine) return;  // (whole groups of eight lanes: units_per_row is a multiple of eight)
    const int b = c4 >> 3, j = c4 & 7;
    float m = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
    m = max_over_8(m);
    const float s = act_scale(m);
    const float inv = m == 0.0f ? 0.0f : 1.0f / s;
    const int q0 = act_quant(v.x, inv), q1 = act_quant(v.y, inv);
    const int q2 = act_quant(v.z, inv), q3 = act_quant(v.w, inv);
    const int half = kByteOrder ? (j >> 1) & 1 : j >> 2, dw = kByteOrder ? 2 * (j & 1) + (j >> 2) : j & 3;
    const size_t lane_entry = (static_cast<size_t>(r >> 5) * kb + b) * 64 + half * 32 + (r & 31);
    qa[lane_entry * 4 + dw] = (q0 & 0xFF) | ((q1 & 0xFF) << 8) | ((q2 & 0xFF) << 16) | ((q3 & 0xFF) << 24);
    if (j == 0) sa[static_cast<size_t>(b) * padded + r] = r < rows ? s : 0.0f;
}

template <int kType, int kRowTiles, int kLive>
__global__ __launch_bounds__(kBmThreads, kRowTiles == 1 ? 4 : 2) void batch_mfma_kernel(float* __restrict__ dst_a, float* __restrict__ partial_a,
                                                                  const uint32_t* __restrict__ qa, const float* __restrict__ sa,
                                                                  const uint8_t* __restrict__ weight_a, int rows, int in_dim,
                                                                  int out_dim, int share_blocks, Epilogue ep_a, BmSecond second, int accumulate) {
    using F = BmFormat<kType>;
    // blockIdx.z == 1: the second matrix of a pair (same X, same shape)
    const bool is_b = blockIdx.z != 0;
    float* dst = is_b ? second.dst : dst_a;
    const uint8_t* weight = is_b ? second.weight : weight_a;
    const Epilogue ep = is_b ? second.ep : ep_a;
    float* partial = partial_a == nullptr ? nullptr : partial_a + (is_b ? static_cast<size_t>(gridDim.y) * rows * out_dim : 0);
    constexpr int kQB = F::kQuantBytes, kWB = F::kWaveBlocks, kPairs = kWB / 2;
    constexpr int kAhead = kRowTiles == 1 ? 8 : (kRowTiles == 2 ? 4 : 2);  // A fragments in registers per row tile
    static_assert(kWB % kAhead == 0 && kAhead % 2 == 0, "fragment ring");
    const int kb_full = in_dim >> 5;
    const int padded = kRowTiles * 32;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lj = lane & 31, lh = lane >> 5;
    const int n0 = blockIdx.x * 32;
    // blocks of this wavefront: [blk0, blk0 + nb), nb in 0..kWB; indices past the end are clamped
    // to the last valid block for every load and their scale products are forced to zero
    const int share_begin = static_cast<int>(blockIdx.y) * share_blocks;
    const int share_end = min(share_begin + share_blocks, kb_full);
    const int blk0 = share_begin + wave * kWB;
    const int nb = max(0, min(kWB, share_end - blk0));
    const int last = blk0 + max(nb, 1) - 1 < kb_full ? blk0 + max(nb, 1) - 1 : kb_full - 1;  // a valid block whatever nb is
    auto clamp_blk = [&](int j) { return min(blk0 + j, last); };

    const size_t blocks_total = static_cast<size_t>(out_dim) * kb_full;
    const uint32_t lds_wave = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(bm_lds))) + wave * kBmWaveBytes;

    // ---- 1. loads.  Order matters: a wavefront's loads complete in the order they were issued,
    // and every wavefront of the grid issues at once, so memory serves all first halves before all
    // second halves.  First half of the weights (LDS-direct, four 1 KB loads), then what the first
    // half of the K loop needs (A fragments, scales), then values only the second half needs, then
    // the second half of the weights.  The compiler counts only its own loads when it waits for
    // one: with at least four of its loads issued behind everything the first half needs, its
    // wait lets exactly the four youngest loads -- the second half of the weights -- stay in flight
    // while the first half is computed.  (Its count can only be too strict, never too lax: loads
    // it does not know of only add to the number outstanding.)
    auto issue_weights = [&](int hb) {
        const uint8_t* wbase = weight + static_cast<size_t>(n0) * kb_full * kQB;
        const int c8 = lane >> 3, slot = lane & 7;
#pragma unroll
        for (int cg = 0; cg < 4; ++cg) {
            const int c = 8 * cg + c8;
            const int chunk = slot ^ ((c >> 1) & 7);
            const int cc = min(n0 + c, out_dim - 1) - n0;
            uint32_t off;
            if (kType == 2) {
                off = (static_cast<uint32_t>(cc) * kb_full + clamp_blk(8 * hb + chunk)) * 16u;
            } else {
                off = (static_cast<uint32_t>(cc) * kb_full + clamp_blk(4 * hb + (chunk >> 1))) * 32u + (chunk & 1) * 16u;
            }
            bm_lds_load16(wbase, off, lds_wave + (hb * 4 + cg) * 1024);
        }
    };
    issue_weights(0);

    // Rows that exist live in the first 2 * kLive lanes of each half of a fragment.  The other
    // lanes' values only reach result rows nobody reads, so they repeat a live lane's address
    // instead of fetching their own zeros: a fragment load then touches 2 * kLive * 32 bytes.
    const int lr = lj % (2 * kLive);
    const int alane = lh * 32 + lr;
    // The fragment and scale loads below have to be issued BEHIND the weight requests above (the wait for the first
    // fragment is what says that the first half of the weights has landed).  Their addresses are taken from pointers
    // that pass through a statement ordered after those requests, so no scheduling can lift them above.
    const uint32_t* qa_behind = qa;
    const float* sa_behind = sa;
    asm volatile("" : "+s"(qa_behind), "+s"(sa_behind) : : "memory");
    const bm_v4i* qa4 = reinterpret_cast<const bm_v4i*>(qa_behind);
    auto load_a = [&](int rt, int j) { return qa4[(static_cast<size_t>(rt) * kb_full + clamp_blk(j)) * 64 + alane]; };
    auto load_ta = [&](int rt, int p) { return sa_behind[static_cast<size_t>(clamp_blk(2 * p + lh)) * padded + rt * 32 + lr]; };
    bm_v4i afrag[kRowTiles][kAhead];
    float ta[kRowTiles][kPairs];  // activation scale of row lj, block 2p + lh
    constexpr int kHalfBlocks = kWB / 2, kHalfPairs = kPairs / 2;
#pragma unroll
    for (int rt = 0; rt < kRowTiles; ++rt)
#pragma unroll
        for (int j = 0; j < kAhead; ++j)
            if (j < kHalfBlocks) afrag[rt][j] = load_a(rt, j);
    // Weight scales, fp16 in block order: pair p needs block 2p + lh = half lh of dword p of the
    // wavefront's run of scales.  With rows of whole 16-byte runs (in_dim a multiple of 256) that is
    // one or two 16-byte loads per lane; otherwise one 2-byte load per pair.
    uint32_t tb_word[kPairs];
    {
        const int cc = min(n0 + lj, out_dim - 1);
        const uint16_t* sw = reinterpret_cast<const uint16_t*>(weight + blocks_total * kQB) + static_cast<size_t>(cc) * kb_full;
        if ((kb_full & 7) == 0) {
            // (reads past the wavefront's last valid block stay inside the scale regions; those pairs count for nothing)
            const uint4* run = reinterpret_cast<const uint4*>(sw + min(blk0, kb_full - 8));
#pragma unroll
            for (int q = 0; q < kPairs / 4; ++q) {
                const uint4 v = run[q];
                tb_word[4 * q] = v.x;
                tb_word[4 * q + 1] = v.y;
                tb_word[4 * q + 2] = v.z;
                tb_word[4 * q + 3] = v.w;
            }
        } else {
#pragma unroll
            for (int p = 0; p < kPairs; ++p) tb_word[p] = static_cast<uint32_t>(sw[clamp_blk(2 * p + lh)]) * 0x10001u;
        }
    }
#pragma unroll
    for (int rt = 0; rt < kRowTiles; ++rt)
#pragma unroll
        for (int p = 0; p < kHalfPairs; ++p) ta[rt][p] = load_ta(rt, p);
    // ... and what only the second half needs (at least four loads)
#pragma unroll
    for (int rt = 0; rt < kRowTiles; ++rt)
#pragma unroll
        for (int j = kHalfBlocks; j < kAhead; ++j) afrag[rt][j] = load_a(rt, j);
#pragma unroll
    for (int rt = 0; rt < kRowTiles; ++rt)
#pragma unroll
        for (int p = kHalfPairs; p < kPairs; ++p) ta[rt][p] = load_ta(rt, p);
    // With a fragment ring shorter than half the blocks, fragments of the first half are still
    // requested inside the loop.  Loads complete in order: requested behind the second half of the
    // weights they would arrive behind it and the first half would be computed only after the
    // whole stream.  There the second half of the weights is requested from inside the loop, right
    // after the loads that complete the first half's fragments and the first ones of the second half's
    // (which are the loads the compiler's wait may retire early instead of the weights).
    constexpr int kIssuePair = kAhead >= kHalfBlocks ? -1 : (kHalfBlocks - kAhead) / 2;
    static_assert(kIssuePair >= 0 || kRowTiles * ((kAhead > kHalfBlocks ? kAhead - kHalfBlocks : 0) + kPairs - kHalfPairs) >= 4 || kType == 8,
                  "cover loads");
    if (kIssuePair < 0) issue_weights(1);

    // The first A fragment was requested behind the first half of the weights: once it is here, so
    // are they.  (The statement makes the compiler wait for that fragment and keeps the LDS reads
    // below it.)
    asm volatile("" : "+v"(afrag[0][0]) : : "memory");

    // this lane's fragment position inside a 1 KB load unit: column lj, chunk slot swizzled by the column
    const int frag_unit = lj >> 3;  // cg
    const int frag_row = (lj & 7) * 8, frag_swz = (lj >> 1) & 7;
    const uint4* wlds = reinterpret_cast<const uint4*>(bm_lds + wave * kBmWaveBytes);
    auto read_b = [&](int j) {
        int li, chunk;
        if (kType == 2) {
            li = (j >> 3) * 4 + frag_unit;
            chunk = j & 7;
        } else {
            li = (j >> 2) * 4 + frag_unit;
            chunk = (j & 3) * 2 + lh;
        }
        const uint4 w = wlds[li * 64 + frag_row + (chunk ^ frag_swz)];
        bm_v4i b;
        if (kType == 2) {
            // A nibble n stands for n - 8.  As the HIGH nibble of a byte, n ^ 8 reads as the int8
            // 16 * (n - 8): flip bit 3 of every nibble, move the wanted nibbles (low = values 0..15
            // = k half 0, high = values 16..31) to the high positions and clear the others.  The
            // dots come out multiplied by 16, which the weight scale takes back (exactly).
            const uint32_t sh = 4u * (1 - lh);
            b = bm_v4i{static_cast<int>(((w.x ^ 0x88888888u) << sh) & 0xF0F0F0F0u), static_cast<int>(((w.y ^ 0x88888888u) << sh) & 0xF0F0F0F0u),
                       static_cast<int>(((w.z ^ 0x88888888u) << sh) & 0xF0F0F0F0u), static_cast<int>(((w.w ^ 0x88888888u) << sh) & 0xF0F0F0F0u)};
        } else {
            b = bm_v4i{static_cast<int>(w.x), static_cast<int>(w.y), static_cast<int>(w.z), static_cast<int>(w.w)};
        }
        return b;
    };

    float acc[kRowTiles][kLive];
#pragma unroll
    for (int rt = 0; rt < kRowTiles; ++rt)
#pragma unroll
        for (int v = 0; v < kLive; ++v) acc[rt][v] = 0.0f;

    // ---- 3. the K loop of this wavefront: pairs of blocks, no barrier
    if (nb > 0) {
        const bm_v16i zi = {};
        const bm_v32f zf = {};
#pragma unroll
        for (int p = 0; p < kPairs; ++p) {
            // the second half of the weights (and every fragment requested so far) has to be here
            if (p == kHalfPairs) asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
            const bool live_blk = 2 * p + lh < nb;  // a clamped re-read of the last block counts for nothing
            const float tb = live_blk ? half_bits_to_f32(static_cast<uint16_t>(tb_word[p] >> (16 * lh))) * (kType == 2 ? 0.0625f : 1.0f) : 0.0f;
#pragma unroll
            for (int rt = 0; rt < kRowTiles; ++rt) {
                const bm_v4i a0 = afrag[rt][(2 * p) % kAhead], a1 = afrag[rt][(2 * p + 1) % kAhead];
                const bm_v32f t = __builtin_amdgcn_mfma_f32_32x32x1f32(live_blk ? ta[rt][p] : 0.0f, tb, zf, 0, 0, 0);
                // one block after the other: the second block's dots take the registers the first one's have left
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const bm_v4i a = h == 0 ? a0 : a1, b = read_b(2 * p + h);
                    bm_v16i c = zi;
                    c = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
#pragma unroll
                    for (int v = 0; v < kLive; ++v) acc[rt][v] = __builtin_fmaf(t[16 * h + v], static_cast<float>(c[v]), acc[rt][v]);
                    fence_registers(acc[rt]);
                }
                // the fragments of blocks 2p, 2p + 1 are consumed: fetch the ones kAhead blocks on
                if (2 * p + kAhead < kWB) {
                    afrag[rt][(2 * p) % kAhead] = load_a(rt, 2 * p + kAhead);
                    afrag[rt][(2 * p + 1) % kAhead] = load_a(rt, 2 * p + 1 + kAhead);
                }
            }
            if (p == kIssuePair) issue_weights(1);
        }
    } else {
        asm volatile("s_waitcnt vmcnt(0)" : : : "memory");  // its weight loads still write LDS, which the sums are about to reuse
    }

    // ---- 4. the wavefronts' sums meet in LDS, one row tile at a time (the weight regions are dead
    // after the first barrier; 8 wavefronts x 16 registers x 64 lanes of floats are half the LDS)
    float* red = reinterpret_cast<float*>(bm_lds);  // [wave][v][lane]
    constexpr int kItems = kLive * 64;
#pragma unroll
    for (int rt = 0; rt < kRowTiles; ++rt) {
        __syncthreads();
#pragma unroll
        for (int v = 0; v < kLive; ++v) red[(wave * kLive + v) * 64 + lane] = acc[rt][v];
        __syncthreads();
        for (int i = tid; i < kItems; i += kBmThreads) {
            // the first four wavefronts' sums, the last four's, then both: what two K shares of four wavefronts each
            // add up to (launch_batch_mfma splits a single share there where that is faster, to the same bits)
            float half[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                half[h] = red[(kBmWaves / 2) * h * kItems + i];
#pragma unroll
                for (int w = 1; w < kBmWaves / 2; ++w) half[h] += red[((kBmWaves / 2) * h + w) * kItems + i];
            }
            const float sum = half[0] + half[1];
            const int l = i & 63, v = i >> 6;
            const int m = rt * 32 + 8 * (v >> 2) + 4 * (l >> 5) + (v & 3);
            const int n = n0 + (l & 31);
            if (m < rows && n < out_dim) {
                const size_t at = static_cast<size_t>(m) * out_dim + n;
                if (partial != nullptr) partial[static_cast<size_t>(blockIdx.y) * rows * out_dim + at] = sum;
                else if (accumulate) unsafeAtomicAdd(dst + at, sum);  // (two K shares, no epilogue, the result cleared beforehand: see batch8_mfma_kernel)
                else dst[at] = finish_output(ep, n, at, sum);
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Up to eight rows: v_mfma_i32_16x16x64_i8 on two blocks at once.
//
// The instruction multiplies 16 rows x 64 k by 64 k x 16 columns, twice the k of one block, and two
// blocks cannot share an int32 sum (their scales differ).  With at most eight rows the A operand has
// room to keep them apart: A row 8 * s + r (s = 0, 1) is row r of X with the bytes of block 2P + s
// in its k half s and ZEROS in the other half, the B operand is the weights of block 2P in k half 0
// and of block 2P + 1 in k half 1.  Result row 8 * s + r is then exactly the dot of row r with block
// 2P + s: one instruction of a quarter of the 32x32x32 one's work gives the dots of two blocks for
// 16 columns, and all four of its result registers are live (lane l: column l % 16, lane group
// g = l / 16: block 2P + g / 2, rows 4 * (g % 2) + v).
//
// The scale products sx[row][block] * sw[column][block] come in the same register layout from one
// v_mfma_f32_16x16x4_f32: A row 8 * s + r carries sx of (r, block 2P + s) at k = s and zeros
// elsewhere, B row k carries sw of block 2P + k (k < 2): every entry is one product plus zeros,
// the correctly rounded f32 product.  What is left for the vector unit per MFMA is the nibble
// unpacking, four conversions and four fused multiply-adds; the LDS sees one read.  (Fetching the
// row scales per result register through the lane-exchange crossbar instead made the LDS pipe, one
// per compute unit, the bottleneck.)
//
// The smaller column granule also makes four load stages of a wavefront's eight 1 KB units instead
// of two: (blocks first half, columns 0..15), (first half, 16..31), (second half, 0..15), (second
// half, 16..31), each waited for by itself, so that a quarter of the arithmetic, not half, is left
// when the last byte arrives.

// X f32 [rows <= 8][in_dim] -> qa8: [pair P][32 entries][16 bytes], sa8: f32 [pair][16].
// Entry 16 * s + 8 * h + r holds sixteen int8 of row r, block 2P + s, k half h, in the k order of the
// weight operand (below): what lane 16 * (2 s + h) + 8 * s + r of the A operand needs; the other lanes
// of the operand are zeros and are not stored.  Slot 8 * s + r of sa8 is the block's scale.  Rows
// past `rows` and a block past the last one are zeros with scale 0.  Same scale, reciprocal and
// rounding as quantize_fragments_kernel.
// k order, lane half h = g % 2:  Q8_0: values [16 h, 16 h + 16).  Q4_0: dwords x[8h..8h+3],
// x[16+8h..+3], x[8h+4..8h+7], x[16+8h+4..+7] -- the low and the high nibbles of bytes [8 h, 8 h + 8) of
// the block, dword by dword, so that one lane unpacks whole bytes.
// zero_a (and zero_b): result arrays of zero_count floats that the matmul launch behind this one adds its two K shares'
// sums to; cleared here, by the launch that has to run first anyway.
template <int kType>
__global__ __launch_bounds__(256) void quantize_fragments8_kernel(const float* __restrict__ x, int rows, int in_dim,
                                                                   uint32_t* __restrict__ qa8, float* __restrict__ sa8,
                                                                   float* __restrict__ zero_a, float* __restrict__ zero_b, int zero_count) {
    const int kb = in_dim >> 5, slots = ((kb + 1) >> 1) * 2;  // block slots: whole pairs
    // blockIdx.y: the row of a group of eight and the group (rows 8 .. 15 of X make a second set of fragments and scales behind the
    // first); a thread takes four values of the row, so nothing is divided, and its load leaves before the results are cleared:
    // 5 x 4096 2.8 us as kernel time, a pass of five rows through four matrices' calls 1537 -> 1515 us.
    const int group = blockIdx.y >> 3, r = blockIdx.y & 7;
    const int u = blockIdx.x * blockDim.x + threadIdx.x, j = u & 7, bs = u >> 3;
    const bool real = 8 * group + r < rows && bs < kb;
    float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (real) v = reinterpret_cast<const float4*>(x)[(static_cast<size_t>(blockIdx.y) * in_dim >> 2) + u];
    if (zero_a != nullptr) {
        for (int i = (blockIdx.y * gridDim.x + blockIdx.x) * blockDim.x + threadIdx.x; i < zero_count; i += gridDim.x * gridDim.y * blockDim.x) {
            zero_a[i] = 0.0f;
            if (zero_b != nullptr) zero_b[i] = 0.0f;
        }
    }
    if (bs >= slots) return;  // (whole groups of eight lanes)
    qa8 += static_cast<size_t>(group) * (slots / 2) * 128;
    sa8 += static_cast<size_t>(group) * (slots / 2) * 16;
    float m = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
    m = max_over_8(m);
    const float s = act_scale(m);
    const float inv = m == 0.0f ? 0.0f : 1.0f / s;
    const int q0 = act_quant(v.x, inv), q1 = act_quant(v.y, inv);
    const int q2 = act_quant(v.z, inv), q3 = act_quant(v.w, inv);
    const int pair = bs >> 1, hs = bs & 1, i = hs * 8 + r;
    // values [4 j, 4 j + 4) of the block: which 16-byte half, which dword of it
    const int h2 = kType == 2 ? (j >> 1) & 1 : j >> 2;
    const int dw = kType == 2 ? 2 * (j & 1) + (j >> 2) : j & 3;
    // entry 16 * s + 8 * h2 + r of the pair: sixteen bytes
    qa8[static_cast<size_t>(pair) * 128 + (16 * hs + 8 * h2 + r) * 4 + dw] = (q0 & 0xFF) | ((q1 & 0xFF) << 8) | ((q2 & 0xFF) << 16) | ((q3 & 0xFF) << 24);
    if (j == 0) sa8[pair * 16 + i] = real ? s : 0.0f;
}

// kStamps (bench.py --probe timeline8): the same code, but instead of results every wavefront stores eight readings of the
// 100 MHz clock at dst_a[8 * (8 * workgroup + wavefront)]: [0] entry, [1] .. [4] the first four stages' bytes there, [5] the last
// stage's, [6] K loop done, [7] after the workgroup's reduction.
// kFullCols: a workgroup takes all 16 kCG columns (`cols` is not looked at).
// accumulate: the launch has exactly two K shares and no epilogue; the result array has been cleared (by the quantizer's
// launch) and each share adds its sums with a float atomic -- no partial sums in scratch, no reduce launch behind.
// kHalves: stage rounds of a wavefront -- it owns kHalves runs of eight (Q4_0; four Q8_0) consecutive blocks, and a K share
// is 8 * kHalves of them: a longer K makes fewer shares (K = 14336 of Q4_0: two of 224 blocks at kHalves = 4 instead of
// four of 112), and two shares need no reduce launch.
// kGroups: groups of eight rows (one or two: nine to sixteen rows run every step's two MFMAs once per group on the same
// weight operand; the second group's fragments and row scales lie behind the first's).
// kQuantize: qa8 is X itself, f32 [rows][in_dim] (sa8 is not looked at), and every wavefront quantizes the values of its own
// blocks before the first stage: no quantizer launch.  The wavefronts of a workgroup own different blocks, so within one
// nothing is converted twice; every workgroup converts all of its K share, while its first weights travel.
template <int kType, int kCG, bool kStamps = false, bool kFullCols = false, int kHalves = 2, int kGroups = 1, bool kQuantize = false>
__global__ __launch_bounds__(kBmThreads, kGroups > 1 ? 2 : 4) void batch8_mfma_kernel(float* __restrict__ dst_a, float* __restrict__ partial_a,
                                                                     const uint32_t* __restrict__ qa8, const float* __restrict__ sa8,
                                                                     const uint8_t* __restrict__ weight_a, int rows, int in_dim, int out_dim,
                                                                     int share_blocks, int cols_arg, int accumulate, Epilogue ep_a, BmSecond second) {
    uint32_t stamp[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (kStamps) stamp[0] = static_cast<uint32_t>(__builtin_amdgcn_s_memrealtime());
    using F = BmFormat<kType>;
    const bool is_b = blockIdx.z != 0;
    float* dst = is_b ? second.dst : dst_a;
    const uint8_t* weight = is_b ? second.weight : weight_a;
    const Epilogue ep = is_b ? second.ep : ep_a;
    float* partial = partial_a == nullptr ? nullptr : partial_a + (is_b ? static_cast<size_t>(gridDim.y) * rows * out_dim : 0);
    constexpr int kQB = F::kQuantBytes, kStageBlocks = F::kWaveBlocks / 2, kWB = kHalves * kStageBlocks;
    constexpr int kPairs = kWB / 2, kHalfPairs = kStageBlocks / 2;  // pairs of blocks: of the wavefront, of a stage
    constexpr int kCols = 16 * kCG, kStages = kHalves * kCG, kSteps = kStages * kHalfPairs;
    const int kb_full = in_dim >> 5, pairs_total = (kb_full + 1) >> 1;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, g = lane >> 4, par = g >> 1, kh = g & 1;  // column, lane group, block parity, k half
    // a workgroup's columns: `cols` of them, a multiple of 8 in (16 kCG - 16, 16 kCG] (the host picks what spreads the matrix
    // evenly over the compute units); the arithmetic runs on all 16 kCG, the last ones on a copy of column cols - 1
    const int cols = kFullCols ? 16 * kCG : cols_arg;
    const int n0 = blockIdx.x * cols;
    const int share_begin = static_cast<int>(blockIdx.y) * share_blocks;  // a multiple of kWB: even
    const int share_end = min(share_begin + share_blocks, kb_full);
    const int blk0 = share_begin + wave * kWB;
    const int nb = max(0, min(kWB, share_end - blk0));
    const int last = blk0 + max(nb, 1) - 1 < kb_full ? blk0 + max(nb, 1) - 1 : kb_full - 1;
    auto clamp_blk = [&](int j) { return min(blk0 + j, last); };
    const size_t blocks_total = static_cast<size_t>(out_dim) * kb_full;
    const uint32_t lds_wave = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(bm_lds))) + wave * kBmWaveBytes;

    // ---- 1. loads.  Stage s = (half hb = s / kCG of the wavefront's blocks, column group cg =
    // s % kCG) is two 1 KB units of weights (8 columns x 8 chunks each), written to slot s % 4 of
    // the wavefront's 8 KB of LDS.  What a compute unit can keep in flight is a small part of what
    // its wavefronts want, and a wavefront that cannot issue a load cannot compute either, so a
    // wavefront requests two stages ahead of the one it works on, not everything at once.
    // Order of the requests (a compute unit has one address unit, all its wavefronts queue there and are
    // served in order): what the quantizer's launch left in the L2 -- the operand fragments in their compact form
    // (two pairs a load) and one or two 4-byte loads for the row scales of the wavefront's pairs -- for the whole
    // workgroup, a barrier, then the first stage, an 8-byte load per column group for the weight scales, two
    // spares; then the second stage.
    // A wavefront's loads complete in the order issued, so "all but the youngest n have completed"
    // says that a stage is there.  The compiler counts only its own loads when it waits for one of
    // them, which can only be too strict: it retires as many more of the oldest younger loads as
    // there are loads it does not know of (two at that point: the second stage).  The two spare
    // loads are those (they are looked at once, after the loop).
    auto issue_stage = [&](int st) {
        const int hb = st / kCG, cg = st % kCG;
        const uint8_t* wbase = weight + static_cast<size_t>(n0) * kb_full * kQB;
        const int c8 = lane >> 3, slot = lane & 7;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int c = 16 * cg + 8 * u + c8;
            const int chunk = slot ^ ((c >> 1) & 7);
            const int cc = min(n0 + min(c, cols - 1), out_dim - 1) - n0;
            uint32_t off;
            if (kType == 2) {
                off = (static_cast<uint32_t>(cc) * kb_full + clamp_blk(8 * hb + chunk)) * 16u;
            } else {
                off = (static_cast<uint32_t>(cc) * kb_full + clamp_blk(4 * hb + (chunk >> 1))) * 32u + (chunk & 1) * 16u;
            }
            bm_lds_load16(wbase, off, lds_wave + ((st & 3) * 2 + u) * 1024);
        }
    };
    const int pair0 = blk0 >> 1;
    // What comes from the L2 goes first, for the whole workgroup: the operand fragments and row scales (written by the
    // quantizer's launch, read by every workgroup) come back in a fraction of the time a weight byte takes, but a compute
    // unit serves its requests in the order issued -- behind the first weight requests they would wait for HBM.  One
    // barrier, reached within a few instructions, keeps every wavefront's weight requests behind all of these.
    // row scales: 64 bytes a pair; lane L of load q takes slot L % 16 of pair 4 q + L / 16
    // operand fragments, compact: 512 bytes a pair, two pairs a load; lane L of load q holds entry
    // L % 32 of pair 2 q + L / 32
    // (Inline assembly: the compiler may move its own loads from read-only memory across the barrier; waited for by
    // hand before the first stage is used.)
    constexpr int kScaleLoads = (kPairs + 3) / 4;
    float sx_part[kGroups][kScaleLoads];
    bm_v4i packed[kGroups][kPairs / 2];
    // (kQuantize: X instead.  A load is eight blocks of one row, eight lanes a block and four values a lane: whole lines)
    typedef float bm_v4f __attribute__((ext_vector_type(4)));
    constexpr int kRowLoads = kQuantize ? kWB / 8 : 1;
    bm_v4f xv[kQuantize ? 8 : 1][kRowLoads];
    const int live = nb > 0 ? rows : 0;
    if constexpr (kQuantize) {
        static_assert(kGroups == 1 && kWB % 8 == 0 && kWB <= 16, "the operand's place in the ring");
        uint32_t x_off[kRowLoads];
#pragma unroll
        for (int c = 0; c < kRowLoads; ++c) {
            x_off[c] = static_cast<uint32_t>(min(blk0 + 8 * c + (lane >> 3), kb_full - 1)) * 128u + (lane & 7) * 16u;
            asm volatile("" : "+v"(x_off[c]));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < 8; r += 2) {
            if (r < live) {
                const float* row0 = reinterpret_cast<const float*>(qa8) + static_cast<size_t>(r) * in_dim;
                const float* row1 = r + 1 < live ? row0 + in_dim : row0;  // (an odd last row twice)
#pragma unroll
                for (int c = 0; c < kRowLoads; ++c) asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(xv[r][c]) : "v"(x_off[c]), "s"(row0) : "memory");
#pragma unroll
                for (int c = 0; c < kRowLoads; ++c) asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(xv[r + 1][c]) : "v"(x_off[c]), "s"(row1) : "memory");
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    } else {
        uint32_t frag_off[kPairs / 2], scale_off[kScaleLoads];
#pragma unroll
        for (int q = 0; q < kPairs / 2; ++q) frag_off[q] = static_cast<uint32_t>(min(pair0 + 2 * q + (lane >> 5), pairs_total - 1) * 32 + (lane & 31)) * 16u;
#pragma unroll
        for (int q = 0; q < kScaleLoads; ++q) scale_off[q] = static_cast<uint32_t>(min(pair0 + 4 * q + g, pairs_total - 1) * 16 + l16) * 4u;
#pragma unroll
        for (int q = 0; q < kPairs / 2; ++q) asm volatile("" : "+v"(frag_off[q]));
#pragma unroll
        for (int q = 0; q < kScaleLoads; ++q) asm volatile("" : "+v"(scale_off[q]));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int grp = 0; grp < kGroups; ++grp) {
            const uint32_t* qa_g = qa8 + static_cast<size_t>(grp) * pairs_total * 128;
            const float* sa_g = sa8 + static_cast<size_t>(grp) * pairs_total * 16;
#pragma unroll
            for (int q = 0; q < kPairs / 2; ++q) asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(packed[grp][q]) : "v"(frag_off[q]), "s"(qa_g) : "memory");
#pragma unroll
            for (int q = 0; q < kScaleLoads; ++q) asm volatile("global_load_dword %0, %1, %2" : "=v"(sx_part[grp][q]) : "v"(scale_off[q]), "s"(sa_g) : "memory");
        }
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    }
    // Weight scales, fp16 in block order (rows of whole 16-byte runs: the host sends no other shape here): word p of a
    // column's run holds blocks 2p and 2p + 1.
    // Tiles of three column groups and more: the workgroup's scales of this K share -- up to 64 columns x 256 bytes (Q4_0;
    // 128 for Q8_0) -- go through LDS.  Thread t fetches sixteen bytes (eight blocks) per round, sixteen (eight) threads a
    // column: whole 128-byte lines, each asked for once per workgroup and ahead of the first weight stage.  (A wavefront
    // fetching the scales of its own blocks of every column asks for 64 pieces of 32 (16) bytes; with the eight
    // wavefronts' 512 requests per compute unit a Q4_0 launch on 14336 columns took 0.4 us longer, a pair of them 0.9,
    // Q8_0 0.6.)  In LDS a column's chunks are stored at chunk ^ (column % chunks): the sixteen columns a step reads one
    // word of then sit in different banks.  Smaller tiles keep the register form (Q4_0, 16 columns on 4096: 7.14
    // against 7.26 us; Q8_0, 32 columns in 2.7 rounds on 11008: 15.6 against 16.1; Q4_0 24 columns on 6144: no difference).
    constexpr bool kScalesInLds = kCG >= 3 || kHalves > 2;
    constexpr int kChunks = kBmWaves * kWB / 8;
    constexpr int kScaleRounds = (16 * kCG * kChunks + kBmThreads - 1) / kBmThreads;  // rounds of the workgroup's threads over the tile's columns
    constexpr int kAheadStages = 2;  // requested beyond the stage being worked on (the ring has four slots)
    unsigned char* lds_scales = bm_lds + kBmLdsBytes;
    bm_v4i scale_run[kScaleRounds];
    if (kScalesInLds) {
        const uint8_t* sbase = weight + blocks_total * kQB + static_cast<size_t>(n0) * kb_full * 2;
        uint32_t run_off[kScaleRounds];
#pragma unroll
        for (int r = 0; r < kScaleRounds; ++r) {
            const int c = tid / kChunks + r * (kBmThreads / kChunks), chunk = tid % kChunks;
            const int cc = min(n0 + min(c, cols - 1), out_dim - 1) - n0;
            run_off[r] = static_cast<uint32_t>(cc * kb_full + min(share_begin + 8 * chunk, kb_full - 8)) * 2u;
            asm volatile("" : "+v"(run_off[r]));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < kScaleRounds; ++r) {
            scale_run[r] = bm_v4i{0, 0, 0, 0};
            if (tid / kChunks + r * (kBmThreads / kChunks) < 16 * kCG)
                asm volatile("global_load_dwordx4 %0, %1, %2" : "+v"(scale_run[r]) : "v"(run_off[r]), "s"(sbase) : "memory");
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    // (kQuantize: Q8_0 requests its second stage in front of the conversions, K = 4096, eight rows: 14336 columns 14.4 -> 13.7 us,
    // 11008 columns 12.3 -> 11.8; Q4_0 loses, a pair of 14336 columns 17.0 .. 17.3 -> 17.7 .. 18.6)
    constexpr bool kStageOneEarly = kQuantize && kScalesInLds && kStages > 1 && kType == 8;
    issue_stage(0);
    if (kStageOneEarly) issue_stage(1);
    if constexpr (kQuantize) {
        // X is there when at most the first stages' requests and the rounds of scale runs that every wavefront takes part in are
        // in flight.  Quantized as quantize_fragments8_kernel does it, bit for bit.  kN vectors are converted together: of their
        // kN maxima over eight lanes a lane ends with one (`pick`: lane % kN, mirrored in the upper four of the eight so that the
        // last exchange, a mirror, stays within one maximum), divides for that one, and the quad hands the reciprocals round.
        // The dwords go to the operand's order through LDS: the ring's slots 2 and 3, whose stages are requested once this has
        // been read back.  Row r of block b is stored in row r ^ (b % 8) of the eight: the 64 lanes' dwords in 64 banks.
        constexpr int kN = 2 * kRowLoads;
        constexpr int kFullRounds = kScalesInLds ? 16 * kCG * kChunks / kBmThreads : 0;
        asm volatile("s_waitcnt vmcnt(%0)" : : "n"((kStageOneEarly ? 4 : 2) + kFullRounds) : "memory");
        unsigned char* own = bm_lds + wave * kBmWaveBytes + 4096;
        const int bl = lane >> 3, j = lane & 7, pick = (j & 4 ? 7 - j : j) & (kN - 1);
        const int h2 = kType == 2 ? (j >> 1) & 1 : j >> 2, dw = kType == 2 ? 2 * (j & 1) + (j >> 2) : j & 3;
        const uint32_t q_base = (bl >> 1) * 512 + (16 * (bl & 1) + 8 * h2 + bl) * 16 + dw * 4;
        float row_scale[4];  // of the lane's own pick
        // (numbers or quiet NaNs on both sides: nothing to quieten first, which fmaxf would do.  The two wait states that a lane
        // exchange of the result needs stand with it: the compiler does not look into the assembly)
        auto max_with = [](float a, float other) { float m; asm("v_max_f32 %0, %1, %2\n\ts_nop 1" : "=v"(m) : "v"(a), "v"(other)); return m; };
#pragma unroll
        for (int r = 0; r < 8; r += 2) {
            row_scale[r / 2] = 0.0f;
            if (r < live) {
                float m[kN];
#pragma unroll
                for (int i = 0; i < kN; ++i) {
                    bm_v4f& v = xv[r + i / kRowLoads][i % kRowLoads];
                    asm volatile("" : "+v"(v));
                    m[i] = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
                }
                float mine = pick & 1 ? m[1] : m[0], other = pick & 1 ? m[0] : m[1];
                mine = max_with(mine, dpp_move<kDppXor1>(other));
                if constexpr (kN == 4) {
                    float mine2 = pick & 1 ? m[3] : m[2], other2 = pick & 1 ? m[2] : m[3];
                    mine2 = max_with(mine2, dpp_move<kDppXor1>(other2));
                    other = pick & 2 ? mine : mine2;
                    mine = pick & 2 ? mine2 : mine;
                } else {
                    other = mine;
                }
                mine = max_with(mine, dpp_move<kDppXor2>(other));
                mine = max_with(mine, dpp_move<kDppHalfMirror>(mine));
                const float s = act_scale(mine);
                row_scale[r / 2] = s;
                const float inv_mine = mine == 0.0f ? 0.0f : 1.0f / s;
                // (the upper four lanes of eight back in order)
                const float inv = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(inv_mine), __float_as_int(inv_mine), 0x1B, 0xF, 0xA, false));
                auto convert = [&](int i, float inv_i) {
                    const bm_v4f v = xv[r + i / kRowLoads][i % kRowLoads];
                    const uint32_t q0 = act_quant(v[0], inv_i), q1 = act_quant(v[1], inv_i), q2 = act_quant(v[2], inv_i), q3 = act_quant(v[3], inv_i);
                    const uint32_t low = __builtin_amdgcn_perm(q1, q0, 0x0C0C0400u), high = __builtin_amdgcn_perm(q3, q2, 0x0C0C0400u);
                    *reinterpret_cast<uint32_t*>(own + (q_base ^ ((r + i / kRowLoads) << 4)) + (i % kRowLoads) * 2048) = low | high << 16;
                };
                convert(0, dpp_move<0x00>(inv));
                convert(1, dpp_move<0x55>(inv));
                if constexpr (kN == 4) {
                    convert(2, dpp_move<0xAA>(inv));
                    convert(3, dpp_move<0xFF>(inv));
                }
            }
        }
        // slot l16 of pair 4 q + g: row l16 % 8 of block 8 q + (2 g + l16 / 8), from the lane of that block that picked it
#pragma unroll
        for (int q = 0; q < kScaleLoads; ++q) {
            const int from = 4 * ((2 * g + (l16 >> 3)) * 8 + (l16 & 1) * kRowLoads + q);
            int got[4];
#pragma unroll
            for (int p = 0; p < 4; ++p) got[p] = __builtin_amdgcn_ds_bpermute(from, __float_as_int(row_scale[p]));
            sx_part[0][q] = __int_as_float(l16 & 4 ? (l16 & 2 ? got[3] : got[2]) : (l16 & 2 ? got[1] : got[0]));
        }
        asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
#pragma unroll
        for (int q = 0; q < kPairs / 2; ++q) {
            const int swz = (4 * q + 2 * (lane >> 5) + ((lane >> 4) & 1)) & 7;
            packed[0][q] = *reinterpret_cast<const bm_v4i*>(own + (2 * q + (lane >> 5)) * 512 + ((lane & 24) + ((lane & 7) ^ swz)) * 16);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
    }
    if (kScalesInLds) {
        // the scale runs are there when at most the first stage's two requests are in flight; the workgroup meets once they
        // are in LDS (the first stage is waited for behind that, with nothing else of the wavefront outstanding: behind
        // the second stage's requests the wait would also have to see those accepted by the memory pipeline, which for
        // the last wavefronts of a unit is well into the stream)
        asm volatile("s_waitcnt vmcnt(%0)" : : "n"(kStageOneEarly ? 4 : 2) : "memory");
#pragma unroll
        for (int r = 0; r < kScaleRounds; ++r) {
            asm volatile("" : "+v"(scale_run[r]));
            const int c = tid / kChunks + r * (kBmThreads / kChunks), chunk = tid % kChunks;
            if (c < 16 * kCG) *reinterpret_cast<bm_v4i*>(lds_scales + c * (kChunks * 16) + ((chunk ^ (c & (kChunks - 1))) << 4)) = scale_run[r];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    }
    // Q8_0: lane group g takes words [g * kWpl, +kWpl) of its wavefront's blocks and the lane exchange hands word p
    // out when its stage comes
    constexpr int kWpl = kPairs / 4;
    uint32_t tb_part[kCG][kWpl];
#pragma unroll
    for (int cg = 0; cg < (kScalesInLds ? 0 : kCG); ++cg) {
        const int cc = min(n0 + min(16 * cg + l16, cols - 1), out_dim - 1);
        const uint16_t* sw = reinterpret_cast<const uint16_t*>(weight + blocks_total * kQB) + static_cast<size_t>(cc) * kb_full;
        const uint32_t* run = reinterpret_cast<const uint32_t*>(sw + min(blk0, kb_full - 8)) + g * kWpl;
        if constexpr (kWpl == 2) {
            const uint2 v = *reinterpret_cast<const uint2*>(run);
            tb_part[cg][0] = v.x;
            tb_part[cg][1] = v.y;
        } else {
            tb_part[cg][0] = run[0];
        }
    }
    constexpr int kSpares = 2;
    uint32_t spare[kSpares] = {0, 0};
    if (!kScalesInLds) {  // (Q4_0 has no load of the compiler's left: nothing to keep its waits from)
#pragma unroll
        for (int k = 0; k < kSpares; ++k) spare[k] = __builtin_nontemporal_load(qa8 + k * 32 + (lane & 31));  // inside the first pair's entries
    }
    // Q4_0 asks for the second stage only when the first one and the register loads are there (below); Q8_0, whose
    // stages are half as many blocks, measured better with the second stage requested up front.
    constexpr bool kStartupAlone = (kType == 2 || kQuantize) && !kStageOneEarly;
    if (!kStartupAlone && !kStageOneEarly) {
#pragma unroll
        for (int st = 1; st < kAheadStages; ++st) issue_stage(st);
    }

    // this lane's B operand: column 16 * cg + l16, block 2p + par, k half kh.  Q8_0: bytes
    // [16 kh, +16) of the block.  Q4_0: bytes [8 kh, +8), low nibbles and high nibbles dword by
    // dword; a nibble n stands for n - 8: with bit 3 flipped and in the high half of a byte it reads as
    // the int8 16 * (n - 8).  Its address inside a stage's slot (the column group does not enter:
    // 16 columns are two whole units and the swizzle repeats every 16 columns).
    uint32_t baddr[kHalfPairs];
#pragma unroll
    for (int q = 0; q < kHalfPairs; ++q) {
        const int j = 2 * q + par;
        const int unit = l16 >> 3, row = (l16 & 7) * 8, swz = (l16 >> 1) & 7;
        const int chunk = kType == 2 ? j : j * 2 + kh;
        baddr[q] = lds_wave + (unit * 64 + row + (chunk ^ swz)) * 16 + (kType == 2 ? 8 * kh : 0);
    }

    float acc[kGroups][kCG][4];
#pragma unroll
    for (int grp = 0; grp < kGroups; ++grp)
#pragma unroll
        for (int cg = 0; cg < kCG; ++cg)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[grp][cg][v] = 0.0f;

    // ---- 2. the stages, software-pipelined by hand over the steps (one step = a pair of blocks,
    // sixteen columns: one int8 MFMA and one scale-product MFMA).  A step's weight bytes are
    // requested from LDS one step ahead and its results are scaled one step behind, after the next
    // MFMAs have been issued: no step waits for the LDS or for the matrix unit's latency.  (The
    // weight bytes of a stage's first step cannot be requested before the stage is there.)  The
    // scheduling barriers keep the compiler from undoing that order.
    if (nb > 0) {
        typedef unsigned bm_v2u __attribute__((ext_vector_type(2)));
        typedef unsigned bm_v4u __attribute__((ext_vector_type(4)));
        typedef typename std::conditional<kType == 2, bm_v2u, bm_v4u>::type Raw;
        typedef __attribute__((address_space(3))) const Raw LdsRaw;
        Raw raw[2];
        bm_v4i afrag[kGroups][kHalfPairs];
        float sxm[kGroups][kHalfPairs], tbm[kHalfPairs];
        bm_v4i cres[kGroups][2];
        bm_v4f tres[kGroups][2];
        auto stage_of = [&](int it) { return it / kHalfPairs; };
        auto fetch_weights = [&](int it) { raw[it & 1] = *reinterpret_cast<LdsRaw*>(baddr[it % kHalfPairs] + (stage_of(it) & 3) * 2048); };
        auto scale = [&](int it) {
            const int cg = stage_of(it) % kCG;
#pragma unroll
            for (int grp = 0; grp < kGroups; ++grp)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    acc[grp][cg][v] = __builtin_fmaf(tres[grp][it & 1][v], static_cast<float>(cres[grp][it & 1][v]), acc[grp][cg][v]);
        };
#pragma unroll
        for (int it = 0; it < kSteps; ++it) {
            if (it % kHalfPairs == 0) {
                const int st = stage_of(it), hb = st / kCG, cg = st % kCG;
                if (st == 0) {
                    if (kStartupAlone) asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
                    else asm volatile("s_waitcnt vmcnt(%0)" : : "n"(2 * (kAheadStages - 1)) : "memory");
#pragma unroll
                    for (int grp = 0; grp < kGroups; ++grp) {
#pragma unroll
                        for (int q = 0; q < kPairs / 2; ++q) asm volatile("" : "+v"(packed[grp][q]));
#pragma unroll
                        for (int q = 0; q < kScaleLoads; ++q) asm volatile("" : "+v"(sx_part[grp][q]));  // (one operand a statement: never the same register twice)
                    }
#pragma unroll
                    for (int c = 0; c < (kScalesInLds ? 0 : kCG); ++c)
#pragma unroll
                        for (int q = 0; q < kWpl; ++q) asm volatile("" : "+v"(tb_part[c][q]));
                }
                if (kStartupAlone && st == 0) {
#pragma unroll
                    for (int ahead = 1; ahead < kAheadStages; ++ahead) issue_stage(ahead);
                }
                if (st + kAheadStages < kStages) issue_stage(st + kAheadStages);
                // operands of this stage's scale products (in the shadow of the wait below).
                // A: lane (slot i = l16, k = g) carries sx of slot i if k is the slot's block (i / 8), else 0
                // B: lane (column l16, k = g) carries sw of block 2p + k for k < 2 (zero if that block is not
                //    this wavefront's: a clamped re-read of the last block counts for nothing), else 0;
                //    Q4_0: times 1/16, the nibbles enter the dots as 16 * (n - 8)
#pragma unroll
                for (int q = 0; q < kHalfPairs; ++q) {
                    const int p = hb * kHalfPairs + q;
                    uint32_t word;
                    if (kScalesInLds) {
                        const int c = 16 * cg + l16, pw = wave * kPairs + p;  // column of the tile, pair of the share
                        word = *reinterpret_cast<const uint32_t*>(lds_scales + c * (kChunks * 16) + (((pw >> 2) ^ (c & (kChunks - 1))) << 4) + ((pw & 3) << 2));
                    } else {
                        word = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(4 * (16 * (p / kWpl) + l16), static_cast<int>(tb_part[cg][p % kWpl])));
                    }
                    const float sw = half_bits_to_f32(static_cast<uint16_t>(word >> (16 * kh))) * (kType == 2 ? 0.0625f : 1.0f);
                    tbm[q] = (g < 2 && 2 * p + g < nb) ? sw : 0.0f;
                }
                if (cg == 0) {
                    // first stage of a half: the half's row scales and A operands.  Lane (g, slot i) takes
                    // entry 8 g + i % 8 of its pair through the lane exchange if the slot's block is the lane
                    // group's, else zeros
#pragma unroll
                    for (int grp = 0; grp < kGroups; ++grp)
#pragma unroll
                        for (int q = 0; q < kHalfPairs; ++q) {
                            const int p = hb * kHalfPairs + q;
                            const float sx = __int_as_float(__builtin_amdgcn_ds_bpermute(4 * (16 * (p & 3) + l16), __float_as_int(sx_part[grp][p >> 2])));
                            sxm[grp][q] = g == (l16 >> 3) ? sx : 0.0f;
                            const int from = 4 * (32 * (p & 1) + 8 * g + (l16 & 7));
#pragma unroll
                            for (int d = 0; d < 4; ++d) {
                                const int got = __builtin_amdgcn_ds_bpermute(from, packed[grp][p >> 1][d]);
                                afrag[grp][q][d] = (l16 >> 3) == par ? got : 0;
                            }
                        }
                }
                // this stage is there when at most the stages requested behind it are in flight
                {
                    const int younger = 2 * ((kStages - 1 - st) < kAheadStages ? (kStages - 1 - st) : kAheadStages);
                    if (younger == 6) asm volatile("s_waitcnt vmcnt(6)" : : : "memory");
                    else if (younger == 4) asm volatile("s_waitcnt vmcnt(4)" : : : "memory");
                    else if (younger == 2) asm volatile("s_waitcnt vmcnt(2)" : : : "memory");
                    else asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
                }
                fetch_weights(it);
                if (kStamps && st < 4) stamp[1 + st] = static_cast<uint32_t>(__builtin_amdgcn_s_memrealtime());
                if (kStamps && st == kStages - 1) stamp[5] = static_cast<uint32_t>(__builtin_amdgcn_s_memrealtime());
            }
            __builtin_amdgcn_sched_barrier(0);
            if (it + 1 < kSteps && (it + 1) % kHalfPairs != 0) fetch_weights(it + 1);
            bm_v4i b;
            {
                const Raw w = raw[it & 1];
                if constexpr (kType == 2) {
                    const uint32_t x = w[0] ^ 0x88888888u, y = w[1] ^ 0x88888888u;
                    b = bm_v4i{static_cast<int>((x << 4) & 0xF0F0F0F0u), static_cast<int>(x & 0xF0F0F0F0u), static_cast<int>((y << 4) & 0xF0F0F0F0u),
                               static_cast<int>(y & 0xF0F0F0F0u)};
                } else {
                    b = bm_v4i{static_cast<int>(w[0]), static_cast<int>(w[1]), static_cast<int>(w[kType == 2 ? 0 : 2]), static_cast<int>(w[kType == 2 ? 1 : 3])};
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            const int q = it % kHalfPairs;
#pragma unroll
            for (int grp = 0; grp < kGroups; ++grp) {
                cres[grp][it & 1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(afrag[grp][q], b, bm_v4i{0, 0, 0, 0}, 0, 0, 0);
                tres[grp][it & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(sxm[grp][q], tbm[q], bm_v4f{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (it > 0) scale(it - 1);
            __builtin_amdgcn_sched_barrier(0);
        }
        scale(kSteps - 1);
        if (kStamps) stamp[6] = static_cast<uint32_t>(__builtin_amdgcn_s_memrealtime());
    } else {
        asm volatile("s_waitcnt vmcnt(0)" : : : "memory");  // nothing may still be writing LDS when the region is reused
    }
    asm volatile("" : : "v"(spare[0]), "v"(spare[1]));

    // ---- 3. the wavefronts' sums (and the two block parities) meet in LDS
    float* red = reinterpret_cast<float*>(bm_lds);  // [wave][cg * 4 + v][lane], one group of rows at a time
#pragma unroll
    for (int grp = 0; grp < kGroups; ++grp) {
        __syncthreads();
#pragma unroll
        for (int cg = 0; cg < kCG; ++cg)
#pragma unroll
            for (int v = 0; v < 4; ++v) red[(wave * kCG * 4 + cg * 4 + v) * 64 + lane] = acc[grp][cg][v];
        __syncthreads();
        if (tid < 8 * kCols) {
            const int m8 = tid / kCols, c = tid % kCols, m = 8 * grp + m8;
            const int item = ((c >> 4) * 4 + (m8 & 3)) * 64 + 16 * (m8 >> 2) + (c & 15);
            float sum = 0.0f;
#pragma unroll
            for (int w = 0; w < kBmWaves; ++w) sum += red[w * kCG * 256 + item] + red[w * kCG * 256 + item + 32];
            const int n = n0 + c;
            if (kStamps) {
                asm volatile("" : : "v"(sum));  // (keeps the arithmetic alive)
            } else if (m < rows && c < cols && n < out_dim) {
                const size_t at = static_cast<size_t>(m) * out_dim + n;
                if (partial != nullptr) partial[static_cast<size_t>(blockIdx.y) * rows * out_dim + at] = sum;
                // two K shares, no epilogue: both add to the zeroed result; 0 + a + b = 0 + b + a to the bit, whoever comes first
                else if (accumulate) unsafeAtomicAdd(dst + at, sum);
                else dst[at] = finish_output(ep, n, at, sum);
            }
        }
    }
    if (kStamps) {
        __syncthreads();
        stamp[7] = static_cast<uint32_t>(__builtin_amdgcn_s_memrealtime());
        if (lane == 0) {
            uint32_t* o = reinterpret_cast<uint32_t*>(dst_a) + (static_cast<size_t>(blockIdx.x) * kBmWaves + wave) * 8;
#pragma unroll
            for (int q = 0; q < 8; ++q) o[q] = stamp[q];
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Nine to 64 rows (one or two row tiles) on a matrix wide enough for 64-column tiles: batch_mfma_kernel's arithmetic
// (v_mfma_i32_32x32x32_i8 per block, scale products of a pair of blocks from one
// v_mfma_f32_32x32x1_2b_f32, one convert and one multiply-add per live result register) with what
// the eight-row kernel showed to matter:
//   * 64 columns per workgroup (two groups of 32): the A fragments -- 16 KB per wavefront, as much
//     as the weights per 32 columns -- are read once for both groups, and there is one workgroup
//     per compute unit with the whole register file (no second workgroup to leave room for);
//   * weights staged: stage (half hb of the wavefront's blocks, column group cg) is four 1 KB
//     units in one of two 4 KB slots; a stage is requested when the stage two before it has been
//     computed, so one stage travels while one is worked on (requesting all at once leaves a
//     wavefront stuck issuing loads while the data it could work on is already there);
//   * the A fragments of the second half of the blocks are requested block by block during the
//     last stage that uses the first half's (behind the weight requests already out, in front of
//     the last one);
//   * a lane unpacks whole bytes of Q4_0 nibbles (low and high: 8 operations per block instead of
//     12; the fragments' k order follows, quantize_fragments_kernel<true>);
//   * the arithmetic of a pair of blocks is ordered by hand: both int8 MFMAs and the scale MFMA
//     first, then the conversions and multiply-adds of both blocks, with the next pair's LDS reads
//     in flight meanwhile.
template <int kType, int kRT, int kLive>
__global__ __launch_bounds__(kBmThreads, 2) void batch32_mfma_kernel(float* __restrict__ dst_a, float* __restrict__ partial_a,
                                                                      const uint32_t* __restrict__ qa, const float* __restrict__ sa,
                                                                      const uint8_t* __restrict__ weight_a, int rows, int in_dim, int out_dim,
                                                                      int share_blocks, Epilogue ep_a, BmSecond second, int accumulate) {
    using F = BmFormat<kType>;
    const bool is_b = blockIdx.z != 0;
    float* dst = is_b ? second.dst : dst_a;
    const uint8_t* weight = is_b ? second.weight : weight_a;
    const Epilogue ep = is_b ? second.ep : ep_a;
    float* partial = partial_a == nullptr ? nullptr : partial_a + (is_b ? static_cast<size_t>(gridDim.y) * rows * out_dim : 0);
    constexpr int kQB = F::kQuantBytes, kWB = F::kWaveBlocks, kHB = kWB / 2, kPairs = kWB / 2, kHalfPairs = kPairs / 2;
    const int kb_full = in_dim >> 5;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lj = lane & 31, lh = lane >> 5;
    const int n0 = blockIdx.x * 64;
    const int share_begin = static_cast<int>(blockIdx.y) * share_blocks;
    const int share_end = min(share_begin + share_blocks, kb_full);
    const int blk0 = share_begin + wave * kWB;
    const int nb = max(0, min(kWB, share_end - blk0));
    const int last = blk0 + max(nb, 1) - 1 < kb_full ? blk0 + max(nb, 1) - 1 : kb_full - 1;
    auto clamp_blk = [&](int j) { return min(blk0 + j, last); };
    const size_t blocks_total = static_cast<size_t>(out_dim) * kb_full;
    const uint32_t lds_wave = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(bm_lds))) + wave * kBmWaveBytes;

    // stage st = 2 * hb + cg -> slot st % 2
    auto issue_stage = [&](int st) {
        const int hb = st >> 1, cg = st & 1;
        const uint8_t* wbase = weight + static_cast<size_t>(n0) * kb_full * kQB;
        const int c8 = lane >> 3, slot = lane & 7;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int c = 32 * cg + 8 * u + c8;
            const int chunk = slot ^ ((c >> 1) & 7);
            const int cc = min(n0 + c, out_dim - 1) - n0;
            uint32_t off;
            if (kType == 2) {
                off = (static_cast<uint32_t>(cc) * kb_full + clamp_blk(8 * hb + chunk)) * 16u;
            } else {
                off = (static_cast<uint32_t>(cc) * kb_full + clamp_blk(4 * hb + (chunk >> 1))) * 32u + (chunk & 1) * 16u;
            }
            bm_lds_load16(wbase, off, lds_wave + ((st & 1) * 4 + u) * 1024);
        }
    };
    issue_stage(0);
    // weight scales of both column groups (fp16, block order; rows of whole 16-byte runs): word p of a
    // column's run holds blocks 2p and 2p + 1
    uint32_t tb_word[2][kPairs];
#pragma unroll
    for (int cg = 0; cg < 2; ++cg) {
        const int cc = min(n0 + 32 * cg + lj, out_dim - 1);
        const uint16_t* sw = reinterpret_cast<const uint16_t*>(weight + blocks_total * kQB) + static_cast<size_t>(cc) * kb_full;
        const uint4* run = reinterpret_cast<const uint4*>(sw + min(blk0, kb_full - 8));
#pragma unroll
        for (int q = 0; q < kPairs / 4; ++q) {
            const uint4 v = run[q];
            tb_word[cg][4 * q] = v.x;
            tb_word[cg][4 * q + 1] = v.y;
            tb_word[cg][4 * q + 2] = v.z;
            tb_word[cg][4 * q + 3] = v.w;
        }
    }
    // A fragments and row scales of the first half of the blocks.  Rows that exist live in the first
    // 2 * kLive lanes of each half of a fragment; the other lanes repeat a live lane's address.
    const int lr = lj % (2 * kLive);
    const int alane = lh * 32 + lr;
    const bm_v4i* qa4 = reinterpret_cast<const bm_v4i*>(qa);
    auto load_a = [&](int rt, int j) { return qa4[(static_cast<size_t>(rt) * kb_full + clamp_blk(j)) * 64 + (rt + 1 < kRT ? lane : alane)]; };
    auto load_ta = [&](int rt, int p) { return sa[static_cast<size_t>(clamp_blk(2 * p + lh)) * (32 * kRT) + rt * 32 + (rt + 1 < kRT ? lj : lr)]; };
    bm_v4i afrag[kRT][kHB];
    float ta[kRT][kHalfPairs];
#pragma unroll
    for (int rt = 0; rt < kRT; ++rt) {
#pragma unroll
        for (int j = 0; j < kHB; ++j) afrag[rt][j] = load_a(rt, j);
#pragma unroll
        for (int p = 0; p < kHalfPairs; ++p) ta[rt][p] = load_ta(rt, p);
    }
    issue_stage(1);

    // this lane's B operand inside a slot: column lj of the group, block j of the half, k half lh
    uint32_t baddr[kHB];
#pragma unroll
    for (int j = 0; j < kHB; ++j) {
        const int unit = lj >> 3, row = (lj & 7) * 8, swz = (lj >> 1) & 7;
        const int chunk = kType == 2 ? j : 2 * j + lh;
        baddr[j] = lds_wave + (unit * 64 + row + (chunk ^ swz)) * 16 + (kType == 2 ? 8 * lh : 0);
    }
#pragma unroll
    for (int j = 0; j < kHB; ++j) asm volatile("" : "+v"(baddr[j]));

    // (a full row tile has all 16 result registers live; kLive counts those of the last one)
    float acc[2][kRT][16];
#pragma unroll
    for (int cg = 0; cg < 2; ++cg)
#pragma unroll
        for (int rt = 0; rt < kRT; ++rt)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[cg][rt][v] = 0.0f;

    if (nb > 0) {
        typedef unsigned bm_v2u __attribute__((ext_vector_type(2)));
        typedef unsigned bm_v4u __attribute__((ext_vector_type(4)));
        typedef typename std::conditional<kType == 2, bm_v2u, bm_v4u>::type Raw;
        typedef __attribute__((address_space(3))) const Raw LdsRaw;
        auto unpack = [&](const Raw& w) {
            bm_v4i b;
            if constexpr (kType == 2) {
                const uint32_t x = w[0] ^ 0x88888888u, y = w[1] ^ 0x88888888u;
                b = bm_v4i{static_cast<int>((x << 4) & 0xF0F0F0F0u), static_cast<int>(x & 0xF0F0F0F0u), static_cast<int>((y << 4) & 0xF0F0F0F0u),
                           static_cast<int>(y & 0xF0F0F0F0u)};
            } else {
                b = bm_v4i{static_cast<int>(w[0]), static_cast<int>(w[1]), static_cast<int>(w[kType == 2 ? 0 : 2]), static_cast<int>(w[kType == 2 ? 1 : 3])};
            }
            return b;
        };
        const bm_v16i zi = {};
        const bm_v32f zf = {};
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            const int hb = st >> 1, cg = st & 1;
            // this stage is there when at most the stage requested behind it is in flight
            if (st < 3) asm volatile("s_waitcnt vmcnt(4)" : : : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
            Raw raw0 = *reinterpret_cast<LdsRaw*>(baddr[0] + (st & 1) * 4096);
            Raw raw1 = *reinterpret_cast<LdsRaw*>(baddr[1] + (st & 1) * 4096);
            bm_v4i b0 = unpack(raw0), b1 = unpack(raw1);
            if (kHalfPairs > 1) {
                raw0 = *reinterpret_cast<LdsRaw*>(baddr[2] + (st & 1) * 4096);
                raw1 = *reinterpret_cast<LdsRaw*>(baddr[3] + (st & 1) * 4096);
            }
#pragma unroll
            for (int q = 0; q < kHalfPairs; ++q) {
                const int p = hb * kHalfPairs + q;
                const bool live_blk = 2 * p + lh < nb;  // a clamped re-read of the last block counts for nothing
                const float tb = live_blk ? half_bits_to_f32(static_cast<uint16_t>(tb_word[cg][p] >> (16 * lh))) * (kType == 2 ? 0.0625f : 1.0f) : 0.0f;
#pragma unroll
                for (int rt = 0; rt < kRT; ++rt) {
                    constexpr int kFull = 16;
                    const int live_regs = rt + 1 < kRT ? kFull : kLive;
                    __builtin_amdgcn_sched_barrier(0);
                    const bm_v32f t = __builtin_amdgcn_mfma_f32_32x32x1f32(live_blk ? ta[rt][q] : 0.0f, tb, zf, 0, 0, 0);
                    const bm_v16i c0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(afrag[rt][2 * q], b0, zi, 0, 0, 0);
                    const bm_v16i c1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(afrag[rt][2 * q + 1], b1, zi, 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    if (cg == 1 && hb == 0) {
                        // last use of the first half's fragments of this pair: the second half's take their place
                        afrag[rt][2 * q] = load_a(rt, kHB + 2 * q);
                        afrag[rt][2 * q + 1] = load_a(rt, kHB + 2 * q + 1);
                        ta[rt][q] = load_ta(rt, kHalfPairs + q);
                    }
                    // while the matrix unit works (last row tile: its operands are no longer needed): the next
                    // pair's weights out of their nibbles, the pair after that out of LDS
                    if (rt == kRT - 1 && q + 1 < kHalfPairs) {
                        b0 = unpack(raw0);
                        b1 = unpack(raw1);
                        if (q + 2 < kHalfPairs) {
                            raw0 = *reinterpret_cast<LdsRaw*>(baddr[(2 * q + 4) % kHB] + (st & 1) * 4096);
                            raw1 = *reinterpret_cast<LdsRaw*>(baddr[(2 * q + 5) % kHB] + (st & 1) * 4096);
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int v = 0; v < kFull; ++v)
                        if (v < live_regs) acc[cg][rt][v] = __builtin_fmaf(t[v], static_cast<float>(c0[v]), acc[cg][rt][v]);
#pragma unroll
                    for (int v = 0; v < kFull; ++v)
                        if (v < live_regs) acc[cg][rt][v] = __builtin_fmaf(t[16 + v], static_cast<float>(c1[v]), acc[cg][rt][v]);
                    fence_registers(acc[cg][rt]);
                }
            }
            // the slot is free: the stage two on takes it
            if (st + 2 < 4) issue_stage(st + 2);
        }
    } else {
        asm volatile("s_waitcnt vmcnt(0)" : : : "memory");  // nothing may still be writing LDS when the region is reused
    }

    // ---- the wavefronts' sums meet in LDS, one row tile at a time: [wave][cg][v][lane] (8 x 2 x 16 x 64 floats = the whole 64 KB)
    float* red = reinterpret_cast<float*>(bm_lds);
    constexpr int kItems = 2 * 16 * 64;
#pragma unroll
    for (int rt = 0; rt < kRT; ++rt) {
        __syncthreads();
#pragma unroll
        for (int cg = 0; cg < 2; ++cg)
#pragma unroll
            for (int v = 0; v < 16; ++v) red[((wave * 2 + cg) * 16 + v) * 64 + lane] = acc[cg][rt][v];
        __syncthreads();
        for (int i = tid; i < kItems; i += kBmThreads) {
            const int l = i & 63, v = (i >> 6) & 15, cg = i >> 10;
            const int m = rt * 32 + 8 * (v >> 2) + 4 * (l >> 5) + (v & 3);
            const int n = n0 + 32 * cg + (l & 31);
            if (m < rows && n < out_dim) {
                float half[2];
#pragma unroll
                for (int h = 0; h < 2; ++h) {  // (batch_mfma_kernel's order, for the same bits)
                    half[h] = red[(kBmWaves / 2) * h * kItems + i];
#pragma unroll
                    for (int w = 1; w < kBmWaves / 2; ++w) half[h] += red[((kBmWaves / 2) * h + w) * kItems + i];
                }
                const float sum = half[0] + half[1];
                const size_t at = static_cast<size_t>(m) * out_dim + n;
                if (partial != nullptr) partial[static_cast<size_t>(blockIdx.y) * rows * out_dim + at] = sum;
                else if (accumulate) unsafeAtomicAdd(dst + at, sum);  // (two K shares, no epilogue, the result cleared beforehand: see batch8_mfma_kernel)
                else dst[at] = finish_output(ep, n, at, sum);
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Nine to 64 rows, one round of workgroups, a compute unit each: a workgroup takes 32 rows and walks over as many groups of 32 (64)
// columns as that round needs, its operand fragments staying in registers.  The arithmetic is the kernels' above; what is
// different is what stands around it, which is what such calls spend their time on:
//   * K is shared out over the wavefronts in runs: every wavefront fetches its fragments once, whatever the number of columns, the first
//     run's ahead of everybody's other requests;
//   * weights and scales (from the tile-order copy: one request brings 32 columns') go through a ring of three stages in LDS that nothing
//     but hand-counted waits stands before;
//   * the matrix instructions of a pair of blocks leave between the conversions and multiply-adds of the pair before (two sets of result
//     registers; runs of four stages, whose fragments fill the registers, keep one set);
//   * the wavefronts' sums meet in LDS behind counters, half a column group later: no barrier in the loop.
// Bound by the vector unit beside the matrix unit, about 200 SIMD cycles per 32 x 32 outputs and block (176 by the instructions alone), and
// by the first bytes' way from memory, 5000 cycles until a wavefront can start.  Q4_0, weights from memory, against the two kernels above
// (us): 32 rows, K = 4096, 4096 columns 10.5 -> 9.8, 6144 12.0 -> 10.7, a pair of 14336 27.9 -> 24.8; 48 rows, 2048 x 2048 11.9 -> 7.4;
// 64 rows, a pair of 14336 columns 51.0 -> 35.6.
//
// kRows: the most rows a call has, 32 (one group of rows), 64 or (Q4_0) 96.  kChains: 0, a wavefront's blocks are added up one after
// the other (a single run's even and odd ones apart); 1, even and odd ones apart; 2, and the sums of its runs too.
template <int kType, int kLive, int kHalves, int kParts, int kChains, int kRows, bool kOne>
__global__ __launch_bounds__(kBmThreads, 2) void batch_groups_mfma_kernel(float* __restrict__ dst_a, float* __restrict__ partial_a,
                                                                      const uint32_t* __restrict__ qa, const float* __restrict__ sa,
                                                                      const uint8_t* __restrict__ weight_a, int rows, int in_dim, int out_dim,
                                                                      int share_blocks, int row_groups, int col_groups, Epilogue ep_a,
                                                                      BmSecond second, int accumulate) {
    using B = BatchGroups<kType, kLive, kHalves, kParts>;
    constexpr bool kShared = kRows > 32, kApart = kChains == 2;
    const bool is_b = blockIdx.z != 0;
    float* dst = is_b ? second.dst : dst_a;
    const uint8_t* weight = is_b ? second.weight : weight_a;
    const Epilogue ep = is_b ? second.ep : ep_a;
    float* partial = partial_a == nullptr ? nullptr : partial_a + (is_b ? static_cast<size_t>(gridDim.y) * rows * out_dim : 0);
    constexpr int kQB = kType == 2 ? 16 : 32, kHB = B::kStageBlocks, kPairs = kHB / 2, kRun = B::kRun;
    constexpr int kSlots = B::kSlots, kSets = B::kSets, kSteps = kHalves * kPairs;
    static_assert(kSteps % 2 == 0, "the two register sets alternate over a column group");
    const int kb_full = in_dim >> 5;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lj = lane & 31, lh = lane >> 5;
    // row groups of the same columns on one XCD (workgroup ids go round-robin over the eight), so that an L2 reads a weight once
    int col_tile = blockIdx.x, group = 0;
    if (kShared) {
        const int slot = blockIdx.x >> 3;
        group = slot % row_groups;
        col_tile = slot / row_groups * 8 + (blockIdx.x & 7);
    }
    const int n_first = col_tile * B::kGroupCols * (kOne ? 1 : col_groups);
    if (n_first >= out_dim) return;
    const int groups_here = kOne ? 1 : min(col_groups, (out_dim - n_first + B::kGroupCols - 1) / B::kGroupCols);
    const int padded = row_groups * 32, row0 = group * 32;
    const int share_begin = static_cast<int>(blockIdx.y) * share_blocks;
    const int share_end = min(share_begin + share_blocks, kb_full);
    const int part = wave % kParts, side = wave / kParts;  // of K; of the group's columns
    // Run hb of this wavefront is the kHB blocks first_of(hb) + [0, kHB).  Two runs follow on each other, a slice of blocks as
    // batch_mfma_kernel's; four, and two in chains of their own, are a row of all wavefronts' each.  Indices past the end are
    // clamped to a valid block for every load; their activation scales are zero.
    auto first_of = [&](int hb) { return share_begin + (kHalves == 2 && kChains == 0 ? (part * 2 + hb) * kHB : hb * kRun + part * kHB); };
    auto clamp_blk = [&](int hb, int j) { return min(first_of(hb) + j, share_end - 1); };
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(bm_lds)));
    const uint32_t lds_slots = lds0 + wave * (kSlots * B::kSlotBytes);

    auto load16 = [&](const uint8_t* base, uint32_t off, uint32_t at) {
        if (kShared) bm_lds_load16_kept(base, off, at);
        else bm_lds_load16(base, off, at);
    };
    // Requests of a stage: the columns' whole 128-byte lines (eight lanes each), chunk slots XOR-swizzled by the column; the scales in
    // the tile order (tile_scale_index) -- of a tile of four (Q8_0: two) columns and 128 blocks the stage's blocks are 128 (64) bytes on
    // end, so one request brings those of 32 columns -- in 16-byte units XOR-swizzled by the tile.
    const size_t blocks_total = static_cast<size_t>(out_dim) * kb_full;
    const uint8_t* scale_tiles = weight + ((blocks_total * (kQB + 2) + 15) & ~static_cast<size_t>(15));
    constexpr int kTileCols = kType == 2 ? 4 : 2, kTileBytes = kType == 2 ? 1024 : 512, kUnits = kType == 2 ? 8 : 4;
    const int slices = (kb_full + 127) >> 7, last_tile = (out_dim - 1) / kTileCols;
    // (a unit of eight columns is eight times the row pitch on, its chunks an XOR by four in the odd ones: two offsets a lane serve every
    // stage but those at the matrix's last columns)
    const int c8 = lane >> 3, s8 = lane & 7;
    const uint32_t pitch = static_cast<uint32_t>(kb_full) * kQB;
    const int unit_tile = lane / kUnits, unit_at = (lane % kUnits) ^ (kType == 2 ? unit_tile >> 1 : unit_tile >> 2);
    const uint32_t weights_at = c8 * pitch + (s8 ^ (c8 >> 1)) * 16;  // (the pitch is a multiple of 128)
    const uint32_t scales_lane = static_cast<uint32_t>(unit_tile * slices) * kTileBytes + unit_at * 16;
    auto issue = [&](int cg, int hb, int slot) {
        const int n0 = min(n_first + cg * B::kGroupCols + side * 32, out_dim - 1) & ~31;  // (a side past the matrix repeats its last columns)
        const uint32_t at = lds_slots + slot * B::kSlotBytes;
        const int first = min(first_of(hb), share_end - kHB);  // (shares and K are whole stages; what is read for one past the end counts for nothing)
        const uint8_t* sbase = scale_tiles + (static_cast<size_t>(n0 / kTileCols) * slices + (first >> 7)) * kTileBytes + (first & (kType == 2 ? 63 : 31)) * 16;
        const uint8_t* wbase = weight + static_cast<size_t>(n0) * pitch + static_cast<size_t>(first) * kQB;
        if (n0 + 32 <= out_dim) {
            load16(sbase, scales_lane, at + 4096);
#pragma unroll
            for (int u = 0; u < 4; ++u) load16(wbase + static_cast<size_t>(8 * u) * pitch, weights_at ^ (u & 1 ? 64u : 0u), at + u * 1024);
        } else {  // rows clamped to the matrix
            int l = lane;
            asm volatile("" : "+v"(l));  // (nothing of this takes registers in the loop)
            const int t = l / kUnits, tile = min(t, last_tile - n0 / kTileCols);
            load16(sbase, static_cast<uint32_t>(tile * slices) * kTileBytes + ((l % kUnits) ^ (kType == 2 ? t >> 1 : t >> 2)) * 16, at + 4096);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int c = 8 * u + (l >> 3);
                load16(wbase, static_cast<uint32_t>(min(c, out_dim - 1 - n0)) * pitch + ((l & 7) ^ ((c >> 1) & 7)) * 16, at + u * 1024);
            }
        }
    };
    // stage st is run st % kHalves of column group st / kHalves
    const int stages = groups_here * kHalves;
    auto issue_stage = [&](int st, int slot) { issue(st / kHalves, st % kHalves, slot); };

    typedef __attribute__((address_space(3))) volatile uint32_t LdsCount;
    const uint32_t counters = lds0 + B::kCountersAt;
    if (tid < 2) *reinterpret_cast<LdsCount*>(counters + 4 * tid) = 0;
    issue_stage(0, 0);
    // A fragments and row scales: all of the wavefront's share, for every column group.  Rows that exist live in the first
    // 2 * kLive lanes of each half of a fragment; the other lanes repeat a live lane's address.
    const int lr = lj % (2 * kLive);
    typedef const __attribute__((address_space(1))) bm_v4i* Fragments;
    typedef const __attribute__((address_space(1))) float* Scales;
    Fragments fragments_at = reinterpret_cast<Fragments>(reinterpret_cast<uintptr_t>(qa));
    Scales scales_at = reinterpret_cast<Scales>(reinterpret_cast<uintptr_t>(sa));
    bm_v4i afrag[kHalves][kHB];
    float ta[kHalves][kPairs];
    auto load_run = [&](int hb) {
#pragma unroll
        for (int j = 0; j < kHB; ++j) afrag[hb][j] = fragments_at[(static_cast<size_t>(group) * kb_full + clamp_blk(hb, j)) * 64 + lh * 32 + lr];
#pragma unroll
        for (int p = 0; p < kPairs; ++p) ta[hb][p] = scales_at[static_cast<size_t>(clamp_blk(hb, 2 * p + lh)) * padded + row0 + lr];
    };
    // A packed nibble in its byte is sixteen times its value, which the weight scale takes back.  A sixteenth of a product of scales
    // below 2^-122 is subnormal where the product may not be, though, and loses up to four of its bits.  Beyond 64 rows, where the other
    // route is the GEMM, which keeps them, a wavefront that holds an activation scale below 2^-98 (the smallest fp16 scale is 2^-24; a
    // block of activations below 4e-28, not all zeros) forms its sums again (form_again).  Up to 64 rows the kernels above, whose bits
    // these are, lose them too.
    constexpr bool kAgain = kType == 2 && kRows > 64;
    bool small_scales = false;  // of the wavefront
    // The compiler counts only its own loads: a wait of its for one of them would be a wait for every request that left in
    // between.  So they are taken here, before the requests of the later stages leave.
    auto take_run = [&](int hb) {
#pragma unroll
        for (int j = 0; j < kHB; ++j) asm volatile("" : "+v"(afrag[hb][j]) : : "memory");
#pragma unroll
        for (int p = 0; p < kPairs; ++p) {
            asm volatile("" : "+v"(ta[hb][p]) : : "memory");
            if (first_of(hb) + 2 * p + lh >= share_end) ta[hb][p] = 0.0f;
        }
        if (kAgain) {
            uint32_t least = ~0u;  // (a zero is no small scale: it wraps round to the largest)
#pragma unroll
            for (int p = 0; p < kPairs; ++p) least = min(least, __float_as_uint(ta[hb][p]) - 1u);
            small_scales = small_scales || __ballot(least < 0x0E800000u - 1u) != 0;  // 2^-98
        }
    };
    // The first run's of all wavefronts go first: a barrier, reached within a few instructions, keeps the others behind them.  (Their
    // addresses pass through it, so that the compiler cannot lift them.)
    load_run(0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : "+s"(fragments_at), "+s"(scales_at) : : "memory");
#pragma unroll
    for (int hb = 1; hb < kHalves; ++hb) load_run(hb);
#pragma unroll
    for (int hb = 0; hb < 1; ++hb) take_run(hb);  // (the others where they are needed)
#pragma unroll
    for (int st = 1; st < kSlots; ++st)
        if (st < stages) issue_stage(st, st);

    typedef unsigned bm_v2u __attribute__((ext_vector_type(2)));
    typedef unsigned bm_v4u __attribute__((ext_vector_type(4)));
    typedef typename std::conditional<kType == 2, bm_v2u, bm_v4u>::type Raw;
    typedef __attribute__((address_space(3))) const Raw LdsRaw;
    typedef __attribute__((address_space(3))) const uint16_t LdsHalf;
    // this lane's B operand inside a slot: column lj, block j of the run (chunk j, or 2j + lh), k half lh -- an XOR away from block 0's
    const uint32_t frag0 = lj * 128 + (((lj >> 1) & 7) ^ (kType == 2 ? 0 : lh)) * 16 + (kType == 2 ? 8 * lh : 0);
    // ... and its scale: unit 2q + lh of its tile, the half of column lj and of the run's place in the slice
    const int lt = lj / kTileCols;
    const uint32_t scale0 = 4096 + lt * (kUnits * 16) + ((lh ^ (kType == 2 ? lt >> 1 : lt >> 2)) << 4) + (lj % kTileCols) * 2;
    auto place_of_run = [&](int hb) {  // Q4_0: blocks 64 apart share a unit; Q8_0: blocks 32 apart
        return kType == 2 ? ((first_of(hb) >> 6) & 1) * 8 : ((first_of(hb) >> 5) & 3) * 4;
    };
    auto unpack = [&](const Raw& w) {
        bm_v4i b;
        if constexpr (kType == 2) {
            auto byte = [](uint32_t x) { return static_cast<int>((x & 0xF0F0F0F0u) ^ 0x80808080u); };  // 16 (n - 8) of each high nibble n
            b = bm_v4i{byte(w[0] << 4), byte(w[0]), byte(w[1] << 4), byte(w[1])};
        } else {
            b = bm_v4i{static_cast<int>(w[0]), static_cast<int>(w[1]), static_cast<int>(w[kType == 2 ? 0 : 2]), static_cast<int>(w[kType == 2 ? 1 : 3])};
        }
        return b;
    };
    // stage `st` has landed when at most the requests of the stages behind it are in flight
    auto wait_stage = [&](int st) {
        if (st + 2 < stages) asm volatile("s_waitcnt vmcnt(10)" : : : "memory");
        else if (st + 1 < stages) asm volatile("s_waitcnt vmcnt(5)" : : : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
    };

    const bm_v16i zi = {};
    const bm_v32f zf = {};
    Raw raw0, raw1;
    uint16_t half;
    int st_read = 0, slot_read = 0;  // the stage that operands are read from, and its slot
    auto read_step = [&](int p) {
        const int hb = p / kPairs, q = p % kPairs;
        const uint32_t slot_at = lds_slots + slot_read * B::kSlotBytes;
        raw0 = *reinterpret_cast<LdsRaw*>(slot_at + (frag0 ^ ((kType == 2 ? 2 * q : 4 * q) * 16)));
        raw1 = *reinterpret_cast<LdsRaw*>(slot_at + (frag0 ^ ((kType == 2 ? 2 * q + 1 : 4 * q + 2) * 16)));
        half = *reinterpret_cast<LdsHalf*>(slot_at + place_of_run(hb) + (scale0 ^ (32 * q)));
    };
    bm_v32f t[kSets];
    bm_v16i c0[kSets], c1[kSets];
    bm_v4i b0, b1;
    float tb;
    auto take_operands = [&](int hb) {
        b0 = unpack(raw0);
        b1 = unpack(raw1);
        tb = half_bits_to_f32(half) * (kType == 2 ? 0.0625f : 1.0f);
        if (first_of(hb) >= share_end) tb = 0.0f;  // a run past the share (inside one, scales past the matrix are zeros)
    };
    // A chain of additions is at most sixteen blocks long.  Runs of four stages put the first half's sums down in the
    // wavefront's own part of the room below.
    constexpr bool kPutDown = kHalves == 4;
    static_assert(!kPutDown || (kOne && !kAgain), "the room is free for the one column group only");
    constexpr int kSums = kApart ? kHalves : 1;
    // ... and where a run's sums are added up by themselves, four: even and odd blocks apart.
    constexpr bool kOdd = kHalves == 1 || kChains > 0;
    // Two runs' fragments, even and odd sums and two sets of results are more than the registers hold (12 spilled, reloaded in the loop):
    // there the next pair's dots take the registers of this pair's as these are read, half a step before they are needed.
    constexpr bool kOneResult = kHalves == 2 && kChains == 1 && !kOne;
    auto last_of_chain = [](int run) { return kApart || run + 1 == kHalves; };  // where even and odd blocks meet
    float acc[kSums][16], odd[16];

    // ---- the wavefronts' sums meet in LDS: [side][part of K][v][lane]; a thread adds up neighbouring columns of a row.  kApart: the sums
    // of a share's runs are added each for itself, in order.  counters[0]: wavefronts that have stored theirs, counters[1]: that have
    // added up; looked at half a column group later, so that nobody waits who is not a half ahead.
    float* red = reinterpret_cast<float*>(bm_lds + B::kSumsAt);
    constexpr int kSideThreads = 64 * kParts, kPer = kLive * 64 / kSideThreads;
    typedef float Terms __attribute__((ext_vector_type(kPer)));
    Terms total;
    const bool plain = ep.bias == nullptr && ep.residual == nullptr && ep.activation == kActNone && partial == nullptr && !accumulate;
    auto wait_count = [&](int which, uint32_t count) {
        while (static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(*reinterpret_cast<LdsCount*>(counters + 4 * which)))) < count)
            __builtin_amdgcn_s_sleep(1);
        asm volatile("" : : : "memory");
    };
    auto count_up = [&](int which) {
        asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
        if (lane == 0) asm volatile("ds_add_u32 %0, %1" : : "v"(counters + 4 * which), "v"(1u) : "memory");
    };
    auto store_sums = [&](int s) {
#pragma unroll
        for (int v = 0; v < kLive; ++v) red[(wave * kLive + v) * 64 + lane] = acc[s][v];
    };
    // The sums of runs [first, last) of a column group once more from plain products, operands straight from memory, where one of them is
    // small enough to feel what was lost (as in gemm_i8_body: 2^-122 in all, which no sum from 2^-96 on does).
    // Activations of 2^-111, products of scales just above 2^-126: the bits of ordinary ones scaled, as on the GEMM; a call without such
    // scales pays for the test alone (77 rows, 2048 x 2048 7.74 -> 7.78 us, 96 rows, 4096 x 6144 18.4 / 18.3).
    auto form_again = [&](int cg, int first, int last, float (&sum)[16]) {
        int l = lane;
        asm volatile("" : "+v"(l));  // (nothing of this takes registers in the loop)
        const int column = l & 31, half_k = l >> 5;
        float least = __builtin_huge_valf();
#pragma unroll
        for (int v = 0; v < kLive; ++v)
            if (row0 + 8 * (v >> 2) + 4 * half_k + (v & 3) < rows) least = fminf(least, fabsf(sum[v]));
        if (__ballot(least < 0x1p-96f) == 0) return;
        float second[16];  // the odd blocks' sums where they are kept apart
#pragma unroll
        for (int v = 0; v < 16; ++v) sum[v] = second[v] = 0.0f;
        const size_t n = min(n_first + cg * B::kGroupCols + side * 32 + column, out_dim - 1);
        const uint16_t* block_scales = reinterpret_cast<const uint16_t*>(weight + blocks_total * kQB) + n * kb_full;
#pragma unroll 1
        for (int run = first; run < last && first_of(run) < share_end; ++run) {
#pragma unroll 1
            for (int blk = first_of(run); blk < first_of(run) + kHB; blk += 2) {
                const bm_v4i* a = reinterpret_cast<const bm_v4i*>(qa) + (static_cast<size_t>(group) * kb_full + blk) * 64 + l;
                const uint2* w = reinterpret_cast<const uint2*>(weight + (n * kb_full + blk) * kQB) + half_k;
                const float x_scale = sa[static_cast<size_t>(blk + half_k) * padded + row0 + column], w_scale = half_bits_to_f32(block_scales[blk + half_k]);
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const bm_v16f products = __builtin_amdgcn_mfma_f32_32x32x2f32(half_k == h ? x_scale : 0.0f, half_k == h ? w_scale : 0.0f, bm_v16f{}, 0, 0, 0);
                    const uint2 nibbles = w[h * (kQB / 8)];
                    auto byte = [](uint32_t x) { return static_cast<int>((x & 0xF0F0F0F0u) ^ 0x80808080u); };
                    const bm_v4i b = {byte(nibbles.x << 4), byte(nibbles.x), byte(nibbles.y << 4), byte(nibbles.y)};
                    const bm_v16i dot = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[h * 64], b, bm_v16i{}, 0, 0, 0);
                    float(&to)[16] = kOdd && h == 1 ? second : sum;
#pragma unroll
                    for (int v = 0; v < kLive; ++v) to[v] = __builtin_fmaf(products[v], static_cast<float>(dot[v] >> 4), to[v]);
                }
            }
        }
        if (kOdd) {
#pragma unroll
            for (int v = 0; v < kLive; ++v) sum[v] += second[v];
        }
    };
    auto add_up = [&](int cg, int s) {
        int side_tid = tid % kSideThreads;
        asm volatile("" : "+v"(side_tid));  // (its addresses are formed here and take no registers elsewhere)
        Terms term[kParts];
#pragma unroll
        for (int w = 0; w < kParts; ++w) term[w] = reinterpret_cast<const Terms*>(red)[(side * kParts + w) * kSideThreads + side_tid];
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            // (batch_mfma_kernel's order, for the same bits)
            float sum = ((term[0][k] + term[1][k]) + term[2][k]) + term[3][k];
            if constexpr (kParts == 8) sum += ((term[4][k] + term[5][k]) + term[6][k]) + term[7][k];
            total[k] = s == 0 ? sum : total[k] + sum;
        }
        if (s + 1 < kSums) return;
        const int l = side_tid * kPer & 63, v = side_tid * kPer >> 6;
        const int m = row0 + 8 * (v >> 2) + 4 * (l >> 5) + (v & 3);
        const int n = n_first + cg * B::kGroupCols + side * 32 + (l & 31);
        // The frequent ways first, their code straight behind the sums': behind the epilogue's, a pass of 32 rows through eight layers (64
        // launches of different kernels) took 502 us instead of 496, though each kernel by itself took the same time
        if (__builtin_expect(plain && n + kPer <= out_dim, 1)) {
            if (m < rows) {
                float* const to = dst + static_cast<size_t>(m) * out_dim + n;
#pragma unroll
                for (int k = 0; k < kPer; ++k) to[k] = total[k];
            }
            return;
        }
        if (__builtin_expect(accumulate, 1)) {  // (two K shares, no epilogue, the result cleared beforehand: see batch8_mfma_kernel)
#pragma unroll
            for (int k = 0; k < kPer; ++k)
                if (m < rows && n + k < out_dim) unsafeAtomicAdd(dst + static_cast<size_t>(m) * out_dim + n + k, total[k]);
            return;
        }
        // finish_output for neighbouring columns together, the activations out of the way: one column after the other it took 0.7 us of a small
        // call (Q8_0 17 x 256 x 512 with a bias 6.86 -> 6.16, without 5.7; Q4_0 48 x 4096 x 8192 with a bias 17.2 -> 16.65)
        if (__builtin_expect(partial == nullptr, 0)) {
            if (ep.bias != nullptr) {
#pragma unroll
                for (int k = 0; k < kPer; ++k) total[k] += ep.bias[min(n + k, out_dim - 1)];
            }
            if (__builtin_expect(ep.activation != kActNone, 0)) {
#pragma unroll
                for (int k = 0; k < kPer; ++k) total[k] = activate(ep.activation, total[k]);
            }
            if (ep.residual != nullptr) {
#pragma unroll
                for (int k = 0; k < kPer; ++k)
                    total[k] += ep.residual[static_cast<size_t>(min(m, rows - 1)) * out_dim + min(n + k, out_dim - 1)];
            }
        }
        if (m >= rows) return;
        float* const to = (partial != nullptr ? partial + static_cast<size_t>(blockIdx.y) * rows * out_dim : dst) + static_cast<size_t>(m) * out_dim + n;
        if (n + kPer <= out_dim) {
#pragma unroll
            for (int k = 0; k < kPer; ++k) to[k] = total[k];
            return;
        }
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            if (n + k < out_dim) to[k] = total[k];
        }
    };

    wait_stage(0);
    read_step(0);
    if (kSets == 2) {
        take_operands(0);
        c0[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(afrag[0][0], b0, zi, 0, 0, 0);
        t[0] = __builtin_amdgcn_mfma_f32_32x32x1f32(ta[0][0], tb, zf, 0, 0, 0);
        c1[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(afrag[0][1], b1, zi, 0, 0, 0);
        read_step(1);
    }
    // A column group.  The first one stands by itself: the fragments of the later runs are taken there, when they are needed.
    auto column_group = [&](int cg, auto first_one) {
        constexpr bool kFirst = decltype(first_one)::value;
#pragma unroll
        for (int s = 0; s < kSums; ++s)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[s][v] = 0.0f;
        if (kOdd) {
#pragma unroll
            for (int v = 0; v < 16; ++v) odd[v] = 0.0f;
        }
#pragma unroll
        for (int p = 0; p < kSteps; ++p) {
            // The step whose matrix instructions go out here (two sets: the next one, possibly of the next column group), and the one
            // whose operands are read here.
            constexpr int kAhead = kSets - 1;
            const int pm = (p + kAhead) % kSteps, pr = (p + kAhead + 1) % kSteps;
            const int hm = pm / kPairs, qm = pm % kPairs;
            const bool beyond = kOne && p + kAhead >= kSteps;  // nothing follows
            take_operands(hm);
            if (qm == kPairs - 1) {
                // the last operands of a stage are in registers: the stage three on takes its slot
                if (kFirst && hm + 1 < kHalves && p + kAhead < kSteps) take_run(hm + 1);
                const int st = st_read, slot = slot_read;
                slot_read = slot_read + 1 == kSlots ? 0 : slot_read + 1;
                ++st_read;
                if (st + kSlots < stages) {
                    asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
                    issue_stage(st + kSlots, slot);
                }
                if (st_read < stages) wait_stage(st_read);
            }
            if (!beyond) read_step(pr);
            const int set = kSets == 2 ? (p + 1) & 1 : 0, cur = kSets == 2 ? p & 1 : 0;
            auto multiply = [&](const bm_v16i& c, int h, int first, int last) {
                float(&sum)[16] = kOdd && h == 1 ? odd : acc[kApart ? p / kPairs : 0];
#pragma unroll
                for (int v = 0; v < kLive; ++v)
                    if (v >= first && v < last) sum[v] = __builtin_fmaf(t[cur][16 * h + v], static_cast<float>(c[v]), sum[v]);
            };
            if constexpr (kOneResult) {
                multiply(c0[0], 0, 0, kLive / 2);
                __builtin_amdgcn_sched_barrier(0);
                t[set] = __builtin_amdgcn_mfma_f32_32x32x1f32(ta[hm][qm], tb, zf, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                multiply(c0[0], 0, kLive / 2, kLive);
                __builtin_amdgcn_sched_barrier(0);
                c0[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(afrag[hm][2 * qm], b0, zi, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                multiply(c1[0], 1, 0, kLive);
                __builtin_amdgcn_sched_barrier(0);
                c1[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(afrag[hm][2 * qm + 1], b1, zi, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            } else if constexpr (kSets == 2) {
                __builtin_amdgcn_sched_barrier(0);
                if (!beyond) c0[set] = __builtin_amdgcn_mfma_i32_32x32x32_i8(afrag[hm][2 * qm], b0, zi, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                multiply(c0[cur], 0, 0, kLive / 2);
                __builtin_amdgcn_sched_barrier(0);
                if (!beyond) t[set] = __builtin_amdgcn_mfma_f32_32x32x1f32(ta[hm][qm], tb, zf, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                multiply(c0[cur], 0, kLive / 2, kLive);
                multiply(c1[cur], 1, 0, kLive / 2);
                __builtin_amdgcn_sched_barrier(0);
                if (!beyond) c1[set] = __builtin_amdgcn_mfma_i32_32x32x32_i8(afrag[hm][2 * qm + 1], b1, zi, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                multiply(c1[cur], 1, kLive / 2, kLive);
            } else {
                __builtin_amdgcn_sched_barrier(0);
                t[0] = __builtin_amdgcn_mfma_f32_32x32x1f32(ta[hm][qm], tb, zf, 0, 0, 0);
                c0[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(afrag[hm][2 * qm], b0, zi, 0, 0, 0);
                c1[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(afrag[hm][2 * qm + 1], b1, zi, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                multiply(c0[0], 0, 0, kLive);
                multiply(c1[0], 1, 0, kLive);
            }
            fence_registers(acc[kApart ? p / kPairs : 0]);
            if (kOdd) {
                fence_registers(odd);
                if (p % kPairs == kPairs - 1 && last_of_chain(p / kPairs)) {
#pragma unroll
                    for (int v = 0; v < kLive; ++v) {
                        acc[kApart ? p / kPairs : 0][v] += odd[v];
                        odd[v] = 0.0f;
                    }
                }
            }
            if (kAgain && kApart && p % kPairs == kPairs - 1 && small_scales) form_again(cg, p / kPairs, p / kPairs + 1, acc[p / kPairs]);
            if (kPutDown && p == kSteps / 2 - 1) {
                store_sums(0);
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[0][v] = 0.0f;
            }
            if (!kApart && !kOne && !kFirst && p == kSteps / 2 - 1) {
                wait_count(0, cg * kBmWaves);
                add_up(cg - 1, 0);
                count_up(1);
            }
        }
        if (kAgain && !kApart && small_scales) form_again(cg, 0, kHalves, acc[0]);
        if (kPutDown) {
#pragma unroll
            for (int v = 0; v < kLive; ++v) acc[0][v] = red[(wave * kLive + v) * 64 + lane] + acc[0][v];
        }
        if (kApart || kOne) {
#pragma unroll
            for (int s = 0; s < kSums; ++s) {
                if (s > 0 || !kFirst) __syncthreads();
                store_sums(s);
                __syncthreads();
                add_up(cg, s);
            }
        } else {
            if (!kFirst) wait_count(1, cg * kBmWaves);
            store_sums(0);
            count_up(0);
        }
    };
    column_group(0, std::true_type{});
    if (!kOne)
        for (int cg = 1; cg < groups_here; ++cg) column_group(cg, std::false_type{});
    if (!kApart && !kOne) {
        __syncthreads();
        add_up(groups_here - 1, 0);
    }
}

namespace {

template <int kType, int kRowTiles, int kLive>
hipError_t bm_launch(hipStream_t stream, float* dst, float* partial, const uint32_t* qa, const float* sa, const uint8_t* weight,
                     int rows, int in_dim, int out_dim, int shares, int share_blocks, const Epilogue& ep, const BmSecond& second, bool accumulate) {
    const dim3 grid(static_cast<unsigned>((out_dim + 31) / 32), static_cast<unsigned>(shares), second.weight ? 2u : 1u), block(kBmThreads);
    hipLaunchKernelGGL((batch_mfma_kernel<kType, kRowTiles, kLive>), grid, block, kBmLdsBytes, stream, dst,
                       shares > 1 && !accumulate ? partial : nullptr, qa, sa, weight, rows, in_dim, out_dim, share_blocks, ep, second, accumulate ? 1 : 0);
    return hipGetLastError();
}

template <int kType>
hipError_t bm_launch_rows(hipStream_t stream, float* dst, float* partial, const uint32_t* qa, const float* sa, const uint8_t* weight,
                          int rows, int in_dim, int out_dim, int shares, int share_blocks, const Epilogue& ep, const BmSecond& second, bool accumulate) {
#define AFHIP_BM(TILES, LIVE) \
    return bm_launch<kType, TILES, LIVE>(stream, dst, partial, qa, sa, weight, rows, in_dim, out_dim, shares, share_blocks, ep, second, accumulate)
    if (rows <= 8) AFHIP_BM(1, 4);
    if (rows <= 16) AFHIP_BM(1, 8);
    if (rows <= 24) AFHIP_BM(1, 12);
    if (rows <= 32) AFHIP_BM(1, 16);
    if (kType == 8 || rows <= 64) AFHIP_BM(2, 16);
    if constexpr (kType == 2) AFHIP_BM(3, 16);
#undef AFHIP_BM
}

// LDS of an eight-row launch: the wavefronts' rings, and for Q4_0 the workgroup's weight scales of one K share
static size_t bm8_lds_bytes(int tensor_type, int column_groups, int halves = 2) {
    const int share_blocks = (tensor_type == 2 ? BmFormat<2>::kShareBlocks : BmFormat<8>::kShareBlocks) / 2 * halves;
    return kBmLdsBytes + (column_groups >= 3 || halves > 2 ? 16 * column_groups * (share_blocks / 8) * 16 : 0);
}

constexpr bool bm8_can_quantize(int tensor_type, int halves, int groups) { return groups == 1 && halves <= (tensor_type == 2 ? 2 : 4); }

// quantize: qa is X itself (at most sixteen blocks a wavefront: kHalves <= 2 for Q4_0, <= 4 for Q8_0)
template <int kType, int kCG, int kHalves, int kGroups>
hipError_t bm_launch8(hipStream_t stream, float* dst, float* partial, const uint32_t* qa, const float* sa, const uint8_t* weight, int rows,
                      int in_dim, int out_dim, int shares, int share_blocks, int cols, bool accumulate, bool quantize, const Epilogue& ep,
                      const BmSecond& second) {
    const dim3 grid(static_cast<unsigned>((out_dim + cols - 1) / cols), static_cast<unsigned>(shares), second.weight ? 2u : 1u), block(kBmThreads);
    if (accumulate || shares == 1) partial = nullptr;
    const size_t lds = bm8_lds_bytes(kType, kCG, kHalves);
    static LdsLimit lds_limit[4];
    auto launch = [&](auto kernel, LdsLimit* limit) {
        if (hipError_t e = allow_lds(kernel, lds, limit); e != hipSuccess) return e;
        hipLaunchKernelGGL(kernel, grid, block, lds, stream, dst, partial, qa, sa, weight, rows, in_dim, out_dim, share_blocks, cols,
                           accumulate ? 1 : 0, ep, second);
        return hipGetLastError();
    };
    if constexpr (bm8_can_quantize(kType, kHalves, kGroups)) {
        if (quantize) {
            if (cols == 16 * kCG) return launch(batch8_mfma_kernel<kType, kCG, false, true, kHalves, kGroups, true>, &lds_limit[2]);
            return launch(batch8_mfma_kernel<kType, kCG, false, false, kHalves, kGroups, true>, &lds_limit[3]);
        }
    }
    if (cols == 16 * kCG) return launch(batch8_mfma_kernel<kType, kCG, false, true, kHalves, kGroups>, &lds_limit[0]);
    return launch(batch8_mfma_kernel<kType, kCG, false, false, kHalves, kGroups>, &lds_limit[1]);
}


// Column groups of sixteen a workgroup takes: four (64 columns: the activations' share of a
// workgroup's traffic and a wavefront's set-up halve) where that still gives most compute units a
// workgroup, else two.
int bm8_column_groups(int out_dim) { return (out_dim + 63) / 64 >= gemv_compute_units() * 3 / 4 ? 4 : 2; }

int bm_shares(int tensor_type, int in_dim) {
    const int share_max = tensor_type == 2 ? BmFormat<2>::kShareBlocks : BmFormat<8>::kShareBlocks;
    return (in_dim / 32 + share_max - 1) / share_max;
}

// The eight-row kernel's stage rounds per wavefront (its kHalves: 2 or 4, Q8_0 also 8) and the K shares that makes.
// The fewest rounds that leave at most two shares (two add to the result themselves, more need a reduce launch; with
// fewer, longer shares a workgroup takes fewer columns and fetches more operand fragments for them), else the most.
// One share instead of two where the two shares' grid of 64-column tiles would not fit the compute units in one round
// while a single share's may.  (A pair counts as one of its matrices and an epilogue does not enter: each half of a
// pair stays bit-identical to the single op, and an op with a bias to the plain op plus the bias.)
// Measured, five rows, against two rounds everywhere (us): Q4_0 K = 14336 x 4096 columns 11.7 against 13.8 (two shares
// instead of four), 11008 x 4096 11.4 against 13.4, 8192 x 28672 29.3 against 31.2, 28672 x 4096 19.3 against 22.4;
// Q8_0 4096 x 14336 (eight rows) 14.0 against 15.5 (one share in one round), 4096 x 11008 11.8 against 14.0,
// 8192 x 8192 15.1 against 22.3 (16.0 as one share), 14336 x 4096 14.4 against 19.3 (16.7 at four rounds).  Where two
// shares fit one round they stay: Q4_0 8192 x 8192 11.7 (12.6 as one share), 6144 x 4096 8.5 (9.4).
int bm8_halves(int tensor_type, int in_dim, int out_dim) {
    const long kb = in_dim / 32, base = (tensor_type == 2 ? BmFormat<2>::kShareBlocks : BmFormat<8>::kShareBlocks) / 2;
    const int most = tensor_type == 2 ? 4 : 8;
    const long tiles = (out_dim + 63) / 64;
    for (int h = 2; h <= most; h *= 2) {
        const long shares = (kb + h * base - 1) / (h * base);
        if (shares > 2) continue;
        if (shares == 2 && h < most && 2 * tiles > gemv_compute_units()) continue;
        return h;
    }
    return most;
}
int bm8_shares(int tensor_type, int in_dim, int halves) {
    const int share_max = (tensor_type == 2 ? BmFormat<2>::kShareBlocks : BmFormat<8>::kShareBlocks) / 2 * halves;
    return (in_dim / 32 + share_max - 1) / share_max;
}

// A single group of sixteen columns a workgroup: for a matrix whose 32-column tiles (times K shares) leave compute
// units idle while its 16-column tiles fill them in one round -- 4096 columns at K = 4096: 7.9 against 9.0 us on
// batch_mfma_kernel; with a second, partial round (6144 columns: 9.7 against 9.4) it does not pay.
bool bm8_one_column_group(size_t shares, size_t out_dim) {
    const size_t units = static_cast<size_t>(gemv_compute_units());
    const size_t narrow = (out_dim + 15) / 16 * shares;
    return (out_dim + 31) / 32 * shares < units && narrow >= units && narrow <= units + units / 8;
}

// Columns a workgroup of the eight-row kernel takes (a multiple of 8 up to 64).  Where some column count gives a grid of
// no more workgroups than compute units, the smallest such count: every unit gets one workgroup, or nearly every
// one, and none two.  Measured at five and eight rows against the rule below: 11008 columns (K = 4096) 10.6 us on 230
// workgroups of 48 columns against 12.2 on 344 of 32 (172 of 64: 11.6); K = 14336 x 4096 columns 14.7 on 64 x 4 K
// shares against 15.6 on 128 x 4; K = 8192 x 8192 columns 14.4 on 128 x 2 against 15.3 on 256 x 2; Q8_0 6144 columns
// 11.5 on 128 x 2 of 48 against 12.2 on 192 x 2; 14336 columns 12.1 .. 12.3 on 256 of 56 against 12.4 on 224 of 64.
// (A column count that is not a multiple of 16 leaves part of a workgroup's last column group idle.)
// Else the grid takes several rounds whatever the tile, and fewer, larger workgroups fetch the operand fragments less
// often: 64 columns from 12288 columns on, 16 where that is one round and a bit, else 32 (Q8_0, 14336 columns, two
// K shares: 18.0 us on 448 workgroups of 64 against 18.9 on 598 of 48; a pair of those 30.2 against 32.2).
int bm8_columns(long shares, int out_dim, bool pair) {
    const long units = gemv_compute_units();
    for (long cols = 8; cols <= 64; cols += 8)
        if ((out_dim + cols - 1) / cols * shares * (pair ? 2 : 1) <= units) return static_cast<int>(cols);
    if (bm8_column_groups(out_dim) == 4) return 64;
    return bm8_one_column_group(static_cast<size_t>(shares), static_cast<size_t>(out_dim)) ? 16 : 32;
}

template <int kType>
hipError_t bm_launch32(hipStream_t stream, float* dst, float* partial, const uint32_t* qa, const float* sa, const uint8_t* weight, int rows,
                       int in_dim, int out_dim, int shares, int share_blocks, const Epilogue& ep, const BmSecond& second, bool accumulate) {
    const dim3 grid(static_cast<unsigned>((out_dim + 63) / 64), static_cast<unsigned>(shares), second.weight ? 2u : 1u), block(kBmThreads);
#define AFHIP_BM32(RT, LIVE)                                                                                                                 \
    hipLaunchKernelGGL((batch32_mfma_kernel<kType, RT, LIVE>), grid, block, kBmLdsBytes, stream, dst, shares > 1 && !accumulate ? partial : nullptr, \
                       qa, sa, weight, rows, in_dim, out_dim, share_blocks, ep, second, accumulate ? 1 : 0)
    if (rows <= 16) AFHIP_BM32(1, 8);
    else if (rows <= 24) AFHIP_BM32(1, 12);
    else if (rows <= 32) AFHIP_BM32(1, 16);
    else AFHIP_BM32(2, 16);
#undef AFHIP_BM32
    return hipGetLastError();
}

// How a launch of the column-group kernel cuts its work up: workgroups over the rows, column groups a workgroup, wavefronts that share K out,
// stages a wavefront and column group, K shares.
struct BatchGroupsPlan {
    int row_groups, column_groups, parts, halves, shares, share_blocks;
    int chains;  // kChains
    bool own_sums;  // the sums are not formed in the older kernels' order
};

// Whether the column-group kernel exists for a cut: those that batch_groups_plan makes.  Q8_0 of up to 16 rows is the eight-row kernel's
// where K is whole runs, its two runs take one column group, on few columns 33 rows and more; four runs take 25 to 64 rows and one group;
// beyond 64 rows a chain of two runs is left on several groups of eight wavefronts' K alone.
constexpr bool batch_groups_exist(int type, int rows_to, bool sixteen_rows, int halves, int parts, int chains, bool one) {
    if (type == 8 && (rows_to == 96 || sixteen_rows || chains == 1 || halves == 4)) return false;
    if (type == 8 && !one && (halves == 2 || (parts == 8 && rows_to == 32))) return false;
    if (halves == 4) return rows_to != 96 && !sixteen_rows && parts == 8 && chains == 0 && one;
    if (chains == 2) return halves == 2 && parts == 8 && one && (type == 2 || rows_to == 64);
    if (chains == 1) return halves == 2 && rows_to == 96;
    return halves == 1 || rows_to != 96 || (parts == 8 && !one);
}

template <int kType, int kHalves, int kParts, int kChains>
hipError_t bm_launch_groups_of(hipStream_t stream, float* dst, float* partial, const uint32_t* qa, const float* sa, const uint8_t* weight, int rows,
                       int in_dim, int out_dim, const BatchGroupsPlan& plan, const Epilogue& ep, const BmSecond& second, bool accumulate) {
    const int cols = 32 * (kBmWaves / kParts) * plan.column_groups, col_tiles = (out_dim + cols - 1) / cols;
    const dim3 grid(static_cast<unsigned>(plan.row_groups == 1 ? col_tiles : (col_tiles + 7) / 8 * 8 * plan.row_groups), static_cast<unsigned>(plan.shares),
                    second.weight ? 2u : 1u),
        block(kBmThreads);
    static LdsLimit lds_limit[8];
    auto launch = [&](auto kernel, int lds, LdsLimit* limit) {
        if (hipError_t e = allow_lds(kernel, lds, limit); e != hipSuccess) return e;
        hipLaunchKernelGGL(kernel, grid, block, lds, stream, dst, plan.shares > 1 && !accumulate ? partial : nullptr, qa, sa, weight, rows, in_dim,
                           out_dim, plan.share_blocks, plan.row_groups, plan.column_groups, ep, second, accumulate ? 1 : 0);
        return hipGetLastError();
    };
    auto launch_for = [&](auto live, auto rows_to, int at) {
        constexpr int kLive = decltype(live)::value, kRows = decltype(rows_to)::value;
        constexpr int lds = BatchGroups<kType, kLive, kHalves, kParts>::kLdsBytes;
        if (plan.column_groups == 1) {
            if constexpr (batch_groups_exist(kType, kRows, kLive == 8, kHalves, kParts, kChains, true))
                return launch(batch_groups_mfma_kernel<kType, kLive, kHalves, kParts, kChains, kRows, true>, lds, &lds_limit[at]);
        } else {
            if constexpr (batch_groups_exist(kType, kRows, kLive == 8, kHalves, kParts, kChains, false))
                return launch(batch_groups_mfma_kernel<kType, kLive, kHalves, kParts, kChains, kRows, false>, lds, &lds_limit[at + 1]);
        }
        return hipErrorInvalidValue;  // (not among the plans)
    };
    if (rows > 64) return launch_for(std::integral_constant<int, 16>{}, std::integral_constant<int, 96>{}, 6);
    if (rows > 32) return launch_for(std::integral_constant<int, 16>{}, std::integral_constant<int, 64>{}, 0);
    if (rows <= 16) return launch_for(std::integral_constant<int, 8>{}, std::integral_constant<int, 32>{}, 2);
    return launch_for(std::integral_constant<int, 16>{}, std::integral_constant<int, 32>{}, 4);
}

template <int kType>
hipError_t bm_launch_groups(hipStream_t stream, float* dst, float* partial, const uint32_t* qa, const float* sa, const uint8_t* weight, int rows,
                            int in_dim, int out_dim, const BatchGroupsPlan& plan, const Epilogue& ep, const BmSecond& second, bool accumulate) {
#define AFHIP_BMG(H, P, CHAINS) bm_launch_groups_of<kType, H, P, CHAINS>(stream, dst, partial, qa, sa, weight, rows, in_dim, out_dim, plan, ep, second, accumulate)
    switch (plan.parts * 100 + plan.halves * 10 + plan.chains) {
        case 810: return AFHIP_BMG(1, 8, 0);
        case 820: return AFHIP_BMG(2, 8, 0);
        case 821: return AFHIP_BMG(2, 8, 1);
        case 822: return AFHIP_BMG(2, 8, 2);
        case 840: return AFHIP_BMG(4, 8, 0);
        case 410: return AFHIP_BMG(1, 4, 0);
        case 420: return AFHIP_BMG(2, 4, 0);
        case 421: return AFHIP_BMG(2, 4, 1);
        default: return hipErrorInvalidValue;
    }
#undef AFHIP_BMG
}

// The column-group kernel's cut of a call.  Runs and shares depend on one matrix alone, and the sums of an op with an epilogue are formed in
// the plain op's order, so that the halves of a pair and a biased op keep the plain single op's bits; column groups do not enter a sum.
//   * A run that fits four wavefronts is given to four, the others take the next 32 columns (K = 1024, 32 rows, 14336 columns 10.2 -> 8.6,
//     48 rows, a pair of 4096 10.3 -> 8.2); one of up to eight wavefronts on many columns likewise, two stages each, unless eight
//     wavefronts and 32 columns leave fewer rounds (K = 2048: 128256 columns 46 against 51, but 77 rows, 5632 columns 13.8 -> 12.4).
//   * Few columns (a matrix's 32 x 32 tiles fill at most half of the units): K goes to twice the workgroups, two shares that add to the
//     result; an op with an epilogue keeps the two runs' sums apart instead (no reduce launch).  32 rows, 2048 x 2048 9.3 -> 7.7 us.
//   * Two shares of two runs add a reduce launch to an op with an epilogue and take twice the workgroups: on 32 rows only where a pair is one
//     round too (K = 5632: 2048 columns 10.9 -> 10.5, but a pair of 4096 14.6 against 16.8), beyond 64 where one matrix is (1344 columns with
//     a bias 14.7 against 17.1).
//   * Four runs a share on few columns: 25 to 32 rows of more than three eighths of the units' where K fills two shares (K = 14336 x 4096 columns
//     19.1 -> 18.3 .. 18.9 and a pair 34.2 -> 32.4, with the smaller error of shorter chains; an op with an epilogue pays its reduce launch,
//     19.3 against 21.1), 33 to 64 rows where a pair is one round (48 rows, 14336 x 1024 18.6 -> 16.3, with a bias 18.9 -> 18.5; 2048
//     columns 19.4 -> 17.9, but a pair 29.6 against 31.1).  Elsewhere the older kernels' K shares are better (32 rows, 14336 x 1024 14.1
//     against 16.1, a pair of 9216 x 4096 27.2 / 29.6), beyond 64 rows the GEMM's (11008 x 512 15.1 against 16.2, with a bias 15.5 / 18.8).
//   * Beyond 64 rows, where the other route is the GEMM, which shares K out on one group of columns: a wavefront's two runs go into chains
//     of even and odd blocks, and K shares are equal.  Error against the GEMM's, a chain of sixteen in brackets: 77 x 4096 x 2048 0.89
//     (1.01), 96 x 2304 x 1500 0.95 (1.14), 66 x 4352 x 1024 0.95 (1.13), 77 x 2048 x 8192 0.87 (1.00); 10.28 -> 10.33, 9.78 -> 9.91, 10.7 ->
//     10.9, 14.1 -> 14.3 us.  On several groups of columns the GEMM takes K whole, a chain of sixteen has 0.81 .. 1.0 of its error, and
//     the bits are batch_mfma_kernel's.
//   * Q8_0, twice the bytes for the same arithmetic, is bound by the bytes sooner: two runs on few columns only at 33 rows and more (32 rows,
//     1280 x 1024 7.1 -> 6.55, but with a bias 8.0 against 8.4; a pair of 4096 x 4096 columns 13.2 against 14.6); one run of eight wavefronts
//     on many columns likewise (a pair of 8192 columns, K = 1024, 32 rows 10.5 against 10.8).
bool batch_groups_plan(int tensor_type, int rows, int in_dim, int out_dim, bool pair, bool adds, BatchGroupsPlan* plan) {
    const int kb = in_dim / 32, stage_blocks = tensor_type == 2 ? 8 : 4;
    if (kb % 8 != 0) return false;
    const long units = gemv_compute_units();
    BatchGroupsPlan p;
    p.row_groups = (rows + 31) / 32;
    const long columns = (out_dim + 31) / 32;
    const bool few = 2 * columns * p.row_groups <= units;
    // One workgroup a compute unit: each takes as many column groups as that needs.  A launch takes the tiles of `groups` groups of columns
    // (of eight XCDs each where there are row groups) for every row group, K share and matrix.
    auto wide = [&] { return 8 / p.parts; };
    auto grid = [&](long groups, int matrices) {
        const long tiles = (columns + groups * wide() - 1) / (groups * wide());
        return (p.row_groups == 1 ? tiles : (tiles + 7) / 8 * 8) * matrices * p.row_groups * static_cast<long>(p.shares);
    };
    auto groups_for = [&](int matrices) {  // the fewest whose grid is no more than the units, or all columns
        const long each = static_cast<long>(matrices) * p.row_groups * p.shares, most = p.row_groups == 1 ? units / each : units / (8 * each) * 8;
        return most == 0 ? columns : std::min(columns, (columns + most * wide() - 1) / (most * wide()));
    };
    p.parts = 8;
    p.shares = 1;
    if (kb <= 4 * stage_blocks) p.parts = 4;
    else if (columns * p.row_groups > units && kb <= 8 * stage_blocks) {
        const long groups8 = groups_for(1);
        p.parts = 4;
        if (2 * groups_for(1) > groups8) p.parts = 8;
    }
    const int run = p.parts * stage_blocks, runs = (kb + run - 1) / run;
    p.shares = (runs + 3) / 4;
    p.chains = 0;
    if (few && runs > 1 && p.shares == 1) {
        if (adds || runs > 2) p.shares = 2;
        else p.chains = 2;
    }
    p.halves = (runs + p.shares - 1) / p.shares;
    p.share_blocks = p.halves * run;
    if (p.halves == 3) p.halves = 4;
    p.shares = (kb + p.share_blocks - 1) / p.share_blocks;
    p.own_sums = few || p.halves != 2;  // (up to 64 rows)
    if (p.shares == 2 && p.halves == 2 && (p.row_groups == 1 ? grid(1, 2) : (p.row_groups == 3 ? grid(1, 1) : 0)) > units) return false;
    const bool four_runs = p.row_groups == 1 ? rows > 24 && 8 * columns > 3 * units && p.shares == 2 && 8 * kb >= 7 * p.shares * 4 * run
                                             : p.row_groups == 2 && grid(1, 2) <= units;
    if (p.halves == 4 && (!few || tensor_type == 8 || !four_runs)) return false;
    if (tensor_type == 8 && few && runs > 1 && (p.row_groups == 1 || 4 * p.row_groups * columns > units)) return false;
    if (tensor_type == 8 && !few && p.halves == 1 && p.parts == 8 && p.row_groups == 1) return false;
    if (rows > 64 && p.halves == 2 && p.chains == 0 && (p.parts == 4 || groups_for(1) == 1)) {
        p.chains = 1;
        if (p.shares > 1) p.share_blocks = ((kb + p.shares - 1) / p.shares + stage_blocks - 1) / stage_blocks * stage_blocks;
    }
    p.column_groups = p.chains == 2 || p.halves == 4 ? 1 : static_cast<int>(groups_for(pair ? 2 : 1));
    if (!batch_groups_exist(tensor_type, rows > 64 ? 96 : (rows > 32 ? 64 : 32), rows <= 16, p.halves, p.parts, p.chains, p.column_groups == 1)) return false;
    *plan = p;
    return true;
}

}  // namespace

bool batch_mfma_supports(int tensor_type, size_t rows, size_t in_dim, size_t out_dim) {
    if (tensor_type != 2 && tensor_type != 8) return false;
    if (rows < 1 || rows > (tensor_type == 2 ? 96 : 64) || in_dim == 0 || in_dim % 32 != 0 || out_dim == 0) return false;
    // 32-bit lane offsets relative to a column tile, grid.y
    if (in_dim > (1u << 22) || out_dim > 0x7fffffff) return false;
    return true;
}

// The eight-row kernel: at most eight rows -- Q8_0 sixteen, as two groups of eight -- and rows of whole 16-byte runs of
// weight scales.  Nine and sixteen rows against the 32-row kernels (us): Q8_0 K = 4096 x 14336 columns 18.7 -> 15.4,
// 28672 columns 34.7 -> 26.4, K = 14336 x 4096 21.0 -> 16.1, K = N = 8192 23.5 -> 17.1, a pair of 14336 columns
// 35.0 -> 27.1, 4096 x 4096 8.7 -> 8.9, K = 2048 x 8192 columns 8.3 -> 8.8.  Q4_0, whose 32-row kernels are better (half
// the bytes per block, the same MFMA time), loses with two groups -- 14336 columns 13.3 -> 14.6, K = N = 8192
// 13.8 -> 14.7, 128256 columns 74 -> 84; 4096 columns 9.8 -> 9.2 and K = 14336 x 4096 16.8 -> 15.8 are the only gains --
// and keeps one there: a step's MFMAs of two groups (2 x (16 + 32) cycles a SIMD) take as long as its bytes.  On a K
// beyond 8192 and up to 8192 columns Q4_0 takes two groups too -- there the other kernels need three and more K shares
// and a reduce launch, this one two shares that add to the result themselves: sixteen rows, K = 14336 x 4096 columns
// 17.0 -> 15.9 us, 6144 columns 22.7 -> 19.3, 8192 columns 26.5 -> 22.7, a pair of 4096 columns 29.1 -> 22.8, K = 11008
// x 4096 15.9 -> 15.4, K = 28672 x 4096 27.2 -> 26.2 (14336 x 14336 columns loses: 39.3 -> 41.0).
// (It used to be kept to grids
// of at least a workgroup per compute unit; with its tiles sized to the matrix and its first requests in order it also
// wins below that: five rows, K = 4096, against batch_mfma_kernel: 6144 columns 8.5 against 9.6 us, 3072 6.8 against
// 9.0, 1024 6.6 against 8.7.)
bool batch_mfma_eight_rows(int tensor_type, size_t rows, size_t in_dim, size_t out_dim) {
    if (!batch_mfma_supports(tensor_type, rows, in_dim, out_dim)) return false;
    const bool sixteen = tensor_type == 8 || (in_dim > 8192 && out_dim <= 8192);
    return rows <= (sixteen ? 16u : 8u) && (in_dim / 32) % 8 == 0;
}

// Workspace: [qa: 32 * row_tiles * in_dim bytes][sa: (in_dim / 32) * 32 * row_tiles floats][partial sums of K shares, for two matrices]
size_t batch_mfma_workspace_bytes(int tensor_type, size_t rows, size_t in_dim, size_t out_dim) {
    if (!batch_mfma_supports(tensor_type, rows, in_dim, out_dim)) return 0;
    const size_t padded = (rows + 31) / 32 * 32;
    const size_t shares = static_cast<size_t>(bm_shares(tensor_type, static_cast<int>(in_dim)));
    const size_t front = padded * in_dim + (in_dim / 32) * padded * 4;
    return (front + 255) / 256 * 256 + (shares > 1 ? 2 * shares * rows * out_dim * 4 : 0);  // (twice: a pair of matrices)
}

// 65 to 96 rows: the column-group kernel or the tiled GEMM (Q4_0; us, GEMM first).  One matrix's columns decide, also for a pair.  One
// column group: always (77 rows, 2048 x 2048 9.7 -> 7.7, 1024 x 1024 8.7 -> 7.0, K = 4096 x 2048 columns 12.0 -> 10.2).  Several, each with
// what its share of K leaves idle, against the GEMM's rounds: while two of its 32 x 64 tiles a compute unit take the matrix, its one round
// is as long as three column groups and a little more (K = 4096, 96 rows: 4096 columns, two groups, 16.0 -> 14.2; 6144, three, 21.3 -> 18.2;
// 8192, four, 21.7 against 22.2), with one run of K four (K = 2048: 5632 columns 14.4 -> 12.4, a pair 21.0 -> 17.8, 8192 15.0 -> 14.1);
// beyond, it starts another round (K = 4096: 11008 columns 31.8 -> 26.2, 14336 32.4 -> 29.5, a pair 56 -> 49.5; K = 2048 x 16384 22.3 / 22.6,
// 24576 34.4 -> 27.0).  K that fills less than seven eighths of the wavefronts' stages stays with the GEMM (3072 x 8192 18.8 against 21.6).
// From three rounds of the GEMM on (a unit's tiles, of which one is a column group of four wavefronts' K or two of eight's) no more column
// groups than rounds: 80 rows, K = 2048: 14336 columns, three and three, 21.3 -> 19.7, 16384, four and three, 21.4 against 22.5 (with a bias
// 21.9 against 24.2), 18432, four and four, 25.4 -> 22.7; K = 3584 x 16384, seven and three, 32.5 against 32.9 (bias 33.1 against 35.3).  A
// pair in its own rounds where eight XCDs share the tile columns evenly (8192 columns, K = 2048 21.4 against 22.3; 8064 22.8 -> 22.4).
// The error against 64 bits is 0.81 to 1.0 of the GEMM's (5.6e-8 .. 9.8e-8 on 48 shapes, the GEMM's 5.7e-8 .. 1.16e-7).
bool batch_mfma_column_groups(int tensor_type, size_t rows, size_t in_dim, size_t out_dim) {
    BatchGroupsPlan plan;
    if (rows <= 64 || !batch_mfma_supports(tensor_type, rows, in_dim, out_dim) ||
        !batch_groups_plan(tensor_type, static_cast<int>(rows), static_cast<int>(in_dim), static_cast<int>(out_dim), false, true, &plan))
        return false;
    const long room = static_cast<long>(plan.halves) * plan.parts * (tensor_type == 2 ? 8 : 4), kb = static_cast<long>(in_dim / 32);
    const long units = gemv_compute_units(), gemm_cols = static_cast<long>((out_dim + 63) / 64), gemm_grid = static_cast<long>((rows + 31) / 32) * gemm_cols;
    if (plan.column_groups == 1) return true;
    if (plan.shares == 1 && 8 * kb < 7 * room) return false;
    const long per_tile = plan.parts == 8 ? 2 : 1;
    auto fits = [&](long tiles, long groups) { return tiles <= 2 * units || groups <= per_tile * ((tiles + units - 1) / units); };
    if (!fits(gemm_grid, plan.column_groups)) return false;
    BatchGroupsPlan pair;
    if (gemm_cols % 8 == 0 && batch_groups_plan(tensor_type, static_cast<int>(rows), static_cast<int>(in_dim), static_cast<int>(out_dim), true, true, &pair) &&
        !fits(2 * gemm_grid, pair.column_groups))
        return false;
    if (gemm_grid <= 2 * units) return plan.column_groups <= (plan.halves == 2 && plan.parts == 8 ? 3 : 4);
    return true;
}

// Largest grid batch32_mfma_kernel is chosen for; negative: one workgroup per compute unit; 0: neither it nor the column-group kernel.
static std::atomic<long> batch32_bound{-1};
void set_batch32_max_workgroups(long bound) { batch32_bound.store(bound, std::memory_order_relaxed); }

hipError_t launch_batch_mfma(hipStream_t stream, int tensor_type, float* dst, const float* input, const uint8_t* weight_prepared,
                             int rows, int in_dim, int out_dim, uint8_t* workspace, float* dst_b,
                             const uint8_t* weight_b_prepared, const Epilogue& ep, const Epilogue& ep_b, void* quantizer_done) {
    if (!batch_mfma_supports(tensor_type, rows, in_dim, out_dim) || workspace == nullptr) return hipErrorInvalidValue;
    const int row_tiles = (rows + 31) / 32, padded = row_tiles * 32, kb = in_dim / 32;
    uint32_t* qa = reinterpret_cast<uint32_t*>(workspace);
    float* sa = reinterpret_cast<float*>(workspace + static_cast<size_t>(padded) * in_dim);
    const size_t front = static_cast<size_t>(padded) * in_dim + static_cast<size_t>(kb) * padded * 4;
    float* partial = reinterpret_cast<float*>(workspace + (front + 255) / 256 * 256);
    const bool eight = batch_mfma_eight_rows(tensor_type, rows, in_dim, out_dim);
    auto plain = [](const Epilogue& e) { return e.bias == nullptr && e.residual == nullptr && e.activation == kActNone; };
    const bool both_plain = plain(ep) && (weight_b_prepared == nullptr || plain(ep_b));
    const int halves = eight ? bm8_halves(tensor_type, in_dim, out_dim) : 2;
    const int shares = eight ? bm8_shares(tensor_type, in_dim, halves) : bm_shares(tensor_type, in_dim);
    // equal shares, whole wavefront slices: a multiple of the blocks one wavefront owns
    const int wave_blocks = (tensor_type == 2 ? BmFormat<2>::kWaveBlocks : BmFormat<8>::kWaveBlocks) / 2 * halves;
    int share_blocks = (kb + shares - 1) / shares;
    share_blocks = (share_blocks + wave_blocks - 1) / wave_blocks * wave_blocks;
    int real_shares = (kb + share_blocks - 1) / share_blocks;
    // Nine to 64 rows (rows of whole 16-byte runs of scales) where the 64-column tiles times the K shares (times two
    // for a pair) make a grid of five eighths of the compute units up to all of them: batch32_mfma_kernel holds one
    // workgroup per unit, and a second round of them costs more than batch_mfma_kernel's two resident workgroups per
    // unit (N = 20480: 21.1 against 18.5 us).  The grid counts, not the width: a long K on few columns qualifies through
    // its shares (sixteen rows, against batch_mfma_kernel: Q4_0 K = 14336 x 4096 columns 17.9 -> 17.0 us, 64 rows
    // 31.8 -> 27.6, K = N = 8192 15.7 -> 14.0, K = 8192 x 6144 columns 14.3 -> 13.0; Q8_0 K = 4096 x 8192 columns
    // 12.7 -> 11.1, K = 8192 x 4096 columns 15.4 -> 14.4).  Below: 160 and 172 workgroups (K = 4096, 10240 and 11008
    // columns) 13.8 -> 12.7 and 13.9 -> 12.8, Q8_0 160 (5120 columns) 11.0 -> 9.9; 128 workgroups lose (8192 columns
    // 10.6 -> 12.5).  set_batch32_max_workgroups overrides the bound (tests
    // reach the kernel's K shares and pair launches that way; 0 switches the kernel off).
    const size_t x_bytes = static_cast<size_t>(rows) * in_dim * 4, y_bytes = static_cast<size_t>(rows) * out_dim * 4;
    auto apart = [&](const float* y) {
        const uintptr_t a = reinterpret_cast<uintptr_t>(input), b = reinterpret_cast<uintptr_t>(y);
        return b + y_bytes <= a || a + x_bytes <= b;
    };
    const long bound_set = batch32_bound.load(std::memory_order_relaxed);
    const long bound = bound_set >= 0 ? bound_set : gemv_compute_units();
    const long groups32 = static_cast<long>((out_dim + 63) / 64) * real_shares * (weight_b_prepared ? 2 : 1);
    const bool old_thirty_two = !eight && rows <= 64 && kb % 8 == 0 && groups32 >= gemv_compute_units() * 5 / 8 && groups32 <= bound;
    // Column groups: where the plan's sums are its own, for every form of the call (the bits of a pair's halves); elsewhere they are the
    // older kernels' and the faster one takes the call (us, Q4_0, K = 4096): one column group and three and more win (6144 columns
    // 12.0 -> 10.7, a pair of 14336 27.9 -> 24.8, 32000 29.8 -> 26.6), two on up to 32 rows lose (14336 columns 16.4 against 17.1, a pair
    // of 6144 15.2 against 15.9, 24 rows, K = 3072 x 9216 15.1 against 15.7).  Several on a slice that K fills to less than three quarters are a
    // loss of its own, which only more than 48 rows make up for (K = 2304 x 12290 columns, 40 rows 21.2 against 22.2; 64 rows x 32000
    // columns 49.1 -> 39.2).  Q8_0 wins with one column group and such a K (K = 2048 x 8192 columns 9.8 -> 9.2; pairs of 5632 11.7 against
    // 12.6; 17 rows, K = 1280 x 8192 8.7 against 9.0).
    const bool adds = both_plain && apart(dst) && (!weight_b_prepared || apart(dst_b));
    BatchGroupsPlan plan;
    const bool planned = !eight && bound_set != 0 && batch_groups_plan(tensor_type, rows, in_dim, out_dim, weight_b_prepared != nullptr, adds, &plan);
    const bool filled = planned && 4 * kb >= 3 * plan.share_blocks;
    const bool column_groups = planned &&
                               (rows > 64 ? batch_mfma_column_groups(tensor_type, rows, in_dim, out_dim)
                                          : plan.own_sums || (plan.column_groups == 1 && (tensor_type == 2 || filled)) ||
                                                (tensor_type == 2 && (plan.parts == 4 || filled || rows > 48) && (plan.column_groups > 2 || rows > 32)));
    const bool thirty_two = old_thirty_two && !column_groups;
    if (column_groups) {
        real_shares = plan.shares;
        share_blocks = plan.share_blocks;
    }
    // batch_mfma_kernel on a K of one share that more than four of its wavefronts work on, few column tiles (at most
    // half the compute units' worth, one matrix counted) and no epilogue: two shares of four wavefronts each.  The
    // kernel adds its wavefronts' sums as (first four) + (last four), so the two shares' sums are exactly those halves
    // and the result has the same bits as the single share's (which a call with an epilogue keeps: no reduce launch
    // for it).  Four wavefronts a workgroup on twice the workgroups, sixteen rows: 4096 x 4096 columns 9.8 -> 8.8 us,
    // 2048 columns 9.3 -> 8.2, 48 rows 14.5 -> 12.8.  (Beyond one workgroup per compute unit it loses: 6144 columns
    // 10.1 -> 11.8, 8192 columns at 64 rows 15.7 -> 22.4.)
    if (!eight && !thirty_two && !column_groups && real_shares == 1 && adds && kb > (kBmWaves / 2) * wave_blocks &&
        2 * static_cast<long>((out_dim + 31) / 32) <= gemv_compute_units()) {
        share_blocks = (kBmWaves / 2) * wave_blocks;
        real_shares = 2;
    }
    // Two K shares and nothing to do to the sums but add them: the kernel's shares add to the result themselves
    // (cleared by the quantizer's launch, so the result must be apart from X), which saves the reduce launch -- two of them for a pair.
    const bool accumulate = real_shares == 2 && adds;
    const int groups = rows > 8 ? 2 : 1;  // (eight-row kernel) groups of eight rows
    // One K share of at most sixteen blocks a wavefront on up to two workgroups per compute unit: the workgroups quantize X
    // themselves, no quantizer launch.  What they convert they convert once per workgroup, so a grid of many rounds keeps the
    // launch (us, fused against launched; weights from memory): Q4_0 5 x 4096 on 4096 columns 6.9 against 8.1 .. 8.9, 6144 8.4
    // (9.0), 14336 10.2 (11.2), a pair of 14336 16.0 .. 16.7 (16.8 .. 17.9), 5 x 2048 x 8192 6.1 (8.0); 8 x 4096 on 32000 columns
    // (500 workgroups) 18.4 (18.4), on 128256 (2004) 66 (54).  Q8_0 5 x 2048 x 8192 6.1 (8.8), 8 x 2048 x 32000 13.3 (15.3),
    // 8 x 4096 x 14336 13.7 (14.0).  Two K shares keep it too: their result has to be cleared first.  So does a result that
    // overlaps X, which here is read by workgroups that start while others store.
    const long groups8 = !eight ? 0 : [&] {
        const int cols = bm8_columns(real_shares, out_dim, weight_b_prepared != nullptr);
        return static_cast<long>((out_dim + cols - 1) / cols) * (weight_b_prepared ? 2 : 1);
    }();
    const bool quantize = eight && real_shares == 1 && bm8_can_quantize(tensor_type, halves, groups) && groups8 <= 2 * gemv_compute_units() &&
                          apart(dst) && (!weight_b_prepared || apart(dst_b));
    if (quantize) {
        qa = reinterpret_cast<uint32_t*>(const_cast<float*>(input));
    } else if (eight) {  // its own operand layout: 512 + 64 bytes per pair of blocks and group of eight rows, inside the same region
        const int pairs = (kb + 1) / 2;
        sa = reinterpret_cast<float*>(workspace + static_cast<size_t>(groups) * pairs * 512);
        const dim3 qgrid(static_cast<unsigned>((2 * pairs * 8 + 255) / 256), static_cast<unsigned>(8 * groups));
        float* zero_a = accumulate ? dst : nullptr;
        float* zero_b = accumulate && weight_b_prepared ? dst_b : nullptr;
        const int zero_count = rows * out_dim;
        if (tensor_type == 2)
            hipLaunchKernelGGL(quantize_fragments8_kernel<2>, qgrid, dim3(256), 0, stream, input, rows, in_dim, qa, sa, zero_a, zero_b, zero_count);
        else
            hipLaunchKernelGGL(quantize_fragments8_kernel<8>, qgrid, dim3(256), 0, stream, input, rows, in_dim, qa, sa, zero_a, zero_b, zero_count);
        if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    } else {
        const dim3 qgrid(static_cast<unsigned>((in_dim / 4 + 255) / 256), static_cast<unsigned>(padded));
        float* zero_a = accumulate ? dst : nullptr;
        float* zero_b = accumulate && weight_b_prepared ? dst_b : nullptr;
        const size_t zero_count = static_cast<size_t>(rows) * out_dim;
        if ((thirty_two || column_groups) && tensor_type == 2)
            hipLaunchKernelGGL(quantize_fragments_kernel<true>, qgrid, dim3(256), 0, stream, input, rows, in_dim,
                               row_tiles, qa, sa, zero_a, zero_b, zero_count);
        else
            hipLaunchKernelGGL(quantize_fragments_kernel<false>, qgrid, dim3(256), 0, stream, input, rows, in_dim,
                               row_tiles, qa, sa, zero_a, zero_b, zero_count);
        if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    }
    // (an op that is being timed: its activation-quantizer phase ends here)
    if (quantizer_done != nullptr) (void)hipEventRecord(static_cast<hipEvent_t>(quantizer_done), stream);
    const size_t count = static_cast<size_t>(rows) * out_dim;
    // a pair is one launch over both matrices (grid.z)
    const BmSecond second{dst_b, weight_b_prepared, ep_b};
    hipError_t e;
    if (eight) {
        const int cols = bm8_columns(real_shares, out_dim, weight_b_prepared != nullptr), cg = (cols + 15) / 16;
#define AFHIP_BM8(T, CG, H, G) bm_launch8<T, CG, H, G>(stream, dst, partial, qa, sa, weight_prepared, rows, in_dim, out_dim, real_shares, share_blocks, cols, accumulate, quantize, ep, second)
#define AFHIP_BM8_CG(T, H, G) (cg == 4 ? AFHIP_BM8(T, 4, H, G) : (cg == 3 ? AFHIP_BM8(T, 3, H, G) : (cg == 2 ? AFHIP_BM8(T, 2, H, G) : AFHIP_BM8(T, 1, H, G))))
#define AFHIP_BM8_G(T, H) (groups == 2 ? AFHIP_BM8_CG(T, H, 2) : AFHIP_BM8_CG(T, H, 1))
        // (Q4_0: two groups of rows only on a long K, which runs four stage rounds)
        if (tensor_type == 2) e = halves == 4 ? AFHIP_BM8_G(2, 4) : AFHIP_BM8_CG(2, 2, 1);
        else e = halves == 8 ? AFHIP_BM8_G(8, 8) : (halves == 4 ? AFHIP_BM8_G(8, 4) : AFHIP_BM8_G(8, 2));
#undef AFHIP_BM8_G
#undef AFHIP_BM8_CG
#undef AFHIP_BM8
    }
    else if (column_groups)
        e = tensor_type == 2 ? bm_launch_groups<2>(stream, dst, partial, qa, sa, weight_prepared, rows, in_dim, out_dim, plan, ep, second, accumulate)
                             : bm_launch_groups<8>(stream, dst, partial, qa, sa, weight_prepared, rows, in_dim, out_dim, plan, ep, second, accumulate);
    else if (thirty_two)
        e = tensor_type == 2 ? bm_launch32<2>(stream, dst, partial, qa, sa, weight_prepared, rows, in_dim, out_dim, real_shares, share_blocks, ep, second, accumulate)
                             : bm_launch32<8>(stream, dst, partial, qa, sa, weight_prepared, rows, in_dim, out_dim, real_shares, share_blocks, ep, second, accumulate);
    else
        e = tensor_type == 2
                       ? bm_launch_rows<2>(stream, dst, partial, qa, sa, weight_prepared, rows, in_dim, out_dim, real_shares, share_blocks, ep, second, accumulate)
                       : bm_launch_rows<8>(stream, dst, partial, qa, sa, weight_prepared, rows, in_dim, out_dim, real_shares, share_blocks, ep, second, accumulate);
    if (e != hipSuccess) return e;
    if (real_shares > 1 && !accumulate) {
        e = launch_splitk_reduce(stream, dst, partial, count, out_dim, real_shares, ep);
        if (e != hipSuccess) return e;
        if (weight_b_prepared) {
            e = launch_splitk_reduce(stream, dst_b, partial + static_cast<size_t>(real_shares) * count, count, out_dim, real_shares, ep_b);
            if (e != hipSuccess) return e;
        }
    }
    return hipSuccess;
}

// The eight-row kernel's own timeline (Q4_0, one K share, a matrix the kernel takes in tiles of 49 .. 64 columns): the
// compact-fragment quantizer, then the kernel template with its stamps flag, which stores clock readings (32 bytes per
// wavefront, eight wavefronts a workgroup) into `stamps` instead of results.
hipError_t launch_batch8_timeline(hipStream_t stream, uint32_t* stamps, size_t stamps_bytes, const float* input,
                                  const uint8_t* weight_prepared, int rows, int in_dim, int out_dim, uint8_t* workspace, int* workgroups,
                                  int* columns) {
    const int kb = in_dim / 32;
    if (rows < 1 || rows > 8 || in_dim % 256 != 0 || kb > BmFormat<2>::kShareBlocks || workspace == nullptr || stamps == nullptr) return hipErrorInvalidValue;
    if (!batch_mfma_supports(2, rows, in_dim, out_dim)) return hipErrorInvalidValue;
    const int cols = bm8_columns(1, out_dim, false);
    if (cols <= 48) return hipErrorInvalidValue;
    const int groups = (out_dim + cols - 1) / cols;
    if (workgroups) *workgroups = groups;
    if (columns) *columns = cols;
    if (stamps_bytes < static_cast<size_t>(groups) * kBmWaves * 32) return hipErrorInvalidValue;
    uint32_t* qa = reinterpret_cast<uint32_t*>(workspace);
    const int pairs = (kb + 1) / 2;
    float* sa = reinterpret_cast<float*>(workspace + static_cast<size_t>(pairs) * 512);
    hipLaunchKernelGGL(quantize_fragments8_kernel<2>, dim3(static_cast<unsigned>((2 * pairs * 8 + 255) / 256), 8), dim3(256), 0, stream, input, rows, in_dim, qa, sa,
                       static_cast<float*>(nullptr), static_cast<float*>(nullptr), 0);
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    int share_blocks = (kb + BmFormat<2>::kWaveBlocks - 1) / BmFormat<2>::kWaveBlocks * BmFormat<2>::kWaveBlocks;
    static LdsLimit lds_limit;
    if (hipError_t e = allow_lds(batch8_mfma_kernel<2, 4, true>, bm8_lds_bytes(2, 4), &lds_limit); e != hipSuccess) return e;
    hipLaunchKernelGGL((batch8_mfma_kernel<2, 4, true>), dim3(static_cast<unsigned>(groups), 1, 1), dim3(kBmThreads), bm8_lds_bytes(2, 4), stream,
                       reinterpret_cast<float*>(stamps), static_cast<float*>(nullptr), qa, sa, weight_prepared, rows, in_dim, out_dim, share_blocks,
                       cols, 0, Epilogue{}, BmSecond{nullptr, nullptr, Epilogue{}});
    return hipGetLastError();
}

}  // namespace afhip
