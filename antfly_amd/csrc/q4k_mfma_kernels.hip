// GGUF Q4_K on the matrix cores: a tile-major device layout and the GEMV / small-batch
// kernel that reads it.
//
// The engine computes Q4_K on f32 activations against the dequantized weights
// w = (d * sc) * q - (dmin * m) (ops/native_compute.zig:31075-31144, CUDA backend
// ops/cuda/cuda_compute.zig:708); there is no integer route at these shapes.  Done on the
// vector ALU that is a convert and a multiply-add per weight, which bounds the kernel by
// instruction issue at a third of the HBM rate.  Here the per-weight work moves to
// v_mfma_f32_32x32x16_bf16 without giving up f32 accuracy:
//
//   * a byte 0x0n read as an fp8 (e4m3) number is n * 2^-9 (the subnormals and the first
//     binade of that format are one linear ramp), so v_cvt_scalef32_pk_bf16_fp8 with scale
//     2^9 turns two masked nibbles into the bf16 numbers n exactly, two weights per instruction;
//   * an activation x is split once per workgroup into three bf16 numbers hi + mid + lo
//     (each the bf16 rounding of what the previous ones left over), which together carry
//     24 mantissa bits; products of bf16 numbers are exact in the f32 accumulator;
//   * one MFMA pair per 32 output columns and 32-value sub-block leaves, for every
//     activation row, S = sum(n * x); with X = sum(x) of the sub-block (computed in f32 by the
//     prologue) the sub-block's contribution is
//         (d sc) * S - (dmin m) * X  =  sum(x * ((d sc) n - dmin m)).
//
// Operand mapping (D = A * B, 32 x 32 x 16): A rows are "x columns" -- row r of X occupies
// x columns 8 (r / 2) + 4 (r % 2) + {0, 1, 2} for its three parts, so that the results of
// up to eight rows land in D registers 4 (r / 2) + part of lane half r % 2 -- and B columns
// are 32 consecutive output columns.  Lane (column c, half g) supplies the K values
// 16 g + 8 m + 0..7 of the sub-block to MFMA m = 0, 1.  x columns that carry nothing read
// some valid column: every D row depends on its own A row only, and their D rows are not read.
//
// Tile-major layout ("prepared" Q4_K): for every tile of 32 output columns and every
// super-block of 256 values, 4608 bytes: the 32 headers of 16 bytes (d, dmin, 12 scale
// bytes) and then, for each of the four 32-byte chunks of nibbles, lane c + 32 g holds bytes
// 16 g .. 16 g + 15 of column c's chunk.  A wavefront's loads are 1 KiB contiguous each.
// Columns past out_dim are zero (d = dmin = 0).  Same size as the raw layout when out_dim
// is a multiple of 32.
#include <hip/hip_runtime.h>


#include <stdint.h>

#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "antfly_hip_qmatmul.h"
#include "device_common.h"
#include "qmatmul_launch.h"

namespace afhip {

namespace {

constexpr int kQ4kBlockBytes = 144;
constexpr int kQ4kBlockValues = 256;
constexpr int kTileCols = 32;
constexpr int kTileBytes = 4608;        // 32 * 16 + 4 * 64 * 16
constexpr int kTileUnits = kTileBytes / 16;
constexpr int kRowPadBytes = 48;        // LDS stride of an x column: 2 K + 48 spreads the columns over the banks
constexpr int kMaxRowsPerLaunch = 8;
constexpr size_t kLdsBudget = 160 * 1024 - 512;  // of the 160 KiB a workgroup can have

typedef uint32_t t_u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 t_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 t_bf16x2 __attribute__((ext_vector_type(2)));
typedef float t_f32x2 __attribute__((ext_vector_type(2)));
typedef float t_f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float ubyte_to_f32(uint32_t word, int index) {
    return static_cast<float>((word >> (8 * index)) & 0xFFu);  // index is a compile-time constant at every use
}

// ------------------------------------------------------------------ layout
__global__ __launch_bounds__(256) void q4k_tile_repack_kernel(t_u32x4* __restrict__ dst, const uint8_t* __restrict__ src,
                                                              int out_dim, int kb, size_t units) {
    for (size_t u = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; u < units;
         u += static_cast<size_t>(gridDim.x) * blockDim.x) {
        const size_t region = u / kTileUnits;
        const int w = static_cast<int>(u - region * kTileUnits);
        const size_t tile = region / kb;
        const int sb = static_cast<int>(region - tile * kb);
        int c, offset;
        if (w < kTileCols) {
            c = w;
            offset = 0;
        } else {
            const int q = w - kTileCols, chunk = q >> 6, lane = q & 63;
            c = lane & 31;
            offset = 16 + 32 * chunk + 16 * (lane >> 5);
        }
        const size_t o = tile * kTileCols + c;
        t_u32x4 v = {0u, 0u, 0u, 0u};
        if (o < static_cast<size_t>(out_dim))
            v = *reinterpret_cast<const t_u32x4*>(src + (o * kb + sb) * kQ4kBlockBytes + offset);
        dst[u] = v;
    }
}

// get_rows / cpy_q_to_f32 from the tile-major layout; arithmetic as dequantizeQ4K,
// gguf/quant_codec.zig:2624-2663 (see dequantize_q4k_rows_kernel for the raw layout).
__global__ __launch_bounds__(256) void dequantize_q4k_tiled_rows_kernel(float* __restrict__ dst,
                                                                        const uint8_t* __restrict__ weight,
                                                                        const long long* __restrict__ ids, size_t rows,
                                                                        int dim, size_t weight_rows) {
    const size_t per_row = static_cast<size_t>(dim >> 2);
    const size_t units = rows * per_row;
    const size_t kb = static_cast<size_t>(dim / kQ4kBlockValues);
    for (size_t u = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; u < units;
         u += static_cast<size_t>(gridDim.x) * blockDim.x) {
        const size_t t = u / per_row;
        const int g = static_cast<int>(u - t * per_row);  // group of four values in the row
        const long long row = ids ? ids[t] : static_cast<long long>(t);
        if (row < 0 || static_cast<size_t>(row) >= weight_rows) {  // an id outside the weight reads nothing: zeros
            reinterpret_cast<float4*>(dst)[u] = float4{0.0f, 0.0f, 0.0f, 0.0f};
            continue;
        }
        const size_t o = static_cast<size_t>(row);
        const int v0 = (g & 63) * 4;                      // first value inside the super-block
        const int chunk = v0 >> 6, pos = v0 & 63, byte = pos & 31;
        const int sub = chunk * 2 + (pos >> 5);
        const int c = static_cast<int>(o & 31);
        const uint8_t* base = weight + ((o >> 5) * kb + (g >> 6)) * kTileBytes;
        const t_u32x4 header = *reinterpret_cast<const t_u32x4*>(base + 16 * c);
        const uint32_t packed =
            *reinterpret_cast<const uint32_t*>(base + 512 + chunk * 1024 + (c + 32 * (byte >> 4)) * 16 + (byte & 15));
        const uint32_t nib = (pos < 32 ? packed : packed >> 4) & 0x0F0F0F0Fu;
        const int shift = (sub & 3) * 8;
        const uint32_t a = (header.y >> shift) & 0xFFu, b = (header.z >> shift) & 0xFFu, cc = (header.w >> shift) & 0xFFu;
        const uint32_t s = sub < 4 ? (a & 63u) : ((cc & 0x0Fu) | ((a >> 6) << 4));
        const uint32_t m = sub < 4 ? (b & 63u) : ((cc >> 4) | ((b >> 6) << 4));
        const float dsc = half_bits_to_f32(static_cast<uint16_t>(header.x & 0xFFFFu)) * static_cast<float>(s);
        const float dmn = half_bits_to_f32(static_cast<uint16_t>(header.x >> 16)) * static_cast<float>(m);
        float4 out;
        out.x = dsc * ubyte_to_f32(nib, 0) - dmn;
        out.y = dsc * ubyte_to_f32(nib, 1) - dmn;
        out.z = dsc * ubyte_to_f32(nib, 2) - dmn;
        out.w = dsc * ubyte_to_f32(nib, 3) - dmn;
        typedef float f32x4_t __attribute__((ext_vector_type(4)));  // written once, read by someone else: streamed past the caches
        __builtin_nontemporal_store(f32x4_t{out.x, out.y, out.z, out.w}, reinterpret_cast<f32x4_t*>(dst) + u);
    }
}

// ------------------------------------------------------------------ GEMV
// Two floats as a packed pair of bf16 numbers (round to nearest even): v_cvt_pk_bf16_f32.
__device__ __forceinline__ uint32_t bf16_pair(float a, float b) {
    const t_f32x2 v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, t_bf16x2));
}

// What a finite v leaves over after its bf16 rounding (bits in the upper half of `rounded`);
// infinities and NaNs leave nothing (they stay in the first part alone).
__device__ __forceinline__ float bf16_rest(float v, uint32_t rounded_high) {
    return __builtin_fabsf(v) < __builtin_inff() ? v - __uint_as_float(rounded_high) : 0.0f;
}

// hi + mid + lo = (a, b) to 2^-25 of their size: three packed bf16 pairs.
__device__ __forceinline__ void split3_pair(float a, float b, uint32_t* hi, uint32_t* mid, uint32_t* lo) {
    const uint32_t h = bf16_pair(a, b);
    const float ra = bf16_rest(a, h << 16), rb = bf16_rest(b, h & 0xFFFF0000u);
    const uint32_t m = bf16_pair(ra, rb);
    *hi = h;
    *mid = m;
    *lo = bf16_pair(ra - __uint_as_float(m << 16), rb - __uint_as_float(m & 0xFFFF0000u));
}

extern __shared__ __align__(16) unsigned char q4k_mfma_lds[];

// kGroups = ceil(rows / 2) row groups (D registers 0 .. 4 kGroups - 1 are read);
// kFlight super-blocks of weights are requested before any of them is used.
// kOwnSlice (one tile per workgroup: the wavefronts partition K): a wavefront splits the slice of X
// that it alone multiplies, four values per lane, and goes on without waiting for the others --
// no workgroup barrier between the split and the matrix work, so wavefronts whose weights have
// arrived start at once and the vector work spreads over the time the stream takes.
template <int kGroups, int kFlight, int kMaxThreads = 512, bool kOwnSlice = false>
__global__ __launch_bounds__(kMaxThreads) void gemv_q4k_mfma_kernel(float* __restrict__ dst, const float* __restrict__ x,
                                                            const uint8_t* __restrict__ weight, int rows, int in_dim,
                                                            int out_dim, int slices, int sb_per_slice, Epilogue ep) {
    const int kb = in_dim >> 8;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int threads = static_cast<int>(blockDim.x), waves = threads >> 6;
    const int row_stride = in_dim * 2 + kRowPadBytes;  // bytes per x column
    unsigned char* xparts = q4k_mfma_lds;  // [rows * 3][row_stride]: the three parts of every row
    float* xsum = reinterpret_cast<float*>(q4k_mfma_lds + static_cast<size_t>(rows) * 3 * row_stride);  // [rows][kb * 8]
    float* partial = xsum + rows * kb * 8;                                                       // [waves][kGroups][64]

    const int tiles_per_wg = waves / slices;
    const int n_tiles = (out_dim + kTileCols - 1) >> 5;
    const int tile_raw = blockIdx.x * tiles_per_wg + wave / slices;
    const bool tile_ok = tile_raw < n_tiles;
    const int tile = tile_ok ? tile_raw : n_tiles - 1;  // spare wavefronts load nothing and store nothing
    const int slice = wave % slices;
    const int sb_begin = slice * sb_per_slice;
    const int sb_end = min(kb, sb_begin + sb_per_slice);
    const uint8_t* tile_base = weight + static_cast<size_t>(tile) * kb * kTileBytes;

    t_u32x4 hdr[kFlight], qv[kFlight][4];
    auto request = [&](int sb_first) {
#pragma unroll
        for (int f = 0; f < kFlight; ++f) {
            const int sb = sb_first + f;
            if (!(tile_ok && sb < sb_end)) continue;  // wave-uniform; the same test guards the use below
            const uint8_t* base = tile_base + static_cast<size_t>(sb) * kTileBytes;
            hdr[f] = __builtin_nontemporal_load(reinterpret_cast<const t_u32x4*>(base + 16 * (lane & 31)));
#pragma unroll
            for (int t = 0; t < 4; ++t)
                qv[f][t] = __builtin_nontemporal_load(reinterpret_cast<const t_u32x4*>(base + 512 + t * 1024 + 16 * lane));
        }
    };

    if (kOwnSlice) {
        // ---- 1. this wavefront's slice of X: item i = (row i / n_sb, super-block sb_begin + i % n_sb)
        const int n_sb = max(sb_end - sb_begin, 0), n_items = rows * n_sb;
        auto item_ptr = [&](int i) {
            const int r = i / n_sb, sb = sb_begin + (i - r * n_sb);
            return reinterpret_cast<const float4*>(x + static_cast<size_t>(r) * in_dim + sb * kQ4kBlockValues) + lane;
        };
        auto split_item = [&](int i, const float4 v) {
            const int r = i / n_sb, sb = sb_begin + (i - r * n_sb);
            uint32_t p[3][2];
            split3_pair(v.x, v.y, &p[0][0], &p[1][0], &p[2][0]);
            split3_pair(v.z, v.w, &p[0][1], &p[1][1], &p[2][1]);
#pragma unroll
            for (int part = 0; part < 3; ++part)
                *reinterpret_cast<uint2*>(xparts + static_cast<size_t>(r * 3 + part) * row_stride + (sb * kQ4kBlockValues + 4 * lane) * 2) =
                    make_uint2(p[part][0], p[part][1]);
            const float s = sum_over_8((v.x + v.y) + (v.z + v.w));
            if ((lane & 7) == 0) xsum[r * (kb * 8) + sb * 8 + (lane >> 3)] = s;
        };
        constexpr int kAhead = 2;  // items requested before the weights (one row, or two rows, of a one-super-block slice)
        float4 first[kAhead];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) first[i] = i < n_items ? *item_ptr(i) : make_float4(0.f, 0.f, 0.f, 0.f);
        __builtin_amdgcn_sched_barrier(0);
        request(sb_begin);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < kAhead; ++i)
            if (i < n_items) split_item(i, first[i]);
        for (int i = kAhead; i < n_items; ++i) split_item(i, *item_ptr(i));
        // the wavefront reads back what its own lanes wrote: LDS operations of a wavefront complete in order
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
    // ---- 1. X: requested first, split into bf16 parts while the weights are on their way
    const int groups_per_row = in_dim >> 3;
    const int n_groups = rows * groups_per_row;
    int grp = tid;
    float4 xa = make_float4(0.f, 0.f, 0.f, 0.f), xb = xa;
    if (grp < n_groups) {
        xa = reinterpret_cast<const float4*>(x)[grp * 2];
        xb = reinterpret_cast<const float4*>(x)[grp * 2 + 1];
    }
    __builtin_amdgcn_sched_barrier(0);
    request(sb_begin);
    __builtin_amdgcn_sched_barrier(0);
    // every lane of a quad takes part in the sums below, so the loop runs for whole quads
    for (int base_grp = tid & ~3; base_grp < n_groups; base_grp += threads) {
        const bool mine = grp < n_groups;
        const float v[8] = {xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w};
        uint32_t p[3][4];
#pragma unroll
        for (int i = 0; i < 4; ++i) split3_pair(v[2 * i], v[2 * i + 1], &p[0][i], &p[1][i], &p[2][i]);
        float s = mine ? ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7])) : 0.0f;
        s += dpp_move<kDppXor1>(s);
        s += __shfl_xor(s, 2);
        if (mine) {
            const int r = grp / groups_per_row, kg = grp - r * groups_per_row;
#pragma unroll
            for (int part = 0; part < 3; ++part)
                *reinterpret_cast<uint4*>(xparts + static_cast<size_t>(r * 3 + part) * row_stride + kg * 16) =
                    make_uint4(p[part][0], p[part][1], p[part][2], p[part][3]);
            if ((tid & 3) == 0) xsum[r * (kb * 8) + (kg >> 2)] = s;
        }
        grp += threads;
        if (grp < n_groups) {
            xa = reinterpret_cast<const float4*>(x)[grp * 2];
            xb = reinterpret_cast<const float4*>(x)[grp * 2 + 1];
        }
    }
    __syncthreads();
    }

    // ---- 2. this lane's roles
    const int c = lane & 31, g = lane >> 5;
    // A operand: x column c of the MFMA = part (c & 3) of row 2 (c >> 3) + ((c >> 2) & 1)
    const int a_row = 2 * (c >> 3) + ((c >> 2) & 1), a_part = c & 3;
    const bool a_live = a_part < 3 && (c >> 3) < kGroups && a_row < rows;
    // (a lane without a part reads the first column: its D row is never looked at)
    const unsigned char* a_base = xparts + static_cast<size_t>(a_live ? a_row * 3 + a_part : 0) * row_stride + 32 * g;
    // results: D register 4 G + part of this lane belongs to row 2 G + g, output column c of the tile
    float acc[kGroups];
    const float* xsum_row[kGroups];
#pragma unroll
    for (int G = 0; G < kGroups; ++G) {
        acc[G] = 0.0f;
        xsum_row[G] = xsum + min(2 * G + g, rows - 1) * (kb * 8);
    }

    for (int sb_first = sb_begin; sb_first < sb_end; sb_first += kFlight) {
        if (sb_first != sb_begin) request(sb_first);
#pragma unroll
        for (int f = 0; f < kFlight; ++f) {
            const int sb = sb_first + f;
            if (!(tile_ok && sb < sb_end)) continue;  // wave-uniform: nothing was requested for it
            const t_u32x4 h = hdr[f];
            const float d = half_bits_to_f32(static_cast<uint16_t>(h.x & 0xFFFFu));
            const float dmin = half_bits_to_f32(static_cast<uint16_t>(h.x >> 16));
            // the eight 6-bit scales and mins as bytes of four words (unpackQ4KScaleMinsU8,
            // ops/native_compute.zig:33745-33754)
            const uint32_t sc_lo = h.y & 0x3F3F3F3Fu, mn_lo = h.z & 0x3F3F3F3Fu;
            const uint32_t sc_hi = (h.w & 0x0F0F0F0Fu) | ((h.y >> 2) & 0x30303030u);
            const uint32_t mn_hi = ((h.w >> 4) & 0x0F0F0F0Fu) | ((h.z >> 2) & 0x30303030u);
            const unsigned char* a_sb = a_base + sb * 512;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                // bytes 0x0n: the low and the high nibbles of this lane's 16 bytes of chunk t
                const uint32_t w[4] = {qv[f][t].x, qv[f][t].y, qv[f][t].z, qv[f][t].w};
                uint32_t nib[2][4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    nib[0][k] = w[k] & 0x0F0F0F0Fu;
                    nib[1][k] = (w[k] >> 4) & 0x0F0F0F0Fu;
                }
#pragma unroll
                for (int hi = 0; hi < 2; ++hi) {  // low nibbles: sub-block 2 t, high nibbles: 2 t + 1
                    const int sub = 2 * t + hi;
                    // (one accumulator set: a second one for the other sub-block costs a wavefront of occupancy)
                    t_f32x16 D = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int m = 0; m < 2; ++m) {
                        union {
                            t_bf16x8 v;
                            t_bf16x2 pair[4];
                            uint4 u;
                        } a, b;
                        // fp8 0x0n = n * 2^-9; times 2^9: the bf16 numbers n, two per instruction
                        b.pair[0] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(static_cast<int>(nib[hi][2 * m]), 512.0f, false);
                        b.pair[1] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(static_cast<int>(nib[hi][2 * m]), 512.0f, true);
                        b.pair[2] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(static_cast<int>(nib[hi][2 * m + 1]), 512.0f, false);
                        b.pair[3] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(static_cast<int>(nib[hi][2 * m + 1]), 512.0f, true);
                        a.u = *reinterpret_cast<const uint4*>(a_sb + (32 * sub + 8 * m) * 2);
                        D = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.v, b.v, D, 0, 0, 0);
                    }
                    const float sc = ubyte_to_f32(sub < 4 ? sc_lo : sc_hi, sub & 3);
                    const float mn = ubyte_to_f32(sub < 4 ? mn_lo : mn_hi, sub & 3);
                    const float dsc = d * sc, dmn = dmin * mn;
#pragma unroll
                    for (int G = 0; G < kGroups; ++G) {
                        const float X = xsum_row[G][sb * 8 + sub];
                        const float S = (D[4 * G] + D[4 * G + 1]) + D[4 * G + 2];
                        acc[G] = __builtin_fmaf(dsc, S, acc[G]);
                        acc[G] = __builtin_fmaf(-dmn, X, acc[G]);
                    }
                }
            }
        }
    }

    // ---- 3. K-slices meet in LDS, in slice order
#pragma unroll
    for (int G = 0; G < kGroups; ++G) partial[(wave * kGroups + G) * 64 + lane] = acc[G];
    __syncthreads();
    const int cells = tiles_per_wg * kGroups * 64;
    for (int i = tid; i < cells; i += threads) {
        const int ti = i / (kGroups * 64), rem = i - ti * (kGroups * 64);
        const int G = rem >> 6, ln = rem & 63;
        float total = 0.0f;
        for (int sl = 0; sl < slices; ++sl) total += partial[((ti * slices + sl) * kGroups + G) * 64 + ln];
        const int row = 2 * G + (ln >> 5);
        const int o = (blockIdx.x * tiles_per_wg + ti) * kTileCols + (ln & 31);
        if (row < rows && o < out_dim) {
            const size_t idx = static_cast<size_t>(row) * out_dim + o;
            dst[idx] = finish_output(ep, o, idx, total);
        }
    }
}


// ------------------------------------------------------------------ one to four rows on the int8 matrix core
// The masked nibble bytes 0x0n are int8 numbers as they stand, so with integer activations a
// sub-block costs no conversion at all and one v_mfma_i32_32x32x32_i8.  X keeps f32 accuracy as
// fixed point: per super-block of 256 values a power of two 2^s with |x| * 2^s < 2^30, q =
// trunc(x * 2^s) (31 bits with sign) written with four signed base-256 digits q = d3 * 2^24 +
// d2 * 2^16 + d1 * 2^8 + d0, every d in -128..127: they are the bytes of (q + 0x80808080) ^
// 0x80808080 (adding 128 to every byte position with the carries, then taking 128 off every
// byte) -- four int8 planes that take MFMA rows 4 * row + digit.  The digit dots of a sub-block
// are exact int32; the eight sub-blocks of a super-block are added as integers, each times its
// 6-bit scale (at most 63 * 32 * 128 * 15 * 8 < 2^25), and only the super-block's four sums
// become floats:
//   y += d * (2^-s * (((D3 * 256 + D2) * 256 + D1) * 256 + D0))  -  dmin * sum_sub m_sub * X_sub.
// Against the three-part bf16 kernel: no conversions (64 per super-block and wavefront), half the
// MFMAs, integer multiply-adds instead of float sums per sub-block; the truncation error is
// 2^-30 of the super-block's largest |x| per value (the bf16 parts: 2^-25 of each value).
// A super-block that holds an infinity or a NaN gives NaN in every column.
// Every wavefront prepares the K slice it alone multiplies (no workgroup barrier before the matrix
// work); one tile per workgroup, its wavefronts partition K.
typedef int t_i32x4 __attribute__((ext_vector_type(4)));
typedef int t_i32x16 __attribute__((ext_vector_type(16)));

constexpr int kDigitPadBytes = 48;  // LDS stride of a digit plane: K + 48 spreads the planes over the banks

// One super-block of one row, four values a lane: the lane's word of each of the four digit planes, -s as a
// number (NaN for a block with an infinity or a NaN in it), and the f32 sum of the lane's sub-block (lane >> 3).
struct Q4kDigits {
    uint32_t plane[4];
    float minus_s;
    float sub_sum;
};
__device__ __forceinline__ Q4kDigits q4k_digit_planes(const float4 v) {
    float m = fmaxf(fmaxf(__builtin_fabsf(v.x), __builtin_fabsf(v.y)), fmaxf(__builtin_fabsf(v.z), __builtin_fabsf(v.w)));
    m = max_over_8(m);
    m = fmaxf(m, dpp_move<kDppRowMirror>(m));  // 16-lane row maximum in every lane
    const int mb = __builtin_bit_cast(int, m);
    m = fmaxf(fmaxf(__builtin_bit_cast(float, __builtin_amdgcn_readlane(mb, 0)),
                    __builtin_bit_cast(float, __builtin_amdgcn_readlane(mb, 16))),
              fmaxf(__builtin_bit_cast(float, __builtin_amdgcn_readlane(mb, 32)),
                    __builtin_bit_cast(float, __builtin_amdgcn_readlane(mb, 48))));
    // |x| < 2^(e - 126) (subnormals: e = 1): times 2^(156 - e) it stays below 2^30.  The exponent goes by
    // v_ldexp_f32 both ways (2^(156 - e) itself is past the f32 range for small e).
    const int e_raw = (__builtin_bit_cast(int, m) >> 23) & 0xFF;
    const int e = e_raw < 1 ? 1 : e_raw;
    Q4kDigits out;
    out.minus_s = e_raw == 255 ? __builtin_nanf("") : static_cast<float>(e - 156);
    const float vv[4] = {v.x, v.y, v.z, v.w};
    uint32_t t[4];  // the four signed digits of each value, lowest in byte 0
#pragma unroll
    for (int k = 0; k < 4; ++k)
        t[k] = (static_cast<uint32_t>(static_cast<int>(__builtin_ldexpf(vv[k], 156 - e))) + 0x80808080u) ^ 0x80808080u;
    // 4 x 4 byte transpose: plane[d] = digit d of the lane's four values (v_perm_b32: selectors 0..3 take
    // bytes of the second operand, 4..7 of the first)
    const uint32_t lo01 = __builtin_amdgcn_perm(t[1], t[0], 0x05010400u), hi01 = __builtin_amdgcn_perm(t[1], t[0], 0x07030602u);
    const uint32_t lo23 = __builtin_amdgcn_perm(t[3], t[2], 0x05010400u), hi23 = __builtin_amdgcn_perm(t[3], t[2], 0x07030602u);
    out.plane[0] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u);
    out.plane[1] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u);
    out.plane[2] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u);
    out.plane[3] = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u);
    out.sub_sum = sum_over_8((v.x + v.y) + (v.z + v.w));
    return out;
}

// The digit planes of up to eight rows made once, for the kernel below with kPlanesGiven: in MFMA
// operand order -- 1 KB per (super-block, sub-block): lane (MFMA row c = 4 * row + digit, half g) holds
// its 16 bytes (K = 16 g .. 16 g + 15 of the sub-block) at 16 * (32 g + c) -- so a wavefront's operand is
// one contiguous load; then -s per (row, super-block) and the sub-block sums.  One wavefront per item.
// zero_a (and zero_b): result arrays of zero_count floats that the matmul launch behind this one adds its two K shares'
// sums to; cleared here, by the launch that has to run first anyway.
__global__ __launch_bounds__(256) void q4k_digit_planes_kernel(const float* __restrict__ x, int rows, int in_dim,
                                                               uint8_t* __restrict__ frag, float* __restrict__ minus_s,
                                                               float* __restrict__ sub_sums, float* __restrict__ zero_a,
                                                               float* __restrict__ zero_b, int zero_count) {
    if (zero_a != nullptr) {
        for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < zero_count; i += gridDim.x * blockDim.x) {
            zero_a[i] = 0.0f;
            if (zero_b != nullptr) zero_b[i] = 0.0f;
        }
    }
    const int kb = in_dim >> 8, lane = threadIdx.x & 63;
    const int item = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (item >= rows * kb) return;
    const int r = item / kb, sb = item - r * kb;
    const Q4kDigits dg = q4k_digit_planes(reinterpret_cast<const float4*>(x + static_cast<size_t>(r) * in_dim + sb * kQ4kBlockValues)[lane]);
    // the lane's values are K = 4 (lane % 8) .. + 3 of sub-block lane / 8: half g = (lane % 8) / 4, bytes 4 (lane % 4) ..
    uint8_t* base = frag + (static_cast<size_t>(sb) * 8 + (lane >> 3)) * 1024 + (32 * ((lane & 7) >> 2) + 4 * r) * 16 + 4 * (lane & 3);
#pragma unroll
    for (int d = 0; d < 4; ++d) *reinterpret_cast<uint32_t*>(base + 16 * d) = dg.plane[d];
    if ((lane & 7) == 0) sub_sums[(static_cast<size_t>(r) * kb + sb) * 8 + (lane >> 3)] = dg.sub_sum;
    if (lane == 0) minus_s[r * kb + sb] = dg.minus_s;
}

// Clears result arrays ahead of a launch whose two K shares add to them (one or two rows: no launch of its own precedes).
__global__ __launch_bounds__(256) void q4k_zero_results_kernel(float* __restrict__ a, float* __restrict__ b, int count) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < count; i += gridDim.x * blockDim.x) {
        a[i] = 0.0f;
        if (b != nullptr) b[i] = 0.0f;
    }
}

// kGroups = ceil(rows / 2) row groups: row r sits in lane half r % 2, D registers 4 (r / 2) + digit.
// kPlanesGiven: the digit planes, -s and the sub-block sums come from q4k_digit_planes_kernel (`frag`, `frag_scale`,
// `frag_sums`) instead of being made here from `x`: the MFMA operand is then a 16-byte load per lane and sub-block,
// requested with the weights, and nothing of X passes through LDS but the few floats of the wavefront's own slice.
// A second matrix of the same shape on the same X (gate and up: grid.y = 2): one launch for both.
// K shares (grid.z = 2, `accumulate`): a matrix with so few column tiles that half the compute units would stay idle
// gives each tile to two workgroups, each with half of K; both add their sums to the result array, cleared beforehand,
// with a float atomic -- two addends on a zero give the same float in either order.  No epilogue then.
// kHalfTile (one row): a workgroup takes sixteen of a tile's columns and all of K.  Lanes with c < 16 hold those columns of
// one super-block, the others the same columns of the next one; the digits of the two super-blocks are MFMA rows 0 .. 3 and
// 4 .. 7, so that columns 0 .. 15 find theirs in the lower lanes and columns 16 .. 31 theirs in the upper ones: as many live
// results per MFMA as a whole tile gives one row.  Twice the workgroups of whole tiles, without K shares and the launch that
// clears their result.
// kByParity: whole tiles with the sums of half tiles, bit for bit: the even and the odd super-blocks of a slice apart.
struct Q4kSecond {
    float* dst;
    const uint8_t* weight;
    Epilogue ep;
};

template <int kGroups, int kFlight, int kMaxThreads, bool kPlanesGiven = false, bool kHalfTile = false, bool kByParity = false>
__global__ __launch_bounds__(kMaxThreads, kMaxThreads == 1024 && kFlight == 1 && !kHalfTile ? 8 : 4) void gemv_q4k_i8_kernel(float* __restrict__ dst_a, const float* __restrict__ x,
                                                                  const uint8_t* __restrict__ weight_a, int rows, int in_dim,
                                                                  int out_dim, int slices, int sb_per_slice, Epilogue ep_a,
                                                                  const uint8_t* __restrict__ frag, const float* __restrict__ frag_scale,
                                                                  const float* __restrict__ frag_sums, Q4kSecond second, int accumulate) {
    const bool is_b = blockIdx.y != 0;
    float* dst = is_b ? second.dst : dst_a;
    const uint8_t* weight = is_b ? second.weight : weight_a;
    const Epilogue ep = is_b ? second.ep : ep_a;
    const int kb = in_dim >> 8;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int threads = static_cast<int>(blockDim.x);
    const int plane_stride = in_dim + kDigitPadBytes;
    unsigned char* xdig = q4k_mfma_lds;  // [rows * 4][plane_stride]: the digit planes of every row (not with kPlanesGiven)
    float* xscale = reinterpret_cast<float*>(q4k_mfma_lds + (kPlanesGiven ? 0 : static_cast<size_t>(rows) * 4 * plane_stride));  // [rows][kb]: -s
    float* xsum = xscale + ((rows * kb + 3) & ~3);                                                          // [rows][kb * 8], 16-byte aligned
    float* partial = xsum + rows * kb * 8;                                                                  // [waves][kGroups][64]

    static_assert(!(kHalfTile || kByParity) || (kGroups == 1 && !kPlanesGiven), "one row, its digits made here");
    static_assert(!kByParity || (!kHalfTile && kFlight == 2), "a slice begins with an even super-block");
    constexpr int kStep = kHalfTile ? 2 : 1;  // super-blocks a lane set of requests covers
    const int n_tiles = (out_dim + kTileCols - 1) >> 5;
    const int my_tile = kHalfTile ? blockIdx.x >> 1 : blockIdx.x, col0 = kHalfTile ? 16 * (blockIdx.x & 1) : 0;
    const int tile = my_tile < n_tiles ? my_tile : n_tiles - 1;
    const int slice = static_cast<int>(blockIdx.z) * slices + wave;  // one tile per workgroup and K share: blockDim.x = 64 * slices
    const int sb_begin = slice * sb_per_slice;
    const int sb_end = min(kb, sb_begin + sb_per_slice);
    const uint8_t* tile_base = weight + static_cast<size_t>(tile) * kb * kTileBytes;

    // MFMA row c = digit (c & 3) of row (c >> 2); rows past the last read row 0's first plane (their D rows are
    // never looked at).  Lane half g supplies K = 16 g .. 16 g + 15.
    const int c = lane & 31, g = lane >> 5;
    const int a_lane = 32 * g + ((c >> 2) < rows ? c : 0);
    t_u32x4 hdr[kFlight], qv[kFlight][4];
    t_i32x4 av[kPlanesGiven ? kFlight : 1][8];
    auto request = [&](int sb_first) {
#pragma unroll
        for (int f = 0; f < kFlight; ++f) {
            const int sb = sb_first + kStep * f;
            if (sb >= sb_end) continue;  // wave-uniform; the same test guards the use below
            if constexpr (kHalfTile) {
                const uint32_t at = static_cast<uint32_t>(min(sb + (c >> 4), sb_end - 1)) * kTileBytes + 16 * (col0 + (c & 15));
                hdr[f] = __builtin_nontemporal_load(reinterpret_cast<const t_u32x4*>(tile_base + at));
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    qv[f][t] = __builtin_nontemporal_load(reinterpret_cast<const t_u32x4*>(tile_base + (at + 512 * g) + (512 + t * 1024)));
                continue;
            }
            const uint8_t* base = tile_base + static_cast<size_t>(sb) * kTileBytes;
            hdr[f] = __builtin_nontemporal_load(reinterpret_cast<const t_u32x4*>(base + 16 * (lane & 31)));
#pragma unroll
            for (int t = 0; t < 4; ++t)
                qv[f][t] = __builtin_nontemporal_load(reinterpret_cast<const t_u32x4*>(base + 512 + t * 1024 + 16 * lane));
            if (kPlanesGiven) {
#pragma unroll
                for (int sub = 0; sub < 8; ++sub)
                    av[f][sub] = *reinterpret_cast<const t_i32x4*>(frag + (static_cast<size_t>(sb) * 8 + sub) * 1024 + a_lane * 16);
            }
        }
    };

    if (kPlanesGiven) {
        // ---- 1. the weights and operands first, then the few floats of this wavefront's slice: -s and the sub-block sums
        request(sb_begin);
        for (int sb = sb_begin; sb < sb_end; ++sb) {
            if (lane < 8 * rows) xsum[(lane >> 3) * (kb * 8) + sb * 8 + (lane & 7)] = frag_sums[(static_cast<size_t>(lane >> 3) * kb + sb) * 8 + (lane & 7)];
            if (lane < rows) xscale[lane * kb + sb] = frag_scale[lane * kb + sb];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
    // ---- 1. this wavefront's slice of X: item i = (row i / n_sb, super-block sb_begin + i % n_sb), four values a lane
    {
        const int n_sb = max(sb_end - sb_begin, 0), n_items = rows * n_sb;
        auto item_ptr = [&](int i) {
            const int r = i / n_sb, sb = sb_begin + (i - r * n_sb);
            return reinterpret_cast<const float4*>(x + static_cast<size_t>(r) * in_dim + sb * kQ4kBlockValues) + lane;
        };
        auto digits_of_item = [&](int i, const float4 v) {
            const int r = i / n_sb, sb = sb_begin + (i - r * n_sb);
            const Q4kDigits dg = q4k_digit_planes(v);
#pragma unroll
            for (int d = 0; d < 4; ++d)
                *reinterpret_cast<uint32_t*>(xdig + static_cast<size_t>(r * 4 + d) * plane_stride + sb * kQ4kBlockValues + 4 * lane) = dg.plane[d];
            if ((lane & 7) == 0) xsum[r * (kb * 8) + sb * 8 + (lane >> 3)] = dg.sub_sum;
            if (lane == 0) xscale[r * kb + sb] = dg.minus_s;
        };
        constexpr int kAhead = kHalfTile ? 2 * kFlight : 2;  // items requested before the weights (one row, or two rows, of a one-super-block slice; a half tile's whole slice)
        float4 first[kAhead];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) first[i] = i < n_items ? *item_ptr(i) : make_float4(0.f, 0.f, 0.f, 0.f);
        __builtin_amdgcn_sched_barrier(0);
        request(sb_begin);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < kAhead; ++i)
            if (i < n_items) digits_of_item(i, first[i]);
        for (int i = kAhead; i < n_items; ++i) digits_of_item(i, *item_ptr(i));
        // the wavefront reads back what its own lanes wrote: LDS operations of a wavefront complete in order
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    }

    // ---- 2. this lane's roles
    const bool a_live = (c >> 2) < rows;
    const unsigned char* a_base = xdig + static_cast<size_t>(kHalfTile ? c & 3 : (a_live ? c : 0)) * plane_stride + 16 * g;
    // results: D registers 4 G .. 4 G + 3 (digits) of lane half g belong to row 2 G + g, output column c of the tile
    const float* xsum_row[kGroups];
    const float* xscale_row[kGroups];
    float acc[kGroups], odd = 0.0f;  // (odd: kByParity)
#pragma unroll
    for (int G = 0; G < kGroups; ++G) {
        const int my_row = min(2 * G + g, rows - 1);
        xsum_row[G] = xsum + my_row * (kb * 8);
        xscale_row[G] = xscale + my_row * kb;
        acc[G] = 0.0f;
    }

    for (int sb_first = sb_begin; sb_first < sb_end; sb_first += kStep * kFlight) {
        if (sb_first != sb_begin) request(sb_first);
#pragma unroll
        for (int f = 0; f < kFlight; ++f) {
            const int sb_step = sb_first + kStep * f;
            if (sb_step >= sb_end) continue;  // wave-uniform: nothing was requested for it
            const int sb = kHalfTile ? min(sb_step + (c >> 4), sb_end - 1) : sb_step;  // the lane's own
            const int a_sb_at = kHalfTile ? min(sb_step + ((c >> 2) & 1), sb_end - 1) : sb_step;
            const t_u32x4 h = hdr[f];
            const float d = half_bits_to_f32(static_cast<uint16_t>(h.x & 0xFFFFu));
            const float dmin = half_bits_to_f32(static_cast<uint16_t>(h.x >> 16));
            // the eight 6-bit scales and mins as bytes of four words (unpackQ4KScaleMinsU8,
            // ops/native_compute.zig:33745-33754)
            const uint32_t sc_lo = h.y & 0x3F3F3F3Fu, mn_lo = h.z & 0x3F3F3F3Fu;
            const uint32_t sc_hi = (h.w & 0x0F0F0F0Fu) | ((h.y >> 2) & 0x30303030u);
            const uint32_t mn_hi = ((h.w >> 4) & 0x0F0F0F0Fu) | ((h.z >> 2) & 0x30303030u);
            const unsigned char* a_sb = a_base + a_sb_at * kQ4kBlockValues;
            // the sub-block sums of a row group: all eight at once for one or two groups, one by one for more (registers)
            constexpr bool kSumsAhead = kGroups <= 2;
            float xs[kSumsAhead ? kGroups : 1][8];
            int digit_sum[kGroups][4];
            float min_sum[kGroups];
#pragma unroll
            for (int G = 0; G < kGroups; ++G) {
                if (kSumsAhead) {
                    const float4 xs_lo = *reinterpret_cast<const float4*>(xsum_row[G] + sb * 8);
                    const float4 xs_hi = *reinterpret_cast<const float4*>(xsum_row[G] + sb * 8 + 4);
                    xs[G][0] = xs_lo.x, xs[G][1] = xs_lo.y, xs[G][2] = xs_lo.z, xs[G][3] = xs_lo.w;
                    xs[G][4] = xs_hi.x, xs[G][5] = xs_hi.y, xs[G][6] = xs_hi.z, xs[G][7] = xs_hi.w;
                }
                digit_sum[G][0] = digit_sum[G][1] = digit_sum[G][2] = digit_sum[G][3] = 0;
                min_sum[G] = 0.0f;
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
#pragma unroll
                for (int hi = 0; hi < 2; ++hi) {  // low nibbles: sub-block 2 t, high nibbles: 2 t + 1
                    const int sub = 2 * t + hi;
                    const uint32_t w[4] = {qv[f][t].x, qv[f][t].y, qv[f][t].z, qv[f][t].w};
                    t_i32x4 b;
#pragma unroll
                    for (int k = 0; k < 4; ++k) b[k] = static_cast<int>((hi ? w[k] >> 4 : w[k]) & 0x0F0F0F0Fu);
                    const t_i32x4 a = kPlanesGiven ? av[f][sub] : *reinterpret_cast<const t_i32x4*>(a_sb + 32 * sub);
                    const t_i32x16 zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
                    const t_i32x16 D = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, zero, 0, 0, 0);
                    const int sc = static_cast<int>(((sub < 4 ? sc_lo : sc_hi) >> (8 * (sub & 3))) & 0xFFu);
                    const float mn = ubyte_to_f32(sub < 4 ? mn_lo : mn_hi, sub & 3);
#pragma unroll
                    for (int G = 0; G < kGroups; ++G) {
#pragma unroll
                        for (int k = 0; k < 4; ++k) digit_sum[G][k] += __mul24(D[4 * G + k], sc);
                        min_sum[G] = __builtin_fmaf(mn, kSumsAhead ? xs[kSumsAhead ? G : 0][sub] : xsum_row[G][sb * 8 + sub], min_sum[G]);
                    }
                    // three and four row groups: one set of MFMA results at a time (the scheduler would keep two or
                    // three sub-blocks' worth live and spill); the other wavefronts of the SIMD fill the matrix core's latency
                    if (kGroups >= 3) __builtin_amdgcn_sched_barrier(0);
                }
            }
#pragma unroll
            for (int G = 0; G < kGroups; ++G) {
                float S = static_cast<float>(digit_sum[G][3]);
                S = __builtin_fmaf(S, 256.0f, static_cast<float>(digit_sum[G][2]));
                S = __builtin_fmaf(S, 256.0f, static_cast<float>(digit_sum[G][1]));
                S = __builtin_fmaf(S, 256.0f, static_cast<float>(digit_sum[G][0]));
                // times 2^-s (xscale holds -s as a number, NaN for a super-block with an infinity or a NaN in it)
                const float minus_s = xscale_row[G][sb];
                S = __builtin_fmaf(minus_s, 0.0f, __builtin_ldexpf(S, static_cast<int>(minus_s)));
                float& sum = kByParity && (f & 1) ? odd : acc[G];
                const float more = __builtin_fmaf(-dmin, min_sum[G], __builtin_fmaf(d, S, sum));
                if (!kHalfTile || sb_step + (c >> 4) < sb_end) sum = more;
            }
        }
    }

    // ---- 3. K-slices meet in LDS, in slice order
    if (kByParity) acc[0] += odd;
#pragma unroll
    for (int G = 0; G < kGroups; ++G) partial[(wave * kGroups + G) * 64 + lane] = acc[G];
    __syncthreads();
    if constexpr (kHalfTile) {
        if (tid < 16) {
            float total = 0.0f;
            for (int sl = 0; sl < slices; ++sl) total += partial[sl * 64 + tid] + partial[sl * 64 + 48 + tid];
            const int o = static_cast<int>(blockIdx.x) * 16 + tid;
            if (o < out_dim) dst[o] = finish_output(ep, o, o, total);
        }
        return;
    }
    for (int i = tid; i < kGroups * 64; i += threads) {
        const int G = i >> 6, ln = i & 63;
        float total = 0.0f;
        for (int sl = 0; sl < slices; ++sl) total += partial[(sl * kGroups + G) * 64 + ln];
        const int row = 2 * G + (ln >> 5);
        const int o = static_cast<int>(blockIdx.x) * kTileCols + (ln & 31);
        if (row < rows && o < out_dim) {
            const size_t idx = static_cast<size_t>(row) * out_dim + o;
            if (accumulate) unsafeAtomicAdd(dst + idx, total);
            else dst[idx] = finish_output(ep, o, idx, total);
        }
    }
}

size_t q4k_i8_rows_lds_bytes(int rows, int in_dim, int waves) {  // kPlanesGiven: -s, sub-block sums, the slices' partial sums
    return ((static_cast<size_t>(rows) * (in_dim / 256) + 3) & ~static_cast<size_t>(3)) * 4 + static_cast<size_t>(rows) * (in_dim / 32) * 4 +
           static_cast<size_t>(waves) * ((rows + 1) / 2) * 64 * 4;
}

size_t q4k_i8_lds_bytes(int rows, int in_dim, int waves) {
    return static_cast<size_t>(rows) * 4 * (static_cast<size_t>(in_dim) + kDigitPadBytes) +
           ((static_cast<size_t>(rows) * (in_dim / 256) + 3) & ~static_cast<size_t>(3)) * 4 + static_cast<size_t>(rows) * (in_dim / 32) * 4 +
           static_cast<size_t>(waves) * ((rows + 1) / 2) * 64 * 4;
}

// Tuning runs only (the CPU engine exposes TERMITE_QUANT_* knobs the same way,
// ops/native_compute.zig:2902-2945).
int tuning_int(const char* name) {
    const char* v = std::getenv(name);
    return v && *v ? std::atoi(v) : 0;
}

// ------------------------------------------------------------------ short prefill
// More rows than one GEMV launch holds, up to 64 (longer ones: the fp6 GEMM below): X is split once by its own kernel --
// parts bf16 [rows][3][in_dim], sub-block sums as bf16 parts [rows][in_dim / 256][4][8] -- and the GEMM below
// converts every weight once per 32 rows instead of once per launch of six.
__global__ __launch_bounds__(256) void q4k_split_parts_kernel(const float* __restrict__ x, uint32_t* __restrict__ parts,
                                                             uint16_t* __restrict__ sum_parts, size_t groups, int groups_per_row) {
    // one thread per eight consecutive values; whole quads run together (groups is a multiple of four)
    for (size_t grp = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; grp < groups;
         grp += static_cast<size_t>(gridDim.x) * blockDim.x) {
        const float4 xa = reinterpret_cast<const float4*>(x)[grp * 2], xb = reinterpret_cast<const float4*>(x)[grp * 2 + 1];
        const float v[8] = {xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w};
        uint32_t p[3][4];
#pragma unroll
        for (int i = 0; i < 4; ++i) split3_pair(v[2 * i], v[2 * i + 1], &p[0][i], &p[1][i], &p[2][i]);
        float s = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
        s += dpp_move<kDppXor1>(s);
        s += __shfl_xor(s, 2);
        const size_t r = grp / groups_per_row;
        const int kg = static_cast<int>(grp - r * groups_per_row);
#pragma unroll
        for (int part = 0; part < 3; ++part)
            reinterpret_cast<uint4*>(parts)[(r * 3 + part) * groups_per_row + kg] =
                make_uint4(p[part][0], p[part][1], p[part][2], p[part][3]);
        // the sub-block sum, split the same way: 64 bytes per row and super-block,
        // [part 0..2][sub-block 0..7] bf16 and a fourth group of zeros (the K padding of the MFMA)
        uint16_t* cell = sum_parts + (r * (groups_per_row >> 5) + (kg >> 5)) * 32;
        const int sub = (kg >> 2) & 7;
        if ((threadIdx.x & 3) == 0) {
            uint32_t hi, mid, lo;
            split3_pair(s, 0.0f, &hi, &mid, &lo);
            cell[sub] = static_cast<uint16_t>(hi);
            cell[8 + sub] = static_cast<uint16_t>(mid);
            cell[16 + sub] = static_cast<uint16_t>(lo);
        } else if ((kg & 31) == 1) {
            *reinterpret_cast<uint4*>(cell + 24) = make_uint4(0u, 0u, 0u, 0u);
        }
    }
}

// Y[32 rows][256 columns] per workgroup, K walked half a super-block at a time: the X chunk of the
// next half travels global -> registers while the current one is computed from LDS,
// then registers -> the other LDS buffer, one barrier per half.  A wavefront owns a
// 32-column tile for all of K (no K split: nothing to combine).  Here the three parts of X lie
// along K instead of along the MFMA rows: a sub-block is six chained MFMAs (part x half) into
// one D of 32 real rows -- lane (row c, half g) supplies the same K values as in the GEMV
// kernel, from part 0, 1, 2 in turn against the same B -- so a row costs two multiply-adds per
// sub-block and the weights are converted once per 32 rows.  (A first version with the parts
// along the rows, ten rows per MFMA pass and four passes, measured 12-28 % slower.)
// Half super-blocks keep a workgroup at 55 KiB of LDS and 118 registers, so two of them share a compute unit: a SIMD has
// four wavefronts to fill the matrix pipe (200 cycles per 32 x 32 outputs and sub-block) while others convert, accumulate or
// wait at the other workgroup's barrier.  Whole super-blocks with the next sub-block's operands requested by hand took 105 KiB
// and 186 registers, two wavefronts a SIMD, 520 cycles where this takes 440: 333 x 4096 x 14336 187 -> 158 us, 1024 x 4096 x 14336
// 426 -> 369, 333 x 14336 x 4096 201 -> 181.
constexpr int kG32Rows = 32;
constexpr int kG32PartStride = 256 + 16;
constexpr int kG32PartsBytes = kG32Rows * 3 * kG32PartStride;
constexpr int kG32ChunkBytes = kG32PartsBytes + kG32Rows * 64;  // parts, then the parts of the sums: [row][part 0..3][sub-block] bf16
constexpr int kG32Units = kG32Rows * 3 * 16;

__global__ __launch_bounds__(512, 4) void gemm_q4k_rows32_kernel(float* __restrict__ dst, const uint32_t* __restrict__ parts,
                                                              const uint16_t* __restrict__ sum_parts, const uint8_t* __restrict__ weight,
                                                              int rows, int in_dim, int out_dim, int sb_per_split,
                                                              float* __restrict__ partial, Epilogue ep) {
    const int kb = in_dim >> 8;
    // K range of this workgroup: all of it, or (a small problem spread over more compute units)
    // share blockIdx.z, whose sums go to partial[z][rows][out_dim] for splitk_reduce_kernel
    const int sb_begin = blockIdx.z * sb_per_split;
    const int sb_end = min(kb, sb_begin + sb_per_split);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n_tiles = (out_dim + kTileCols - 1) >> 5;
    const int tile_raw = blockIdx.x * 8 + wave;
    const bool tile_ok = tile_raw < n_tiles;
    const int tile = tile_ok ? tile_raw : n_tiles - 1;  // a spare wavefront repeats the last tile and stores nothing
    const int row0 = blockIdx.y * kG32Rows;
    const int rows_here = min(kG32Rows, rows - row0);
    const uint8_t* tile_base = weight + static_cast<size_t>(tile) * kb * kTileBytes;
    const int groups_per_row = in_dim >> 3;

    static_assert(kG32Units == 3 * 512, "three 16-byte units of the X chunk per thread");
    // (named registers, not an array: an array stayed in scratch memory across the two branches that fill and drain it)
    uint4 stage0, stage1, stage2;
    uint4 stage_sum = make_uint4(0u, 0u, 0u, 0u);
    auto fetch_unit = [&](int i, int h) {
        const int u = tid + i * 512;
        const int rp = u >> 4, k16 = u & 15;
        const int r = min(rp / 3, rows_here - 1), part = rp - (rp / 3) * 3;  // rows past the end repeat the last one
        return reinterpret_cast<const uint4*>(parts)[(static_cast<size_t>(row0 + r) * 3 + part) * groups_per_row + h * 16 + k16];
    };
    auto fetch = [&](int h) {  // half super-block h; the sum parts (64 bytes per row) come with the second half
        stage0 = fetch_unit(0, h);
        stage1 = fetch_unit(1, h);
        stage2 = fetch_unit(2, h);
        if ((h & 1) && tid < kG32Rows * 4) {
            const int r = min(tid >> 2, rows_here - 1);
            stage_sum = reinterpret_cast<const uint4*>(sum_parts)[(static_cast<size_t>(row0 + r) * kb + (h >> 1)) * 4 + (tid & 3)];
        }
    };
    auto deposit_unit = [&](unsigned char* chunk, int i, const uint4& v) {
        const int u = tid + i * 512;
        *reinterpret_cast<uint4*>(chunk + (u >> 4) * kG32PartStride + (u & 15) * 16) = v;
    };
    auto deposit = [&](int h) {
        unsigned char* chunk = q4k_mfma_lds + (h & 1) * kG32ChunkBytes;
        deposit_unit(chunk, 0, stage0);
        deposit_unit(chunk, 1, stage1);
        deposit_unit(chunk, 2, stage2);
        if ((h & 1) && tid < kG32Rows * 4) reinterpret_cast<uint4*>(chunk + kG32PartsBytes)[tid] = stage_sum;
    };

    const int c = lane & 31, g = lane >> 5;
    const int a_offset = c * 3 * kG32PartStride + 32 * g;  // A operand: row c of the block, K half g
    float acc[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0f;

    t_u32x4 hdr, qv[2], hdr_next, qv_next[2];
    auto request = [&](int h, t_u32x4& header, t_u32x4 (&q)[2]) {
        const uint8_t* base = tile_base + static_cast<size_t>(h >> 1) * kTileBytes;
        if ((h & 1) == 0) header = __builtin_nontemporal_load(reinterpret_cast<const t_u32x4*>(base + 16 * (lane & 31)));
#pragma unroll
        for (int t = 0; t < 2; ++t)
            q[t] = __builtin_nontemporal_load(reinterpret_cast<const t_u32x4*>(base + 512 + (2 * (h & 1) + t) * 1024 + 16 * lane));
    };

    if (sb_begin >= sb_end) return;  // workgroup-uniform (the host sends no empty shares)
    fetch(2 * sb_begin);
    request(2 * sb_begin, hdr, qv);
    hdr_next = hdr;
    deposit(2 * sb_begin);
    __syncthreads();
    for (int sb = sb_begin; sb < sb_end; ++sb) {
        const float d = half_bits_to_f32(static_cast<uint16_t>(hdr.x & 0xFFFFu));
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const bool more = half == 0 || sb + 1 < sb_end;  // uniform
            if (more) {
                fetch(2 * sb + half + 1);
                request(2 * sb + half + 1, hdr_next, qv_next);
            }
            const unsigned char* chunk = q4k_mfma_lds + half * kG32ChunkBytes;
            // scales of sub-blocks 0..3 (first half) or 4..7
            const uint32_t scales = half == 0 ? hdr.y & 0x3F3F3F3Fu : (hdr.w & 0x0F0F0F0Fu) | ((hdr.y >> 2) & 0x30303030u);
#pragma unroll
            for (int sub = 0; sub < 4; ++sub) {
                t_f32x16 D = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                const int t = sub >> 1, hi = sub & 1;  // low nibbles of chunk t: sub-block 2 t, high nibbles: 2 t + 1
                const uint32_t w[4] = {qv[t].x, qv[t].y, qv[t].z, qv[t].w};
#pragma unroll
                for (int m = 0; m < 2; ++m) {
                    union {
                        t_bf16x8 v;
                        t_bf16x2 pair[4];
                    } b;
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
                        const uint32_t nib = hi ? (w[2 * m + k] >> 4) & 0x0F0F0F0Fu : w[2 * m + k] & 0x0F0F0F0Fu;
                        b.pair[2 * k] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(static_cast<int>(nib), 512.0f, false);
                        b.pair[2 * k + 1] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(static_cast<int>(nib), 512.0f, true);
                    }
#pragma unroll
                    for (int part = 0; part < 3; ++part) {
                        union {
                            t_bf16x8 v;
                            uint4 u;
                        } a;
                        a.u = *reinterpret_cast<const uint4*>(chunk + a_offset + part * kG32PartStride + (32 * sub + 8 * m) * 2);
                        D = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.v, b.v, D, 0, 0, 0);
                    }
                }
                const float dsc = d * ubyte_to_f32(scales, sub);
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[i] = __builtin_fmaf(dsc, D[i], acc[i]);
                // pin the accumulation here: left to itself the compiler keeps every D and its operands alive (spills)
#pragma unroll
                for (int i = 0; i < 16; ++i) asm volatile("" : "+v"(acc[i]));
            }
            if (half == 1) {
                // The min term of the whole super-block, sum over sub-blocks of m[column][sub] * X[row][sub],
                // is one more small product: A = the three bf16 parts of the eight sub-block sums of each
                // row (K = part * 8 + sub, padded with zeros to 32), B = the eight 6-bit mins of each column.
                const unsigned char* sums = chunk + kG32PartsBytes + c * 64 + 16 * g;
                const float dmin = half_bits_to_f32(static_cast<uint16_t>(hdr.x >> 16));
                const uint32_t mn_lo = hdr.z & 0x3F3F3F3Fu, mn_hi = ((hdr.w >> 4) & 0x0F0F0F0Fu) | ((hdr.z >> 2) & 0x30303030u);
                union {
                    t_bf16x8 v;
                    uint4 u;
                } sa0, sa1, mb;
                sa0.u = *reinterpret_cast<const uint4*>(sums);       // parts 0 (g = 0) and 1 (g = 1)
                sa1.u = *reinterpret_cast<const uint4*>(sums + 32);  // part 2 (g = 0) and the zeros (g = 1)
                mb.u = make_uint4(bf16_pair(ubyte_to_f32(mn_lo, 0), ubyte_to_f32(mn_lo, 1)),
                                  bf16_pair(ubyte_to_f32(mn_lo, 2), ubyte_to_f32(mn_lo, 3)),
                                  bf16_pair(ubyte_to_f32(mn_hi, 0), ubyte_to_f32(mn_hi, 1)),
                                  bf16_pair(ubyte_to_f32(mn_hi, 2), ubyte_to_f32(mn_hi, 3)));
                t_f32x16 T = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                T = __builtin_amdgcn_mfma_f32_32x32x16_bf16(sa0.v, mb.v, T, 0, 0, 0);
                T = __builtin_amdgcn_mfma_f32_32x32x16_bf16(sa1.v, mb.v, T, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[i] = __builtin_fmaf(-dmin, T[i], acc[i]);
                hdr = hdr_next;
            }
            if (more) {
                deposit(2 * sb + half + 1);
                qv[0] = qv_next[0];
                qv[1] = qv_next[1];
            }
            __syncthreads();  // the next chunk is in place, and nobody still reads the one about to be replaced
        }
    }

    if (!tile_ok) return;
    const int o = tile * kTileCols + c;
    if (o >= out_dim) return;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int r = 8 * (i >> 2) + 4 * g + (i & 3);
        if (r < rows_here) {
            const size_t at = static_cast<size_t>(row0 + r) * out_dim + o;
            if (partial != nullptr) partial[static_cast<size_t>(blockIdx.z) * rows * out_dim + at] = acc[i];
            else dst[at] = finish_output(ep, o, at, acc[i]);
        }
    }
}

// ------------------------------------------------------------------ prefill
// More than 64 rows: X is split once by its own kernel, then a GEMM on the 6-bit matrix
// instructions.  v_mfma_scale_f32_32x32x64_f8f6f4 multiplies 64 fp6 (e2m3) numbers a column in the 33 cycles that
// v_mfma_f32_32x32x16_bf16 needs for 16 bf16 ones, and to it
//   * the fp6 codes 0 .. 16 are the numbers n / 8 (a sign in front), so a weight nibble is its own code;
//   * an activation is eight digits from -16 to 16: x = sum over d of digit_d * 2^(e - 4 - 5 d), with 2^(e - 1) <= max |x| < 2^e over the
//     sub-block.  Rounded to 2^(e - 39): 24-bit numbers down to 2^(e - 16) are exact, for smaller ones see add_lost; products with the
//     scales that the instruction applies to 32 values at a time are exact.
// A sub-block of 32 values is four such instructions -- lane half g of number p multiplies digit 2 p + g -- against six bf16
// ones, and its result needs no conversion: (d sc) * D is added to the sum.
//
// The order of the 16 values of a lane half inside its three 32-bit words of codes: the one in which nine instructions spread
// the nibbles of the tile-major layout (expand_nibbles).
constexpr int kFp6Order[16] = {0, 12, 5, 10, 3, 15, 4, 9, 2, 14, 7, 8, 1, 13, 6, 11};

// Workspace: the digits, for every 32 rows (the last tile: its rows, rounded up to even) and sub-block the operands of the four
// instructions, each [half g][row] 16 bytes and then [half g][row] 8 bytes (a lane's six words); behind them, for every row and
// super-block 64 bytes: the eight sub-block sums as three bf16 parts, [part][sub-block], the sub-blocks' scale bytes, and in the first
// row of 32 a byte per sub-block that says whether the digits left something of these 32 rows' values behind.
constexpr int kDigitBytes = 192;  // of a row and sub-block
typedef int t_i32x6 __attribute__((ext_vector_type(6)));

__device__ __forceinline__ int rows_of_tile(int rows, int tile) { return (min(kG32Rows, rows - tile * kG32Rows) + 1) & ~1; }

// What the digits leave of a value, exact (at most 2^(e - 40)); `exponent` = e + 126, the biased exponent of the sub-block's largest value.
// In two steps, as the digits are made: together they are the value rounded to 2^(e - 39), to the even neighbour from halfway.
__device__ __forceinline__ float left_behind(float x, int exponent) {
    const float rest = x - __builtin_ldexpf(__builtin_rintf(__builtin_ldexpf(x, 145 - exponent)), exponent - 145);
    return rest - __builtin_ldexpf(__builtin_rintf(__builtin_ldexpf(rest, 165 - exponent)), exponent - 165);
}

// 32 values as 6-bit codes: code f is even[f / 2] (odd[f / 2]) / scale rounded to eighths, the even one from halfway.  (As assembly: with
// the builtin the compiler may give the result the scale's register, which the instruction still reads after its first words.)
__device__ __forceinline__ t_i32x6 fp6_codes(t_f32x16 even, t_f32x16 odd, float scale) {
    t_i32x6 codes;
    asm("v_cvt_scalef32_2xpk16_fp6_f32 %0, %1, %2, %3" : "=&v"(codes) : "v"(even), "v"(odd), "v"(scale));
    return codes;
}

// A workgroup per 32 rows and sub-block, a lane for a row and one of the eight digits: X less what the digits above take of it -- adding
// and subtracting 1.5 * 2^23 units rounds to a unit; from the fifth digit on in two steps, as 24 bits reach no further -- and the
// conversion rounds to the digit itself.  X comes in by whole lines and is handed round in LDS.
// Bound by the launch and a trip to memory on short calls, the vector ALU on long ones.  us of kernel time by rocprofv3, against a lane
// for 16 values and all digits, packed by shifts: 75 x 256 4.1 -> 1.8, 333 x 4096 7.3 -> 6.1, 2048 x 4096 17.7 (four-bit digits 19.0).
__global__ __launch_bounds__(256) void q4k_split_digits_kernel(const float* __restrict__ x, uint8_t* __restrict__ digits,
                                                             uint8_t* __restrict__ sums, int rows, int in_dim) {
    __shared__ float4 staged[kG32Rows * 8];  // [row][chunk ^ row % 8]
    const int tid = threadIdx.x, tile = blockIdx.y, sub = blockIdx.x;
    {
        const int r = tid >> 3, chunk = tid & 7, row = tile * kG32Rows + r;
        float4 q = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (row < rows) q = *reinterpret_cast<const float4*>(x + static_cast<size_t>(row) * in_dim + sub * 32 + chunk * 4);
        staged[r * 8 + (chunk ^ (r & 7))] = q;
    }
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), digit = tid >> 5;
    const int r = tid & 31, row = tile * kG32Rows + r, tile_rows = rows_of_tile(rows, tile);
    float v[32];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const float4 q = staged[r * 8 + (c ^ (r & 7))];
        v[4 * c] = q.x; v[4 * c + 1] = q.y; v[4 * c + 2] = q.z; v[4 * c + 3] = q.w;
    }
    uint32_t peak = 0;
#pragma unroll
    for (int i = 0; i < 32; ++i) peak = max(peak, __float_as_uint(v[i]) & 0x7FFFFFFFu);
    // the biased exponent is the scale byte of digit 0; below 5 (2^-121) the digits reach 2^-160, under every f32, and the scales
    // of the lower ones would leave their range.  255: an infinity or a NaN, which the instruction takes as NaN
    const int exponent = max(static_cast<int>(peak >> 23), 5);
    uint8_t* const cell = sums + (static_cast<size_t>(row) * (in_dim >> 8) + (sub >> 3)) * 64;
    if (wave == 0) {
        float s = 0.0f;
        {
            float part[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) part[i] = v[2 * i] + v[2 * i + 1];
#pragma unroll
            for (int n = 8; n >= 1; n /= 2)
#pragma unroll
                for (int i = 0; i < n; ++i) part[i] = part[2 * i] + part[2 * i + 1];
            s = part[0];
        }
        if (digit == 0 && row < rows) {
            uint32_t hi, mid, lo;
            split3_pair(s, 0.0f, &hi, &mid, &lo);
            uint16_t* part = reinterpret_cast<uint16_t*>(cell) + (sub & 7);
            part[0] = static_cast<uint16_t>(hi);
            part[8] = static_cast<uint16_t>(mid);
            part[16] = static_cast<uint16_t>(lo);
            cell[48 + (sub & 7)] = static_cast<uint8_t>(exponent);
        }
    } else if (wave == 1) {
        // the digits may leave something of a value whose last bit is below 2^(e - 39) (zeros wrap round to the largest number)
        uint32_t least = 0xFFFFFFFFu;
#pragma unroll
        for (int i = 0; i < 32; ++i) least = min(least, (__float_as_uint(v[i]) << 1) - 1u);
        const bool left = least != 0xFFFFFFFFu && static_cast<int>((least + 1) >> 24) < exponent - 15;
        const bool any_left = __builtin_amdgcn_ballot_w64(left) != 0;
        if (tid == 64) cell[56 + (sub & 7)] = any_left;  // (row 0)
    }
    // The units and the scale as floats, for which sub-blocks near the ends of f32 are brought to 2^0.
    const bool far = exponent < 70 || exponent > 220;
    const int base = far ? 127 : exponent;
    if (__builtin_amdgcn_ballot_w64(far && peak != 0) != 0) {
#pragma unroll
        for (int i = 0; i < 32; ++i) v[i] = __builtin_ldexpf(v[i], base - exponent);
    }
    auto take_off = [&](int biased) {  // multiples of 2^(biased - 150)
        const float c = __uint_as_float(static_cast<uint32_t>(biased) << 23 | 0x400000u);
#pragma unroll
        for (int i = 0; i < 32; ++i) v[i] -= (v[i] + c) - c;
    };
    if (wave >= 2) take_off(base + 5);
    take_off(base + 25 - 5 * digit);
    t_f32x16 even, odd;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        even[i] = v[(i & 8) * 2 + kFp6Order[2 * i & 15]];
        odd[i] = v[(i & 8) * 2 + kFp6Order[(2 * i & 15) + 1]];
    }
    const t_i32x6 codes = fp6_codes(even, odd, __uint_as_float(static_cast<uint32_t>(base - 5 * digit) << 23));
    if (r < tile_rows) {
        uint8_t* image = digits + static_cast<size_t>(tile) * kG32Rows * in_dim * 6 + (static_cast<size_t>(sub) * 4 + (digit >> 1)) * tile_rows * 48;
        const int at = (digit & 1) * tile_rows + r;
        reinterpret_cast<int4*>(image)[at] = make_int4(codes[0], codes[1], codes[2], codes[3]);
        reinterpret_cast<int2*>(image + tile_rows * 32)[at] = make_int2(codes[4], codes[5]);
    }
}

// (x & mask) | (y & ~mask) and (x & mask) | y in one instruction at the fast rate (v_bitop3_b32 2.4 cycles; v_and_or_b32 and the
// shifts 4.4, v_permlane32_swap_b32 8.7).
__device__ __forceinline__ uint32_t blend(uint32_t mask, uint32_t x, uint32_t y) {
    return __builtin_amdgcn_bitop3_b32(mask, x, y, 0xCA);
}
__device__ __forceinline__ uint32_t masked_or(uint32_t mask, uint32_t x, uint32_t y) {
    return __builtin_amdgcn_bitop3_b32(mask, x, y, 0xEA);
}

// One 64-lane load of 16 bytes a lane from base + off straight into LDS at lds + at + 16 lane, then off += step (as inline
// assembly, as in gemm_kernels.hip: the compiler would make every later LDS read wait for all of them).  The addition stands
// where M0 needs a wait state before it is used; lds, base and step are wave-uniform, `at` a constant.
__device__ __forceinline__ void q4k_lds_load16(const void* base, uint32_t& off, uint32_t step, uint32_t lds, int at) {
    uint32_t next;
    asm volatile("s_add_u32 m0, %1, %5\n\tv_add_u32 %0, %2, %3\n\tglobal_load_lds_dwordx4 %3, %4"
                 : "=&v"(next)
                 : "s"(__builtin_amdgcn_readfirstlane(lds)), "s"(step), "v"(off), "s"(base), "i"(at)
                 : "memory", "m0", "scc");
    off = next;
}

typedef int t_i32x8 __attribute__((ext_vector_type(8)));
typedef uint32_t t_u32x2 __attribute__((ext_vector_type(2)));

// s_waitcnt for "at most kLeft vector memory operations outstanding".
template <int kLeft>
__device__ __forceinline__ void q4k_wait_vm() {
    static_assert(kLeft < 16, "the count's low four bits");
    __builtin_amdgcn_s_waitcnt(kLeft | (7 << 4) | (15 << 8));
}

template <int kWaves, int kR, int kC>
struct G6Shape {
    static constexpr int kThreads = 64 * kWaves;
    static constexpr int kRows = kG32Rows * kR, kTiles = kC * kWaves, kCols = kTileCols * kTiles;
    static constexpr int kDigits = kR * kG32Rows * kDigitBytes;  // of a sub-block: ring of four
    static constexpr int kChunk = kTiles * 1024;                 // nibbles of two sub-blocks: two
    static constexpr int kHeaders = kTiles * 512;                // of a super-block: one
    static constexpr int kSums = kR * kG32Rows * 64;             // of a super-block: two
    static constexpr int kChunkAt = 4 * kDigits, kHeadersAt = kChunkAt + 2 * kChunk, kSumsAt = kHeadersAt + kHeaders;
    static constexpr int kLdsBytes = kSumsAt + 2 * kSums;
    // 1 KiB loads of a stage, dealt out to the wavefronts in turn
    static constexpr int kUnitsDigits = 6 * kR, kUnitsChunk = kTiles, kUnitsHeaders = kTiles / 2, kUnitsSums = 2 * kR;
    static_assert(kTiles % 2 == 0, "headers are loaded for two column tiles at a time");
};

// Y[32 kR rows][32 kC kWaves columns] per workgroup; a wavefront owns kC column tiles for all rows of the workgroup and the
// whole K of the launch.  A stage is a sub-block: digits and weights travel global -> LDS three stages ahead, and what a stage
// computes with is read from LDS one stage (or row tile) ahead.
// Bound by instruction issue beside the MFMAs and, on a full chip, by its power (1.7 GHz): four MFMAs of 33 cycles, 45 other
// instructions (16 of them the multiply-adds) and about 210 SIMD cycles per 32 x 32 outputs and sub-block, where the bf16 kernel took
// 440.  Against it: 2048 x 4096 x 14336 685 -> 501 us, 333 x 4096 x 14336 twice 290 -> 212, 333 x 14336 x 4096 166 -> 121.
template <int kWaves, int kR, int kC, int kOcc>
__global__ __launch_bounds__(64 * kWaves, kOcc) void gemm_q4k_fp6_kernel(
    float* __restrict__ dst, const uint8_t* __restrict__ digits, const uint8_t* __restrict__ sums,
    const uint8_t* __restrict__ weight, int rows, int in_dim, int out_dim, int m_groups, int n_groups, int band, int sb_per_split,
    float* __restrict__ partial, int first_to_dst, Epilogue ep, Q4kSecond second, const float* __restrict__ x) {
    using S = G6Shape<kWaves, kR, kC>;
    if (blockIdx.z != 0) {  // a second matrix on the same X
        dst = second.dst;
        weight = second.weight;
        ep = second.ep;
    }
    const int kb = in_dim >> 8;
    // K range of this workgroup: all of it, or share blockIdx.y, whose sums go to partial[share][rows][out_dim] (first_to_dst = 1: the
    // first share's to dst, the others' to partial[share - 1])
    const int sb_begin = blockIdx.y * sb_per_split;
    const int sb_end = min(kb, sb_begin + sb_per_split);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = lane & 31, g = lane >> 5;
    // An XCD (consecutive ids go round-robin over the eight) takes an eighth of the list of tiles, in which `band` row groups of a
    // column group follow each other, then the next column group's: what is resident on an XCD shares both operands in its L2.
    const int id = blockIdx.x, index = (id & 7) * (gridDim.x >> 3) + (id >> 3);
    const int band_at = index / (band * n_groups) * band, band_rows = min(band, m_groups - band_at), in_band = index - band_at * n_groups;
    if (index >= m_groups * n_groups || sb_begin >= sb_end) return;  // workgroup-uniform
    const int m_group = band_at + in_band % band_rows, n_group = in_band / band_rows;
    const int n_tiles = (out_dim + kTileCols - 1) >> 5, m_tiles = (rows + kG32Rows - 1) / kG32Rows;
    const int tile0 = n_group * S::kTiles;
    const uint32_t tile_stride = static_cast<uint32_t>(kb) * kTileBytes;
    auto tile_at = [&](int tile) { return weight + static_cast<size_t>(min(tile0 + tile, n_tiles - 1)) * tile_stride; };  // spare ones repeat the last

    // ---- loads: units of each kind, dealt out in turn; where they do not go round, some wavefronts repeat another's, so that all
    // count the same loads and no branch stands between them (branches on the counts cost a wavefront 400 cycles a stage)
    constexpr int kPerDigits = (S::kUnitsDigits + kWaves - 1) / kWaves, kPerChunk = (S::kUnitsChunk + kWaves - 1) / kWaves;
    constexpr int kPerHeaders = (S::kUnitsHeaders + kWaves - 1) / kWaves, kPerSums = (S::kUnitsSums + kWaves - 1) / kWaves;
    const uint32_t lds_base = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(q4k_mfma_lds)));
    // bases stay, this lane's offsets move on with every load
    const uint8_t *digit_base[kPerDigits], *chunk_base[kPerChunk], *header_base[kPerHeaders], *sum_base[kPerSums];
    uint32_t digit_off[kPerDigits], chunk_off[kPerChunk], header_off[kPerHeaders], sum_off[kPerSums], digit_step[kPerDigits];
    uint32_t digit_lds[kPerDigits], chunk_lds[kPerChunk], header_lds[kPerHeaders], sum_lds[kPerSums];
#pragma unroll
    for (int k = 0; k < kPerDigits; ++k) {
        const int u = (wave + k * kWaves) % S::kUnitsDigits, q = u % 6;
        const int mt = min(m_group * kR + u / 6, m_tiles - 1), n = rows_of_tile(rows, mt);
        digit_step[k] = n * kDigitBytes;
        digit_base[k] = digits + static_cast<size_t>(mt) * kG32Rows * in_dim * 6 + static_cast<size_t>(sb_begin) * 8 * digit_step[k];
        digit_lds[k] = lds_base + u * 1024;
        const int o = q * 1024 + lane * 16, p = o / 1536, w = o - p * 1536;  // image offset of this lane's bytes
        int at;
        if (w < 1024) at = ((w >> 9) * n + min((w >> 4) & 31, n - 1)) * 16;
        else at = n * 32 + (((w - 1024) >> 8) * n + min(((w - 1024) >> 3) & 31, n - 2)) * 8;
        digit_off[k] = static_cast<uint32_t>(p * n * 48 + at);
    }
#pragma unroll
    for (int k = 0; k < kPerChunk; ++k) {
        const int u = (wave + k * kWaves) % S::kUnitsChunk;
        chunk_base[k] = tile_at(u) + static_cast<size_t>(sb_begin) * kTileBytes + 512;
        chunk_off[k] = 16 * lane;
        chunk_lds[k] = lds_base + S::kChunkAt + u * 1024;
    }
#pragma unroll
    for (int k = 0; k < kPerHeaders; ++k) {
        const int u = (wave + k * kWaves) % S::kUnitsHeaders;
        header_base[k] = tile_at(2 * u) + static_cast<size_t>(sb_begin) * kTileBytes;
        header_off[k] = (g != 0 && tile0 + 2 * u + 1 < n_tiles ? tile_stride : 0u) + 16 * c;
        header_lds[k] = lds_base + S::kHeadersAt + u * 1024;
    }
#pragma unroll
    for (int k = 0; k < kPerSums; ++k) {
        const int u = (wave + k * kWaves) % S::kUnitsSums, mt = min(m_group * kR + (u >> 1), m_tiles - 1);
        sum_base[k] = sums + (static_cast<size_t>(mt) * kG32Rows * kb + sb_begin) * 64;
        sum_off[k] = static_cast<uint32_t>(min(c, rows - 1 - mt * kG32Rows)) * static_cast<uint32_t>(kb * 64) + (2 * (u & 1) + g) * 16;
        sum_lds[k] = lds_base + S::kSumsAt + u * 1024;
    }
    // load l of stage s (0 .. 7)
    constexpr int kLoadsOdd = kPerDigits, kLoadsEven = kPerDigits + kPerChunk, kLoadsFirst = kLoadsEven + kPerHeaders + kPerSums;
    auto loads_of = [](int s) constexpr { return s == 0 ? kLoadsFirst : ((s & 1) ? kLoadsOdd : kLoadsEven); };
    auto issue_one = [&](int s, int l, int parity) {
        if (l < kPerDigits) {
            const int k = l;
            q4k_lds_load16(digit_base[k], digit_off[k], digit_step[k], digit_lds[k], (s & 3) * S::kDigits);
        } else if (l < kLoadsEven) {
            const int k = l - kPerDigits;
            q4k_lds_load16(chunk_base[k], chunk_off[k], s < 6 ? 1024 : kTileBytes - 3072, chunk_lds[k], ((s >> 1) & 1) * S::kChunk);
        } else if (l < kLoadsEven + kPerHeaders) {
            const int k = l - kLoadsEven;
            q4k_lds_load16(header_base[k], header_off[k], kTileBytes, header_lds[k], 0);
        } else {
            const int k = l - kLoadsEven - kPerHeaders;
            q4k_lds_load16(sum_base[k], sum_off[k], 64, sum_lds[k] + parity * S::kSums, 0);  // [row tile][16-byte chunk][row]
        }
    };
    auto issue = [&](int s, int parity) {
#pragma unroll
        for (int l = 0; l < loads_of(s); ++l) issue_one(s, l, parity);
    };
    auto past_the_end = [&](bool last) {  // the loads that run past the end of K repeat its last super-block: nobody uses them
        const uint32_t back = last ? 1 : 0;
#pragma unroll
        for (int k = 0; k < kPerDigits; ++k) digit_off[k] -= 8 * back * digit_step[k];
#pragma unroll
        for (int k = 0; k < kPerChunk; ++k) chunk_off[k] -= back * kTileBytes;
#pragma unroll
        for (int k = 0; k < kPerHeaders; ++k) header_off[k] -= back * kTileBytes;
#pragma unroll
        for (int k = 0; k < kPerSums; ++k) sum_off[k] -= back * 64;
    };

    t_f32x16 acc[kR][kC];
#pragma unroll
    for (int i = 0; i < kR; ++i)
#pragma unroll
        for (int j = 0; j < kC; ++j) acc[i][j] = t_f32x16{};

    // Statements below that only name registers ("+v") hold what follows, or what made them, in its place.
    typedef const __attribute__((address_space(3))) t_u32x4* lds16_ptr;
    typedef const __attribute__((address_space(3))) t_u32x2* lds8_ptr;
    uint32_t lane16 = lds_base + 16 * lane, lane8 = lds_base + 1024 + 8 * lane;
    const uint32_t own_tiles = 1024 * wave * kC;
    t_u32x4 qv[kC];
    uint32_t nib[kC][2], e[kC][3];
    t_i32x6 a[4], b[2][kC];
    auto read_digits = [&](int s, int i, int p) {
        asm volatile("" : "+v"(lane16), "+v"(lane8));
        const int at = (s & 3) * S::kDigits + i * 6144 + p * 1536;
        const t_u32x4 wide = *reinterpret_cast<lds16_ptr>(lane16 + at);
        const t_u32x2 rest = *reinterpret_cast<lds8_ptr>(lane8 + at);
        a[p] = t_i32x6{static_cast<int>(wide.x), static_cast<int>(wide.y), static_cast<int>(wide.z), static_cast<int>(wide.w),
                       static_cast<int>(rest.x), static_cast<int>(rest.y)};
    };
    auto read_chunk = [&](int s) {  // nibbles of sub-blocks s and s + 1, s even
        asm volatile("" : "+v"(lane16));
#pragma unroll
        for (int j = 0; j < kC; ++j)
            qv[j] = *reinterpret_cast<lds16_ptr>(lane16 + own_tiles + (S::kChunkAt + ((s >> 1) & 1) * S::kChunk + j * 1024));
    };
    // The weights of sub-block s in three parts: nibbles of the sub-block alone, sixteen 6-bit codes in three words, all 32 values
    // in both lane halves.
    auto convert = [&](int s, int j, int piece) {
        constexpr uint32_t kLow = 0x0F0F0F0Fu;
        if (piece == 0) {
            t_u32x4 w = qv[j];
            asm volatile("" : "+v"(w));
            if ((s & 1) == 0) {
                nib[j][0] = blend(kLow, w.x, w.y << 4);
                nib[j][1] = blend(kLow, w.z, w.w << 4);
            } else {
                nib[j][0] = blend(kLow, w.x >> 4, w.y);
                nib[j][1] = blend(kLow, w.z >> 4, w.w);
            }
            asm volatile("" : "+v"(nib[j][0]), "+v"(nib[j][1]));
        } else if (piece == 1) {
            const uint32_t n = nib[j][0], x = nib[j][1] << 2;
            e[j][0] = masked_or(0xC03C03C0u, x, n & 0x0F00F00Fu);
            e[j][1] = masked_or(0x03C03C00u, x, n & 0xF00F00F0u) | (nib[j][1] >> 30);
            e[j][2] = masked_or(0x3C03C03Cu, x, n & 0x00F00F00u);
            asm volatile("" : "+v"(e[j][0]), "+v"(e[j][1]), "+v"(e[j][2]));
        } else {
            t_i32x6& to = b[s & 1][j];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const auto both = __builtin_amdgcn_permlane32_swap(e[j][k], e[j][k], false, false);
                to[k] = static_cast<int>(both[0]);
                to[k + 3] = static_cast<int>(both[1]);
            }
            asm volatile("" : "+v"(to));
        }
    };

    const int b_scale = 130 | 120 << 8 | 110 << 16 | 100 << 24;  // 2^(3 - 10 p): codes are eighths, digit pair p weighs 2^(-10 p)
    issue(0, sb_begin & 1);
    issue(1, 0);
    issue(2, 0);
    q4k_wait_vm<kLoadsEven>();  // loads complete in order: stages 0 and 1 have landed
    __syncthreads();
    read_chunk(0);
#pragma unroll
    for (int p = 0; p < 4; ++p) read_digits(0, 0, p);
#pragma unroll
    for (int j = 0; j < kC; ++j)
#pragma unroll
        for (int piece = 0; piece < 3; ++piece) convert(0, j, piece);

    // A step is one row tile and sub-block: kC times four chained MFMAs into D.  A slot is one MFMA and what stands behind it: the
    // matrix pipe takes 33 cycles an instruction and only what is issued in between overlaps it.  That is a share of the
    // multiply-adds of the step before (its D times its factor), the reads of the next step's digits, the conversion of the next
    // sub-block's weights and the loads of the stage three ahead.  Eight sub-blocks are followed by the min term, a step of two bf16
    // MFMAs per row tile.
    t_f32x16 D[2][kC];
    float factor[2][kC];
#pragma unroll
    for (int j = 0; j < kC; ++j) {
        D[1][j] = t_f32x16{};
        factor[1][j] = 0.0f;
    }
    int a_scale[kR], a_scale_next[kR];
    uint32_t first_half = g == 0 ? 0xFFFFFFFFu : 0u;
    asm volatile("" : "+v"(first_half));  // (a select here would become a branch around an MFMA)
    auto read_scales = [&](int sb, int half) {
#pragma unroll
        for (int i = 0; i < kR; ++i)
            a_scale_next[i] = *reinterpret_cast<const int*>(q4k_mfma_lds + S::kSumsAt + (sb & 1) * S::kSums + i * 2048 + 1536 + 16 * c + 4 * half);
    };
    auto accumulate = [&](int before, int i, int j, int first, int last) {
#pragma unroll
        for (int v = first; v < last; ++v) acc[i][j][v] = __builtin_fmaf(factor[before][j], D[before][j][v], acc[i][j][v]);
        asm volatile("" : "+v"(acc[i][j]));
    };
    read_scales(sb_begin, 0);
    // whether the min terms outweigh what the digits leave behind (see add_lost): bit 7 of every byte while no 6-bit min is zero, and
    // the least of 16 |dmin| - |d|
    uint32_t mins_live[kC];
    float slack[kC];
#pragma unroll
    for (int j = 0; j < kC; ++j) {
        mins_live[j] = 0xFFFFFFFFu;
        slack[j] = 0.0f;
    }
    for (int sb = sb_begin; sb < sb_end; ++sb) {
        const unsigned char* cell = q4k_mfma_lds + S::kSumsAt + (sb & 1) * S::kSums;
        t_u32x4 hdr[kC];
        uint4 mins[kC], sum_parts[2];
        float d[kC];
#pragma unroll
        for (int j = 0; j < kC; ++j) hdr[j] = *reinterpret_cast<const t_u32x4*>(q4k_mfma_lds + S::kHeadersAt + (wave * kC + j) * 512 + 16 * c);
        auto read_sums = [&](int i) {
            sum_parts[0] = *reinterpret_cast<const uint4*>(cell + i * 2048 + g * 512 + 16 * c);  // parts 0 (g = 0) and 1 (g = 1)
            sum_parts[1] = *reinterpret_cast<const uint4*>(cell + i * 2048 + 1024 + 16 * c);     // part 2
        };
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            if (s == 5) past_the_end(sb + 1 == sb_end);
            constexpr int kSlots = 4 * kR * kC;
            const int to_issue = loads_of((s + 3) & 7);
            if ((s & 3) == 0) {
#pragma unroll
                for (int i = 0; i < kR; ++i) a_scale[i] = a_scale_next[i] - 0x05050505 * g;
            }
#pragma unroll
            for (int i = 0; i < kR; ++i) {
                const int step = s * kR + i, now = step & 1, before = now ^ 1, i_before = (i + kR - 1) % kR;
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    const t_i32x8 a8 = __builtin_shufflevector(a[p], a[p], 0, 1, 2, 3, 4, 5, -1, -1);
#pragma unroll
                    for (int j = 0; j < kC; ++j) {
                        const t_i32x8 b8 = __builtin_shufflevector(b[s & 1][j], b[s & 1][j], 0, 1, 2, 3, 4, 5, -1, -1);
                        const t_f32x16 from = p == 0 ? t_f32x16{} : D[now][j];
                        // Highest digits first: added to a smaller sum, the large products always round the same way, 2.9e-8 of a
                        // sub-block but with a mean of -8.8e-8 that grows with K (333 x 14336 x 4096: 6.3e-7 against 4.5e-7).
#define AFHIP_STEP(P, W) \
    if (p == P && (s & 3) == W) D[now][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a8, b8, from, 2, 2, W, a_scale[i], P, b_scale)
                        AFHIP_STEP(0, 0); AFHIP_STEP(0, 1); AFHIP_STEP(0, 2); AFHIP_STEP(0, 3);
                        AFHIP_STEP(1, 0); AFHIP_STEP(1, 1); AFHIP_STEP(1, 2); AFHIP_STEP(1, 3);
                        AFHIP_STEP(2, 0); AFHIP_STEP(2, 1); AFHIP_STEP(2, 2); AFHIP_STEP(2, 3);
                        AFHIP_STEP(3, 0); AFHIP_STEP(3, 1); AFHIP_STEP(3, 2); AFHIP_STEP(3, 3);
#undef AFHIP_STEP
                        __builtin_amdgcn_sched_barrier(0);
                        const int at = (i * 4 + p) * kC + j;  // slot of the stage
#pragma unroll
                        for (int l = 0; l < to_issue; ++l)
                            if (l * kSlots / to_issue == at) issue_one((s + 3) & 7, l, (sb + 1) & 1);
                        if (j == kC - 1) read_digits(i + 1 < kR ? s : s + 1, (i + 1) % kR, p);
                        if (at == 0 && (s & 1)) read_chunk((s + 1) & 7);
                        if (at == kC && (s & 3) == 3) read_scales(s == 3 ? sb : sb + 1, s == 3);
                        if (s == 7 && at == kSlots - 1) read_sums(0);
                        accumulate(before, i_before, j, 4 * p, 4 * p + 4);
                        if (s == 0 && i == 0 && p == 2) asm volatile("" : "+v"(hdr[j]));
                        if (s == 0 && i == 0 && p == 2) d[j] = half_bits_to_f32(static_cast<uint16_t>(hdr[j].x & 0xFFFFu));
                        if (p == 3) {
                            const uint32_t scales = s < 4 ? hdr[j].y & 0x3F3F3F3Fu : (hdr[j].w & 0x0F0F0F0Fu) | ((hdr[j].y >> 2) & 0x30303030u);
                            factor[now][j] = d[j] * ubyte_to_f32(scales, s & 3);
                        }
                        if (i == kR - 1 && p > 0) convert((s + 1) & 7, j, p - 1);
                        if (s == 6 && i == 0 && p == 0) {
                            asm volatile("" : "+v"(hdr[j]));
                            const uint32_t mn_lo = hdr[j].z & 0x3F3F3F3Fu, mn_hi = ((hdr[j].w >> 4) & 0x0F0F0F0Fu) | ((hdr[j].z >> 2) & 0x30303030u);
                            mins[j] = make_uint4(bf16_pair(ubyte_to_f32(mn_lo, 0), ubyte_to_f32(mn_lo, 1)),
                                                 bf16_pair(ubyte_to_f32(mn_lo, 2), ubyte_to_f32(mn_lo, 3)),
                                                 bf16_pair(ubyte_to_f32(mn_hi, 0), ubyte_to_f32(mn_hi, 1)),
                                                 bf16_pair(ubyte_to_f32(mn_hi, 2), ubyte_to_f32(mn_hi, 3)));
                            asm volatile("" : "+v"(mins[j].x), "+v"(mins[j].y), "+v"(mins[j].z), "+v"(mins[j].w));
                            mins_live[j] &= (mn_lo + 0x7F7F7F7Fu) & (mn_hi + 0x7F7F7F7Fu);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
            if (s == 7) {
                // The min term of the whole super-block, sum over sub-blocks of m[column][sub] * X[row][sub]: A = the three bf16
                // parts of the eight sub-block sums of each row (K = part * 8 + sub), B = the eight 6-bit mins of each column
                // (nothing for the last eight K).
#pragma unroll
                for (int i = 0; i < kR; ++i) {
                    const int now = i & 1, before = now ^ 1, i_before = (i + kR - 1) % kR;  // (step 8 kR + i)
#pragma unroll
                    for (int m = 0; m < 2; ++m) {
                        union {
                            t_bf16x8 v;
                            uint4 u;
                        } sa, mb;
                        sa.u = sum_parts[m];
#pragma unroll
                        for (int j = 0; j < kC; ++j) {
                            mb.u = mins[j];
                            if (m == 1) mb.u = make_uint4(mb.u.x & first_half, mb.u.y & first_half, mb.u.z & first_half, mb.u.w & first_half);
                            D[now][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(sa.v, mb.v, m == 0 ? t_f32x16{} : D[now][j], 0, 0, 0);
                            __builtin_amdgcn_sched_barrier(0);
                            if (m == 1 && j == kC - 1 && i + 1 < kR) read_sums(i + 1);
                            accumulate(before, i_before, j, 8 * m, 8 * (m + 1));
                            if (m == 1) {
                                factor[now][j] = -half_bits_to_f32(static_cast<uint16_t>(hdr[j].x >> 16));
                                if (i == 0) slack[j] = fminf(slack[j], __builtin_fmaf(16.0f, __builtin_fabsf(factor[now][j]), -__builtin_fabsf(d[j])));
                            }
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                }
                if (kR & 1) {  // an odd number of steps: the next super-block expects the last one in the second set
#pragma unroll
                    for (int j = 0; j < kC; ++j) {
                        D[1][j] = D[0][j];
                        factor[1][j] = factor[0][j];
                    }
                }
            }
            // stage s + 2 has landed for every wavefront: the next stage reads its operands ahead
            if (s == 5) q4k_wait_vm<kLoadsFirst>();
            else if (s & 1) q4k_wait_vm<kLoadsEven>();
            else q4k_wait_vm<kLoadsOdd>();
            __syncthreads();
        }
    }
#pragma unroll
    for (int j = 0; j < kC; ++j) accumulate(1, kR - 1, j, 0, 16);
    q4k_wait_vm<0>();  // what is still on its way to LDS lands before the workgroup ends

    // add_lost: what the digits left behind of an activation, at most 2^(e - 40), where it can count.  A sub-block's dot holds the
    // values near 2^e with their nibbles and loses more than that when it is rounded -- unless those nibbles are zero; then the
    // products are (-dmin m) x, and where dmin m is at least d sc / 1024 their own rounding in 24 bits is the larger.  Columns
    // of which no super-block is below that line (16 |dmin| >= |d|, no m of zero) end the call here: all of ordinary weights,
    // whose min is about 8 steps of d sc.  The others look for sub-blocks with something left, take it from X itself, in three bf16
    // parts as gemm_q4k_rows32_kernel multiplies them, and decide by 32 rows x 32 columns x sub-block, so that
    // a result does not depend on the workgroup's tile.  Without this a channel 2^16 times the others, on weights that are zero,
    // would cost 1.8e-7 of a row's largest result, at 2^20 3.3e-6, at 2^30 3e-3.  us before / with this: 512 x 4096 x 14336 141.6 / 141.3, 333 x 14336
    // x 4096 120.4 / 119.7; weights of random bytes, where a 64th of the mins is zero, 148 / 174 and 125 / 146.
    // (a tile's columns past the matrix are zeros, which are below every line: they do not count.  us, counted / not: a pair of
    // 130 x 14336 x 1877 115 / 100, 917 x 1024 x 1512 32.3 / 29.5)
    bool below = false;
#pragma unroll
    for (int j = 0; j < kC; ++j)
        below |= (tile0 + wave * kC + j) * kTileCols + c < out_dim && ((mins_live[j] & 0x80808080u) != 0x80808080u || slack[j] < 0.0f);
    if (__builtin_amdgcn_ballot_w64(below) != 0) {
#pragma unroll
        for (int i = 0; i < kR; ++i) {
            const int mt = min(m_group * kR + i, m_tiles - 1), row = min(mt * kG32Rows + c, rows - 1);
            const uint8_t* const left_at = sums + static_cast<size_t>(mt) * kG32Rows * kb * 64 + 56;
            const uint8_t* const exponent_at = sums + static_cast<size_t>(row) * kb * 64 + 48;
            const float* const xrow = x + static_cast<size_t>(row) * in_dim + 16 * g;
#pragma unroll 1
            for (int sb0 = sb_begin; sb0 < sb_end; sb0 += 64) {
                uint64_t some = 0;  // a lane's super-block: the eight flags
                if (sb0 + lane < sb_end) some = *reinterpret_cast<const uint64_t*>(left_at + static_cast<size_t>(sb0 + lane) * 64);
                uint64_t todo = __builtin_amdgcn_ballot_w64(some != 0);
#pragma unroll 1
                while (todo != 0) {
                    const int from = __builtin_ctzll(todo), sb = sb0 + from;
                    todo &= todo - 1;
                    const uint64_t flags = static_cast<uint64_t>(__builtin_amdgcn_readlane(static_cast<uint32_t>(some >> 32), from)) << 32 |
                                           static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<uint32_t>(some), from));
                    const uint8_t* base[kC];
                    t_u32x4 h[kC];
#pragma unroll
                    for (int j = 0; j < kC; ++j) {
                        base[j] = tile_at(wave * kC + j) + static_cast<size_t>(sb) * kTileBytes;
                        h[j] = *reinterpret_cast<const t_u32x4*>(base[j] + 16 * c);
                    }
#pragma unroll 1
                    for (int sub = 0; sub < 8; ++sub) {
                        if ((flags >> (8 * sub) & 0xFFu) == 0) continue;
                        // everything is requested ahead of the look at the headers: this pass is a chain of trips to memory
                        const int exponent = exponent_at[static_cast<size_t>(sb) * 64 + sub];
                        float4 v[4];
#pragma unroll
                        for (int k = 0; k < 4; ++k) v[k] = reinterpret_cast<const float4*>(xrow + sb * kQ4kBlockValues + sub * 32)[k];
                        t_u32x4 q[kC];
#pragma unroll
                        for (int j = 0; j < kC; ++j) q[j] = *reinterpret_cast<const t_u32x4*>(base[j] + 512 + (sub >> 1) * 1024 + 16 * lane);
                        const int shift = 8 * (sub & 3);
                        float dsc[kC];
                        bool counts[kC], any = false;
#pragma unroll
                        for (int j = 0; j < kC; ++j) {
                            const uint32_t sc = sub < 4 ? h[j].y & 0x3F3F3F3Fu : (h[j].w & 0x0F0F0F0Fu) | ((h[j].y >> 2) & 0x30303030u);
                            const uint32_t mn = sub < 4 ? h[j].z & 0x3F3F3F3Fu : ((h[j].w >> 4) & 0x0F0F0F0Fu) | ((h[j].z >> 2) & 0x30303030u);
                            dsc[j] = half_bits_to_f32(static_cast<uint16_t>(h[j].x & 0xFFFFu)) * static_cast<float>(sc >> shift & 0xFFu);
                            const float min_term = half_bits_to_f32(static_cast<uint16_t>(h[j].x >> 16)) * static_cast<float>(mn >> shift & 0xFFu);
                            counts[j] = __builtin_amdgcn_ballot_w64(1024.0f * __builtin_fabsf(min_term) < __builtin_fabsf(dsc[j])) != 0;
                            any |= counts[j];
                        }
                        if (!any) continue;
                        union {
                            t_bf16x8 v;
                            uint32_t u[4];
                        } part[3][2];
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            const float r[4] = {left_behind(v[k].x, exponent), left_behind(v[k].y, exponent), left_behind(v[k].z, exponent),
                                                left_behind(v[k].w, exponent)};
#pragma unroll
                            for (int e = 0; e < 2; ++e)
                                split3_pair(r[2 * e], r[2 * e + 1], &part[0][k >> 1].u[2 * (k & 1) + e], &part[1][k >> 1].u[2 * (k & 1) + e],
                                            &part[2][k >> 1].u[2 * (k & 1) + e]);
                        }
#pragma unroll
                        for (int j = 0; j < kC; ++j) {
                            if (!counts[j]) continue;
                            t_f32x16 dot = t_f32x16{};
#pragma unroll
                            for (int m = 0; m < 2; ++m) {
                                union {
                                    t_bf16x8 v;
                                    t_bf16x2 pair[4];
                                } w;
#pragma unroll
                                for (int k = 0; k < 2; ++k) {
                                    const int nibbles = static_cast<int>(q[j][2 * m + k] >> (4 * (sub & 1)) & 0x0F0F0F0Fu);
                                    w.pair[2 * k] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(nibbles, 512.0f, false);
                                    w.pair[2 * k + 1] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(nibbles, 512.0f, true);
                                }
#pragma unroll
                                for (int t = 2; t >= 0; --t) dot = __builtin_amdgcn_mfma_f32_32x32x16_bf16(part[t][m].v, w.v, dot, 0, 0, 0);
                            }
#pragma unroll
                            for (int e = 0; e < 16; ++e)  // (dsc may be an infinity)
                                if (dot[e] != 0.0f) acc[i][j][e] = __builtin_fmaf(dsc[j], dot[e], acc[i][j][e]);
                        }
                    }
                }
            }
        }
    }

    // Results, from the registers.  A bias is a float a column.  All residuals are requested at once, and an activation is a loop over
    // a copy in LDS, not 64 copies of its code in a row (45 KB).  us of a call with a bias, gelu and a residual, against a loop that
    // took everything a value at a time, one trip to memory each (in brackets the bias alone): 75 x 256 x 2048 14.7 -> 11.4
    // (11.1 -> 8.1), 670 x 1024 x 5632 65 -> 44 (42 -> 34), 512 x 4096 x 14336 185 -> 163 (159 -> 150).
    const int row0 = m_group * S::kRows + 4 * g, col0 = (tile0 + wave * kC) * kTileCols + c;
    if (partial == nullptr && (ep.bias != nullptr || ep.residual != nullptr || ep.activation != kActNone)) {
        float bias[kC], residual[kR][kC][16];
        if (ep.bias != nullptr) {
#pragma unroll
            for (int j = 0; j < kC; ++j) bias[j] = ep.bias[min(col0 + j * kTileCols, out_dim - 1)];
        }
        if (ep.residual != nullptr) {  // (past the end: the last row's, the last column's; not stored)
#pragma unroll
            for (int i = 0; i < kR; ++i)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const float* from = ep.residual + static_cast<size_t>(min(row0 + i * kG32Rows + 8 * (v >> 2) + (v & 3), rows - 1)) * out_dim;
#pragma unroll
                    for (int j = 0; j < kC; ++j) residual[i][j][v] = from[min(col0 + j * kTileCols, out_dim - 1)];
                }
        }
        asm volatile("" : : : "memory");  // (requested here, not where they are used)
        if (ep.bias != nullptr) {
#pragma unroll
            for (int j = 0; j < kC; ++j)
#pragma unroll
                for (int i = 0; i < kR; ++i)
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc[i][j][v] += bias[j];
        }
        if (ep.activation != kActNone) {
            __syncthreads();  // every wavefront's loads have landed: the ring is free
            static_assert(kR * kC * kWaves * 4096 <= S::kLdsBytes, "a tile of results is 4 KB");
            float* copy = reinterpret_cast<float*>(q4k_mfma_lds) + wave * (kR * kC * 1024) + lane;  // a lane reads back what it wrote
#pragma unroll
            for (int i = 0; i < kR; ++i)
#pragma unroll
                for (int j = 0; j < kC; ++j)
#pragma unroll
                    for (int v = 0; v < 16; ++v) copy[((i * kC + j) * 16 + v) * 64] = acc[i][j][v];
#pragma unroll 1
            for (int n = 0; n < kR * kC * 4; ++n)
#pragma unroll
                for (int u = 0; u < 4; ++u) copy[(4 * n + u) * 64] = activate(ep.activation, copy[(4 * n + u) * 64]);
#pragma unroll
            for (int i = 0; i < kR; ++i)
#pragma unroll
                for (int j = 0; j < kC; ++j)
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc[i][j][v] = copy[((i * kC + j) * 16 + v) * 64];
        }
        if (ep.residual != nullptr) {
#pragma unroll
            for (int i = 0; i < kR; ++i)
#pragma unroll
                for (int j = 0; j < kC; ++j)
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc[i][j][v] += residual[i][j][v];
        }
    }
    float* out = partial == nullptr || (blockIdx.y == 0 && first_to_dst != 0) ? dst
                                                                              : partial + static_cast<size_t>(blockIdx.y - first_to_dst) * rows * out_dim;
#pragma unroll
    for (int j = 0; j < kC; ++j) {
        if (col0 + j * kTileCols >= out_dim) continue;
#pragma unroll
        for (int i = 0; i < kR; ++i) {
            float* to = out + static_cast<size_t>(row0 + i * kG32Rows) * out_dim + col0 + j * kTileCols;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int r = 8 * (v >> 2) + (v & 3);
                if (row0 + i * kG32Rows + r < rows) to[static_cast<size_t>(r) * out_dim] = acc[i][j][v];
            }
        }
    }
}

size_t q4k_mfma_lds_bytes(int rows, int in_dim, int waves, int groups) {
    return static_cast<size_t>(rows) * 3 * (static_cast<size_t>(in_dim) * 2 + kRowPadBytes) +
           static_cast<size_t>(rows) * (in_dim / 32) * 4 + static_cast<size_t>(waves) * groups * 64 * 4;
}

template <int kGroups>
hipError_t launch_q4k_mfma_rows(hipStream_t stream, float* dst, const float* x, const uint8_t* weight, int rows, int in_dim,
                                int out_dim, const Epilogue& ep, const Q4kSecond* second = nullptr) {
    // a second matrix on the same X: one launch where the int8 kernel serves the rows, else one after the other
    if (second != nullptr && kGroups > 2) {
        if (hipError_t e = launch_q4k_mfma_rows<kGroups>(stream, dst, x, weight, rows, in_dim, out_dim, ep); e != hipSuccess) return e;
        return launch_q4k_mfma_rows<kGroups>(stream, second->dst, x, second->weight, rows, in_dim, out_dim, second->ep);
    }
    const int kb = in_dim / kQ4kBlockValues;
    const int n_tiles = (out_dim + kTileCols - 1) / kTileCols;
    // One or two rows: sixteen K slices per tile (one tile, sixteen wavefronts a workgroup) -- the
    // most wavefronts, the shortest dependent chain each.  More rows: four slices and two tiles
    // a workgroup of eight wavefronts (their register need rules out sixteen), so that many
    // threads share the splitting of X.  (Measured on 14336 x 4096, 4096 x 14336, 4096 x 4096
    // and 128256 x 4096.)
    const int max_waves = kGroups == 1 ? 16 : 8;
    static const int env_shared = tuning_int("AFHIP_Q4K_SHARED_SPLIT"), env_bf16 = tuning_int("AFHIP_Q4K_BF16_DECODE");
    // one or two rows: fixed-point activations on the int8 matrix core (the bf16 kernel when a tuning run asks
    // for it and its three copies of X fit)
    // ... three or four rows too (eight slices, 512 threads) while their digit planes fit LDS and every workgroup has a
    // compute unit to itself: each workgroup makes the digits of all rows itself, which two workgroups sharing a unit's
    // vector ALUs cannot afford (N = 14336: 12.9 / 14.0 us against 12.6 / 13.0 on the bf16 kernel; 8192 x 8192: 15.2
    // against 18.3; 4096 x 4096: 8.9 against 11.1)
    const bool use_i8 = kGroups == 1 ? !((env_bf16 != 0 || env_shared != 0) && q4k_mfma_lds_bytes(rows, in_dim, 16, 1) <= kLdsBudget)
                                     : (kGroups == 2 && env_bf16 == 0 && n_tiles <= gemv_compute_units() &&
                                        q4k_i8_lds_bytes(rows, in_dim, 8) <= kLdsBudget);
    int slices = kGroups == 1 ? 16 : (use_i8 ? 8 : 4);
    // bf16 kernel: long rows (three or more super-blocks a slice) and vocabulary-sized matrices did better with
    // eight; the int8 kernel with sixteen everywhere (K = 14336: 12.5 against 13.8 us, K = 11008: 10.3 against 12.0)
    if (!use_i8 && slices == 16 && (kb > 32 || n_tiles > 2048)) slices = 8;
    while (slices > kb) slices /= 2;
    static const int env_slices = tuning_int("AFHIP_Q4K_SLICES"), env_tiles = tuning_int("AFHIP_Q4K_TILES_PER_WG");
    if (env_slices >= 1 && env_slices <= max_waves && (env_slices & (env_slices - 1)) == 0 && env_slices <= kb) slices = env_slices;
    // The int8 kernel at two rows on a matrix whose column tiles occupy at most half the compute units (one matrix
    // counted, so that each half of a pair takes the single op's path and has its bits), K long enough for a
    // super-block per wavefront of two workgroups, no epilogue: two K shares.  A call with an epilogue keeps one share and sums in
    // another order.  One row takes half tiles there, or their order of sums.
    auto plain = [](const Epilogue& e) { return e.bias == nullptr && e.residual == nullptr && e.activation == kActNone; };
    // One row of such a matrix, from seventeen super-blocks on: half tiles, all of K (us, against one share of whole tiles up to
    // 31 super-blocks and two shares with their clearing launch beyond; weights from memory): 4352 x 4096 columns 5.8 (6.1),
    // 5120 5.5 (6.4), 7168 6.4 (7.2), 8192 6.5 (8.4), 11008 8.8 (9.9), 14336 10.3 (10.7), 16384 10.5 (11.1), 14336 x 1024 8.2
    // (8.9), 8192 x 2048 5.6 (8.4).  4096 x 4096 columns is even (5.5) and stays.  A slice is whole pairs of super-blocks.  A
    // pair whose half tiles would take two rounds (5120 x 4096 columns each 8.9, 14336 20) takes whole tiles that add in the
    // half tiles' order (against one share, or two with their clearing launch): 5120 x 4096 7.2 (7.2), 8192 9.1 (10.0), 14336
    // 15.6 (17.1).
    const bool half_sums = kGroups == 1 && rows == 1 && use_i8 && env_slices == 0 && slices == 16 && kb > 16 &&
                           2 * n_tiles <= gemv_compute_units();
    const bool half_tiles = half_sums && (second == nullptr || 4 * n_tiles <= gemv_compute_units());
    const bool two_shares = kGroups == 1 && use_i8 && env_slices == 0 && slices == 16 && kb >= 32 && plain(ep) &&
                            (second == nullptr || plain(second->ep)) && !half_sums &&
                            2 * n_tiles <= gemv_compute_units();
    if (half_sums && kb < 32) slices = (kb + 1) / 2;
    const int sb_per_slice = half_sums ? ((kb + slices - 1) / slices + 1) / 2 * 2
                                       : (kb + (two_shares ? 2 : 1) * slices - 1) / ((two_shares ? 2 : 1) * slices);
    int tiles_per_wg = use_i8 ? 1 : (slices > 8 ? 16 : 8) / slices;  // (the int8 kernel: its wavefronts partition K, nothing else)
    if (!use_i8 && env_tiles >= 1 && env_tiles * slices <= max_waves) tiles_per_wg = env_tiles;
    const int waves = slices * tiles_per_wg;
    const int grid = half_tiles ? (out_dim + 15) / 16 : (n_tiles + tiles_per_wg - 1) / tiles_per_wg;
    const size_t lds = q4k_mfma_lds_bytes(rows, in_dim, waves, kGroups);
    // super-blocks requested ahead: all of a short slice (fewer registers, more wavefronts
    // resident), four at a time of a long one
    const int steps = half_tiles ? sb_per_slice / 2 : sb_per_slice;
    const int flight = steps <= 1 ? 0 : (steps <= 2 ? 1 : 2);
    const int variant = (waves > 8 ? 3 : 0) + flight;
    const bool own_slice = kGroups == 1 && tiles_per_wg == 1 && env_shared == 0;
    if constexpr (kGroups <= 2) {
        if (use_i8) {
            if (tiles_per_wg != 1) return hipErrorInvalidValue;  // (a tuning knob asked for a shape this kernel does not have)
            void (*k8)(float*, const float*, const uint8_t*, int, int, int, int, int, Epilogue, const uint8_t*, const float*, const float*, Q4kSecond, int) = nullptr;
            if constexpr (kGroups == 1) {
                switch (variant) {
                    case 0:
                    case 1: k8 = gemv_q4k_i8_kernel<1, 2, 512>; break;
                    case 2: k8 = gemv_q4k_i8_kernel<1, 2, 512>; break;  // (four in flight do not fit 128 registers here)
                    case 3: k8 = gemv_q4k_i8_kernel<1, 1, 1024>; break;
                    case 4: k8 = gemv_q4k_i8_kernel<1, 2, 1024>; break;
                    default: k8 = gemv_q4k_i8_kernel<1, 2, 1024>; break;  // (a longer slice: two super-blocks at a time)
                }
            } else {
                k8 = gemv_q4k_i8_kernel<2, 2, 512>;
            }
            if constexpr (kGroups == 1) {
                if (half_sums) k8 = gemv_q4k_i8_kernel<1, 2, 1024, false, false, true>;
                if (half_tiles) k8 = steps <= 1 ? gemv_q4k_i8_kernel<1, 1, 1024, false, true> : gemv_q4k_i8_kernel<1, 2, 1024, false, true>;
            }
            const size_t lds8 = q4k_i8_lds_bytes(rows, in_dim, waves);
            static LdsLimit lds_limit8[13];
            const int limit8 = half_tiles ? variant + 6 : (half_sums ? 12 : variant);
            if (hipError_t e = allow_lds(k8, lds8, &lds_limit8[limit8]); e != hipSuccess) return e;
            if (two_shares) {
                const int count = rows * out_dim;
                hipLaunchKernelGGL(q4k_zero_results_kernel, dim3((count + 1023) / 1024), dim3(256), 0, stream, dst,
                                   second ? second->dst : static_cast<float*>(nullptr), count);
                if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
            }
            hipLaunchKernelGGL(k8, dim3(grid, second ? 2 : 1, two_shares ? 2 : 1), dim3(waves * 64), lds8, stream, dst, x, weight, rows, in_dim,
                               out_dim, slices, sb_per_slice, ep, static_cast<const uint8_t*>(nullptr), static_cast<const float*>(nullptr),
                               static_cast<const float*>(nullptr), second ? *second : Q4kSecond{nullptr, nullptr, Epilogue{}}, two_shares ? 1 : 0);
            return hipGetLastError();
        }
    }
    if (second != nullptr) {  // (the bf16 kernel: one matrix a launch)
        if (hipError_t e = launch_q4k_mfma_rows<kGroups>(stream, dst, x, weight, rows, in_dim, out_dim, ep); e != hipSuccess) return e;
        return launch_q4k_mfma_rows<kGroups>(stream, second->dst, x, second->weight, rows, in_dim, out_dim, second->ep);
    }
    void (*kernel)(float*, const float*, const uint8_t*, int, int, int, int, int, Epilogue) = nullptr;
    switch (variant) {
        case 0:
        case 1:
            if constexpr (kGroups == 1) kernel = own_slice ? gemv_q4k_mfma_kernel<1, 2, 512, true> : gemv_q4k_mfma_kernel<1, 2>;
            else kernel = gemv_q4k_mfma_kernel<kGroups, 2>;
            break;
        case 2:
            if constexpr (kGroups == 1) kernel = own_slice ? gemv_q4k_mfma_kernel<1, 4, 512, true> : gemv_q4k_mfma_kernel<1, 4>;
            else kernel = gemv_q4k_mfma_kernel<kGroups, 4>;
            break;
        default:
            if constexpr (kGroups == 1) {  // sixteen wavefronts: at most 128 registers each
                if (own_slice)
                    kernel = variant == 3 ? gemv_q4k_mfma_kernel<1, 1, 1024, true>
                                          : (variant == 4 ? gemv_q4k_mfma_kernel<1, 2, 1024, true> : gemv_q4k_mfma_kernel<1, 4, 1024, true>);
                else
                    kernel = variant == 3 ? gemv_q4k_mfma_kernel<1, 1, 1024>
                                          : (variant == 4 ? gemv_q4k_mfma_kernel<1, 2, 1024> : gemv_q4k_mfma_kernel<1, 4, 1024>);
            }
            break;
    }
    if (kernel == nullptr) return hipErrorInvalidValue;
    static LdsLimit lds_limit[12];
    if (hipError_t e = allow_lds(kernel, lds, &lds_limit[variant + (own_slice ? 6 : 0)]); e != hipSuccess) return e;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(waves * 64), lds, stream, dst, x, weight, rows, in_dim, out_dim, slices,
                       sb_per_slice, ep);
    return hipGetLastError();
}

}  // namespace

size_t q4k_tiled_bytes(size_t out_dim, size_t in_dim) {
    return (out_dim + kTileCols - 1) / kTileCols * (in_dim / kQ4kBlockValues) * kTileBytes;
}

hipError_t launch_q4k_tile_repack(hipStream_t stream, uint8_t* dst, const uint8_t* src_raw, int out_dim, int in_dim) {
    const int kb = in_dim / kQ4kBlockValues;
    const size_t units = q4k_tiled_bytes(static_cast<size_t>(out_dim), static_cast<size_t>(in_dim)) / 16;
    if (units == 0) return hipSuccess;
    size_t grid = (units + 255) / 256;
    if (grid > 65536) grid = 65536;
    hipLaunchKernelGGL(q4k_tile_repack_kernel, dim3(static_cast<unsigned>(grid)), dim3(256), 0, stream,
                       reinterpret_cast<t_u32x4*>(dst), src_raw, out_dim, kb, units);
    return hipGetLastError();
}

hipError_t launch_dequantize_q4k_tiled_rows(hipStream_t stream, float* dst, const uint8_t* weight, const long long* ids,
                                            size_t rows, int dim, size_t weight_rows) {
    if (rows == 0 || dim == 0) return hipSuccess;
    size_t grid = (rows * static_cast<size_t>(dim >> 2) + 255) / 256;
    if (grid > 65536) grid = 65536;
    hipLaunchKernelGGL(dequantize_q4k_tiled_rows_kernel, dim3(static_cast<unsigned>(grid)), dim3(256), 0, stream, dst, weight,
                       ids, rows, dim, weight_rows);
    return hipGetLastError();
}

int gemv_q4k_tiled_rows_per_launch(int in_dim) {
    int per_launch = kMaxRowsPerLaunch;
    while (per_launch > 1 && q4k_mfma_lds_bytes(per_launch, in_dim, 8, (per_launch + 1) / 2) > kLdsBudget) --per_launch;
    // two rows on the int8 kernel: four one-byte digit planes a row instead of three bf16 copies
    if (per_launch < 2 && q4k_i8_lds_bytes(2, in_dim, 16) <= kLdsBudget) per_launch = 2;
    return per_launch;
}

// From this many rows on -- more than one launch of the GEMV kernel holds (LDS bounds its rows:
// six at K = 4096, one at K = 14336), and at least three -- the GEMM is the faster way (measured
// against two GEMV launches: 23 us against 26-29 at K = 4096, N = 14336; 34 us against 61-180 for
// 4-12 rows at K = 14336): small problems split K over up to eight workgroups whose sums a
// second kernel adds up.
int gemm_q4k_min_rows(int in_dim) {
    const int one_launch = gemv_q4k_tiled_rows_per_launch(in_dim);
    return one_launch + 1 > 3 ? one_launch + 1 : 3;
}

namespace {
int device_units() {
    static const int cus = []() {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
            n = 256;
        return n;
    }();
    return cus;
}

// What serves a GEMM call: the bf16 kernel (kParts), or the fp6 kernel with one of its tiles; and over how many workgroups K is
// shared out (at most eight, at least two super-blocks each, no empty one; kParts: a power of two).
enum Q4kGemmKind { kParts, kFp6Tile64x256, kFp6Tile64x128, kFp6Tile32x128 };
struct Q4kGemmPlan {
    Q4kGemmKind kind;
    int splits;
};

// Time of a call in us, from the rounds of the busiest XCD's compute units.  `steps[n]`: a sub-block of a wavefront's tiles with n + 1
// workgroups on the unit; `base`: launches, start and drain; `shares`, `share_mb`: the reduce launch and its MB; `split`: per million
// values of X; `out`: per MB of Y.  Fitted to 5400 timed plans of 420 calls (65 .. 2048 rows, K 256 .. 14336, N 64 .. 14336; 7 % rms);
// over these the choice is 1 % from the best tile and share count on the mean, 17 % at worst.
struct Q4kGemmCost {
    int rows, cols, tiles, resident;
    double steps[4], base, shares, share_mb, split, out;
    double us(double m, double k, double n, int s) const {
        const long long groups = static_cast<long long>((m + rows - 1) / rows) * static_cast<long long>((n + cols - 1) / cols);
        const long long units = device_units() >= 8 ? device_units() / 8 : 1;
        const long long per_unit = ((groups + 7) / 8 * s + units - 1) / units, kb = static_cast<long long>(k / kQ4kBlockValues);
        const double work = static_cast<double>(tiles * 8 * ((kb + s - 1) / s)), mb = m * n * 4e-6;
        const long long full = per_unit / resident, rest = per_unit % resident;
        double t = static_cast<double>(full) * work * steps[resident - 1] + base;
        if (rest > 0) t += work * steps[rest - 1];
        if (s > 1) t += shares + share_mb * (s + 1) * mb;
        return t + split * m * k * 1e-6 + out * mb;
    }
};
constexpr Q4kGemmCost kQ4kGemmCosts[4] = {
    {32, 256, 1, 2, {0.377, 0.664, 0, 0}, 6.1, 1.3, 0.63, 1.8, 0.41},
    {64, 256, 4, 2, {0.110, 0.214, 0, 0}, 8.3, 4.0, 0.26, 2.0, 0.30},
    {64, 128, 2, 2, {0.141, 0.255, 0, 0}, 7.0, 3.9, 0.27, 2.2, 0.295},
    {32, 128, 1, 4, {0.225, 0.319, 0.480, 0.620}, 6.6, 3.7, 0.24, 2.0, 0.27},
};

// The parts or digits of X with the sub-block sums behind them (the fp6 kernel's rows are padded to even), and the partial sums of
// K shares behind those.
size_t gemm_q4k_digit_bytes(size_t rows, size_t in_dim) { return (rows + 1) / 2 * 2 * in_dim * 6; }
size_t gemm_q4k_split_bytes(Q4kGemmKind kind, size_t rows, size_t in_dim) {
    const size_t values = kind == kParts ? rows * in_dim * 6 : gemm_q4k_digit_bytes(rows, in_dim);
    return (values + rows * (in_dim / 32) * 8 + 255) / 256 * 256;
}
// (the fp6 kernel's first share stores where the result goes: one array of sums fewer)
size_t gemm_q4k_sum_arrays(const Q4kGemmPlan& plan) {
    return plan.splits <= 1 ? 0 : static_cast<size_t>(plan.kind == kParts ? plan.splits : plan.splits - 1);
}
size_t gemm_q4k_plan_bytes(const Q4kGemmPlan& plan, size_t rows, size_t in_dim, size_t out_dim) {
    return gemm_q4k_split_bytes(plan.kind, rows, in_dim) + gemm_q4k_sum_arrays(plan) * rows * out_dim * 4;
}

bool gemm_q4k_shares_allowed(int splits, size_t in_dim) {
    const size_t kb = in_dim / kQ4kBlockValues, s = static_cast<size_t>(splits), each = (kb + s - 1) / s;
    return splits == 1 || (splits <= 8 && kb / s >= 2 && (kb + each - 1) / each == s);
}

// The bf16 kernel's own shares: one when its workgroups fill the compute units anyway, else as many as spread it over them.
Q4kGemmPlan gemm_q4k_parts_plan(size_t rows, size_t in_dim, size_t out_dim) {
    Q4kGemmPlan parts{kParts, 1};
    const long long workgroups = static_cast<long long>((out_dim + 255) / 256) * static_cast<long long>((rows + kG32Rows - 1) / kG32Rows);
    while (workgroups * parts.splits * 2 <= device_units() && parts.splits < 8 && in_dim / kQ4kBlockValues / (2 * parts.splits) >= 2) parts.splits *= 2;
    return parts;
}

// The scratch that a call may take: the cost of a plan says nothing of the memory it asks callers for (without a limit 129 x 5120 x 13824
// took 31 MB where X is 4, 512 x 8192 x 28672 137 where X is 25).  A call whose bf16 plan fits the static entry's array keeps
// fitting it; past that the partial sums may take twice what the bf16 plan takes.  By the cost model the limit is 0.5 % on the mean of
// 4000 shapes (65 .. 2048 rows), 128 of them more than 5 % -- 815, and 2.7 %, with powers of two alone and an array for every share.
// us with the limit / eight shares allowed without one: 113 x 11008 x 6144 62 / 60, 333 x 4096 x 6144 71 / 69, but 167 x 12288 x 2580
// 54 / 47, 176 x 7680 x 11008 119 / 103 (one share), 243 x 8448 x 5375 109 / 81.
size_t gemm_q4k_most_bytes(size_t rows, size_t in_dim, size_t out_dim) {
    const size_t parts = gemm_q4k_plan_bytes(gemm_q4k_parts_plan(rows, in_dim, out_dim), rows, in_dim, out_dim);
    return parts <= AFHIP_STATIC_SCRATCH_BYTES ? static_cast<size_t>(AFHIP_STATIC_SCRATCH_BYTES) : 3 * parts;
}

// The plan of a call that lends `room` bytes (splits = 0: none fits).  Whoever lends gemm_q4k_workspace_bytes or more gets the
// same one: the choice is over what fits, and the best of all that fits the most a call may take is the best of fewer.
// A result's bits depend on the shares alone, and a pair's halves have the single call's, while a pair is one launch on one share only.
// Columns of at least twice K, which mostly come in pairs (gate and up): a quarter of the pair's time counts beside the call's own
// (99 x 2816 x 9728 twice: one share 51 us, two 59, a call 29.7 and 28.8; 99 x 2048 x 4096 a call 17.4 on the bf16 kernel's shares and 21
// on one of the 6-bit kernel's).  Other shapes: the call's own, one share where that costs at most 3 % more.
// `pair`: the tile may be another than the single call's (333 x 4096 x 14336 twice: 64 x 256 tiles 212 us, 64 x 128 231; once 124 / 119).
// An activation is sixteen values and more a lane of the matrix kernels, about 3 us, and one a thread of the reduce launch: a third of
// that is counted (65 x 1024 x 4096 plain 13.7 us on the bf16 kernel's shares and 13.3 on one of the 6-bit kernel's, with gelu 14.5 and 16.7).
// Up to 64 rows the bf16 kernel is the faster one (64 x 4096 x 4096 17.5 against 19.4 us, 32 x 4096 x 14336 21.4 / 22.4), above where it is
// expected within 3 %.
constexpr double kEpilogueUs = 1.0;
Q4kGemmPlan gemm_q4k_plan(size_t rows, size_t in_dim, size_t out_dim, size_t room, bool pair = false) {
    const double m = static_cast<double>(rows), k = static_cast<double>(in_dim), n = static_cast<double>(out_dim);
    room = std::min(room, gemm_q4k_most_bytes(rows, in_dim, out_dim));
    auto fits = [&](const Q4kGemmPlan& p) { return gemm_q4k_plan_bytes(p, rows, in_dim, out_dim) <= room; };
    const Q4kGemmPlan none{kParts, 0}, parts = gemm_q4k_parts_plan(rows, in_dim, out_dim);
    if (rows <= 64) return fits(parts) ? parts : none;
    Q4kGemmKind pair_kind = kFp6Tile64x256;  // of one share
    double pair_us = 1e30;
    for (int kind = kFp6Tile64x256; kind <= kFp6Tile32x128; ++kind)
        if (const double us = kQ4kGemmCosts[kind].us(m, k, 2 * n, 1); us < pair_us) {
            pair_us = us;
            pair_kind = static_cast<Q4kGemmKind>(kind);
        }
    auto cost = [&](const Q4kGemmPlan& plan) {
        const double epilogue = plan.splits == 1 ? kEpilogueUs : 0.0;
        const double us = kQ4kGemmCosts[plan.kind].us(m, k, n, plan.splits) * (plan.kind == kParts ? 0.97 : 1.0) + epilogue;
        if (out_dim < 2 * in_dim) return us * (plan.kind != kParts && plan.splits > 1 ? 1.03 : 1.0);
        const bool together = plan.kind != kParts && plan.splits == 1;
        return us + 0.25 * (together ? pair_us + epilogue : 2 * us - kQ4kGemmCosts[plan.kind].split * m * k * 1e-6);
    };
    Q4kGemmPlan best = none;
    double best_cost = 1e60;
    for (int s = 1; s <= 8; ++s) {
        if (!gemm_q4k_shares_allowed(s, in_dim)) continue;
        for (int kind = kFp6Tile64x256; kind <= kFp6Tile32x128; ++kind) {
            const Q4kGemmPlan plan{static_cast<Q4kGemmKind>(kind), s};
            if (const double c = cost(plan); c < best_cost && fits(plan)) {
                best_cost = c;
                best = plan;
            }
        }
    }
    if (fits(parts) && cost(parts) < best_cost) return parts;
    if (pair && best.splits == 1) best.kind = pair_kind;
    return best;
}

struct Q4kGemmCall {
    hipStream_t stream;
    const float* x;
    float* dst;
    const uint8_t *digits, *sums, *weight;
    int rows, in_dim, out_dim, sb_per_split, shares;
    float* partial;
    bool first_to_dst;
    const Epilogue& ep;
    const Q4kSecond* second;
};

template <int kWaves, int kR, int kC, int kOcc>
hipError_t launch_fp6_tile(const Q4kGemmCall& q) {
    using S = G6Shape<kWaves, kR, kC>;
    const int m_groups = (q.rows + S::kRows - 1) / S::kRows, n_groups = (q.out_dim + S::kCols - 1) / S::kCols;
    const long long grid = (static_cast<long long>(n_groups) * m_groups + 7) / 8 * 8;
    if (grid > 0x7fffffffLL) return hipErrorInvalidValue;
    auto kernel = gemm_q4k_fp6_kernel<kWaves, kR, kC, kOcc>;
    static LdsLimit lds_limit;
    if (hipError_t e = allow_lds(kernel, S::kLdsBytes, &lds_limit); e != hipSuccess) return e;
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid), q.shares, q.second ? 2 : 1), dim3(S::kThreads), S::kLdsBytes, q.stream, q.dst,
                       q.digits, q.sums, q.weight, q.rows, q.in_dim, q.out_dim, m_groups, n_groups, 8, q.sb_per_split, q.partial, q.first_to_dst ? 1 : 0, q.ep,
                       q.second ? *q.second : Q4kSecond{nullptr, nullptr, Epilogue{}}, q.x);
    return hipGetLastError();
}
}  // namespace

size_t gemm_q4k_workspace_bytes(size_t rows, size_t in_dim, size_t out_dim) {
    return gemm_q4k_plan_bytes(gemm_q4k_plan(rows, in_dim, out_dim, SIZE_MAX), rows, in_dim, out_dim);
}

bool gemm_q4k_fits(size_t rows, size_t in_dim, size_t out_dim, size_t workspace_bytes) {
    return gemm_q4k_plan(rows, in_dim, out_dim, workspace_bytes).splits != 0;
}

hipError_t launch_gemm_q4k_tiled(hipStream_t stream, float* dst, const float* x, const uint8_t* weight, void* workspace,
                                 size_t workspace_bytes, int rows, int in_dim, int out_dim, const Epilogue& ep, float* dst_b,
                                 const uint8_t* weight_b, const Epilogue& ep_b) {
    if (in_dim % kQ4kBlockValues != 0 || rows < 1 || workspace == nullptr) return hipErrorInvalidValue;
    const size_t m = rows, k = in_dim, n = out_dim;
    Q4kGemmPlan plan = gemm_q4k_plan(m, k, n, workspace_bytes, dst_b != nullptr);
    if (plan.splits == 0) return hipErrorInvalidValue;
    // the fp6 kernel may look at X again when other workgroups have stored results
    auto over_x = [&](const float* y) {
        const uintptr_t a = reinterpret_cast<uintptr_t>(x), b = reinterpret_cast<uintptr_t>(y);
        return y != nullptr && b < a + m * k * 4 && a < b + m * n * 4;
    };
    if (plan.kind != kParts && (over_x(dst) || over_x(dst_b))) {
        plan = gemm_q4k_parts_plan(m, k, n);
        if (gemm_q4k_plan_bytes(plan, m, k, n) > workspace_bytes) plan.splits = 1;
    }
    // (a residual in the result's place has to outlast the first share: the sums take an array each then, and fewer shares where
    // those have no room)
    const bool over_residual = ep.residual != nullptr && reinterpret_cast<uintptr_t>(ep.residual) < reinterpret_cast<uintptr_t>(dst) + m * n * 4 &&
                               reinterpret_cast<uintptr_t>(dst) < reinterpret_cast<uintptr_t>(ep.residual) + m * n * 4;
    const bool first_to_dst = plan.kind != kParts && plan.splits > 1 && !over_residual;
    if (plan.kind != kParts && over_residual)
        while (plan.splits > 1 && gemm_q4k_split_bytes(plan.kind, m, k) + plan.splits * m * n * 4 > workspace_bytes) --plan.splits;
    const int kb = in_dim / kQ4kBlockValues;
    const int sb_per_split = (kb + plan.splits - 1) / plan.splits;
    const int shares = (kb + sb_per_split - 1) / sb_per_split;  // no empty share
    uint8_t* const space = static_cast<uint8_t*>(workspace);
    float* partial = shares > 1 ? reinterpret_cast<float*>(space + gemm_q4k_split_bytes(plan.kind, rows, in_dim)) : nullptr;
    const int m_tiles = (rows + kG32Rows - 1) / kG32Rows;
    if (m_tiles > 65535) return hipErrorInvalidValue;
    uint32_t* parts = static_cast<uint32_t*>(workspace);
    uint16_t* part_sums = reinterpret_cast<uint16_t*>(space + static_cast<size_t>(rows) * in_dim * 6);
    uint8_t* digit_sums = space + gemm_q4k_digit_bytes(rows, in_dim);
    if (plan.kind == kParts) {
        const size_t groups = static_cast<size_t>(rows) * (in_dim >> 3);
        size_t split_grid = (groups + 255) / 256;
        if (split_grid > 65536) split_grid = 65536;
        hipLaunchKernelGGL(q4k_split_parts_kernel, dim3(static_cast<unsigned>(split_grid)), dim3(256), 0, stream, x, parts, part_sums,
                           groups, in_dim >> 3);
    } else {
        hipLaunchKernelGGL(q4k_split_digits_kernel, dim3(in_dim / 32, m_tiles), dim3(256), 0, stream, x, space, digit_sums, rows, in_dim);
    }
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    const Q4kSecond second{dst_b, weight_b, ep_b};
    auto multiply = [&](float* y, const uint8_t* w, const Epilogue& epilogue, const Q4kSecond* with) {
        const Q4kGemmCall q{stream, x, y, space, digit_sums, w, rows, in_dim, out_dim, sb_per_split, shares, partial, first_to_dst, epilogue, with};
        hipError_t e;
        if (plan.kind == kFp6Tile64x256) e = launch_fp6_tile<4, 2, 2, 2>(q);
        else if (plan.kind == kFp6Tile64x128) e = launch_fp6_tile<4, 2, 1, 2>(q);
        else if (plan.kind == kFp6Tile32x128) e = launch_fp6_tile<4, 1, 1, 3>(q);
        else {
            static_assert(2 * kG32ChunkBytes <= 64 * 1024, "no raised LDS limit");
            const unsigned grid_x = static_cast<unsigned>((out_dim + 255) / 256);
            hipLaunchKernelGGL(gemm_q4k_rows32_kernel, dim3(grid_x, m_tiles, shares), dim3(512), 2 * kG32ChunkBytes, stream, y, parts,
                               part_sums, w, rows, in_dim, out_dim, sb_per_split, partial, epilogue);
            e = hipGetLastError();
        }
        if (e != hipSuccess || shares == 1) return e;
        return launch_splitk_reduce(stream, y, partial, static_cast<size_t>(rows) * out_dim, out_dim, shares, epilogue, first_to_dst);
    };
    if (dst_b == nullptr) return multiply(dst, weight, ep, nullptr);
    if (shares == 1 && plan.kind != kParts) return multiply(dst, weight, ep, &second);
    // (the partial sums have room for one matrix)
    if (hipError_t e = multiply(dst, weight, ep, nullptr); e != hipSuccess) return e;
    return multiply(dst_b, weight_b, ep_b, nullptr);
}

// Three to eight rows with the caller's scratch: the digit planes of X made once by their own kernel
// (launch_q4k_digit_planes), then one launch per matrix of the int8 kernel with its operands read from them.
bool q4k_i8_rows_supports(size_t rows, size_t in_dim) {
    return rows >= 3 && rows <= 8 && in_dim % kQ4kBlockValues == 0 && in_dim <= static_cast<size_t>(gemv_q4k_max_in_dim());
}

// [operand fragments: 8 KB a super-block][-s: 8 rows x super-blocks][sub-block sums: 8 rows x super-blocks x 8]
size_t q4k_i8_rows_workspace_bytes(size_t in_dim) {
    const size_t kb = in_dim / kQ4kBlockValues;
    return kb * 8192 + kb * 8 * 4 + kb * 8 * 8 * 4;
}

// Whether launch_gemv_q4k_i8_rows shares K out over two workgroups per column tile, which add to the result arrays: then
// launch_q4k_digit_planes has to clear them.  Column tiles that occupy at most half the compute units (one matrix
// counted: each half of a pair then has the single op's bits), a super-block per wavefront of both shares, no epilogue.
bool q4k_i8_rows_two_shares(size_t rows, size_t in_dim, size_t out_dim, bool pair, const Epilogue& ep, const Epilogue& ep_b) {
    auto plain = [](const Epilogue& e) { return e.bias == nullptr && e.residual == nullptr && e.activation == kActNone; };
    if (!q4k_i8_rows_supports(rows, in_dim) || !plain(ep) || (pair && !plain(ep_b))) return false;
    const size_t n_tiles = (out_dim + kTileCols - 1) / kTileCols;
    return in_dim / kQ4kBlockValues >= 16 && 2 * n_tiles <= static_cast<size_t>(gemv_compute_units());
}

hipError_t launch_q4k_digit_planes(hipStream_t stream, const float* x, int rows, int in_dim, void* workspace, float* zero_a,
                                   float* zero_b, size_t zero_count) {
    if (!q4k_i8_rows_supports(static_cast<size_t>(rows), static_cast<size_t>(in_dim)) || workspace == nullptr) return hipErrorInvalidValue;
    const int kb = in_dim / kQ4kBlockValues;
    uint8_t* frag = static_cast<uint8_t*>(workspace);
    float* minus_s = reinterpret_cast<float*>(frag + static_cast<size_t>(kb) * 8192);
    float* sums = minus_s + static_cast<size_t>(kb) * 8;
    const int items = rows * kb;
    hipLaunchKernelGGL(q4k_digit_planes_kernel, dim3((items + 3) / 4), dim3(256), 0, stream, x, rows, in_dim, frag, minus_s, sums, zero_a,
                       zero_b, static_cast<int>(zero_count));
    return hipGetLastError();
}

hipError_t launch_gemv_q4k_i8_rows(hipStream_t stream, float* dst, const void* workspace, const uint8_t* weight, int rows, int in_dim,
                                   int out_dim, const Epilogue& ep, float* dst_b, const uint8_t* weight_b, const Epilogue& ep_b,
                                   bool results_cleared) {
    if (!q4k_i8_rows_supports(static_cast<size_t>(rows), static_cast<size_t>(in_dim)) || workspace == nullptr) return hipErrorInvalidValue;
    if (out_dim == 0) return hipSuccess;
    const int kb = in_dim / kQ4kBlockValues;
    const uint8_t* frag = static_cast<const uint8_t*>(workspace);
    const float* minus_s = reinterpret_cast<const float*>(frag + static_cast<size_t>(kb) * 8192);
    const float* sums = minus_s + static_cast<size_t>(kb) * 8;
    int slices = 8;
    while (slices > kb) slices /= 2;
    // (two K shares only when the caller had the result arrays cleared by the digit planes' launch)
    const bool two_shares = results_cleared && q4k_i8_rows_two_shares(static_cast<size_t>(rows), static_cast<size_t>(in_dim),
                                                                      static_cast<size_t>(out_dim), weight_b != nullptr, ep, ep_b);
    const int shares = two_shares ? 2 : 1, accumulate = two_shares ? 1 : 0;
    const int sb_per_slice = (kb + shares * slices - 1) / (shares * slices);
    const int n_tiles = (out_dim + kTileCols - 1) / kTileCols;
    const size_t lds = q4k_i8_rows_lds_bytes(rows, in_dim, slices);
    const float* no_x = nullptr;
    const Q4kSecond second{dst_b, weight_b, ep_b};
    const dim3 grid(n_tiles, weight_b != nullptr ? 2 : 1, shares);
    switch ((rows + 1) / 2) {
        case 2:
            hipLaunchKernelGGL((gemv_q4k_i8_kernel<2, 1, 512, true>), grid, dim3(64 * slices), lds, stream, dst, no_x, weight, rows, in_dim,
                               out_dim, slices, sb_per_slice, ep, frag, minus_s, sums, second, accumulate);
            break;
        case 3:
            hipLaunchKernelGGL((gemv_q4k_i8_kernel<3, 1, 512, true>), grid, dim3(64 * slices), lds, stream, dst, no_x, weight, rows, in_dim,
                               out_dim, slices, sb_per_slice, ep, frag, minus_s, sums, second, accumulate);
            break;
        default:
            hipLaunchKernelGGL((gemv_q4k_i8_kernel<4, 1, 512, true>), grid, dim3(64 * slices), lds, stream, dst, no_x, weight, rows, in_dim,
                               out_dim, slices, sb_per_slice, ep, frag, minus_s, sums, second, accumulate);
            break;
    }
    return hipGetLastError();
}

hipError_t launch_gemv_q4k_tiled(hipStream_t stream, float* dst, const float* x, const uint8_t* weight, int rows, int in_dim,
                                 int out_dim, const Epilogue& ep0, float* dst_b, const uint8_t* weight_b, const Epilogue& ep_b0) {
    if (in_dim % kQ4kBlockValues != 0 || in_dim > gemv_q4k_max_in_dim()) return hipErrorInvalidValue;
    // as many rows per launch as LDS holds (three bf16 copies of each), at most eight
    const int per_launch = gemv_q4k_tiled_rows_per_launch(in_dim);
    if (per_launch > 2 && q4k_mfma_lds_bytes(per_launch, in_dim, 8, 1) > kLdsBudget) return hipErrorInvalidValue;
    if (per_launch <= 2 && q4k_i8_lds_bytes(per_launch, in_dim, 16) > kLdsBudget) return hipErrorInvalidValue;
    for (int r0 = 0; r0 < rows; r0 += per_launch) {
        const int nr = rows - r0 < per_launch ? rows - r0 : per_launch;
        float* d = dst + static_cast<size_t>(r0) * out_dim;
        const float* xr = x + static_cast<size_t>(r0) * in_dim;
        Epilogue ep = ep0;
        if (ep.residual) ep.residual += static_cast<size_t>(r0) * out_dim;
        Q4kSecond second{dst_b ? dst_b + static_cast<size_t>(r0) * out_dim : nullptr, weight_b, ep_b0};
        if (second.ep.residual) second.ep.residual += static_cast<size_t>(r0) * out_dim;
        const Q4kSecond* sec = weight_b != nullptr ? &second : nullptr;
        hipError_t e;
        switch ((nr + 1) / 2) {
            case 1: e = launch_q4k_mfma_rows<1>(stream, d, xr, weight, nr, in_dim, out_dim, ep, sec); break;
            case 2: e = launch_q4k_mfma_rows<2>(stream, d, xr, weight, nr, in_dim, out_dim, ep, sec); break;
            case 3: e = launch_q4k_mfma_rows<3>(stream, d, xr, weight, nr, in_dim, out_dim, ep, sec); break;
            default: e = launch_q4k_mfma_rows<4>(stream, d, xr, weight, nr, in_dim, out_dim, ep, sec); break;
        }
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace afhip
