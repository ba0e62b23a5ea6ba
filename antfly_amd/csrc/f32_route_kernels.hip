// The f32 route (fewer than 512 columns, or K below 96: narrow key / value projections) on the matrix cores, PREPARED
// layout: y[r][o] = sum over blocks of d[o][b] * sum_i x[r][32 b + i] * q[o][32 b + i], f32 activations.
//
// What bounded the one-wavefront-per-output kernel (linear_f32_route_kernel, still used for few outputs and the raw layout):
// every output read its whole row of X and row of W again and converted every weight again -- one convert and one
// multiply-add per weight and row on the vector ALU.  Here an activation is split once per workgroup column group into
// three bf16 numbers hi + mid + lo, each the leading eight bits of what the previous ones left over: together all 24 bits
// of the f32, so the products q * x (q is exact in bf16) are exact in the accumulator and nothing is lost against f32.
// (Below about 2^-110 the last part is a subnormal, which holds fewer than eight bits: a wavefront that met such a value goes
// over its blocks once more for what was left.  Without that the error at 2^-116 was 6e-6 of the row's largest output, at 2^-124
// 1.8e-3; now 2.4e-7 and 3.1e-7.)
// Three v_mfma_f32_16x16x32_bf16 per 16 rows x 16 columns x block then leave the block's dots, and one multiply-add per
// element applies the scale, as before.
//
// A workgroup owns 16 rows x 16 * kTiles columns and all of K; its wavefronts (sixteen where K allows) take a run of blocks each
// and their sums meet in LDS in wavefront order.  kTiles column tiles share one split of X: the split is about 70 of 100 vector
// instructions at one tile, but a short prompt has too few tiles to give up workgroups for it.
// What bounded it on most shapes was neither the split nor latency but the address unit: with every lane loading the values it
// multiplies, a load of X asks for sixteen lines, one a lane of a quad, and so does a load of weights -- about 800 cycles of
// address work a wavefront and four blocks.  One column tile therefore loads whole lines and lets its lanes exchange them
// through LDS (2 KB of X, up to 2 KB of weights a wavefront, where the sums go afterwards): about 180.
// us, loaded by its user / by lines, Q4_0: a pair of 256 columns at K = 2048, 77 rows 9.8 / 6.6, 300 rows 24 / 13.5, 2048 rows 73 / 62;
// 333 x 4096 x 100 17.3 / 11.5, 20 x 4096 x 500 16.5 / 9.6.  Now the vector ALU (the split) on many rows, launch and latency on few.
// Relative error against 64 bits 1.0e-7.
#include <hip/hip_runtime.h>

#include "device_common.h"
#include "qmatmul_launch.h"

namespace afhip {

namespace {

typedef float r_f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 r_bf16x8 __attribute__((ext_vector_type(8)));
union Bf16x8 {
    r_bf16x8 v;
    uint32_t u[4];
};

constexpr int kRouteRows = 16;   // rows of a workgroup, and columns of a tile
constexpr int kWaveFloats = 1024;  // of LDS: a block of X (2 KB), one tile's weights of four blocks (2 KB); at the end the sums

// What a wavefront's own lanes hand each other through LDS: the operations of a wavefront complete in order, only the compiler
// has to keep theirs.
__device__ __forceinline__ void wave_order() {
    asm volatile("" : : : "memory");
}

__device__ __forceinline__ uint32_t upper_halves(float a, float b) {  // bf16 bits of a, b (already exact in bf16): a low, b high
    return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, b), __builtin_bit_cast(uint32_t, a), 0x07060302u);
}
__device__ __forceinline__ float leading8(float v) { return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v) & 0xFFFF0000u); }

// x = hi + mid + lo exactly (truncation: no rounding can overflow).  An infinity is its own hi with nothing left over, so that
// it reaches the sum as an infinity; a NaN leaves a NaN behind even where its payload lies in the low bits.
// `left` collects the lanes whose lo has bits in the half that a bf16 does not hold: values below about 2^-110 only.
__device__ __forceinline__ void split_pair(float x0, float x1, uint32_t* hi, uint32_t* mid, uint32_t* lo, uint64_t* left) {
    const float h0 = leading8(x0), h1 = leading8(x1);
    const float r0 = __builtin_isinf(x0) ? 0.0f : x0 - h0, r1 = __builtin_isinf(x1) ? 0.0f : x1 - h1;
    const float m0 = leading8(r0), m1 = leading8(r1);
    *hi = upper_halves(h0, h1);
    *mid = upper_halves(m0, m1);
    const float l0 = r0 - m0, l1 = r1 - m1;
    *lo = upper_halves(l0, l1);
    *left |= __ballot(static_cast<uint16_t>(__builtin_bit_cast(uint32_t, l0) | __builtin_bit_cast(uint32_t, l1)) != 0);
}

// What hi + mid + lo leave of x, at most sixteen bits of a subnormal, times 2^100: a normal number, in two bf16 parts.
__device__ __forceinline__ void left_pair(float x0, float x1, uint32_t* hi, uint32_t* lo) {
    const float x[2] = {x0, x1};
    float h[2], l[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const float r = __builtin_isinf(x[i]) ? 0.0f : x[i] - leading8(x[i]);
        const float lo_part = r - leading8(r);
        const float e = (lo_part - leading8(lo_part)) * 0x1p100f;
        h[i] = leading8(e);
        l[i] = e - h[i];
    }
    *hi = upper_halves(h[0], h[1]);
    *lo = upper_halves(l[0], l[1]);
}

// Where in a block's bytes the eight values 8 g .. 8 g + 7 lie; Q4_0: values 0..15 are the low nibbles of the 16 bytes, 16..31
// the high ones.
template <int kType>
__device__ __forceinline__ int quant_offset(int g) { return 8 * (kType == 2 ? g & 1 : g); }

// Eight weights of a lane as bf16: bytes biased to unsigned (nibbles are so already), converted, the bias taken off: integers
// below 2^8, exact.
template <int kType>
__device__ __forceinline__ r_bf16x8 weights_bf16(uint2 packed, int g) {
    const uint32_t p[2] = {packed.x, packed.y};
    Bf16x8 w;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint32_t biased = kType == 2 ? (p[i] >> (4 * (g >> 1))) & 0x0F0F0F0Fu : p[i] ^ 0x80808080u;
        constexpr float kBias = kType == 2 ? 8.0f : 128.0f;
        const float f0 = static_cast<float>(biased & 0xFFu) - kBias, f1 = static_cast<float>((biased >> 8) & 0xFFu) - kBias;
        const float f2 = static_cast<float>((biased >> 16) & 0xFFu) - kBias, f3 = static_cast<float>(biased >> 24) - kBias;
        w.u[2 * i] = upper_halves(f0, f1);
        w.u[2 * i + 1] = upper_halves(f2, f3);
    }
    return w.v;
}

}  // namespace

// A second matrix of the same shape on the same X: grid.z = 2.
struct RouteSecond {
    float* dst;
    const uint8_t* weight;
    Epilogue ep;
};

// kDepth: blocks a wavefront requests ahead of its arithmetic.
template <int kType, int kTiles, int kDepth>
__global__ __launch_bounds__(1024, 8) void linear_f32_rows_kernel(float* __restrict__ dst_a, const float* __restrict__ x,
                                                               const uint8_t* __restrict__ weight_a, int rows, int in_dim, int out_dim,
                                                               Epilogue ep_a, RouteSecond second) {
    extern __shared__ __align__(16) float route_sums[];  // a wavefront's kWaveFloats; sums: [tile][4][64]
    const bool is_b = blockIdx.z != 0;
    float* dst = is_b ? second.dst : dst_a;
    const uint8_t* weight = is_b ? second.weight : weight_a;
    const Epilogue ep = is_b ? second.ep : ep_a;
    constexpr int kQuantBytes = kType == 2 ? 16 : 32;
    const int kb = in_dim >> 5;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6;
    const int c = lane & 15, g = lane >> 4;  // operand row / column, and the eight values 8 g .. 8 g + 7 of a block
    const int m0 = blockIdx.y * kRouteRows, n0 = blockIdx.x * (16 * kTiles);
    // rows and columns past the end repeat the last one; their results are not stored
    // One tile: X is loaded eight lanes a row and block (rows r8 and r8 + 8), whole lines, and goes to the operand's lanes through
    // LDS, as the weights do.  A lane that loads what it multiplies asks for sixteen lines a load, four a quad of lanes, and the
    // address unit was what bounded the kernel (with four tiles the registers do not allow it; loaded by its user there).
    constexpr bool kStaged = kTiles == 1;
    const int r8 = lane >> 3, ch = lane & 7;
    const float* xrow[2];
    if constexpr (kStaged) {
#pragma unroll
        for (int i = 0; i < 2; ++i) xrow[i] = x + static_cast<size_t>(min(m0 + r8 + 8 * i, rows - 1)) * in_dim + 4 * ch;
    } else {
        xrow[0] = x + static_cast<size_t>(min(m0 + c, rows - 1)) * in_dim + 8 * g;
        xrow[1] = xrow[0] + 4;
    }
    float* own = route_sums + wave * kWaveFloats;
    float4* own_x = reinterpret_cast<float4*>(own);                       // [row][chunk ^ row / 2], 16 bytes each: a read in 16 banks' groups
    // [block][16-byte half][column ^ 2 * place of block and half]: written by lanes of one column and all places, read by all columns
    // of one place, in different banks both times
    unsigned char* own_w = reinterpret_cast<unsigned char*>(own) + 2048;
    auto weight_slot = [](int place, int column) { return place * 16 + (column ^ (2 * place & 15)); };
    const size_t blocks = static_cast<size_t>(out_dim) * kb;
    const uint16_t* scales = reinterpret_cast<const uint16_t*>(weight + blocks * kQuantBytes);
    size_t first[kTiles];  // first block of this lane's column in each tile
#pragma unroll
    for (int t = 0; t < kTiles; ++t) first[t] = static_cast<size_t>(min(n0 + 16 * t + c, out_dim - 1)) * kb;

    // (one tile) a column's four blocks are one load of 64 bytes (Q8_0: two loads of 64 lanes, 128 bytes a column), its four scales are
    // four lanes'
    constexpr int kWeightLoads = kType == 2 ? 1 : 2;
    const uint8_t* wcol[kWeightLoads];
    const uint16_t* scol = scales + static_cast<size_t>(min(n0 + (lane >> 2), out_dim - 1)) * kb;
#pragma unroll
    for (int i = 0; i < kWeightLoads; ++i) {
        const int col = kType == 2 ? lane >> 2 : 8 * i + r8, half = kType == 2 ? 0 : ch & 1;
        wcol[i] = weight + static_cast<size_t>(min(n0 + col, out_dim - 1)) * kb * kQuantBytes + 16 * half;
    }

    r_f32x4 acc[kTiles];
#pragma unroll
    for (int t = 0; t < kTiles; ++t) acc[t] = r_f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    uint64_t left_behind = 0;  // lanes that met a value below about 2^-110
    // a wavefront's blocks follow each other, parts of the same lines of weights; the first kb % waves wavefronts have one more
    const int per_wave = kb / waves, more = kb - per_wave * waves, begin = wave * per_wave + min(wave, more), end = begin + per_wave + (wave < more);
    for (int b0 = begin; b0 < end; b0 += kDepth) {
        float4 xv[kDepth][2];
        uint2 wq[kDepth][kTiles];
        uint16_t ws[kDepth][kTiles];
        int sraw = 0;
        uint4 wraw[kWeightLoads];
        if constexpr (kStaged) {
#pragma unroll
            for (int i = 0; i < kWeightLoads; ++i)
                wraw[i] = *reinterpret_cast<const uint4*>(wcol[i] + min(b0 + (kType == 2 ? lane & 3 : ch >> 1), end - 1) * kQuantBytes);
            sraw = scol[min(b0 + (lane & 3), end - 1)];
        }
#pragma unroll
        for (int u = 0; u < kDepth; ++u) {
            const int b = min(b0 + u, end - 1);  // past the end: the last block again, not used
            xv[u][0] = *reinterpret_cast<const float4*>(xrow[0] + b * 32);
            xv[u][1] = *reinterpret_cast<const float4*>(xrow[1] + b * 32);
#pragma unroll
            for (int t = 0; t < (kStaged ? 0 : kTiles); ++t) {
                wq[u][t] = *reinterpret_cast<const uint2*>(weight + (first[t] + b) * kQuantBytes + quant_offset<kType>(g));
                ws[u][t] = scales[first[t] + b];
            }
        }
        if constexpr (kStaged) {
#pragma unroll
            for (int i = 0; i < kWeightLoads; ++i)
                *reinterpret_cast<uint4*>(own_w + 16 * (kType == 2 ? weight_slot(lane & 3, lane >> 2) : weight_slot(ch, 8 * i + r8))) = wraw[i];
        }
#pragma unroll
        for (int u = 0; u < kDepth; ++u) {
            if (b0 + u >= end) break;  // wavefront-uniform
            Bf16x8 part[3];
            float4 x0 = xv[u][0], x1 = xv[u][1];
            if constexpr (kStaged) {
                own_x[r8 * 8 + (ch ^ (r8 >> 1))] = x0;
                own_x[(r8 + 8) * 8 + (ch ^ ((r8 + 8) >> 1))] = x1;
                wave_order();
                x0 = own_x[c * 8 + ((2 * g) ^ (c >> 1))];
                x1 = own_x[c * 8 + ((2 * g + 1) ^ (c >> 1))];
                const int slot = weight_slot(kType == 2 ? u : u * 2 + (g >> 1), c);
                wq[u][0] = *reinterpret_cast<const uint2*>(own_w + 16 * slot + 8 * (g & 1));
                ws[u][0] = static_cast<uint16_t>(__builtin_amdgcn_ds_bpermute(4 * (4 * c + u), sraw));
                wave_order();
            }
            const float v[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) split_pair(v[2 * i], v[2 * i + 1], &part[0].u[i], &part[1].u[i], &part[2].u[i], &left_behind);
#pragma unroll
            for (int t = 0; t < kTiles; ++t) {
                const r_bf16x8 w = weights_bf16<kType>(wq[u][t], g);
                r_f32x4 dot = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int q = 2; q >= 0; --q) dot = __builtin_amdgcn_mfma_f32_16x16x32_bf16(part[q].v, w, dot, 0, 0, 0);
                const float d = half_bits_to_f32(ws[u][t]);
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[t][i] = __builtin_fmaf(d, dot[i], acc[t][i]);
            }
        }
    }
#pragma unroll
    for (int t = 0; t < kTiles; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) own[(t * 4 + i) * 64 + lane] = acc[t][i];
    // A second pass over the wavefront's blocks where a value left something behind, added to its own sums in LDS: no activation
    // of a model does, and nothing of this may take registers in the loop above: four tiles keep to the 64 that give a compute
    // unit two workgroups (as a branch in the loop 128; one workgroup: 4096 rows of K = 288 x 288 columns 11.0 -> 12.1 us).
    if (left_behind != 0) {
        int again = lane;
        asm volatile("" : "+v"(again));  // addresses are formed anew
        const int c2 = again & 15, g2 = again >> 4;
        const float* row = x + static_cast<size_t>(min(m0 + c2, rows - 1)) * in_dim + 8 * g2;
#pragma unroll 1
        for (int b = begin; b < end; ++b) {
            const float4 x0 = reinterpret_cast<const float4*>(row + b * 32)[0], x1 = reinterpret_cast<const float4*>(row + b * 32)[1];
            Bf16x8 rest[2];
            left_pair(x0.x, x0.y, &rest[0].u[0], &rest[1].u[0]);
            left_pair(x0.z, x0.w, &rest[0].u[1], &rest[1].u[1]);
            left_pair(x1.x, x1.y, &rest[0].u[2], &rest[1].u[2]);
            left_pair(x1.z, x1.w, &rest[0].u[3], &rest[1].u[3]);
#pragma unroll 1
            for (int t = 0; t < kTiles; ++t) {
                const size_t at = static_cast<size_t>(min(n0 + 16 * t + c2, out_dim - 1)) * kb + b;
                const r_bf16x8 w = weights_bf16<kType>(*reinterpret_cast<const uint2*>(weight + at * kQuantBytes + quant_offset<kType>(g2)), g2);
                r_f32x4 dot = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int q = 1; q >= 0; --q) dot = __builtin_amdgcn_mfma_f32_16x16x32_bf16(rest[q].v, w, dot, 0, 0, 0);
                const float d = half_bits_to_f32(scales[at]);
                float* sums = own + t * 256 + again;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (dot[i] != 0.0f) sums[64 * i] += d * dot[i] * 0x1p-100f;  // (d may be an infinity)
            }
        }
    }
    __syncthreads();
    for (int at = tid; at < kTiles * 256; at += blockDim.x) {
        float total = 0.0f;
        for (int w = 0; w < waves; ++w) total += route_sums[w * kWaveFloats + at];
        const int l = at & 63, i = (at >> 6) & 3, t = at >> 8;
        const int m = m0 + 4 * (l >> 4) + i, n = n0 + 16 * t + (l & 15);
        if (m < rows && n < out_dim) {
            const size_t to = static_cast<size_t>(m) * out_dim + n;
            dst[to] = finish_output(ep, n, to, total);
        }
    }
}

hipError_t launch_linear_f32_rows(hipStream_t stream, int tensor_type, float* dst, const float* x, const uint8_t* weight_prepared,
                                  int rows, int in_dim, int out_dim, const Epilogue& ep0, float* dst_b, const uint8_t* weight_b,
                                  const Epilogue& ep_b0) {
    if (rows <= 0 || out_dim <= 0) return hipSuccess;
    const int kb = in_dim / 32, matrices = weight_b != nullptr ? 2 : 1;
    int waves = 16;
    while (waves > 1 && waves > kb) waves /= 2;
    constexpr int kRowsPerLaunch = 16 * 65535;  // grid.y
    for (int r0 = 0; r0 < rows; r0 += kRowsPerLaunch) {
        const int nr = rows - r0 < kRowsPerLaunch ? rows - r0 : kRowsPerLaunch;
        const unsigned groups = static_cast<unsigned>((nr + 15) / 16);
        // One column tile, whose loads go through LDS, or four, which share a split of X but not those loads (the two add alike).  Four
        // where their workgroups fill the compute units' rounds: to 65 % up to K = 1024, 75 % up to 4096, 90 % beyond (Q8_0; Q4_0 not at
        // all), and not where K is a multiple of 256 past 1024, or of 512 (the rows that a load of X touches meet in the caches).  us, one /
        // four: Q8_0, pairs, 1917 x 1376 x 411 72 / 53, 671 x 672 x 292 14.3 / 10.4, Q4_0 1090 x 1120 x 305 28 / 21, 1764 x 352 x 384
        // 19.9 / 13.0, but 478 x 992 x 256 (47 % full) 10 / 13, 863 x 2816 x 256 40 / 42, 927 x 1536 x 223 25 / 31.  Over 1200 shapes (16 ..
        // 2048 rows, K 256 .. 8192, 64 .. 511 columns) 0.3 % above the better of the two on the mean.
        const long units = gemv_compute_units(), wide = static_cast<long>(groups) * ((out_dim + 63) / 64) * matrices;
        const long fill = 100 * wide / (units * ((wide + units - 1) / units));
        const bool apart = in_dim % 256 != 0 || (in_dim <= 1024 && in_dim % 512 != 0);
        const long least = in_dim <= 1024 && in_dim % 256 != 0 ? 65 : (in_dim <= 4096 ? 75 : (tensor_type == 8 ? 90 : 101));
        const int tiles = apart && fill >= least ? 4 : 1;
        const dim3 grid(static_cast<unsigned>((out_dim + 16 * tiles - 1) / (16 * tiles)), groups, matrices), block(64 * waves);
        const size_t lds = static_cast<size_t>(waves) * kWaveFloats * 4;  // at most 64 KiB
        Epilogue ep = ep0, ep_b = ep_b0;
        if (ep.residual) ep.residual += static_cast<size_t>(r0) * out_dim;
        if (ep_b.residual) ep_b.residual += static_cast<size_t>(r0) * out_dim;
        float* d = dst + static_cast<size_t>(r0) * out_dim;
        const float* in = x + static_cast<size_t>(r0) * in_dim;
        const RouteSecond second{dst_b ? dst_b + static_cast<size_t>(r0) * out_dim : nullptr, weight_b, ep_b};
        const int per_wave = (kb + waves - 1) / waves;
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, block, lds, stream, d, in, weight_prepared, nr, in_dim, out_dim, ep, second);
        };
        if (tensor_type == 2) {
            if (tiles == 4) launch(linear_f32_rows_kernel<2, 4, 4>);
            else if (per_wave == 1) launch(linear_f32_rows_kernel<2, 1, 1>);
            else if (per_wave == 2) launch(linear_f32_rows_kernel<2, 1, 2>);
            else launch(linear_f32_rows_kernel<2, 1, 4>);
        } else {
            if (tiles == 4) launch(linear_f32_rows_kernel<8, 4, 4>);
            else if (per_wave == 1) launch(linear_f32_rows_kernel<8, 1, 1>);
            else if (per_wave == 2) launch(linear_f32_rows_kernel<8, 1, 2>);
            else launch(linear_f32_rows_kernel<8, 1, 4>);
        }
        if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace afhip
