// A per-layer token input.  token_gate_kernel is the gate product with its epilogue,
//     g[t] = gelu_tanh(gate x_t) * side[token_t],
// spread over as many workgroups as there are 16 x 16 tiles of g; token_parts_kernel and token_proj_kernel share the gate out over the chip
// and make the projection too (bf16, few rows).  token_side_kernel is the end of a
// layer in one launch (bf16), for prompts, where there are rows enough to fill the chip with 16 each:
//     x <- x + y / rms(y) * post_w                       (the feed-forward's result)
//     g  = gelu_tanh(gate x) * side[token]
//     x <- x + p / rms(p) * side_norm,  p = proj g
//     out = x / rms(x) * next_w, or x                    (what the next layer reads)
// A workgroup takes up to 16 rows of the float32 stream.  A row belongs to one wave in the element-wise phases (its sums
// are wave reductions, no barriers); in between, the rows' bf16 copy in LDS is the first operand of the gate product,
// whose k range the eight waves share out, and p, rounded to bf16, takes that copy's place for the last phase.  Bound: the
// bytes of the rows and, in between, the address unit that serves the weights' fragments.  Packed weights lie in operand order,
// a wave's load is 1 KB that lies whole instead of 16 half-used lines, and what this saves in registers keeps the rows, which
// were read twice before (8192 rows, with the packing: W = 1024 46.9 -> 32.7 us, 2048 84.2 -> 67.8, 4096 215 -> 145).
#include <algorithm>

#include "decoder.h"
#include "mma.h"

namespace em {
namespace {

constexpr int kThreads = 512;
constexpr int kWaves = kThreads / kWave;
constexpr int kTileRows = 16;
constexpr int kGateTiles = 4;  // 16-column tiles of the gate product that a wave accumulates at a time

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

__device__ __forceinline__ void load4(const uint16_t* p, float (&v)[4]) {
    const u32x2_t w = *reinterpret_cast<const u32x2_t*>(p);
    v[0] = bf16_lo(w[0]);
    v[1] = bf16_hi(w[0]);
    v[2] = bf16_lo(w[1]);
    v[3] = bf16_hi(w[1]);
}
__device__ __forceinline__ void store4(uint16_t* p, const float (&v)[4]) {
    *reinterpret_cast<u32x2_t*>(p) = u32x2_t{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
}

// One workgroup per 16 x 16 tile of g; its waves share out the k range.
template <typename Elem>
__global__ __launch_bounds__(kThreads) void token_gate_kernel(const typename Elem::storage* __restrict__ x,
                                                              const typename Elem::storage* __restrict__ gate,
                                                              const int32_t* __restrict__ tokens,
                                                              const typename Elem::storage* __restrict__ table,
                                                              int64_t table_stride, int column0,
                                                              typename Elem::storage* __restrict__ g, int64_t T, int W, int dim) {
    typedef Mma<Elem> M;
    constexpr int kAhead = 4;
    __shared__ float part[kWaves][256];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, lq = lane >> 4;
    const int64_t t0 = static_cast<int64_t>(blockIdx.x) * 16;
    const int d0 = blockIdx.y * 16;
    const int steps = (W + 31) / 32;
    const bool vec = W % 8 == 0, row_ok = t0 + l16 < T, col_ok = d0 + l16 < dim;
    const typename Elem::storage* xr = x + (row_ok ? t0 + l16 : t0) * W;
    const typename Elem::storage* wr = gate + static_cast<int64_t>(col_ok ? d0 + l16 : d0) * W;  // (extra columns are not stored)
    f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int s = wave; s < steps; s += kWaves * kAhead) {
        typename M::frag fx[kAhead], fw[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u)
            if (s + u * kWaves < steps) {
                const int k = (s + u * kWaves) * 32 + lq * 8;
                fx[u] = load_frag<Elem>(xr + k, W - k, vec);
                fw[u] = load_frag<Elem>(wr + k, W - k, vec);
            }
#pragma unroll
        for (int u = 0; u < kAhead; ++u)
            if (s + u * kWaves < steps) acc = M::mac(fx[u], fw[u], acc);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) part[wave][(lq * 4 + r) * 16 + l16] = acc[r];
    __syncthreads();
    if (tid < 256) {
        const int r = tid >> 4, d = d0 + (tid & 15);
        if (t0 + r < T && d < dim) {
            float z = 0.0f;
#pragma unroll
            for (int w = 0; w < kWaves; ++w) z += part[w][tid];
            const float e = Elem::load(table[static_cast<int64_t>(tokens[t0 + r]) * table_stride + column0 + d]);
            g[(t0 + r) * dim + d] = Elem::store(gelu_tanh(z) * e);
        }
    }
}

// The same and the projection behind it, p = proj g, in two launches of which neither waits for one CU's share of the weights: the gate product's
// k is shared out over workgroups, which leave partial sums, and every workgroup of the projection adds up those of its tokens, a
// few KB, in front of the gelu.  (As token_gate_kernel takes it, 23 tokens of 4096 columns are eight workgroups that bring in 256 KB each,
// and more tokens are read once per 16 rows of the gate.)  ND: 16-row tiles of the gate.
template <int ND>
__global__ __launch_bounds__(256) void token_parts_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ gate, float* __restrict__ parts,
                                                          int64_t T, int W) {
    typedef Mma<BF16Elem> M;
    constexpr int kAhead = ND <= 4 ? 4 : 2, kWavesHere = 4, kCols = ND * 16;
    __shared__ __attribute__((aligned(16))) float sums[kWavesHere][16][kCols + 4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, lq = lane >> 4;
    const int64_t t0 = static_cast<int64_t>(blockIdx.x) * 16;
    const int steps = W / 32, first = static_cast<int>(static_cast<int64_t>(steps) * blockIdx.y / gridDim.y),
              end = static_cast<int>(static_cast<int64_t>(steps) * (blockIdx.y + 1) / gridDim.y);
    const uint16_t *xr = x + min(t0 + l16, T - 1) * W + lq * 8, *wr[ND];
#pragma unroll
    for (int n = 0; n < ND; ++n) wr[n] = gate + static_cast<int64_t>(n * 16 + l16) * W + lq * 8;
    f32x4_t acc[ND];
#pragma unroll
    for (int n = 0; n < ND; ++n) acc[n] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    for (int s = first + wave; s < end; s += kWavesHere * kAhead) {
        M::frag fx[kAhead], fw[kAhead][ND];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int k = min(s + u * kWavesHere, end - 1) * 32;
            fx[u] = M::load(xr + k);
#pragma unroll
            for (int n = 0; n < ND; ++n) fw[u][n] = M::load(wr[n] + k);
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            if (s + u * kWavesHere >= end) break;
#pragma unroll
            for (int n = 0; n < ND; ++n) acc[n] = M::mac(fw[u][n], fx[u], acc[n]);
        }
    }
    // element i of a fragment: token l16, gate row lq * 4 + i
#pragma unroll
    for (int n = 0; n < ND; ++n) *reinterpret_cast<f32x4_t*>(&sums[wave][l16][n * 16 + lq * 4]) = acc[n];
    __syncthreads();
    float* out = parts + (static_cast<int64_t>(blockIdx.y) * T + t0) * kCols;
    for (int i = tid; i < 16 * (kCols / 4); i += 256) {
        const int t = i / (kCols / 4), c = (i - t * (kCols / 4)) * 4;
        if (t0 + t >= T) break;
        f32x4_t v = *reinterpret_cast<const f32x4_t*>(&sums[0][t][c]);
#pragma unroll
        for (int w = 1; w < kWavesHere; ++w) v += *reinterpret_cast<const f32x4_t*>(&sums[w][t][c]);
        *reinterpret_cast<f32x4_t*>(out + t * kCols + c) = v;
    }
}

// MT: 16-token tiles of a workgroup; ND: 32-element steps of g; NT: 16-column tiles of a wave
template <int MT, int ND, int NT>
__global__ __launch_bounds__(256) void token_proj_kernel(const float* __restrict__ parts, int n_parts, const int32_t* __restrict__ tokens,
                                                         const uint16_t* __restrict__ table, int64_t table_stride, int column0,
                                                         const uint16_t* __restrict__ proj, uint16_t* __restrict__ out, int64_t T, int W) {
    typedef Mma<BF16Elem> M;
    constexpr int kCols = ND * 32, LPG = kCols + 8, kPieces = MT * 16 * (kCols / 4) / 256, kMost = 8;
    __shared__ __attribute__((aligned(16))) uint16_t Gs[MT * 16 * LPG];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, lq = lane >> 4;
    const int64_t t0 = static_cast<int64_t>(blockIdx.x) * (16 * MT);
    M::frag fw[NT][ND];
    auto fetch = [&](int n0) {
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int k = 0; k < ND; ++k) fw[n][k] = M::load(proj + static_cast<int64_t>(min(n0 + n * 16 + l16, W - 1)) * kCols + k * 32 + lq * 8);
    };
    const int first = (static_cast<int>(blockIdx.y) * 4 + wave) * (NT * 16), step = static_cast<int>(gridDim.y) * (NT * 64);
    fetch(first);
    static_assert(MT * 16 * (kCols / 4) % 256 == 0 || MT * 16 * (kCols / 4) == 128, "pieces of four to a thread");
    constexpr bool kHalf = kPieces == 0;                 // (16 tokens of 32 columns: every other wave)
#pragma unroll
    for (int i = 0; i < (kHalf ? 1 : kPieces); ++i) {
        const int e = tid + i * 256, t = e / (kCols / 4), c = (e - t * (kCols / 4)) * 4;
        if (kHalf && tid >= 128) break;
        const int64_t row = min(t0 + t, T - 1);
        const float* from = parts + row * kCols + c;
        u32x2_t side;
        __builtin_memcpy(&side, __builtin_assume_aligned(table + static_cast<int64_t>(tokens[row]) * table_stride + column0 + c, 8), 8);
        f32x4_t z = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int p0 = 0; p0 < n_parts; p0 += kMost) {
            f32x4_t v[kMost];
#pragma unroll
            for (int j = 0; j < kMost; ++j) v[j] = *reinterpret_cast<const f32x4_t*>(from + static_cast<int64_t>(min(p0 + j, n_parts - 1)) * T * kCols);
#pragma unroll
            for (int j = 0; j < kMost; ++j)
                if (p0 + j < n_parts) z += v[j];
        }
        const u32x2_t g = {pack_bf16(gelu_tanh(z[0]) * bf16_lo(side[0]), gelu_tanh(z[1]) * bf16_hi(side[0])),
                           pack_bf16(gelu_tanh(z[2]) * bf16_lo(side[1]), gelu_tanh(z[3]) * bf16_hi(side[1]))};
        *reinterpret_cast<u32x2_t*>(Gs + t * LPG + c) = g;
    }
    __syncthreads();
    M::frag fg[MT][ND];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int k = 0; k < ND; ++k) fg[m][k] = M::load(Gs + (m * 16 + l16) * LPG + k * 32 + lq * 8);
    for (int n0 = first; n0 < W; n0 += step) {
        f32x4_t acc[NT][MT];
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                acc[n][m] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int k = 0; k < ND; ++k) acc[n][m] = M::mac(fw[n][k], fg[m][k], acc[n][m]);
            }
        if (n0 + step < W) fetch(n0 + step);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int64_t t = t0 + m * 16 + l16;
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                const int c = n0 + n * 16 + lq * 4;
                if (t < T && c < W) *reinterpret_cast<u32x2_t*>(out + t * W + c) = u32x2_t{pack_bf16(acc[n][m][0], acc[n][m][1]), pack_bf16(acc[n][m][2], acc[n][m][3])};
            }
        }
    }
}

// The weights in operand order: 16 rows x 32 columns, each piece as an MFMA takes it, 16 bytes per thread.  Made in front of every
// call that reads them, so that there is no second copy to keep up with weights that are written later (0.25 MB each for
// 2048 x 64: 2.0 us beside the 66 of 8192 rows).
__global__ __launch_bounds__(256) void token_side_pack_kernel(const uint16_t* __restrict__ gate, const uint16_t* __restrict__ proj,
                                                              uint16_t* __restrict__ gate_out, uint16_t* __restrict__ proj_out, int W, int dim) {
    const int i = blockIdx.x * 256 + threadIdx.x, piece = i / 64, row = i % 16, c = i % 64 / 16 * 8;
    if (i >= W / 8 * dim) return;
    const int d0 = piece % (dim / 16) * 16, k = piece / (dim / 16) * 32;       // gate: steps of W outside
    const int w0 = piece / (dim / 32) * 16, e = piece % (dim / 32) * 32;       // proj: steps of dim inside
    const bf16x8_t g = Mma<BF16Elem>::load(gate + static_cast<int64_t>(d0 + row) * W + k + c);
    const bf16x8_t v = Mma<BF16Elem>::load(proj + static_cast<int64_t>(w0 + row) * dim + e + c);
    store_frag<BF16Elem>(gate_out + static_cast<int64_t>(i) * 8, g);
    store_frag<BF16Elem>(proj_out + static_cast<int64_t>(i) * 8, v);
}

// NV: four-element pieces of a row per lane (W <= 256 * NV).  FULL: W % 128 == 0 and dim % 32 == 0, no operand piece is
// ragged and several weight fragments are fetched together.
template <int NV, bool FULL, int RPW, bool PACKED>
__global__ __launch_bounds__(kThreads, NV <= 8 && (!PACKED || NV * RPW <= 8) ? 4 : 2) void token_side_kernel(TokenSideProblem p) {
    typedef Mma<BF16Elem> M;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_raw[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, lq = lane >> 4;
    const int W = p.W, LPX = (W + 31) / 32 * 32 + 8, dim = p.dim, DP = (dim + 31) / 32 * 32, LPG = DP + 8;
    uint16_t* Xs = reinterpret_cast<uint16_t*>(lds_raw);          // [16][LPX] rows in bf16; later p
    float* Part = reinterpret_cast<float*>(lds_raw);              // [8][16][64] partial gate products, in the same place
    uint16_t* Gs = reinterpret_cast<uint16_t*>(lds_raw + p.g_offset);  // [16][LPG]
    const int64_t row0 = static_cast<int64_t>(blockIdx.x) * p.rows_per_group;
    const int n = static_cast<int>(min(static_cast<int64_t>(p.rows_per_group), p.T - row0));
    const float inv_w = 1.0f / static_cast<float>(W);

    // ---- x + normed y: as bf16 into LDS, and (KEEP) as it is in registers ----
    constexpr bool KEEP = PACKED;
    constexpr int R = KEEP ? RPW : 1;
    float keep[KEEP ? R : 1][KEEP ? NV : 1][4], y_rstd[2] = {0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int r = wave + i * kWaves;
        if (i < RPW && r < n) {
            const uint16_t* yr = p.y + (row0 + r) * W;
            float y[NV][4], sum = 0.0f;
            f32x4_t x[NV];
#pragma unroll
            for (int j = 0; j < NV; ++j) {
                const int c = (lane + j * 64) * 4;
                if (c < W) {
                    load4(yr + c, y[j]);
                    x[j] = *reinterpret_cast<const f32x4_t*>(p.x + (row0 + r) * W + c);
                }
            }
#pragma unroll
            for (int j = 0; j < NV; ++j)
                if ((lane + j * 64) * 4 < W) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) sum = fmaf(y[j][e], y[j][e], sum);
                }
            y_rstd[i] = 1.0f / sqrtf(wave_sum(sum) * inv_w + p.eps);
#pragma unroll
            for (int j = 0; j < NV; ++j) {
                const int c = (lane + j * 64) * 4;
                if (c < W) {
                    const f32x4_t w4 = *reinterpret_cast<const f32x4_t*>(p.post_w + c);
                    float v[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        v[e] = x[j][e] + y[j][e] * y_rstd[i] * w4[e];
                        if (KEEP) keep[i % R][j % (KEEP ? NV : 1)][e] = v[e];
                    }
                    store4(Xs + r * LPX + c, v);
                }
            }
        } else if (r < kTileRows) {
            const float z[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            for (int c = lane * 4; c < W; c += 256) store4(Xs + r * LPX + c, z);
        }
    }
    for (int i = tid; i < kTileRows * (LPX - W); i += kThreads) {   // the columns up to a multiple of 32
        const int w = LPX - W, r = i / w;
        Xs[r * LPX + W + (i - r * w)] = 0;
    }
    for (int i = tid; i < kTileRows * (DP - dim); i += kThreads) {
        const int w = DP - dim, r = i / w;
        Gs[r * LPG + dim + (i - r * w)] = 0;
    }
    // ---- gate product, 64 columns at a time ----
    const int steps = (W + 31) / 32;
    for (int d0 = 0; d0 < dim; d0 += kGateTiles * 16) {
        __syncthreads();
        f32x4_t acc[kGateTiles];
#pragma unroll
        for (int t = 0; t < kGateTiles; ++t) acc[t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        if (FULL) {
            constexpr int kAhead = KEEP ? 2 : 4;
            for (int s = wave; s < steps; s += kWaves * kAhead) {
                typename M::frag fw[kAhead][kGateTiles];
#pragma unroll
                for (int u = 0; u < kAhead; ++u)
                    if (s + u * kWaves < steps) {
#pragma unroll
                        for (int t = 0; t < kGateTiles; ++t)
                            if (d0 + t * 16 < dim)
                                fw[u][t] = M::load(PACKED ? p.gate + (static_cast<int64_t>(s + u * kWaves) * (dim / 16) + d0 / 16 + t) * 512 + lane * 8
                                                          : p.gate + static_cast<int64_t>(d0 + t * 16 + l16) * W + (s + u * kWaves) * 32 + lq * 8);
                    }
#pragma unroll
                for (int u = 0; u < kAhead; ++u)
                    if (s + u * kWaves < steps) {
                        const typename M::frag fx = M::load(Xs + l16 * LPX + (s + u * kWaves) * 32 + lq * 8);
#pragma unroll
                        for (int t = 0; t < kGateTiles; ++t)
                            if (d0 + t * 16 < dim) acc[t] = M::mac(fx, fw[u][t], acc[t]);
                    }
            }
        } else for (int s = wave; s < steps; s += kWaves) {
            const int k = s * 32 + lq * 8;
            const typename M::frag fx = M::load(Xs + l16 * LPX + k);
#pragma unroll
            for (int t = 0; t < kGateTiles; ++t) {
                const int d = d0 + t * 16 + l16;
                // (W is a multiple of four: the last piece of a row may be half)
                if (d0 + t * 16 < dim)
                    acc[t] = M::mac(fx, d < dim ? load_frag<BF16Elem>(p.gate + static_cast<int64_t>(d) * W + k, W - k, W % 8 == 0) : M::zero(), acc[t]);
            }
        }
        // the partial products lie where the rows did: for more columns than one turn takes they lie behind everything
        float* part = p.part_offset == 0 ? Part : reinterpret_cast<float*>(lds_raw + p.part_offset);
        __syncthreads();
#pragma unroll
        for (int t = 0; t < kGateTiles; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) part[(wave * kTileRows + lq * 4 + r) * 64 + t * 16 + l16] = acc[t][r];
        __syncthreads();
        for (int i = tid; i < kTileRows * 64; i += kThreads) {
            const int r = i / 64, d = d0 + i % 64;
            if (d < dim) {
                float z = 0.0f;
#pragma unroll
                for (int w = 0; w < kWaves; ++w) z += part[w * kTileRows * 64 + i];
                float e = 0.0f;
                if (r < n) e = bf16_bits_to_f32(p.table[static_cast<int64_t>(p.tokens[row0 + r]) * p.table_stride + p.column0 + d]);
                Gs[r * LPG + d] = f32_to_bf16_bits(gelu_tanh(z) * e);
            }
        }
    }
    __syncthreads();
    // ---- p = proj g: every wave a share of the columns ----
    const int col_tiles = (W + 15) / 16;
    if (FULL) {
        constexpr int kAhead = KEEP ? 4 : 8;  // column tiles whose weights are fetched together
        for (int t = wave; t < col_tiles; t += kWaves * kAhead) {
            f32x4_t acc[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; ++u) acc[u] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
            for (int k = lq * 8; k < DP; k += 32) {
                typename M::frag fw[kAhead];
#pragma unroll
                for (int u = 0; u < kAhead; ++u)
                    if (t + u * kWaves < col_tiles)
                        fw[u] = M::load(PACKED ? p.proj + (static_cast<int64_t>(t + u * kWaves) * (dim / 32) + k / 32) * 512 + lane * 8
                                               : p.proj + static_cast<int64_t>((t + u * kWaves) * 16 + l16) * dim + k);
                const typename M::frag fg = M::load(Gs + l16 * LPG + k);
#pragma unroll
                for (int u = 0; u < kAhead; ++u)
                    if (t + u * kWaves < col_tiles) acc[u] = M::mac(fg, fw[u], acc[u]);
            }
#pragma unroll
            for (int u = 0; u < kAhead; ++u)
                if (t + u * kWaves < col_tiles) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) Xs[(lq * 4 + r) * LPX + (t + u * kWaves) * 16 + l16] = f32_to_bf16_bits(acc[u][r]);
                }
        }
    } else for (int t = wave; t < col_tiles; t += kWaves) {
        const int c = t * 16 + l16;
        f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int k = lq * 8; k < DP; k += 32) {
            const typename M::frag fg = M::load(Gs + l16 * LPG + k);
            acc = M::mac(fg, c < W ? load_frag<BF16Elem>(p.proj + static_cast<int64_t>(c) * dim + k, dim - k, dim % 8 == 0) : M::zero(), acc);
        }
        if (c < W) {
#pragma unroll
            for (int r = 0; r < 4; ++r) Xs[(lq * 4 + r) * LPX + c] = f32_to_bf16_bits(acc[r]);
        }
    }
    __syncthreads();
    // ---- the stream and the next layer's input ----
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
        const int r = wave + i * kWaves;
        if (r >= n) continue;
        const int64_t row = row0 + r;
        float sum = 0.0f;
        float x[NV][4];
        if (KEEP) {
#pragma unroll
            for (int j = 0; j < NV; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) x[j][e] = keep[i % R][j % (KEEP ? NV : 1)][e];
        } else {
            f32x4_t x4[NV];
            float y[NV][4];
#pragma unroll
            for (int j = 0; j < NV; ++j) {
                const int c = (lane + j * 64) * 4;
                if (c >= W) continue;
                load4(p.y + row * W + c, y[j]);
                x4[j] = *reinterpret_cast<const f32x4_t*>(p.x + row * W + c);
            }
#pragma unroll
            for (int j = 0; j < NV; ++j) {
                const int c = (lane + j * 64) * 4;
                if (c >= W) continue;
                const f32x4_t w4 = *reinterpret_cast<const f32x4_t*>(p.post_w + c);
#pragma unroll
                for (int e = 0; e < 4; ++e) x[j][e] = x4[j][e] + y[j][e] * y_rstd[i] * w4[e];
            }
        }
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int c = (lane + j * 64) * 4;
            if (c < W) {
                float v[4];
                load4(Xs + r * LPX + c, v);
#pragma unroll
                for (int e = 0; e < 4; ++e) sum = fmaf(v[e], v[e], sum);
            }
        }
        const float rstd = 1.0f / sqrtf(wave_sum(sum) * inv_w + p.eps);
        sum = 0.0f;
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int c = (lane + j * 64) * 4;
            if (c < W) {
                float v[4];
                load4(Xs + r * LPX + c, v);
                const f32x4_t s4 = *reinterpret_cast<const f32x4_t*>(p.side_norm + c);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    x[j][e] += v[e] * rstd * s4[e];
                    sum = fmaf(x[j][e], x[j][e], sum);
                }
            }
        }
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int c = (lane + j * 64) * 4;
            if (c < W) *reinterpret_cast<f32x4_t*>(p.x + row * W + c) = f32x4_t{x[j][0], x[j][1], x[j][2], x[j][3]};
        }
        const float x_rstd = p.next_w != nullptr ? 1.0f / sqrtf(wave_sum(sum) * inv_w + p.eps) : 1.0f;
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int c = (lane + j * 64) * 4;
            if (c < W) {
                float v[4];
                if (p.next_w != nullptr) {
                    const f32x4_t w4 = *reinterpret_cast<const f32x4_t*>(p.next_w + c);
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = x[j][e] * x_rstd * w4[e];
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = x[j][e];
                }
                store4(p.out + row * p.out_stride + c, v);
            }
        }
    }
}

constexpr int kPartBytes = kWaves * kTileRows * 64 * 4;

// LDS: the rows (or, when one turn takes all gate columns, the partial products in their place), the gate's result, and
// the partial products if they need room of their own.
size_t lds_bytes(int W, int dim, int* g_offset, int* part_offset) {
    const int rows = static_cast<int>(round_up(W, 32) + 8) * kTileRows * 2;
    const bool one_turn = dim <= kGateTiles * 16;
    const int first = one_turn && rows < kPartBytes ? kPartBytes : rows;
    *g_offset = first;
    const int g = static_cast<int>(round_up(dim, 32) + 8) * kTileRows * 2;
    *part_offset = one_turn ? 0 : first + g;
    return static_cast<size_t>(first) + g + (one_turn ? 0 : kPartBytes);
}

template <int NV, bool FULL, int RPW, bool PACKED>
int launch_rows(TokenSideProblem p, size_t lds, hipStream_t s) {
    p.rows_per_group = RPW * kWaves;
    const int rc = allow_lds(reinterpret_cast<const void*>(token_side_kernel<NV, FULL, RPW, PACKED>), lds);
    if (rc != 0) return rc;
    launch((token_side_kernel<NV, FULL, RPW, PACKED>), dim3(static_cast<unsigned>(ceil_div(p.T, p.rows_per_group))), dim3(kThreads), lds, s, p);
    return launch_status();
}

// One row per wave while two do not fill the chip; and with eight pieces a lane, whose two rows in registers take a CU to themselves, where
// the LDS lets a second workgroup in: phases of one then run while the other waits (us for 8192 rows, one / two: W = 1024 37 / 31,
// 2048 66 / 79, 4096 200 / 160).  With LDS for one workgroup only (W = 1536 from dim 96, 1280 from 256) half of a tile's rows would be
// empty for nothing: W = 1536, dim 96 98.8 / 69.1, 3072 rows 47.2 / 34.4 (40.2 before the weights were packed), 2048 x 256 191 / 126.
template <int NV, bool FULL>
int launch_side(const TokenSideProblem& p, size_t lds, hipStream_t s) {
    if constexpr (FULL)
        if (p.packed) return p.T <= 512 || (NV == 8 && 2 * lds <= kLdsPerCu) ? launch_rows<NV, FULL, 1, true>(p, lds, s) : launch_rows<NV, FULL, 2, true>(p, lds, s);
    return p.T <= 512 ? launch_rows<NV, FULL, 1, false>(p, lds, s) : launch_rows<NV, FULL, 2, false>(p, lds, s);
}

}  // namespace

int launch_token_gate(const void* x, const void* gate, const int32_t* tokens, const void* table, int64_t table_stride,
                      int column0, void* g, int64_t T, int W, int dim, int dtype, hipStream_t s) {
    const dim3 grid(static_cast<unsigned>(ceil_div(T, 16)), static_cast<unsigned>(ceil_div(dim, 16)));
    if (dtype == EM_DTYPE_BF16)
        launch((token_gate_kernel<BF16Elem>), grid, dim3(kThreads), 0, s, static_cast<const uint16_t*>(x),
               static_cast<const uint16_t*>(gate), tokens, static_cast<const uint16_t*>(table), table_stride, column0,
               static_cast<uint16_t*>(g), T, W, dim);
    else
        launch((token_gate_kernel<F32Elem>), grid, dim3(kThreads), 0, s, static_cast<const float*>(x),
               static_cast<const float*>(gate), tokens, static_cast<const float*>(table), table_stride, column0,
               static_cast<float*>(g), T, W, dim);
    return launch_status();
}

// How many ranges of W the gate product is shared out over: a workgroup for every CU (of 16 tokens, or the tiled product's of 64), 256
// columns at least, and as few sums to add up as still pay; 0: what this does not take, and numbers of tokens that leave the tiled product few
// workgroups (gates of 64, W = 2048, 700 tokens one by one 10.7, this 11.8; 1000 11.0 / 11.7).
constexpr int64_t kFewTokens = 64, kSomeTokens = 512;
int token_input_parts(int64_t T, int W, int dim) {
    if (T <= 0 || W <= 0 || W % 64 != 0 || (dim != 32 && dim != 64 && dim != 128) || (T > kFewTokens && !tile_gemm_supported(T, dim, W))) return 0;
    if (T > kSomeTokens && T < 1280 && W <= 2048) return 0;
    const int64_t groups = T > kFewTokens ? ceil_div(T, 64) * ceil_div(dim, 64) : ceil_div(T, 16), most = std::max(W / 256, 1);
    return static_cast<int>(std::min<int64_t>({most, std::max<int64_t>(1, 256 / groups), T > kSomeTokens ? 4 : T > kFewTokens ? 8 : 16}));
}

// Where this is faster than the gate and the projection one by one: from this width on, by the gate's rows and the tokens (us, one by one / this.
// Gates of 32: 1 x 256 6.0 / 5.2, 64 x 2048 9.1 / 5.8; 300 x 512 6.7 / 7.1, x 1024 8.0 / 7.3; 1280 x 512 7.0 / 7.6, x 1024 8.5 / 7.9.  Of 64: 1 x 1024
// 5.9 / 6.1, x 2048 6.8 / 6.1, x 4096 9.3 / 6.7, 23 x 512 5.9 / 6.3, x 1024 6.7 / 6.3, x 4096 12.2 / 8.4; 300 x 1024 7.8 / 8.3, x 2048 9.7 / 9.1, x 4096
// 13.9 / 11.2; 1280 x 1024 10.6 / 10.7, 4000 18.2 / 16.6, 2244 x 2048 20.9 / 19.0, x 4096 33.7 / 24.6.  Of 128: 1 x 8192 14.1 / 15.1, 23 x 3072 10.9 /
// 12.3, x 4096 12.6 / 12.4; 128 x 3072 11.6 / 11.3, x 4096 13.2 / 11.8, 300 x 4096 14.4 / 15.0, x 8192 23.1 / 21.3; 1000 x 3072 20.3 / 19.4; 1280 x 1024
// 12.8 / 14.7, x 2048 19.6 / 18.5, 4000 41.1 / 30.6).
bool token_input_pays(int64_t T, int W, int dim) {
    if (token_input_parts(T, W, dim) == 0) return false;
    constexpr int kNever = 1 << 30;
    int least;
    if (T <= kFewTokens) least = dim == 32 ? 256 : dim == 64 ? (T < 16 ? 2048 : 1024) : (T < 16 ? kNever : 4096);
    else if (T <= kSomeTokens) least = dim == 32 ? 1024 : dim == 64 ? 2048 : T <= 128 ? 4096 : 8192;
    else least = dim == 32 || (dim == 64 && T >= 4000) ? 1024 : 2048;
    return W >= least;
}

// The most ranges that the kernel of the gate product makes: none of them empty (its steps are of 32 columns, the tiled product's of 64).
int token_input_most_parts(int64_t T, int W) { return T > kFewTokens ? std::min(W / 64, kMostSplits) : std::min(W / 32, 65535); }

int launch_token_input(const TokenInputProblem& p, hipStream_t s) {
    if (p.T > kFewTokens) {
        TileGemm g{};
        g.x = p.x; g.x_stride = p.W; g.w = p.gate; g.w_stride = p.W; g.out = p.parts; g.f32 = true;
        g.splits = p.n_parts; g.T = static_cast<int>(p.T); g.N = p.dim; g.K = p.W;
        const int rc = launch_tile_gemm(g, s);
        if (rc != 0) return rc;
    }
#define EM_PARTS(ND) launch((token_parts_kernel<ND>), dim3(static_cast<unsigned>(ceil_div(p.T, 16)), static_cast<unsigned>(p.n_parts)), dim3(256), 0, s, p.x, p.gate, p.parts, p.T, p.W)
    // how many workgroups share a row's columns: two to a CU, as every one adds up its tokens' sums anew
    auto columns = [&](int mt, int nt) {
        const int64_t groups = ceil_div(p.T, 16 * mt), all = ceil_div(p.W, 64 * nt);
        return static_cast<unsigned>(std::min<int64_t>(all, std::max<int64_t>(1, ceil_div(512, groups))));
    };
#define EM_PROJ(MT, ND, NT)                                                                                                              \
    launch((token_proj_kernel<MT, ND, NT>), dim3(static_cast<unsigned>(ceil_div(p.T, 16 * MT)), columns(MT, NT)), dim3(256), 0, s, \
           p.parts, p.n_parts, p.tokens, p.table, p.table_stride, p.column0, p.proj, p.out, p.T, p.W)
#define EM_BOTH(ND)                                         \
    do {                                                    \
        if (p.T <= kFewTokens) {                            \
            EM_PARTS(2 * ND);                               \
            EM_PROJ(1, ND, 1);                              \
        } else if (p.T <= kSomeTokens) {                    \
            EM_PROJ(1, ND, 4);                              \
        } else {                                            \
            EM_PROJ(2, ND, 4);                              \
        }                                                   \
    } while (0)
    if (p.dim == 32) EM_BOTH(1);
    else if (p.dim == 64) EM_BOTH(2);
    else EM_BOTH(4);
#undef EM_BOTH
#undef EM_PROJ
#undef EM_PARTS
    return launch_status();
}

bool token_side_supported(int W, int dim) {
    int a, b;
    return W > 0 && W % 4 == 0 && W <= 4096 && dim > 0 && dim <= 1024 && lds_bytes(W, dim, &a, &b) <= kLdsPerCu;
}

// Packing is a launch of its own, 0.5 to 2 us behind whose rows the loads in operand order have to come out ahead (us, as they are / packed
// and packing): rows of up to 256 with few columns do not (128 x 64, 1024 rows 9.8 / 11.2; 256 x 96, 4096 13.3 / 14.4), 32 columns only
// with long or many rows (512, 4096 rows 13.6 / 14.3, 8192 17.9 / 17.1; 1024, 4096 25.1 / 22.2), and rows of 1152 to 1920 with 32 lose
// where twice as many workgroups, of one row per wave, take a round more (1536, 4000 rows 33 / 24, 6144 41.6 / 44.6, 9216 71.5 / 65.2).
bool token_side_pack_pays(int64_t T, int W, int dim) {
    if (dim >= 64) return W >= 384 || W * dim >= 65536 || (W * dim > 16384 && T > 4096);
    if (W <= 1024) return W >= (T > 4096 ? 384 : 1024);
    return W >= 2048 || T <= 4096 || T > 8192;
}

int launch_token_side_pack(const uint16_t* gate, const uint16_t* proj, uint16_t* gate_out, uint16_t* proj_out, int W, int dim, hipStream_t s) {
    launch(token_side_pack_kernel, dim3(static_cast<unsigned>(ceil_div(W / 8 * dim, 256))), dim3(256), 0, s, gate, proj, gate_out, proj_out, W, dim);
    return launch_status();
}

int launch_token_side(TokenSideProblem p, hipStream_t s) {
    const size_t lds = lds_bytes(p.W, p.dim, &p.g_offset, &p.part_offset);
    if (token_side_packable(p.W, p.dim)) {
        if (p.W <= 1024) return launch_side<4, true>(p, lds, s);
        if (p.W <= 2048) return launch_side<8, true>(p, lds, s);
        return launch_side<16, true>(p, lds, s);
    }
    if (p.W <= 1024) return launch_side<4, false>(p, lds, s);
    if (p.W <= 2048) return launch_side<8, false>(p, lds, s);
    return launch_side<16, false>(p, lds, s);
}

}  // namespace em
