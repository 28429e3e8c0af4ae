// Row kernels of a decoder whose residual stream is float32: embedding, post-norm residual update fused with the next
// layer's pre-norm, squared ReLU, gated SiLU, and the gated norm of a mixer's output.
#include <algorithm>

#include "decoder.h"

namespace em {
namespace {

constexpr int kRowMaxPerThread = 32;  // floats of a row that one thread keeps in registers
constexpr int64_t kFewRows = 256;     // up to so many rows a CU has one at most
constexpr int kPartPiece = 16;        // elements of a partial sum's row that a thread requests at once where it takes them one by one

// Sum over the workgroup, the same value and the same order in every thread.  `scratch`: one float per wave.
template <int THREADS>
__device__ __forceinline__ float block_sum(float v, float* scratch) {
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) v += __shfl_xor(v, off);
    __syncthreads();  // readers of an earlier sum are done
    if (lane_id() == 0) scratch[threadIdx.x / kWave] = v;
    __syncthreads();
    float total = 0.0f;
#pragma unroll
    for (int w = 0; w < THREADS / kWave; ++w) total += scratch[w];
    return total;
}

template <typename Elem, int VEC>
struct RowIo {
    static __device__ __forceinline__ void load(const typename Elem::storage* p, float (&v)[VEC]) {
        typename Elem::storage t[VEC];
        __builtin_memcpy(t, __builtin_assume_aligned(p, VEC * sizeof(t[0])), sizeof(t));
#pragma unroll
        for (int j = 0; j < VEC; ++j) v[j] = Elem::load(t[j]);
    }
    static __device__ __forceinline__ void store(typename Elem::storage* p, const float (&v)[VEC]) {
        typename Elem::storage t[VEC];
#pragma unroll
        for (int j = 0; j < VEC; ++j) t[j] = Elem::store(v[j]);
        __builtin_memcpy(__builtin_assume_aligned(p, VEC * sizeof(t[0])), t, sizeof(t));
    }
};

// x = table[token] * scale in float32; copied, rounded to the compute type, to up to two strided destinations.
template <typename Elem, int VEC>
__global__ __launch_bounds__(256) void embed_kernel(const int32_t* __restrict__ tokens,
                                                    const typename Elem::storage* __restrict__ table, float scale,
                                                    float* __restrict__ x, typename Elem::storage* __restrict__ copy,
                                                    int64_t copy_stride, int W) {
    const int64_t t = blockIdx.x;
    const typename Elem::storage* src = table + static_cast<int64_t>(tokens[t]) * W;
    for (int c = threadIdx.x * VEC; c < W; c += 256 * VEC) {
        float v[VEC];
        RowIo<Elem, VEC>::load(src + c, v);
#pragma unroll
        for (int j = 0; j < VEC; ++j) v[j] *= scale;
        RowIo<F32Elem, VEC>::store(x + t * W + c, v);
        if (copy != nullptr) RowIo<Elem, VEC>::store(copy + t * copy_stride + c, v);
    }
}

// One workgroup per row, N vectors of the row per thread.
// y may be given as float32 partial sums [y_parts, T, W].
//   UPDATE 0: x stays          UPDATE 1: x += y / rms(y) * post_w          UPDATE 2: x = y + post_w
//   then, when out != null: out = next_w ? x / rms(x) * next_w : x, rounded to the compute type
// PARTS: y_parts > 1, of which one is requested at a time, for the whole row (64 rows of 8192 in threes 8.4 -> 7.4 us), or in pieces
// where elements go one by one: a whole row's addresses spill, and short rows would ask 32 times for a few (float32, in eights, element
// by element / whole rows / pieces: 64 rows of 9001 15.1 / 21.3 / 13.8, 300 of 1022 8.7 / 9.7 / 8.6, 64 of 20001 51 / 36 / 27).
template <typename Elem, typename YElem, int UPDATE, int VEC, int THREADS, int N, bool PARTS>
__global__ __launch_bounds__(THREADS) void residual_norm_kernel(
    float* __restrict__ x, const typename YElem::storage* __restrict__ y, int y_parts, const float* __restrict__ post_w,
    const float* __restrict__ next_w, typename Elem::storage* __restrict__ out, int64_t out_stride, int W, float eps) {
    __shared__ float scratch[THREADS / kWave];
    const int64_t row = blockIdx.x;
    float* xr = x + row * W;
    float v[N][VEC];
    if (UPDATE != 0) {
        const typename YElem::storage* yr = y + row * W;
        float sum = 0.0f;
        auto square = [&](int i) {
#pragma unroll
            for (int j = 0; j < VEC; ++j) sum = fmaf(v[i][j], v[i][j], sum);
        };
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int c = (threadIdx.x + i * THREADS) * VEC;
            if (c < W) {
                RowIo<YElem, VEC>::load(yr + c, v[i]);
                if (UPDATE == 1 && !PARTS) square(i);
            }
        }
        if (PARTS) {
            constexpr int kPiece = VEC == 1 ? kPartPiece : N;
#pragma unroll
            for (int i0 = 0; i0 < N; i0 += kPiece) {
                if (i0 * THREADS * VEC >= W) break;
                for (int p = 1; p < y_parts; ++p) {
                    float more[kPiece][VEC];
#pragma unroll
                    for (int i = 0; i < kPiece; ++i) {
                        const int c = (threadIdx.x + (i0 + i) * THREADS) * VEC;
                        if (c < W) RowIo<YElem, VEC>::load(yr + static_cast<int64_t>(p) * gridDim.x * W + c, more[i]);
                    }
#pragma unroll
                    for (int i = 0; i < kPiece; ++i)
#pragma unroll
                        for (int j = 0; j < VEC; ++j) v[i0 + i][j] += more[i][j];
                }
            }
#pragma unroll
            for (int i = 0; i < N; ++i)
                if (UPDATE == 1 && (threadIdx.x + i * THREADS) * VEC < W) square(i);
        }
        float rstd = 0.0f;
        if (UPDATE == 1) rstd = 1.0f / sqrtf(block_sum<THREADS>(sum, scratch) / static_cast<float>(W) + eps);
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int c = (threadIdx.x + i * THREADS) * VEC;
            if (c < W) {
                float pw[VEC];
                if (UPDATE == 1) {
                    float xv[VEC];
                    RowIo<F32Elem, VEC>::load(post_w + c, pw);
                    RowIo<F32Elem, VEC>::load(xr + c, xv);
#pragma unroll
                    for (int j = 0; j < VEC; ++j) v[i][j] = xv[j] + v[i][j] * rstd * pw[j];
                } else if (post_w != nullptr) {
                    RowIo<F32Elem, VEC>::load(post_w + c, pw);
#pragma unroll
                    for (int j = 0; j < VEC; ++j) v[i][j] += pw[j];
                }
                RowIo<F32Elem, VEC>::store(xr + c, v[i]);
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int c = (threadIdx.x + i * THREADS) * VEC;
            if (c < W) RowIo<F32Elem, VEC>::load(xr + c, v[i]);
        }
    }
    if (out == nullptr) return;
    float rstd = 1.0f;
    if (next_w != nullptr) {
        float sum = 0.0f;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int c = (threadIdx.x + i * THREADS) * VEC;
            if (c < W) {
#pragma unroll
                for (int j = 0; j < VEC; ++j) sum = fmaf(v[i][j], v[i][j], sum);
            }
        }
        rstd = 1.0f / sqrtf(block_sum<THREADS>(sum, scratch) / static_cast<float>(W) + eps);
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int c = (threadIdx.x + i * THREADS) * VEC;
        if (c < W) {
            float o[VEC];
            if (next_w != nullptr) {
                float nw[VEC];
                RowIo<F32Elem, VEC>::load(next_w + c, nw);
#pragma unroll
                for (int j = 0; j < VEC; ++j) o[j] = v[i][j] * rstd * nw[j];
            } else {
#pragma unroll
                for (int j = 0; j < VEC; ++j) o[j] = v[i][j];
            }
            RowIo<Elem, VEC>::store(out + row * out_stride + c, o);
        }
    }
}

// The same for short rows that are few.  Bound: the way from the first load to the last store.  Everything that a row needs is
// requested before the first sum over it: loads behind the barriers, and partial sums one by one, cost a way to memory each.
template <typename Elem, typename YElem, int UPDATE, int VEC, int THREADS, int N>
__global__ __launch_bounds__(THREADS) void residual_norm_early_kernel(
    float* __restrict__ x, const typename YElem::storage* __restrict__ y, int y_parts, const float* __restrict__ post_w,
    const float* __restrict__ next_w, typename Elem::storage* __restrict__ out, int64_t out_stride, int W, float eps) {
    __shared__ float scratch[THREADS / kWave];
    constexpr int kParts = 4;          // partial sums requested at once
    const int64_t row = blockIdx.x;
    float* xr = x + row * W;
    float v[N][VEC], xv[N][VEC], pw[N][VEC], nw[N][VEC], sum = 0.0f;
    const bool add_w = UPDATE == 1 || (UPDATE == 2 && post_w != nullptr), norm = out != nullptr && next_w != nullptr;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int c = (threadIdx.x + i * THREADS) * VEC;
        if (c >= W) continue;
        if (UPDATE != 0) RowIo<YElem, VEC>::load(y + row * W + c, v[i]);
        if (UPDATE != 2) RowIo<F32Elem, VEC>::load(xr + c, xv[i]);
        if (add_w) RowIo<F32Elem, VEC>::load(post_w + c, pw[i]);
        if (norm) RowIo<F32Elem, VEC>::load(next_w + c, nw[i]);
    }
    if (UPDATE != 0 && y_parts > 1) {
        for (int p0 = 1; p0 < y_parts; p0 += kParts) {
            float more[kParts][N][VEC];
#pragma unroll
            for (int p = 0; p < kParts; ++p)
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    const int c = (threadIdx.x + i * THREADS) * VEC;
                    if (c < W) RowIo<YElem, VEC>::load(y + (static_cast<int64_t>(min(p0 + p, y_parts - 1)) * gridDim.x + row) * W + c, more[p][i]);
                }
#pragma unroll
            for (int p = 0; p < kParts; ++p)
#pragma unroll
                for (int i = 0; i < N; ++i)
#pragma unroll
                    for (int j = 0; j < VEC; ++j) v[i][j] += p0 + p < y_parts ? more[p][i][j] : 0.0f;
        }
    }
    if (UPDATE == 1) {
#pragma unroll
        for (int i = 0; i < N; ++i)
            if ((threadIdx.x + i * THREADS) * VEC < W) {
#pragma unroll
                for (int j = 0; j < VEC; ++j) sum = fmaf(v[i][j], v[i][j], sum);
            }
    }
    float rstd = 0.0f;
    if (UPDATE == 1) rstd = 1.0f / sqrtf(block_sum<THREADS>(sum, scratch) / static_cast<float>(W) + eps);
    sum = 0.0f;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int c = (threadIdx.x + i * THREADS) * VEC;
        if (c >= W) continue;
#pragma unroll
        for (int j = 0; j < VEC; ++j) {
            if (UPDATE == 0) v[i][j] = xv[i][j];
            if (UPDATE == 1) v[i][j] = xv[i][j] + v[i][j] * rstd * pw[i][j];
            if (UPDATE == 2 && add_w) v[i][j] += pw[i][j];
            sum = fmaf(v[i][j], v[i][j], sum);
        }
        if (UPDATE != 0) RowIo<F32Elem, VEC>::store(xr + c, v[i]);
    }
    if (out == nullptr) return;
    rstd = 1.0f;
    if (norm) rstd = 1.0f / sqrtf(block_sum<THREADS>(sum, scratch) / static_cast<float>(W) + eps);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int c = (threadIdx.x + i * THREADS) * VEC;
        if (c >= W) continue;
        if (norm) {
#pragma unroll
            for (int j = 0; j < VEC; ++j) v[i][j] = v[i][j] * rstd * nw[i][j];
        }
        RowIo<Elem, VEC>::store(out + row * out_stride + c, v[i]);
    }
}

// u = relu(u)^2 in place
template <typename Elem, int VEC>
__global__ __launch_bounds__(256) void relu_squared_kernel(typename Elem::storage* __restrict__ u, int64_t n) {
    const int64_t i = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * VEC;
    if (i >= n) return;
    float v[VEC];
    RowIo<Elem, VEC>::load(u + i, v);
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
        const float r = fmaxf(v[j], 0.0f);
        v[j] = r * r;
    }
    RowIo<Elem, VEC>::store(u + i, v);
}

// out [T, ff] = silu(u[:, :ff]) * u[:, ff:]
template <typename Elem, int VEC>
__global__ __launch_bounds__(256) void silu_gate_kernel(const typename Elem::storage* __restrict__ u, typename Elem::storage* __restrict__ out,
                                                        int64_t n, int ff) {
    const int64_t i = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * VEC;
    if (i >= n) return;
    const int64_t row = i / ff, c = i - row * ff;
    float g[VEC], v[VEC];
    RowIo<Elem, VEC>::load(u + row * 2 * ff + c, g);
    RowIo<Elem, VEC>::load(u + row * 2 * ff + ff + c, v);
#pragma unroll
    for (int j = 0; j < VEC; ++j) v[j] *= silu(g[j]);
    RowIo<Elem, VEC>::store(out + i, v);
}

// y = y silu(z), normed in equal parts of `size` elements, times w, in place: one workgroup per (row, part).  EARLY: everything is
// requested before the sum; else the product is taken as it comes and the weights wait.  Rows of more than 4096 elements would not keep
// both operands in registers (float32, 300 rows of 9001: 35.8 us that way, spilled, 13.2 now; bf16, 3505 of 8192: 36.2, 31.2); rows
// of 1025 to 4096 elements of 16 bits that fill the chip are better off with more rows in flight (early / in turn: 3000 of 4096 17.1 /
// 16.2, 8192 of 2048 21.7 / 20.8), in 32 bits and shorter ones not (3000 of 3000 17.8 / 18.4, 8192 of 1000 bf16 13.3 / 13.5).
template <typename Elem, int VEC, int THREADS, int N, bool EARLY>
__global__ __launch_bounds__(THREADS) void gated_norm_kernel(typename Elem::storage* __restrict__ y, const typename Elem::storage* __restrict__ z,
                                                             int64_t z_stride, const float* __restrict__ w, int size, float eps) {
    __shared__ float scratch[THREADS / kWave];
    const int64_t row = blockIdx.x;
    const int c0 = blockIdx.y * size;
    typename Elem::storage* yr = y + (row * gridDim.y + blockIdx.y) * size;
    const typename Elem::storage* zr = z + row * z_stride + c0;
    constexpr int M = EARLY ? N : 1;
    float v[N][VEC], g[M][VEC], wv[M][VEC], sum = 0.0f;
    auto times_silu = [&](int i) {
#pragma unroll
        for (int j = 0; j < VEC; ++j) {
            v[i][j] *= silu(g[i % M][j]);
            sum = fmaf(v[i][j], v[i][j], sum);
        }
    };
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int c = (threadIdx.x + i * THREADS) * VEC;
        if (c >= size) continue;
        RowIo<Elem, VEC>::load(yr + c, v[i]);
        RowIo<Elem, VEC>::load(zr + c, g[i % M]);
        if (EARLY) RowIo<F32Elem, VEC>::load(w + c0 + c, wv[i % M]);
        else times_silu(i);
    }
    if (EARLY) {
#pragma unroll
        for (int i = 0; i < N; ++i)
            if ((threadIdx.x + i * THREADS) * VEC < size) times_silu(i);
    }
    const float rstd = 1.0f / sqrtf(block_sum<THREADS>(sum, scratch) / static_cast<float>(size) + eps);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int c = (threadIdx.x + i * THREADS) * VEC;
        if (c < size) {
            if (!EARLY) RowIo<F32Elem, VEC>::load(w + c0 + c, wv[i % M]);
#pragma unroll
            for (int j = 0; j < VEC; ++j) v[i][j] *= rstd * wv[i % M][j];
            RowIo<Elem, VEC>::store(yr + c, v[i]);
        }
    }
}

// Place of the largest value of a row, the first one where several are equal; a NaN is larger than every number.  One
// workgroup per row, up to AHEAD vectors to a thread requested at once: 32000 columns take a way to memory and a pass over 32
// values a thread: the maximum of a piece first, two values to an instruction, its first place only where it brings anything, and over the
// wave without LDS (us: one row 7.8 -> 5.1, 64 rows 8.7 -> 5.9, 128256 columns 22.7 -> 14.1; the library 10.7 and 11.3 for 32000).
constexpr int kArgmaxThreads = 1024;
template <int ROTATE>
__device__ __forceinline__ int rotated(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x120 + ROTATE, 0xf, 0xf, true); }
__device__ __forceinline__ float wave_max(float v) {
    v = fmaxf(v, __int_as_float(rotated<8>(__float_as_int(v))));
    v = fmaxf(v, __int_as_float(rotated<4>(__float_as_int(v))));
    v = fmaxf(v, __int_as_float(rotated<2>(__float_as_int(v))));
    return column_max(fmaxf(v, __int_as_float(rotated<1>(__float_as_int(v)))));
}
__device__ __forceinline__ int wave_min(int v) {
    v = min(v, rotated<8>(v));
    v = min(v, rotated<4>(v));
    v = min(v, rotated<2>(v));
    v = min(v, rotated<1>(v));
    const auto a = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    v = min(static_cast<int>(a[0]), static_cast<int>(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return min(static_cast<int>(b[0]), static_cast<int>(b[1]));
}
// the place of the largest of the wave's values, in all lanes; `value` becomes it
__device__ __forceinline__ int wave_argmax(float& value, int place) {
    const bool nan = value != value;
    if (__ballot(nan) != 0) {
        place = wave_min(nan ? place : INT_MAX);
        value = NAN;
        return place;
    }
    const float most = wave_max(value);
    place = wave_min(value == most ? place : INT_MAX);
    value = most;
    return place;
}
template <int VEC, int AHEAD>
__global__ __launch_bounds__(kArgmaxThreads) void argmax_kernel(const float* __restrict__ x, int V, int32_t* __restrict__ out) {
    __shared__ float best_v[kArgmaxThreads / kWave];
    __shared__ int best_i[kArgmaxThreads / kWave];
    const int step = static_cast<int>(blockDim.x) * VEC, waves = static_cast<int>(blockDim.x) / kWave;
    const float* row = x + static_cast<int64_t>(blockIdx.x) * V;
    float value = -INFINITY;
    int place = V;
    for (int c0 = threadIdx.x * VEC; c0 < V; c0 += AHEAD * step) {
        float v[AHEAD][VEC], most = -INFINITY;
        bool nan = false;
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) RowIo<F32Elem, VEC>::load(row + min(c0 + i * step, V - VEC), v[i]);
#pragma unroll
        for (int i = 0; i < AHEAD; ++i)
#pragma unroll
            for (int j = 0; j < VEC; ++j) {
                if (c0 + i * step >= V) v[i][j] = -INFINITY;      // (V is a multiple of VEC)
                most = fmaxf(most, v[i][j]);
                nan = nan || v[i][j] != v[i][j];
            }
        // the first place of it, where this piece of the row brings anything: a NaN, something larger, or the first values at all
        const bool seek = value == value && (nan || most > value || place == V);
        if (!seek) continue;
#pragma unroll
        for (int i = AHEAD - 1; i >= 0; --i)
#pragma unroll
            for (int j = VEC - 1; j >= 0; --j)
                if (nan ? v[i][j] != v[i][j] : v[i][j] == most) place = c0 + i * step + j;
        value = nan ? NAN : most;
    }
    place = wave_argmax(value, place);
    if (lane_id() == 0) {
        best_v[threadIdx.x / kWave] = value;
        best_i[threadIdx.x / kWave] = place;
    }
    __syncthreads();
    if (threadIdx.x >= kWave) return;
    value = best_v[threadIdx.x % waves];
    place = wave_argmax(value, best_i[threadIdx.x % waves]);
    if (threadIdx.x == 0) out[blockIdx.x] = place;
}

template <typename Elem, int VEC>
int launch_gated(void* y, const void* z, int64_t z_stride, const float* w, int64_t T, int parts, int size, float eps, hipStream_t s) {
    typedef typename Elem::storage S;
    const dim3 grid(static_cast<unsigned>(T), static_cast<unsigned>(parts));
#define EM_GATED(THREADS, N, EARLY) \
    launch((gated_norm_kernel<Elem, VEC, THREADS, N, EARLY>), grid, dim3(THREADS), 0, s, static_cast<S*>(y), static_cast<const S*>(z), z_stride, w, size, eps)
    const bool few = T * parts <= kFewRows;
    if (size <= 512) EM_GATED(64, 8 / VEC, true);
    else if (VEC == 4 && few && size > 1024 && size <= 4096) EM_GATED(1024, 4 / VEC, true);
    else if (VEC == 4 && !few && size > 1024 && size <= 4096 && sizeof(S) == 2) EM_GATED(256, 16 / VEC, false);
    else if (VEC == 4 && size <= 4096) EM_GATED(256, 16 / VEC, true);
    else if (size <= 256 * kRowMaxPerThread) EM_GATED(256, kRowMaxPerThread / VEC, false);
    else EM_GATED(1024, kRowMaxPerThread / VEC, false);
#undef EM_GATED
    return launch_status();
}

// Few rows leave CUs without one, and a row is over sooner with one vector per thread and everything requested at once (us, 64 rows
// of 2048 in fours 4.6 -> 3.9, one of 4096 in twos 5.2 -> 4.5).  Where rows fill the chip, their bytes are the bound and rows in flight
// count for more than a row's way: the normed update, which keeps four rows of floats that way, waits with its weights and the
// stream (rows of 4096, at once / in turn: 300 6.0 / 5.8, 1024 11.0 / 8.6, 3505 32.0 / 26.9, 16384 206 / 148; 8192 of 2048 31.8 / 30.4);
// y + w, which keeps three, does so for long rows in large numbers only (rows of 4096: 768 6.6 / 6.9, 1500 10.9 / 9.7, 16384 133 / 113;
// 8192 of 2048 21.4 / 21.9), and not with partial sums, which it requests in fours (300 of 4096 in twos 6.0 / 5.1), x alone never (8192 of
// 4096 29.6 / 30.8).
template <typename Elem, typename YElem, int UPDATE, int VEC>
int launch_residual(float* x, const void* y, int y_parts, const float* post_w, const float* next_w, void* out, int64_t out_stride,
                    int64_t T, int W, float eps, hipStream_t s) {
#define EM_ROWS(THREADS, ...)                                                                                                             \
    do {                                                                                                                                  \
        launch((__VA_ARGS__), dim3(static_cast<unsigned>(T)), dim3(THREADS), 0, s, x, static_cast<const typename YElem::storage*>(y), y_parts, \
               post_w, next_w, static_cast<typename Elem::storage*>(out), out_stride, W, eps);                                            \
        return launch_status();                                                                                                           \
    } while (0)
#define EM_EARLY(THREADS, N) EM_ROWS(THREADS, residual_norm_early_kernel<Elem, YElem, UPDATE, VEC, THREADS, N>)
#define EM_LATE(THREADS, N)                                                                                       \
    do {                                                                                                          \
        if constexpr (UPDATE != 0 && sizeof(typename YElem::storage) == 4)                                        \
            if (y_parts > 1) EM_ROWS(THREADS, residual_norm_kernel<Elem, YElem, UPDATE, VEC, THREADS, N, true>);  \
        EM_ROWS(THREADS, residual_norm_kernel<Elem, YElem, UPDATE, VEC, THREADS, N, false>);                      \
    } while (0)
    if constexpr (VEC == 4) {
        if (T <= kFewRows && W > 1024 && W <= 2048) EM_EARLY(512, 1);
        if (T <= kFewRows && W > 1024 && W <= 4096) EM_EARLY(1024, 1);
        const bool early = T <= kFewRows || UPDATE == 0 || (UPDATE == 2 && y_parts == 1 && (W <= 2048 || T <= 4 * kFewRows));
        if (early && W <= 2048) EM_EARLY(256, 2);
        if (early && W <= 4096) EM_EARLY(256, 4);
        if (W <= 2048) EM_LATE(256, 2);
        if (W <= 4096) EM_LATE(256, 4);
    }
    if (W <= 256 * kRowMaxPerThread) EM_LATE(256, kRowMaxPerThread / VEC);
    EM_LATE(1024, kRowMaxPerThread / VEC);
#undef EM_LATE
#undef EM_EARLY
#undef EM_ROWS
}

template <typename Elem, typename YElem, int VEC>
int dispatch_residual(int update, float* x, const void* y, int y_parts, const float* post_w, const float* next_w, void* out,
                      int64_t out_stride, int64_t T, int W, float eps, hipStream_t s) {
    if (update == 0) return launch_residual<Elem, YElem, 0, VEC>(x, y, y_parts, post_w, next_w, out, out_stride, T, W, eps, s);
    if (update == 1) return launch_residual<Elem, YElem, 1, VEC>(x, y, y_parts, post_w, next_w, out, out_stride, T, W, eps, s);
    return launch_residual<Elem, YElem, 2, VEC>(x, y, y_parts, post_w, next_w, out, out_stride, T, W, eps, s);
}

}  // namespace

bool row_width_ok(int W) { return W > 0 && W <= 1024 * kRowMaxPerThread; }

int launch_embed(const int32_t* tokens, const void* table, float scale, float* x, void* copy, int64_t copy_stride,
                 int64_t T, int W, int dtype, hipStream_t s) {
    const dim3 grid(static_cast<unsigned>(T));
    const bool vec = W % 4 == 0 && copy_stride % 4 == 0;
    if (dtype == EM_DTYPE_BF16) {
        const uint16_t* e = static_cast<const uint16_t*>(table);
        uint16_t* c = static_cast<uint16_t*>(copy);
        if (vec) launch((embed_kernel<BF16Elem, 4>), grid, dim3(256), 0, s, tokens, e, scale, x, c, copy_stride, W);
        else launch((embed_kernel<BF16Elem, 1>), grid, dim3(256), 0, s, tokens, e, scale, x, c, copy_stride, W);
    } else {
        const float* e = static_cast<const float*>(table);
        float* c = static_cast<float*>(copy);
        if (vec) launch((embed_kernel<F32Elem, 4>), grid, dim3(256), 0, s, tokens, e, scale, x, c, copy_stride, W);
        else launch((embed_kernel<F32Elem, 1>), grid, dim3(256), 0, s, tokens, e, scale, x, c, copy_stride, W);
    }
    return launch_status();
}

int launch_residual_norm(int update, float* x, const void* y, int y_dtype, int y_parts, const float* post_w, const float* next_w,
                         void* out, int64_t out_stride, int64_t T, int W, float eps, int dtype, hipStream_t s) {
    const bool vec = W % 4 == 0 && out_stride % 4 == 0;
#define EM_RESIDUAL(E, Y)                                                                                        \
    return vec ? dispatch_residual<E, Y, 4>(update, x, y, y_parts, post_w, next_w, out, out_stride, T, W, eps, s)         \
               : dispatch_residual<E, Y, 1>(update, x, y, y_parts, post_w, next_w, out, out_stride, T, W, eps, s)
    if (dtype == EM_DTYPE_F32) { EM_RESIDUAL(F32Elem, F32Elem); }
    if (y_dtype == EM_DTYPE_F32) { EM_RESIDUAL(BF16Elem, F32Elem); }
    EM_RESIDUAL(BF16Elem, BF16Elem);
#undef EM_RESIDUAL
}

int launch_relu_squared(void* u, int64_t n, int dtype, hipStream_t s) {
    const int vec = n % 8 == 0 ? 8 : 1;
    const dim3 grid(static_cast<unsigned>(ceil_div(ceil_div(n, vec), 256)));
    if (dtype == EM_DTYPE_BF16) {
        if (vec == 8) launch((relu_squared_kernel<BF16Elem, 8>), grid, dim3(256), 0, s, static_cast<uint16_t*>(u), n);
        else launch((relu_squared_kernel<BF16Elem, 1>), grid, dim3(256), 0, s, static_cast<uint16_t*>(u), n);
    } else {
        if (vec == 8) launch((relu_squared_kernel<F32Elem, 8>), grid, dim3(256), 0, s, static_cast<float*>(u), n);
        else launch((relu_squared_kernel<F32Elem, 1>), grid, dim3(256), 0, s, static_cast<float*>(u), n);
    }
    return launch_status();
}

int launch_silu_gate(const void* u, void* out, int64_t T, int ff, int dtype, hipStream_t s) {
    const int64_t n = T * ff;
    const int vec = ff % 8 == 0 ? 8 : 1;
    const dim3 grid(static_cast<unsigned>(ceil_div(ceil_div(n, vec), 256)));
    if (dtype == EM_DTYPE_BF16) {
        if (vec == 8) launch((silu_gate_kernel<BF16Elem, 8>), grid, dim3(256), 0, s, static_cast<const uint16_t*>(u), static_cast<uint16_t*>(out), n, ff);
        else launch((silu_gate_kernel<BF16Elem, 1>), grid, dim3(256), 0, s, static_cast<const uint16_t*>(u), static_cast<uint16_t*>(out), n, ff);
    } else {
        if (vec == 8) launch((silu_gate_kernel<F32Elem, 8>), grid, dim3(256), 0, s, static_cast<const float*>(u), static_cast<float*>(out), n, ff);
        else launch((silu_gate_kernel<F32Elem, 1>), grid, dim3(256), 0, s, static_cast<const float*>(u), static_cast<float*>(out), n, ff);
    }
    return launch_status();
}

// No more vectors to a thread than a row has for it: a pass over places that are not there takes as long as one over others (us, eight to a thread
// / as here: one row of 1000 3.8 / 2.3, 5000 5.3 / 3.0, 16384 5.3 / 3.8; 1000 rows of 1000 11.7 / 3.2, 4096 18.2 / 5.4, 8192 18.2 / 6.6); where rows
// fill the chip the next workgroup hides a row's way (256 of 32000 7.1 / 6.9, of 128256 24.8 / 22.0, 1000 of 32000 27.3 / 21.7).
int launch_argmax(const float* x, int64_t T, int V, int32_t* out, hipStream_t s) {
    const bool vec = V % 4 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0;
    const dim3 grid(static_cast<unsigned>(T)), block(vec ? static_cast<unsigned>(std::min<int64_t>(kArgmaxThreads, round_up(V / 4, kWave))) : kArgmaxThreads);
    if (!vec) launch((argmax_kernel<1, 8>), grid, block, 0, s, x, V, out);
    else if (V <= 4 * kArgmaxThreads) launch((argmax_kernel<4, 1>), grid, block, 0, s, x, V, out);
    else if (V <= 8 * kArgmaxThreads) launch((argmax_kernel<4, 2>), grid, block, 0, s, x, V, out);
    else if (V <= 16 * kArgmaxThreads || T >= 256) launch((argmax_kernel<4, 4>), grid, block, 0, s, x, V, out);
    else launch((argmax_kernel<4, 8>), grid, block, 0, s, x, V, out);
    return launch_status();
}

int launch_gated_norm(void* y, const void* z, int64_t z_stride, const float* w, int64_t T, int parts, int size, float eps, int dtype,
                      hipStream_t s) {
    const bool vec = size % 4 == 0 && z_stride % 4 == 0;
    if (dtype == EM_DTYPE_BF16)
        return vec ? launch_gated<BF16Elem, 4>(y, z, z_stride, w, T, parts, size, eps, s)
                   : launch_gated<BF16Elem, 1>(y, z, z_stride, w, T, parts, size, eps, s);
    return vec ? launch_gated<F32Elem, 4>(y, z, z_stride, w, T, parts, size, eps, s)
               : launch_gated<F32Elem, 1>(y, z, z_stride, w, T, parts, size, eps, s);
}

}  // namespace em
