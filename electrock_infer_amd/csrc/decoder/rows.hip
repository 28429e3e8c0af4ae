// Row kernels of a decoder whose residual stream is float32: embedding, post-norm residual update fused with the next
// layer's pre-norm, squared ReLU, gated SiLU, and the gated norm of a mixer's output.
#include "decoder.h"

namespace em {
namespace {

constexpr int kRowMaxPerThread = 32;  // floats of a row that one thread keeps in registers
constexpr int64_t kFewRows = 256;     // up to so many rows a CU has one at most

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
// Bound: bytes for prompts, the way from the first load to the last store for a few rows.  Everything that a row needs is
// requested before the first sum over it: loads behind the barriers, and partial sums one by one, cost a way to memory
// each (four partial sums of 64 rows of 2048: 5.5 us that way, 4.9 now; two of 24 rows of 4096: 6.8, 4.9; 8192 rows of 2048:
// 35.3, 34.5).
template <typename Elem, typename YElem, int UPDATE, int VEC, int THREADS, int N>
__global__ __launch_bounds__(THREADS) void residual_norm_kernel(
    float* __restrict__ x, const typename YElem::storage* __restrict__ y, int y_parts, const float* __restrict__ post_w,
    const float* __restrict__ next_w, typename Elem::storage* __restrict__ out, int64_t out_stride, int W, float eps) {
    __shared__ float scratch[THREADS / kWave];
    constexpr bool kEarly = N * VEC <= 16;          // (longer rows do not fit in the registers twice)
    constexpr int kParts = kEarly ? 4 : 1, M = kEarly ? N : 1;      // partial sums requested at once; rows of early loads
    const int64_t row = blockIdx.x;
    float* xr = x + row * W;
    float v[N][VEC], xv[M][VEC], pw[M][VEC], nw[M][VEC], sum = 0.0f;
    const bool add_w = UPDATE == 1 || (UPDATE == 2 && post_w != nullptr), norm = out != nullptr && next_w != nullptr;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int c = (threadIdx.x + i * THREADS) * VEC;
        if (c >= W) continue;
        if (UPDATE != 0) RowIo<YElem, VEC>::load(y + row * W + c, v[i]);
        if (!kEarly) continue;
        if (UPDATE != 2) RowIo<F32Elem, VEC>::load(xr + c, xv[i % M]);
        if (add_w) RowIo<F32Elem, VEC>::load(post_w + c, pw[i % M]);
        if (norm) RowIo<F32Elem, VEC>::load(next_w + c, nw[i % M]);
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
        if (!kEarly && UPDATE != 2) RowIo<F32Elem, VEC>::load(xr + c, xv[i % M]);
        if (!kEarly && add_w) RowIo<F32Elem, VEC>::load(post_w + c, pw[i % M]);
#pragma unroll
        for (int j = 0; j < VEC; ++j) {
            if (UPDATE == 0) v[i][j] = xv[i % M][j];
            if (UPDATE == 1) v[i][j] = xv[i % M][j] + v[i][j] * rstd * pw[i % M][j];
            if (UPDATE == 2 && add_w) v[i][j] += pw[i % M][j];
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
            if (!kEarly) RowIo<F32Elem, VEC>::load(next_w + c, nw[i % M]);
#pragma unroll
            for (int j = 0; j < VEC; ++j) v[i][j] = v[i][j] * rstd * nw[i % M][j];
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

// y = y silu(z), normed in equal parts of `size` elements, times w, in place: one workgroup per (row, part)
template <typename Elem, int VEC, int THREADS, int N>
__global__ __launch_bounds__(THREADS) void gated_norm_kernel(typename Elem::storage* __restrict__ y, const typename Elem::storage* __restrict__ z,
                                                             int64_t z_stride, const float* __restrict__ w, int size, float eps) {
    __shared__ float scratch[THREADS / kWave];
    const int64_t row = blockIdx.x;
    const int c0 = blockIdx.y * size;
    typename Elem::storage* yr = y + (row * gridDim.y + blockIdx.y) * size;
    const typename Elem::storage* zr = z + row * z_stride + c0;
    constexpr bool kEarly = N * VEC <= 16;
    constexpr int M = kEarly ? N : 1;
    float v[N][VEC], g[M][VEC], wv[M][VEC], sum = 0.0f;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int c = (threadIdx.x + i * THREADS) * VEC;
        if (c >= size) continue;
        RowIo<Elem, VEC>::load(yr + c, v[i]);
        if (!kEarly) continue;
        RowIo<Elem, VEC>::load(zr + c, g[i % M]);
        RowIo<F32Elem, VEC>::load(w + c0 + c, wv[i % M]);
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int c = (threadIdx.x + i * THREADS) * VEC;
        if (c >= size) continue;
        if (!kEarly) RowIo<Elem, VEC>::load(zr + c, g[i % M]);
#pragma unroll
        for (int j = 0; j < VEC; ++j) {
            v[i][j] *= silu(g[i % M][j]);
            sum = fmaf(v[i][j], v[i][j], sum);
        }
    }
    const float rstd = 1.0f / sqrtf(block_sum<THREADS>(sum, scratch) / static_cast<float>(size) + eps);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int c = (threadIdx.x + i * THREADS) * VEC;
        if (c < size) {
            if (!kEarly) RowIo<F32Elem, VEC>::load(w + c0 + c, wv[i % M]);
#pragma unroll
            for (int j = 0; j < VEC; ++j) v[i][j] *= rstd * wv[i % M][j];
            RowIo<Elem, VEC>::store(yr + c, v[i]);
        }
    }
}

// Place of the largest value of a row, the first one where several are equal; a NaN is larger than every number.  One
// workgroup per row, eight vectors of it requested at once: 32000 columns take a way to memory and the sum over the workgroup
// (4.5 us; the library's two passes 15).
constexpr int kArgmaxThreads = 1024;
__device__ __forceinline__ bool argmax_before(float a, int ia, float b, int ib) {
    const bool na = a != a, nb = b != b;
    if (na != nb) return na;
    return (!na && a != b) ? a > b : ia < ib;
}
template <int VEC>
__global__ __launch_bounds__(kArgmaxThreads) void argmax_kernel(const float* __restrict__ x, int V, int32_t* __restrict__ out) {
    constexpr int kAhead = 8;
    __shared__ float best_v[kArgmaxThreads / kWave];
    __shared__ int best_i[kArgmaxThreads / kWave];
    const float* row = x + static_cast<int64_t>(blockIdx.x) * V;
    float value = -INFINITY;
    int place = V;
    for (int c0 = threadIdx.x * VEC; c0 < V; c0 += kAhead * kArgmaxThreads * VEC) {
        float v[kAhead][VEC];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) RowIo<F32Elem, VEC>::load(row + min(c0 + i * kArgmaxThreads * VEC, V - VEC), v[i]);
#pragma unroll
        for (int i = 0; i < kAhead; ++i)
#pragma unroll
            for (int j = 0; j < VEC; ++j) {
                const int c = c0 + i * kArgmaxThreads * VEC + j;
                if (c < V && argmax_before(v[i][j], c, value, place)) {
                    value = v[i][j];
                    place = c;
                }
            }
    }
    auto take = [&](float other, int at) {
        if (argmax_before(other, at, value, place)) {
            value = other;
            place = at;
        }
    };
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) take(__shfl_xor(value, off), __shfl_xor(place, off));
    if (lane_id() == 0) {
        best_v[threadIdx.x / kWave] = value;
        best_i[threadIdx.x / kWave] = place;
    }
    __syncthreads();
    if (threadIdx.x >= kWave) return;
    constexpr int kWaves = kArgmaxThreads / kWave;
    value = best_v[threadIdx.x % kWaves];
    place = best_i[threadIdx.x % kWaves];
#pragma unroll
    for (int off = kWaves / 2; off > 0; off >>= 1) take(__shfl_xor(value, off), __shfl_xor(place, off));
    if (threadIdx.x == 0) out[blockIdx.x] = place;
}

template <typename Elem, int VEC>
int launch_gated(void* y, const void* z, int64_t z_stride, const float* w, int64_t T, int parts, int size, float eps, hipStream_t s) {
    typedef typename Elem::storage S;
    const dim3 grid(static_cast<unsigned>(T), static_cast<unsigned>(parts));
#define EM_GATED(THREADS, N) \
    launch((gated_norm_kernel<Elem, VEC, THREADS, N>), grid, dim3(THREADS), 0, s, static_cast<S*>(y), static_cast<const S*>(z), z_stride, w, size, eps)
    if (size <= 512) EM_GATED(64, 8 / VEC);
    else if (VEC == 4 && T * parts <= kFewRows && size > 1024 && size <= 4096) EM_GATED(1024, 4 / VEC);
    else if (VEC == 4 && size <= 4096) EM_GATED(256, 16 / VEC);
    else if (size <= 256 * kRowMaxPerThread) EM_GATED(256, kRowMaxPerThread / VEC);
    else EM_GATED(1024, kRowMaxPerThread / VEC);
#undef EM_GATED
    return launch_status();
}

template <typename Elem, typename YElem, int UPDATE, int VEC, int THREADS, int N>
int launch_rows(float* x, const void* y, int y_parts, const float* post_w, const float* next_w, void* out, int64_t out_stride,
                int64_t T, int W, float eps, hipStream_t s) {
    launch((residual_norm_kernel<Elem, YElem, UPDATE, VEC, THREADS, N>), dim3(static_cast<unsigned>(T)), dim3(THREADS), 0, s, x,
           static_cast<const typename YElem::storage*>(y), y_parts, post_w, next_w, static_cast<typename Elem::storage*>(out), out_stride, W, eps);
    return launch_status();
}

// One vector per thread where the rows do not fill the chip (kFewRows), so that a row is over sooner; 256 threads where they do.
template <typename Elem, typename YElem, int UPDATE, int VEC>
int launch_residual(float* x, const void* y, int y_parts, const float* post_w, const float* next_w, void* out, int64_t out_stride,
                    int64_t T, int W, float eps, hipStream_t s) {
#define EM_ROWS(THREADS, N) return launch_rows<Elem, YElem, UPDATE, VEC, THREADS, N>(x, y, y_parts, post_w, next_w, out, out_stride, T, W, eps, s)
    if constexpr (VEC == 4) {
        if (T <= kFewRows && W > 1024 && W <= 2048) EM_ROWS(512, 1);
        if (T <= kFewRows && W > 1024 && W <= 4096) EM_ROWS(1024, 1);
        if (W <= 2048) EM_ROWS(256, 2);
        if (W <= 4096) EM_ROWS(256, 4);
    }
    if (W <= 256 * kRowMaxPerThread) EM_ROWS(256, kRowMaxPerThread / VEC);
    EM_ROWS(1024, kRowMaxPerThread / VEC);
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

int launch_argmax(const float* x, int64_t T, int V, int32_t* out, hipStream_t s) {
    const dim3 grid(static_cast<unsigned>(T)), block(kArgmaxThreads);
    if (V % 4 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0) launch((argmax_kernel<4>), grid, block, 0, s, x, V, out);
    else launch((argmax_kernel<1>), grid, block, 0, s, x, V, out);
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
