// out[T, N] = act(x[T, K] w[N, K]^T) for a decode batch (T <= 64), bf16: a stream over the weights, for products whose rows or
// ranges of K do not fill the chip with the tiled kernel's workgroups (decode_pays in tile_gemm.hip has the measured line).
//
// A workgroup owns 16 * NT columns of one of `splits` ranges of K; its waves share that range out, add their results up
// in LDS, and one pass applies the activation and stores.  Bound: the weights' bytes, and for the small matrices of a
// layer the way from a launch to the first bytes.
//
// Per 64 elements of k a wave loads eight rows of 128 bytes with one instruction, eight lanes side by side on a row,
// of the weights and of the token rows alike, and turns both into MFMA operands through a stretch of LDS of its own (pitch
// 144 bytes: no conflicts).  Loads straight in operand layout touch sixteen half-used lines each, and the address unit, not
// the memory, sets the pace: with 64 token rows 2048 x 4096 took 23 us that way and takes 7.5 (library: 14), with one
// 6.5 and now 5.1.  The weights, read once, are loaded past the caches' order of use (non-temporal).  Two steps
// are in flight per wave; requesting the next two while these are multiplied was 5-15 % slower (half the waves fit).
// With splits > 1 the results are float32 partial sums [splits, T, N] that the next kernel adds up.  GLU: w is [2 N, K],
// a workgroup makes the same columns of both halves and stores silu(first) * second.
#include "decoder.h"
#include "mma.h"

namespace em {
namespace {

constexpr int kStepK = 64;
constexpr int kPitch = kStepK + 8;       // elements of a row in LDS
constexpr int kSplitGroups = 256;        // a workgroup of eight waves takes a CU

__device__ __forceinline__ u32x4_t load_once(const uint16_t* p) {
    return __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(p));
}
__device__ __forceinline__ bf16x8_t as_frag(u32x4_t w) {
    bf16x8_t f;
    __builtin_memcpy(&f, &w, 16);
    return f;
}

template <int MT, int NT, int WAVES>
constexpr int skinny_lds() {
    constexpr int stage = WAVES * (MT + NT) * 16 * kPitch * 2, sums = WAVES * 16 * MT * (16 * NT + 4) * 4;
    return stage > sums ? stage : sums;
}

// MT: tiles of 16 tokens; NT: tiles of 16 weight rows; AHEAD: steps of k in flight
template <int MT, int NT, int WAVES, int AHEAD, bool F32OUT, bool GLU>
__global__ __launch_bounds__(WAVES * kWave) void skinny_gemm_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
                                                                    void* __restrict__ out, int T, int N, int K, int act) {
    typedef Mma<BF16Elem> M;
    static_assert(!GLU || NT % 2 == 0, "tiles of both halves");
    constexpr int kCols = 16 * NT, kOutCols = GLU ? kCols / 2 : kCols, kSumPitch = kCols + 4;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, lq = lane >> 4, l8 = lane >> 3, c8 = (lane & 7) * 8;
    uint16_t* xs = reinterpret_cast<uint16_t*>(lds) + wave * (MT + NT) * 16 * kPitch;
    uint16_t* ws = xs + MT * 16 * kPitch;
    const int n0 = blockIdx.x * kOutCols;
    const int steps = K / kStepK, splits = gridDim.y, split = blockIdx.y;
    const int g0 = static_cast<int>(static_cast<int64_t>(steps) * split / splits);
    const int g1 = static_cast<int>(static_cast<int64_t>(steps) * (split + 1) / splits);
    const int s0 = g0 + (g1 - g0) * wave / WAVES, s1 = g0 + (g1 - g0) * (wave + 1) / WAVES, last = max(s1 - 1, 0);
    const uint16_t* wr[NT][2];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int c = n0 + (GLU ? n / 2 : n) * 16 + h * 8 + l8;      // (columns beyond N are not stored)
            wr[n][h] = w + (static_cast<int64_t>(c < N ? c : N - 1) + (GLU ? (n & 1) * static_cast<int64_t>(N) : 0)) * K + c8;
        }
    const uint16_t* xr[MT][2];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int h = 0; h < 2; ++h) xr[m][h] = x + static_cast<int64_t>(min(m * 16 + h * 8 + l8, T - 1)) * K + c8;
    f32x4_t acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[m][n] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    for (int s = s0; s < s1; s += AHEAD) {
        // (a step behind the last is the last one again, so that the waits count loads in a straight line)
        u32x4_t fw[AHEAD][NT][2], fx[AHEAD][MT][2];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u)
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int h = 0; h < 2; ++h) fw[u][n][h] = load_once(wr[n][h] + min(s + u, last) * kStepK);
#pragma unroll
        for (int u = 0; u < AHEAD; ++u)
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int h = 0; h < 2; ++h) fx[u][m][h] = *reinterpret_cast<const u32x4_t*>(xr[m][h] + min(s + u, last) * kStepK);
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            if (s + u >= s1) continue;
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int h = 0; h < 2; ++h) *reinterpret_cast<u32x4_t*>(ws + (n * 16 + h * 8 + l8) * kPitch + c8) = fw[u][n][h];
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int h = 0; h < 2; ++h) *reinterpret_cast<u32x4_t*>(xs + (m * 16 + h * 8 + l8) * kPitch + c8) = fx[u][m][h];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");       // (the stretch is this wave's own)
            typename M::frag ax[MT][2], aw[NT][2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
#pragma unroll
                for (int m = 0; m < MT; ++m) ax[m][h] = as_frag(*reinterpret_cast<const u32x4_t*>(xs + (m * 16 + l16) * kPitch + h * 32 + lq * 8));
#pragma unroll
                for (int n = 0; n < NT; ++n) aw[n][h] = as_frag(*reinterpret_cast<const u32x4_t*>(ws + (n * 16 + l16) * kPitch + h * 32 + lq * 8));
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int m = 0; m < MT; ++m)
#pragma unroll
                    for (int n = 0; n < NT; ++n) acc[m][n] = M::mac(ax[m][h], aw[n][h], acc[m][n]);
        }
    }
    __syncthreads();
    float* sums = reinterpret_cast<float*>(lds);                         // [WAVES][16 * MT][kSumPitch]
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int r = 0; r < 4; ++r) sums[(wave * 16 * MT + m * 16 + lq * 4 + r) * kSumPitch + n * 16 + l16] = acc[m][n][r];
    __syncthreads();
    for (int i = tid; i < 16 * MT * kOutCols; i += WAVES * kWave) {
        const int t = i / kOutCols, c = i % kOutCols;
        if (t >= T || n0 + c >= N) continue;
        if (GLU) {
            const float* at = sums + t * kSumPitch + c / 16 * 32 + c % 16;
            float g = 0.0f, u = 0.0f;
#pragma unroll
            for (int k = 0; k < WAVES; ++k) {
                g += at[k * 16 * MT * kSumPitch];
                u += at[k * 16 * MT * kSumPitch + 16];
            }
            static_cast<uint16_t*>(out)[static_cast<int64_t>(t) * N + n0 + c] = f32_to_bf16_bits(silu(g) * u);
            continue;
        }
        float v = 0.0f;
#pragma unroll
        for (int k = 0; k < WAVES; ++k) v += sums[(k * 16 * MT + t) * kSumPitch + c];
        if (act == 1) {
            v = fmaxf(v, 0.0f);
            v *= v;
        }
        const int64_t at = (static_cast<int64_t>(split) * T + t) * N + n0 + c;
        if (F32OUT) static_cast<float*>(out)[at] = v;
        else static_cast<uint16_t*>(out)[at] = f32_to_bf16_bits(v);
    }
}

template <int MT, int NT, int WAVES, int AHEAD, bool F32OUT, bool GLU>
int launch_one(const uint16_t* x, const uint16_t* w, void* out, int splits, int T, int N, int K, int act, hipStream_t s) {
    const int rc = allow_lds(reinterpret_cast<const void*>(skinny_gemm_kernel<MT, NT, WAVES, AHEAD, F32OUT, GLU>), skinny_lds<MT, NT, WAVES>());
    if (rc != 0) return rc;
    launch((skinny_gemm_kernel<MT, NT, WAVES, AHEAD, F32OUT, GLU>),
           dim3(static_cast<unsigned>(ceil_div(N, (GLU ? 8 : 16) * NT)), static_cast<unsigned>(splits)), dim3(WAVES * kWave),
           (skinny_lds<MT, NT, WAVES>()), s, x, w, out, T, N, K, act);
    return launch_status();
}

template <int MT, int NT, int WAVES, int AHEAD>
int launch_form(const uint16_t* x, const uint16_t* w, void* out, bool f32, int splits, int T, int N, int K, int act, hipStream_t s) {
    if constexpr (NT > 1)
        if (act == 2) return launch_one<MT, NT, WAVES, AHEAD, false, true>(x, w, out, splits, T, N, K, 0, s);
    return f32 ? launch_one<MT, NT, WAVES, AHEAD, true, false>(x, w, out, splits, T, N, K, act, s)
               : launch_one<MT, NT, WAVES, AHEAD, false, false>(x, w, out, splits, T, N, K, act, s);
}

// Ranges of K that fill the chip with `groups` workgroups each, a step of k for every wave at least.
int ranges_of(int groups, int K) {
    const int want = kSplitGroups / groups, most = K / (kStepK * 8), s = want < most ? want : most;
    return s < 1 ? 1 : s > 8 ? 8 : s;
}

// 64 rows of weights to a workgroup for partial sums, instead of 32: where K is long enough for as many workgroups.
bool wide_parts(int T, int N, int K) {
    const int narrow = static_cast<int>(ceil_div(N, 32)), wide = static_cast<int>(ceil_div(N, 64));
    return T > 32 && N >= 4096 && wide * ranges_of(wide, K) >= narrow * ranges_of(narrow, K);
}

// Tiles of weight rows per workgroup: as few as leave one workgroup of eight waves to a CU (us, with 64 tokens: 3072 rows of
// 2048 in ones 8.8, in twos 10.7; 6176 in twos 11.9, ones 17.4, fours 15.3; 8512 in fours 16.9, twos 19.5; with up to 32
// tokens two such workgroups share a CU, and the few beyond the first 256 cost less than half of the chip without work: 8512,
// T = 1, twos 10.0, fours 11.8).  Beyond 64 rows to a CU workgroups of four waves, of which two share a CU (32000 x 2048,
// T = 32: 25.0 / 29.3 with eight).  With three or four tiles of tokens those carry one step of k instead of two (T = 64:
// 31.5 / 38.4), and partial sums take 64 rows as soon as four ranges of K fill the chip that way, since the token rows are
// read by half as many workgroups (4096 x 12288, T = 64: 26.8 / 30.5; T = 32: 22.6 / 22.6); K too short for that many ranges would leave
// CUs without work (4096 x 1024, T = 64, with the norm that adds the ranges up 13.9 / 12.0; 4096 x 1536 15.0 / 12.9).
template <int MT>
int launch_tokens(const uint16_t* x, const uint16_t* w, void* out, bool f32, int splits, int T, int N, int K, int act, hipStream_t s) {
    const int rows = act == 2 ? 2 * N : N;
    if (splits > 1) {
        if (MT > 2 && wide_parts(T, N, K)) return launch_form<MT, 4, 8, 2>(x, w, out, f32, splits, T, N, K, act, s);
        return launch_form<MT, 2, 8, 2>(x, w, out, f32, splits, T, N, K, act, s);
    }
    if (rows <= 16 * kSplitGroups && act != 2) return launch_form<MT, 1, 8, 2>(x, w, out, f32, splits, T, N, K, act, s);
    if (rows <= (MT > 2 ? 32 : 36) * kSplitGroups) return launch_form<MT, 2, 8, 2>(x, w, out, f32, splits, T, N, K, act, s);
    if (MT > 2 && rows <= 64 * kSplitGroups) return launch_form<MT, 4, 8, 2>(x, w, out, f32, splits, T, N, K, act, s);
    return launch_form<MT, 4, 4, (MT > 2 ? 1 : 2)>(x, w, out, f32, splits, T, N, K, act, s);
}

}  // namespace

// The range of ed_skinny_gemm.
bool skinny_supported(int64_t T, int N, int K) {
    if (!decode_gemm_supported(T, N, K)) return false;
    const int64_t weights = static_cast<int64_t>(N) * K;
    return T <= 4 || (T <= 16 && weights <= (int64_t{1} << 25)) || (T <= 32 && weights <= (int64_t{1} << 24)) ||
           (T <= 64 && weights <= (int64_t{1} << 22));
}

bool decode_gemm_supported(int64_t T, int N, int K) { return T > 0 && T <= 64 && N > 0 && K > 0 && K % kStepK == 0; }

// Where a product without partial sums is faster this way than by the library (and the kernel of its activation): measured at rows
// of 1024 to 24576, k of 1024 to 16384, T of 2 to 64, weights read from memory; 0.86 / 0.86 / 0.77 / 0.80 of the library's time on the
// average (bf16, float32, squared ReLU, gated), at most a tenth more anywhere but float32 sums of 24576 rows.  The library shares k
// out over the chip, so it is ahead where here
//   * rows are few and k is long: a quarter or half of the CUs walk through all of it (us, this / library, T = 64: 1024 x 8192
//     21.0 / 14.1; gated, 2048 rows x 12288, T = 40 34.4 / 23.3), or one tile to a CU still takes 16384 steps;
//   * rows of 64 to a workgroup leave CUs without one (9216 to 15360; 12288 x 4096, T = 24 28.5 / 26.5, T = 8 26.4 / 30.4);
//   * there are more than 48 tokens, whose rows every workgroup reads: unless the weights are small or an activation comes along.
// (Layers ask for the tiled kernel first: ungated products of more than 8192 rows, and of 6144 from 33 tokens on, come here through
// ed_decode_gemm and ed_skinny_gemm only.)
bool decode_gemm_pays(int64_t T, int rows, int K, int act, bool f32) {
    if (!decode_gemm_supported(T, rows, K)) return false;
    if (rows <= 2048) {
        if (T <= 16) return act != 2 || K <= 8192;
        if (act == 1 && T <= 32) return true;
        if (f32 && rows <= 1024 && T > 32) return K <= 2048;
        return K <= (T > 32 || rows <= 1024 ? 4096 : 6144);
    }
    if (K > 12288 && rows < 8192) return false;
    if (act == 2) return rows > 4096 || K <= (T > 48 ? 3072 : rows > 3072 || T <= 32 ? 8192 : 6144);
    if (act == 1) return true;
    const bool small = static_cast<int64_t>(rows) * K <= (int64_t{1} << 24);
    if (T > 48 && rows < 16384) return (small && K <= 4096) || (rows >= 6144 && rows <= 8192 && K <= 3072);
    if (T > 48) return f32 || small;
    if (rows >= 9216 && rows < 15360) {
        if (T <= 16) return K <= (f32 ? 2048 : 4096) || (rows >= 12288 && K > 4096 && K <= 6144);
        if (T <= 32) return K <= 2048;
        return rows < 12288 || K <= 2048 || K >= 6144;
    }
    return true;
}

// Ranges of K for results that may stay partial sums: enough workgroups for the chip, a step of k for every wave.
int skinny_splits(int T, int N, int K) { return ranges_of(static_cast<int>(ceil_div(N, wide_parts(T, N, K) ? 64 : 32)), K); }

int launch_skinny_gemm(const void* x, const void* w, void* out, bool f32, int splits, int T, int N, int K, int act, hipStream_t s) {
    const uint16_t* xp = static_cast<const uint16_t*>(x);
    const uint16_t* wp = static_cast<const uint16_t*>(w);
    if (T <= 16) return launch_tokens<1>(xp, wp, out, f32, splits, T, N, K, act, s);
    if (T <= 32) return launch_tokens<2>(xp, wp, out, f32, splits, T, N, K, act, s);
    if (T <= 48) return launch_tokens<3>(xp, wp, out, f32, splits, T, N, K, act, s);
    return launch_tokens<4>(xp, wp, out, f32, splits, T, N, K, act, s);
}

}  // namespace em
