// Recurrences with one decay per head and token, behind short causal convolutions:
//     S <- g S;   u = beta (v - S^T k)  (delta rule)   or   u = beta v  (additive rule);   S <- S + k u^T;   o = S^T q
// with a float32 state S [dim, vdim] per head and sequence; q and k are shared by heads / kv_heads heads.  The gated
// delta rule has beta = sigmoid(b) and unit vectors q and k, the state-space form has k = B, q = C, beta = dt and a skip
// o + D v; both have log g = -exp(A_log) softplus(a + dt_bias), where dt is that softplus.
//
// Convolutions.  q, k and v are sums over the last `taps` projections of a channel, then SiLU.  A sequence keeps its last
// projections in a ring of `taps` rows, position p in row p % taps: a step reads other rows than the one it writes, so
// that workgroups which share channels need no order among them.
//
// Prompts.  A sequence's tokens are cut into chunks and a chunk into blocks of 16.  With c_t the product of the decays
// from the block's first token to t and S the state in front of the block,
//     (I + A) U = diag(beta) (V - diag(c) K S),        A_ts = beta_t (c_t / c_s) k_t . k_s   for s < t   (0: additive)
//     o_t = c_t S^T q_t + sum_{s <= t} (c_t / c_s) (q_t . k_s) u_s
//     S  <- c_16 S + sum_s (c_16 / c_s) k_s u_s^T
// block_kernel makes (I + A)^-1 diag(beta) and the 16 x 16 scores of every block, all blocks in parallel.  chunk_kernel
// walks through the blocks of a chunk, a wave holding 16 columns of the float32 state in the registers in which an MFMA
// leaves them, which, split into bf16 parts, are the next MFMA's second operand as they lie.  With several chunks in a sequence a
// first pass starts every chunk from zero, and for the delta rule, whose chunks multiply the state by a matrix, runs the
// identity's columns along, which gives that matrix; a scan over the chunks makes the states in front of them, and the
// output pass starts from there.  Ratios of decays are powers of differences of logarithms, never positive ones.
//
// Decoding.  One workgroup per (sequence, head): convolutions, decay, update, read-out, norm and gate; the state is read
// and written once.
#include <algorithm>

#include "decoder.h"

namespace em {
namespace {

constexpr int kBlock = 16;
constexpr float kLog2e = 1.4426950408889634f;
constexpr int kConvPiece = 256;      // channels of one wave of the convolution
constexpr int kMaxTaps = 16;

// A block's record, in floats: 16 x 16 scores, c_t, c_16 / c_t, beta_t, log2 of c_16 (16 of them); delta rule: the inverse
constexpr int kRecScores = 0, kRecDecay = 256, kRecRest = 272, kRecBeta = 288, kRecLog = 304, kRecInverse = 320;
static_assert(recur_record(false) == kRecInverse && recur_record(true) == kRecInverse + 256, "a block's record");

__device__ __forceinline__ float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }
// with the hardware's exponential, reciprocal and square root, 1 ulp each
__device__ __forceinline__ float silu_fast(float g) { return g * __builtin_amdgcn_rcpf(1.0f + exp2_fast(-g * kLog2e)); }
__device__ __forceinline__ float softplus(float z) { return fmaxf(z, 0.0f) + log1pf(expf(-fabsf(z))); }
__device__ __forceinline__ float sigmoid(float z) { return 1.0f / (1.0f + expf(-z)); }

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// log2 of the decay, and beta (dt for the additive rule)
template <typename Elem>
__device__ __forceinline__ f32x2_t decay_and_beta(const RecurProblem& p, int64_t row, int h) {
    typedef typename Elem::storage S;
    const float sp = softplus(Elem::load(static_cast<const S*>(p.decay_in)[row * p.stride + h]) + p.dt_bias[h]);
    const float log_g = -expf(p.a_log[h]) * sp * kLog2e;
    return f32x2_t{log_g, p.beta_in ? sigmoid(Elem::load(static_cast<const S*>(p.beta_in)[row * p.stride + h])) : sp};
}

template <typename Elem, bool VEC>
__device__ __forceinline__ void load_channels(const typename Elem::storage* src, int c, int count, float (&v)[4]) {
    if (VEC) {
        if (c < count) {
            typename Elem::storage t[4];
            __builtin_memcpy(t, __builtin_assume_aligned(src + c, sizeof(t)), sizeof(t));
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = Elem::load(t[j]);
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = 0.0f;
        }
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = c + j < count ? Elem::load(src[c + j]) : 0.0f;
    }
}

// ---- prompts: convolutions, unit vectors, decays ----
// every value's sum over `lanes` neighbouring lanes (a power of two), in all of them
template <int N>
__device__ __forceinline__ void add_heads(float (&v)[N], int lanes) {
    if (lanes >= 16) {
#pragma unroll
        for (int i = 0; i < N; ++i) v[i] = row_sum(v[i]);
    }
    for (int off = lanes >= 16 ? 16 : 1; off < lanes; off *= 2) {
#pragma unroll
        for (int i = 0; i < N; ++i) v[i] += __shfl_xor(v[i], off);
    }
}
// A wave takes TOKENS tokens of kConvPiece channels: four per lane, of as many q or k heads as fit (a head has a power of two of
// lanes, `head_lanes`) or of v; the last waves' share is decays and betas, one per lane.  K >= taps: rows that a lane keeps; TOKENS >= K - 1,
// so that only a portion's first piece reads the ring.  VEC: all counts and offsets are multiples of four.
template <typename Elem, int K, bool VEC, int TOKENS>
__global__ __launch_bounds__(256) void recur_conv_kernel(RecurProblem p, int head_lanes) {
    static_assert(TOKENS >= K - 1 && kBlock % TOKENS == 0, "the ring's readers");
    typedef typename Elem::storage S;
    const int4 ch = p.chunks[blockIdx.x];
    const int first = blockIdx.y * TOKENS;
    if (first >= ch.z) return;
    const int n = min(TOKENS, ch.z - first), seq = ch.x;
    const int64_t row0 = static_cast<int64_t>(ch.y) + first;
    const int q_begin = p.q_begin[seq], n_seq = p.q_begin[seq + 1] - q_begin;
    const int at0 = static_cast<int>(row0) - q_begin;          // in this step's portion of the sequence
    const int start = p.starts[seq], pos0 = start + at0;
    const int lane = threadIdx.x & 63;
    const int v_count = p.heads * p.vdim, v_units = (v_count + kConvPiece - 1) / kConvPiece;
    const int fit = kWave / head_lanes, head_units = (p.kv_heads + fit - 1) / fit;
    const int unit = blockIdx.z * 4 + (threadIdx.x >> 6);
    if (unit >= 2 * head_units + v_units) {
        const int i = (unit - 2 * head_units - v_units) * kWave + lane, t = i / p.heads, h = i - t * p.heads;
        if (t < n) *reinterpret_cast<f32x2_t*>(p.rates + ((row0 + t) * p.heads + h) * 2) = decay_and_beta<Elem>(p, row0 + t, h);
        return;
    }
    const bool is_v = unit >= 2 * head_units, is_q = unit < head_units;
    const int g = is_v ? 0 : (is_q ? unit : unit - head_units) * fit + lane / head_lanes;      // this lane's q or k head
    const int begin = is_v ? (unit - 2 * head_units) * kConvPiece : g * p.dim;
    const int count = is_v ? min(kConvPiece, v_count - begin) : g < p.kv_heads ? p.dim : 0;
    const S* src = static_cast<const S*>(is_v ? p.v : is_q ? p.q : p.k) + begin;
    const int c = (is_v ? lane : lane % head_lanes) * 4;
    const int channels = 2 * p.kv_heads * p.dim + v_count;
    const int channel0 = (is_v ? 2 * p.kv_heads * p.dim : is_q ? 0 : p.kv_heads * p.dim) + begin;
    S* ring = static_cast<S*>(p.ring) + static_cast<int64_t>(p.slots[seq]) * p.taps * channels + channel0;

    float cur[TOKENS][4];
#pragma unroll
    for (int t = 0; t < TOKENS; ++t) load_channels<Elem, VEC>(src + (row0 + min(t, n - 1)) * p.stride, c, count, cur[t]);
    float w[K][4], bias[4];                                     // w[i]: of the row K - 1 - i tokens back
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        bias[j] = p.conv_b != nullptr && c + j < count ? p.conv_b[channel0 + c + j] : 0.0f;
        if (K == 4 && p.taps == 4) {
            f32x4_t row = {0.0f, 0.0f, 0.0f, 0.0f};
            if (c + j < count) row = *reinterpret_cast<const f32x4_t*>(p.conv_w + static_cast<int64_t>(channel0 + c + j) * 4);
#pragma unroll
            for (int i = 0; i < K; ++i) w[i][j] = row[i & 3];
            continue;
        }
#pragma unroll
        for (int i = 0; i < K; ++i)
            w[i][j] = K - 1 - i < p.taps && c + j < count ? p.conv_w[static_cast<int64_t>(channel0 + c + j) * p.taps + p.taps - K + i] : 0.0f;
    }
    float hist[K][4];                                           // hist[i]: the row K - 1 - i back, hist[K - 1] unused
#pragma unroll
    for (int i = 0; i < K; ++i) {
        const int back = K - 1 - i;
#pragma unroll
        for (int j = 0; j < 4; ++j) hist[i][j] = 0.0f;
        if (back > 0 && back < p.taps) {
            if (at0 >= back) load_channels<Elem, VEC>(src + (row0 - back) * p.stride, c, count, hist[i]);
            else if (pos0 >= back) load_channels<Elem, VEC>(ring + static_cast<int64_t>((pos0 - back) % p.taps) * channels, c, count, hist[i]);
        }
    }
    // (results take the projections' registers, so that the sums of all tokens' vectors are added up side by side)
    float ss[TOKENS];
#pragma unroll
    for (int t = 0; t < TOKENS; ++t) {
        ss[t] = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float y = bias[j];
#pragma unroll
            for (int i = 0; i < K - 1; ++i) {
                y = fmaf(w[i][j], hist[i][j], y);
                hist[i][j] = i + 1 < K - 1 ? hist[i + 1][j] : cur[t][j];
            }
            cur[t][j] = silu_fast(fmaf(w[K - 1][j], cur[t][j], y));
            ss[t] = fmaf(cur[t][j], cur[t][j], ss[t]);
        }
    }
    if (is_v) {
        S* dst = static_cast<S*>(p.v_f) + row0 * v_count + begin;
#pragma unroll
        for (int t = 0; t < TOKENS; ++t, dst += v_count) {
            if (VEC) {
                if (c < count && t < n) {
                    S s4[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) s4[j] = Elem::store(cur[t][j]);
                    __builtin_memcpy(__builtin_assume_aligned(dst + c, sizeof(s4)), s4, sizeof(s4));
                }
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (c + j < count && t < n) dst[c + j] = Elem::store(cur[t][j]);
            }
        }
    } else {
        const int dp = (p.dim + 15) / 16 * 16;
        float scale[TOKENS];
        if (p.unit_eps > 0.0f) add_heads(ss, head_lanes);
#pragma unroll
        for (int t = 0; t < TOKENS; ++t) scale[t] = (is_q ? p.q_scale : 1.0f) * (p.unit_eps > 0.0f ? __builtin_amdgcn_rsqf(ss[t] + p.unit_eps) : 1.0f);
        // (channels beyond dim are zero: their weights are)
        float* dst = (is_q ? p.q_f : p.k_f) + (row0 * p.kv_heads + g) * dp;
#pragma unroll
        for (int t = 0; t < TOKENS; ++t, dst += p.kv_heads * dp)
            if (c < dp && count > 0 && t < n)
                *reinterpret_cast<f32x4_t*>(dst + c) = f32x4_t{cur[t][0] * scale[t], cur[t][1] * scale[t], cur[t][2] * scale[t], cur[t][3] * scale[t]};
    }
    if (at0 != 0) return;
    // (the lane that reads the ring's old rows of these channels is the one that replaces them)
    S last[K][4];
#pragma unroll
    for (int back = 1; back < K; ++back)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            last[back][j] = back < p.taps && back <= n_seq && c + j < count ? src[(static_cast<int64_t>(q_begin) + n_seq - back) * p.stride + c + j] : S(0);
#pragma unroll
    for (int back = 1; back < K; ++back) {
        if (back >= p.taps || back > n_seq) continue;
        S* dst = ring + static_cast<int64_t>((start + n_seq - back) % p.taps) * channels;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (c + j < count) dst[c + j] = last[back][j];
    }
}

// ---- prompts: every block's scores and inverse ----
// A wave takes one block and up to kBlockHeads of the heads that share q and k.
constexpr int kBlockHeads = 8;
template <bool DELTA>
__global__ __launch_bounds__(256) void recur_block_kernel(RecurProblem p, int heads_per_wave) {
    constexpr int kPitch = 20;
    __shared__ __attribute__((aligned(16))) float lds[4][kBlock * kPitch];
    const int4 ch = p.chunks[blockIdx.x];
    const int first = blockIdx.y * kBlock;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, lq = lane >> 4;
    const int share = p.heads / p.kv_heads, h0 = (blockIdx.z * 4 + wave) * heads_per_wave;   // (a divisor of `share`)
    if (first >= ch.z || h0 >= p.heads) return;                 // (waves share nothing)
    const int n = min(kBlock, ch.z - first);
    const int64_t row0 = static_cast<int64_t>(ch.y) + first;
    const int dp = (p.dim + 15) / 16 * 16, g = h0 / share;
    const int64_t pitch = static_cast<int64_t>(p.kv_heads) * dp;
    const bool ok = l16 < n;
    const float* kr = p.k_f + (row0 + (ok ? l16 : 0)) * pitch + g * dp + lq * 4;
    const float* qr = p.q_f + (row0 + (ok ? l16 : 0)) * pitch + g * dp + lq * 4;
    f32x4_t qk = {0.0f, 0.0f, 0.0f, 0.0f}, kk = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
    for (int d = 0; d < dp; d += 16) {
        const f32x4_t q4 = *reinterpret_cast<const f32x4_t*>(qr + d), k4 = *reinterpret_cast<const f32x4_t*>(kr + d);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            qk = __builtin_amdgcn_mfma_f32_16x16x4f32(q4[r], k4[r], qk, 0, 0, 0);
            if (DELTA) kk = __builtin_amdgcn_mfma_f32_16x16x4f32(k4[r], k4[r], kk, 0, 0, 0);
        }
    }
    const int64_t nb = p.chunk_tokens / kBlock;
    float* am = lds[wave];
    for (int h = h0; h < h0 + heads_per_wave; ++h) {
        f32x2_t rate = {0.0f, 0.0f};
        if (ok) rate = *reinterpret_cast<const f32x2_t*>(p.rates + ((row0 + l16) * p.heads + h) * 2);
        float bl = rate[0];
#pragma unroll
        for (int off = 1; off < kBlock; off <<= 1) {
            const float up = __shfl_up(bl, off, kBlock);
            if (l16 >= off) bl += up;
        }
        const float tot = __shfl(bl, kBlock - 1, kBlock);
        float* rec = p.blocks + ((blockIdx.x * nb + blockIdx.y) * p.heads + h) * recur_record(DELTA);
        if (lq == 0) {
            rec[kRecDecay + l16] = exp2_fast(bl);
            rec[kRecRest + l16] = exp2_fast(tot - bl);
            rec[kRecBeta + l16] = rate[1];
            rec[kRecLog + l16] = tot;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int t = lq * 4 + r;
            const float ratio = exp2_fast(fminf(__shfl(bl, t, kBlock) - bl, 0.0f)), beta = __shfl(rate[1], t, kBlock);
            rec[kRecScores + t * kBlock + l16] = l16 <= t && t < n ? qk[r] * ratio : 0.0f;
            if (DELTA) am[t * kPitch + l16] = l16 < t && t < n ? beta * kk[r] * ratio : 0.0f;
        }
        if (!DELTA) continue;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        // column l16 of the inverse of the unit lower triangular matrix, row by row (each few of the wave on its own)
        float inv[kBlock];
#pragma unroll
        for (int t = 0; t < kBlock; ++t) {
            float v = t == l16 ? 1.0f : 0.0f;
#pragma unroll
            for (int s0 = 0; s0 < t; s0 += 4) {
                const f32x4_t a = *reinterpret_cast<const f32x4_t*>(am + t * kPitch + s0);
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (s0 + j < t) v = fmaf(-a[j], inv[s0 + j], v);
            }
            inv[t] = v;
        }
#pragma unroll
        for (int t = 0; t < kBlock; ++t)
            if ((t >> 2) == lq) rec[kRecInverse + t * kBlock + l16] = inv[t] * rate[1];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
}

// ---- prompts: a chunk's blocks, one after the other ----
// Products with the state (but the additive rule's read-out) run on the bf16 matrix units, every float32 operand as the sum of three
// bf16 values: 8 bits each, rounded to nearest, together all 24 (the second is 2^-8 of the first at most, the third 2^-17).  Of the nine
// products the six down to 2^-17 of the first are added up, in float32, the smallest first; the others are 2^-25 of it at most.  Against
// float64 this is no further off than float32 products (1536 tokens, 4 heads of 128 x 128, this / those: 8.3e-7 / 8.5e-7 where everything is
// kept, 7.06e-7 / 7.06e-7 with decays of e^-2.7 a token; over five mixers and four decays at most 1.001 of theirs); six bf16 products take 96 cycles where eight float32 ones take 256.  The parts of an infinite value, or one beyond the largest
// bf16, are no numbers, and a key, an update or a state with such parts leaves NaN in the state until the chunk ends (a query's are asked
// for): such a chunk is computed once more, with float32 products.  No time without one (8192 tokens: 407 / 409 and 332 / 334 us a call).
constexpr float kMostPart = 3.3895314e38f;            // the largest bf16
//
// What bounds the kernel now is instructions: a block is 60-80 matrix and 130-500 vector instructions per wave (splitting the state 180,
// scaling it 32, a share of the keys 50), and the chain from the barrier through LDS, sums, u and update.  So operands are read from LDS
// ahead of their products, row sums rotate inside the vector unit (16 shuffles through LDS before), addresses are kept from block to
// block, and the passes that fit 128 registers run with four waves per SIMD.  us at 8192 tokens, 16 heads of 128 x 128 (delta) and 64 of
// 128 x 64 with one key, before / now: first pass 206 / 138 and 103 / 72, output pass 193 / 135 and 222 / 170.
struct Split2 {
    uint32_t part[3];
};
__device__ __forceinline__ Split2 split2(float a, float b) {
    Split2 s;
    s.part[0] = pack_bf16(a, b);
    asm("" : "+v"(s.part[0]));        // (else the compiler converts every value once more instead of shifting it back)
    const float a1 = a - bf16_lo(s.part[0]), b1 = b - bf16_hi(s.part[0]);
    s.part[1] = pack_bf16(a1, b1);
    asm("" : "+v"(s.part[1]));
    s.part[2] = pack_bf16(a1 - bf16_lo(s.part[1]), b1 - bf16_hi(s.part[1]));
    return s;
}
struct Split4 {
    u32x2_t part[3];
};
__device__ __forceinline__ Split4 split4(f32x4_t v) {
    const Split2 lo = split2(v[0], v[1]), hi = split2(v[2], v[3]);
    Split4 s;
#pragma unroll
    for (int i = 0; i < 3; ++i) s.part[i] = u32x2_t{lo.part[i], hi.part[i]};
    return s;
}
// two packed halves side by side
__device__ __forceinline__ bf16x8_t join(u32x2_t lo, u32x2_t hi) {
    const u32x4_t w = {lo[0], lo[1], hi[0], hi[1]};
    bf16x8_t f;
    __builtin_memcpy(&f, &w, 16);
    return f;
}
struct Split8 {
    bf16x8_t part[3];
};
__device__ __forceinline__ Split8 split8(f32x4_t lo, f32x4_t hi) {
    const Split4 l = split4(lo), h = split4(hi);
    Split8 s;
#pragma unroll
    for (int i = 0; i < 3; ++i) s.part[i] = join(l.part[i], h.part[i]);
    return s;
}
__device__ __forceinline__ f32x4_t mma(bf16x8_t a, bf16x8_t b, f32x4_t c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
// four rows of a column: ds_read_b64_tr_b16, for which the 16 lanes of a group name the four-element pieces of four rows
__device__ __forceinline__ u32x2_t read_column(const uint16_t* piece) {
    typedef short s16x4_t __attribute__((ext_vector_type(4)));
    const s16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)(piece));
    u32x2_t w;
    __builtin_memcpy(&w, &v, 8);
    return w;
}

// Whether a kernel multiplies by parts.  Not the 16 waves that a delta rule's values beyond 128 need for their norm: 128 registers a lane are
// too few for the parts, and what they spill costs more than the products (us of a call, 8192 tokens, 16 heads: 128 x 256 1086 by parts,
// 770 as they are; 64 x 256 663 / 423); unless the state alone spills (256 x 256 2392 / 2481).
constexpr bool chunk_parts(int threads, int ndt) { return threads <= 512 || ndt > 8; }

// One workgroup per (chunk, head, group of column tiles), one wave per tile of 16 state columns; waves without a tile help
// with the loads.  Additive rule: a workgroup may take all columns of several heads that share keys (`group`), which then are split
// once.  OUTPUT: from the state in front of the chunk; else from zero, with the identity's columns behind the state's for the
// delta rule.  True, for the whole workgroup and without a state written, where the parts did not hold a value (`kParts`).
template <typename Elem, int NDT, bool DELTA, bool OUTPUT, int THREADS, bool kParts>
__device__ __forceinline__ bool chunk_pass(const RecurProblem& p, int group, int tid, dim3 block) {
    typedef typename Elem::storage S;
    constexpr int D = NDT * 16, DP = D + 8, kPieces = (NDT + 7) / 8;   // four-float pieces of a block's k (q) per thread
    constexpr int kPart = kBlock * DP, kTile = 3 * kPart;
    static_assert(NDT % 2 == 0, "a step of the products is two tiles");
    constexpr bool kRoom = THREADS <= 512 && NDT <= 8;                 // for operands ahead of their products in registers
    const int waves = blockDim.x / kWave;
    extern __shared__ __attribute__((aligned(16))) uint16_t operands[];
    uint16_t* Ks = operands;                               // [2][3 parts][16][DP]
    // Q by its parts as well, [2][3 parts][16][DP], where the delta rule splits the state for K anyway; for the additive rule as it is,
    // [2][16][D + 4]: splitting the state costs more than the float32 products it saves
    constexpr int kPitch = D + 4, kFloatTile = kBlock * kPitch;
    uint16_t* Qs = Ks + 2 * kTile;
    float* Kf = reinterpret_cast<float*>(operands);        // !kParts: both as they are, [2][16][D + 4]
    float* Qf = kParts ? reinterpret_cast<float*>(Qs) : Kf + 2 * kFloatTile;
    float* Rs = kParts ? reinterpret_cast<float*>(Qs + 2 * kTile) : Qf + 2 * kFloatTile;      // [2][THREADS / 64][16] partial sums of squares (delta rule)

    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, lq = lane >> 4;
    const int4 ch = p.chunks[block.x];
    const int dim = p.dim, vdim = p.vdim, dp = (dim + 15) / 16 * 16, v_tiles = (vdim + 15) / 16;
    const bool several = !DELTA && group > 1;
    const int h = several ? static_cast<int>(block.y) * group + min(wave / v_tiles, group - 1) : static_cast<int>(block.y), tile = several ? wave % v_tiles : static_cast<int>(block.z) * waves + wave;
    const int g = h / (p.heads / p.kv_heads);
    const bool identity = !OUTPUT && DELTA && tile >= v_tiles;
    const bool has_tile = (several ? wave < group * v_tiles : tile < v_tiles) || (identity && tile < v_tiles + dp / 16);
    const int col = (identity ? tile - v_tiles : tile) * 16 + l16;
    const bool v_ok = has_tile && tile < v_tiles && col < vdim;
    const int64_t kq_pitch = static_cast<int64_t>(p.kv_heads) * dp, v_pitch = static_cast<int64_t>(p.heads) * vdim;
    const float* kg = p.k_f + g * dp;
    const float* qg = p.q_f + g * dp;
    const S* vg = static_cast<const S*>(p.v_f) + h * vdim + tile * 16;
    const S* gate = OUTPUT && DELTA ? static_cast<const S*>(p.gate) + h * vdim + tile * 16 : nullptr;
    const int n_blocks = (ch.z + kBlock - 1) / kBlock;
    const int64_t rec_pitch = static_cast<int64_t>(p.heads) * recur_record(DELTA);
    const float* rec0 = p.blocks + (static_cast<int64_t>(block.x) * (p.chunk_tokens / kBlock) * p.heads + h) * recur_record(DELTA);

    // Column `col` of the state, rows lq * D / 4 + dt * 4 + r: two tiles are eight rows of a lane that lie side by side, as a
    // product over the state takes them, and the pieces of a key that one tile takes lie a few of its row apart (so that they,
    // and 16 rows of either operand, fall on different banks).  !kParts: a tile's 16 rows side by side.
    f32x4_t st[NDT];
    auto row_of = [&](int dt) { return kParts ? lq * (D / 4) + dt * 4 : dt * 16 + lq * 4; };
    const int64_t head_state = static_cast<int64_t>(dim) * vdim;
    float* slot = p.states + (static_cast<int64_t>(p.slots[ch.x]) * p.heads + h) * head_state;
    const bool chunked = p.chunk_states != nullptr;
    float* mine = chunked ? p.chunk_states + (static_cast<int64_t>(block.x) * p.heads + h) * head_state : slot;
    const bool from_zero = !OUTPUT || (!chunked && p.starts[ch.x] == 0);
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int d = row_of(dt) + r;
            st[dt][r] = identity ? (d == col ? 1.0f : 0.0f) : (!from_zero && v_ok && d < dim) ? mine[static_cast<int64_t>(d) * vdim + col] : 0.0f;
        }
    const float norm_w = OUTPUT && DELTA && v_ok ? p.norm_w[col] : 0.0f;
    const float skip = OUTPUT && p.skip != nullptr ? p.skip[h] : 0.0f;
    const float inv_vdim = 1.0f / static_cast<float>(vdim);

    // A block's operands, in flight while the one before is computed: loads of rows and columns that exist, without conditions around
    // them (what does not exist is made zero where it is used).
    // (The additive rule's output pass and the delta rule's first one ask for a block's record when they start on it: one set of registers instead of two is what lets
    // a CU have four waves per SIMD.)
    constexpr bool kAhead = kParts || THREADS > 512, kLate = OUTPUT != DELTA || !kAhead;     // (a second pass loads a block when it starts on it)
    f32x4_t rk[kPieces], rq[kPieces], scores, inverse, decay, rest, beta;
    float block_decay, block_log;
    S v[4] = {}, gt[4] = {};                          // (as stored: a conversion here would wait for the load)
    int k_at[kPieces], v_at[4];                       // a lane's elements, from a block's first row
    int64_t gate_at[4];
    auto place = [&](int last) {                      // ... of whose rows `last` is the last
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            const int e = tid + i * static_cast<int>(blockDim.x), t = e / (D / 4), d = (e - t * (D / 4)) * 4;
            k_at[i] = min(t, last) * static_cast<int>(kq_pitch) + min(d, dp - 4);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int t = min(lq * 4 + r, last), c = v_ok ? l16 : 0;
            v_at[r] = t * static_cast<int>(v_pitch) + c;
            if (OUTPUT && DELTA) gate_at[r] = t * p.stride + c;
        }
    };
    auto records = [&](int b) {
        const float* rec = rec0 + b * rec_pitch;
        if (OUTPUT) scores = *reinterpret_cast<const f32x4_t*>(rec + kRecScores + l16 * kBlock + lq * 4);
        if (DELTA) inverse = *reinterpret_cast<const f32x4_t*>(rec + kRecInverse + l16 * kBlock + lq * 4);
        else beta = *reinterpret_cast<const f32x4_t*>(rec + kRecBeta + lq * 4);
        decay = *reinterpret_cast<const f32x4_t*>(rec + kRecDecay + lq * 4);
        rest = *reinterpret_cast<const f32x4_t*>(rec + kRecRest + lq * 4);
        block_decay = rec[kRecDecay + kBlock - 1];
        block_log = rec[kRecLog];
    };
    auto fetch = [&](int b) {
        const int64_t row0 = static_cast<int64_t>(ch.y) + b * kBlock;
        if (!kParts || b == 0 || b == n_blocks - 1) place(min(kBlock, ch.z - b * kBlock) - 1);
        const float *k0 = kg + row0 * kq_pitch, *q0 = qg + row0 * kq_pitch;
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            rk[i] = *reinterpret_cast<const f32x4_t*>(k0 + k_at[i]);
            if (OUTPUT) rq[i] = *reinterpret_cast<const f32x4_t*>(q0 + k_at[i]);
        }
        if (!kLate) records(b);
        if (tile >= v_tiles) return;
        const S *v0 = vg + row0 * v_pitch, *gate0 = gate + (OUTPUT && DELTA ? row0 * p.stride : 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            v[r] = v0[v_at[r]];
            if (OUTPUT && DELTA) gt[r] = gate0[gate_at[r]];
        }
    };
    // a block's results wait for the row sums of the other waves until the next barrier
    f32x4_t held = {0.0f, 0.0f, 0.0f, 0.0f};
    float held_gate[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    auto finish = [&](int b) {
        const int n = min(kBlock, ch.z - b * kBlock);
        const int64_t row0 = static_cast<int64_t>(ch.y) + b * kBlock;
        f32x4_t ss = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w0 = 0; w0 < THREADS / kWave; w0 += 4) {
            f32x4_t part[4];
#pragma unroll
            for (int w = 0; w < 4; ++w) part[w] = *reinterpret_cast<const f32x4_t*>(Rs + ((b & 1) * (THREADS / kWave) + w0 + w) * kBlock + lq * 4);
#pragma unroll
            for (int w = 0; w < 4; ++w) ss += part[w];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int t = lq * 4 + r;
            const float y = held[r] * __builtin_amdgcn_rsqf(ss[r] * inv_vdim + p.eps) * norm_w * silu_fast(held_gate[r]);
            if (v_ok && t < n) static_cast<S*>(p.out)[(row0 + t) * v_pitch + h * vdim + col] = Elem::store(y);
        }
    };
    if (OUTPUT && DELTA)              // (waves that do not exist add nothing)
        for (int i = tid; i < 2 * THREADS / kWave * kBlock; i += static_cast<int>(blockDim.x)) Rs[i] = 0.0f;
    float log_sum = 0.0f, largest_q = 0.0f;
    if (kAhead) fetch(0);
    for (int b = 0; b < n_blocks; ++b) {
        uint16_t* kb = Ks + (b & 1) * kTile;
        uint16_t* qb = Qs + (b & 1) * kTile;
        float *kf = Kf + (b & 1) * kFloatTile, *qf = Qf + (b & 1) * kFloatTile;
        const int n = min(kBlock, ch.z - b * kBlock);
        if (!kAhead) fetch(b);
        auto keep = [&](uint16_t* to, f32x4_t v, bool exists) {
            const f32x4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
            const Split4 s = split4(exists ? v : zero);
#pragma unroll
            for (int i = 0; i < 3; ++i) *reinterpret_cast<u32x2_t*>(to + i * kPart) = s.part[i];
        };
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            const int e = tid + i * static_cast<int>(blockDim.x), t = e / (D / 4), d = (e - t * (D / 4)) * 4;
            if (t < kBlock) {
                const bool exists = t < n && d < dp;
                const f32x4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
                if (kParts) keep(kb + t * DP + d, rk[i], exists);
                else *reinterpret_cast<f32x4_t*>(kf + t * kPitch + d) = exists ? rk[i] : zero;
                if (kParts && DELTA && OUTPUT) {
                    keep(qb + t * DP + d, rq[i], exists);
                    largest_q = fmaxf(fmaxf(fmaxf(largest_q, fabsf(rq[i][0])), fmaxf(fabsf(rq[i][1]), fabsf(rq[i][2]))), fabsf(rq[i][3]));
                }
                if (OUTPUT && !(kParts && DELTA)) *reinterpret_cast<f32x4_t*>(qf + t * kPitch + d) = exists ? rq[i] : zero;
            }
        }
        f32x4_t scores_b, inverse_b, decay_b, rest_b, beta_b;
        float whole;
        auto take = [&]() {
            scores_b = scores, inverse_b = inverse, decay_b = decay, rest_b = rest, beta_b = beta;
            whole = block_decay;
            log_sum += block_log;
        };
        if (!kLate) take();
        float v_b[4], gt_b[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const bool ok = v_ok && lq * 4 + r < n;
            v_b[r] = ok ? Elem::load(v[r]) : 0.0f;
            gt_b[r] = OUTPUT && DELTA && ok ? Elem::load(gt[r]) : 0.0f;
        }
        __syncthreads();              // (the block before last, in the same half, has been used)
        if (kLate) {
            records(b);
            take();
        }
        if (kAhead && b + 1 < n_blocks) fetch(b + 1);
        if (OUTPUT && DELTA && b > 0 && (!kParts || !has_tile)) finish(b - 1);
        if (!has_tile) continue;
        // Operands from LDS a step ahead of the products, K's and Q's sums in turn: every product of a sum waits for the one before.
        f32x4_t u, ks = {0.0f, 0.0f, 0.0f, 0.0f}, o = {0.0f, 0.0f, 0.0f, 0.0f};
        if (DELTA && kParts) {
            constexpr int kTwo = kRoom && OUTPUT ? 1 : 0;
            Split8 ka[1 + kTwo], qa[1 + kTwo];
            auto rows = [&](int k) {
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    const int at = i * kPart + l16 * DP + lq * (D / 4) + k * 8;
                    ka[k & kTwo].part[i] = *reinterpret_cast<const bf16x8_t*>(kb + at);
                    if (OUTPUT) qa[k & kTwo].part[i] = *reinterpret_cast<const bf16x8_t*>(qb + at);
                }
            };
            Split8 s8[1 + kTwo];
            if (kTwo) {
                rows(0);
                s8[0] = split8(st[0], st[1]);
            }
#pragma unroll
            for (int k = 0; k < NDT / 2; ++k) {
                if (!kTwo) rows(k);
                else if (k + 1 < NDT / 2) rows(k + 1);
                if (kRoom) __builtin_amdgcn_sched_barrier(0);
                if (!kTwo) s8[0] = split8(st[2 * k], st[2 * k + 1]);
                else if (k + 1 < NDT / 2) s8[(k + 1) & kTwo] = split8(st[2 * k + 2], st[2 * k + 3]);
                // the smallest products first
                constexpr int kFirst[6] = {2, 1, 0, 1, 0, 0}, kSecond[6] = {0, 1, 2, 0, 1, 0};
#pragma unroll
                for (int i = 0; i < 6; ++i) {
                    ks = mma(ka[k & kTwo].part[kFirst[i]], s8[k & kTwo].part[kSecond[i]], ks);
                    if (OUTPUT) o = mma(qa[k & kTwo].part[kFirst[i]], s8[k & kTwo].part[kSecond[i]], o);
                }
            }
        }
        if (!kParts) {
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) {
                const f32x4_t k4 = *reinterpret_cast<const f32x4_t*>(kf + l16 * kPitch + row_of(dt));
#pragma unroll
                for (int r = 0; r < 4; ++r) ks = __builtin_amdgcn_mfma_f32_16x16x4f32(k4[r], st[dt][r], ks, 0, 0, 0);
            }
        }
        if ((!DELTA || !kParts) && OUTPUT) {
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) {
                const f32x4_t q4 = *reinterpret_cast<const f32x4_t*>(qf + l16 * kPitch + row_of(dt));
#pragma unroll
                for (int r = 0; r < 4; ++r) o = __builtin_amdgcn_mfma_f32_16x16x4f32(q4[r], st[dt][r], o, 0, 0, 0);
                if (kRoom && dt % 2 != 0) __builtin_amdgcn_sched_barrier(0);      // (all of them at once do not fit the registers)
            }
        }
        if (kParts && OUTPUT && DELTA && b > 0) finish(b - 1);
        // the keys by column, for the update: on their way while u is made
        const uint16_t* kc = kb + (lq * 4 + (l16 >> 2)) * DP + (l16 & 3) * (D / 4);
        constexpr int kRing = !kRoom ? 1 : OUTPUT || DELTA ? 2 : 4;
        u32x2_t kt[kRing][3];
        auto columns = [&](int dt) {
#pragma unroll
            for (int i = 0; i < 3; ++i) kt[dt % kRing][i] = read_column(kc + i * kPart + dt * 4);
        };
        if (kRoom) {
#pragma unroll
            for (int dt = 0; dt < kRing && dt < NDT; ++dt) columns(dt);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (DELTA) {
            f32x4_t right;
#pragma unroll
            for (int r = 0; r < 4; ++r) right[r] = v_b[r] - decay_b[r] * ks[r];
            u = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int r = 0; r < 4; ++r) u = __builtin_amdgcn_mfma_f32_16x16x4f32(inverse_b[r], right[r], u, 0, 0, 0);
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) u[r] = beta_b[r] * v_b[r];
        }
        if (OUTPUT) {
            o *= decay_b;
#pragma unroll
            for (int r = 0; r < 4; ++r) o = __builtin_amdgcn_mfma_f32_16x16x4f32(scores_b[r], u[r], o, 0, 0, 0);
        }
        u *= rest_b;
        // A product over 16 tokens fills half of an instruction: the halves take two of the six products of parts.
        const Split4 us = split4(u);
        const bf16x8_t u32 = join(us.part[2], us.part[1]), u21 = join(us.part[1], us.part[0]), u11 = join(us.part[0], us.part[0]);
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) {
            if (!kParts) {
                st[dt] *= whole;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    st[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[(lq * 4 + r) * kPitch + dt * 16 + l16], u[r], st[dt], 0, 0, 0);
                continue;
            }
            if (!kRoom) columns(dt);
            const bf16x8_t k12 = join(kt[dt % kRing][0], kt[dt % kRing][1]), k13 = join(kt[dt % kRing][0], kt[dt % kRing][2]);
            if (kRoom && dt + kRing < NDT) columns(dt + kRing);
            st[dt] *= whole;
            st[dt] = mma(k12, u32, st[dt]);           // k1 u3 + k2 u2
            st[dt] = mma(k13, u21, st[dt]);           // k1 u2 + k3 u1
            st[dt] = mma(k12, u11, st[dt]);           // k1 u1 + k2 u1
        }
        if (OUTPUT && DELTA) {
            f32x4_t ss;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                ss[r] = row_sum(o[r] * o[r]);
                held_gate[r] = gt_b[r];
            }
            if (l16 == 0) *reinterpret_cast<f32x4_t*>(Rs + ((b & 1) * (THREADS / kWave) + wave) * kBlock + lq * 4) = ss;
            held = o;
        } else if (OUTPUT) {
            const int64_t row0 = static_cast<int64_t>(ch.y) + b * kBlock;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int t = lq * 4 + r;
                if (v_ok && t < n)
                    static_cast<S*>(p.out)[(row0 + t) * v_pitch + h * vdim + col] = Elem::store(fmaf(skip, v_b[r], o[r]));
            }
        }
    }
    if (OUTPUT && DELTA) {
        __syncthreads();
        finish(n_blocks - 1);
    }
    if (kParts) {
        float sum = 0.0f;             // (NaN if a value is infinite or none)
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int r = 0; r < 4; ++r) sum = fmaf(st[dt][r], 0.0f, sum);
        if (__syncthreads_or(sum != sum || largest_q > kMostPart)) return true;
    }
    if (OUTPUT && chunked) return false;
    if (identity) {
        float* m = p.chunk_trans + (static_cast<int64_t>(block.x) * p.heads + h) * dp * dp;
        if (has_tile) {
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int d = row_of(dt) + r;
                    if (d < dp) m[d * dp + col] = st[dt][r];
                }
        }
        return false;
    }
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int d = row_of(dt) + r;
            if (v_ok && d < dim) mine[static_cast<int64_t>(d) * vdim + col] = st[dt][r];
        }
    if (!OUTPUT && !DELTA && tile == 0 && lane == 0) p.chunk_trans[static_cast<int64_t>(block.x) * p.heads + h] = log_sum;
    return false;
}

template <typename Elem, int NDT, bool DELTA, bool OUTPUT, int THREADS>
__global__ __launch_bounds__(THREADS, (DELTA && OUTPUT) || NDT > 8 ? 2 : 4) void recur_chunk_kernel(RecurProblem p, int group) {
    if constexpr (chunk_parts(THREADS, NDT)) {
        if (!chunk_pass<Elem, NDT, DELTA, OUTPUT, THREADS, true>(p, group, threadIdx.x, blockIdx)) return;
        // Again, as float32.  (Everything is read anew: what the passes shared would be kept in registers during the first.)
        auto args = __builtin_amdgcn_kernarg_segment_ptr();
        int tid = threadIdx.x;
        dim3 block = blockIdx;
        asm volatile("" : "+s"(args), "+v"(tid), "+s"(block.x), "+s"(block.y), "+s"(block.z));
        RecurProblem again;
        __builtin_memcpy(&again, (const void*)args, sizeof(again));
        chunk_pass<Elem, NDT, DELTA, OUTPUT, THREADS, false>(again, group, tid, block);
    } else {
        chunk_pass<Elem, NDT, DELTA, OUTPUT, THREADS, false>(p, group, threadIdx.x, blockIdx);
    }
}

// ---- prompts: contribution of every chunk -> state in front of it; the state behind the last chunk goes to the slot ----
// Additive rule: a chunk multiplies the state by a number.
__global__ __launch_bounds__(256) void recur_scan_kernel(RecurProblem p) {
    constexpr int kAhead = 4;
    const int i = blockIdx.x * 256 + threadIdx.x, n = p.dim * p.vdim;
    if (i >= n) return;
    const int h = blockIdx.y, s = blockIdx.z;
    const int c0 = p.seq_chunks[s], c1 = p.seq_chunks[s + 1];
    const int64_t pitch = static_cast<int64_t>(p.heads) * n;
    float* slot = p.states + (static_cast<int64_t>(p.slots[s]) * p.heads + h) * n + i;
    float* cs = p.chunk_states + static_cast<int64_t>(h) * n + i;
    float state = p.starts[s] == 0 ? 0.0f : *slot;
    for (int c = c0; c < c1; c += kAhead) {
        float u[kAhead], e[kAhead];
#pragma unroll
        for (int j = 0; j < kAhead; ++j)
            if (c + j < c1) {
                u[j] = cs[(c + j) * pitch];
                e[j] = p.chunk_trans[static_cast<int64_t>(c + j) * p.heads + h];
            }
#pragma unroll
        for (int j = 0; j < kAhead; ++j)
            if (c + j < c1) {
                cs[(c + j) * pitch] = state;
                state = fmaf(exp2_fast(e[j]), state, u[j]);
            }
    }
    *slot = state;
}

// Delta rule: by a matrix.  One workgroup per (head, 16 state columns, sequence), one wave per 16 rows.
// A chain of chunks, bound by how fast one CU takes a chunk's matrix in: a wave's 16 rows lie whole in memory and are loaded so, 1 KB an
// instruction, and turned into operands through LDS that is the wave's own (loaded as operands, 16 pieces of 64 bytes an instruction, 16 chunks
// of 16 heads of 128 x 128 took 44.7 us instead of 31.4, five chunks of five sequences 53.0 instead of 38.3; the products alone are 0.9 us a
// chunk.  Matrices of 256 rows have no room there and are loaded as operands).
template <int NDT>
__global__ __launch_bounds__(NDT * kWave) void recur_matrix_scan_kernel(RecurProblem p) {
    constexpr bool kStaged = NDT <= 8;
    constexpr int kPitch = NDT * 16 + 4, kPieces = NDT * 4, kSwap = kPieces < 16 ? kPieces - 1 : 15;       // 16-byte pieces of a row
    __shared__ __attribute__((aligned(16))) float state[2][16 * kPitch];      // column by column
    __shared__ __attribute__((aligned(16))) f32x4_t rows[kStaged ? NDT : 1][kStaged ? 16 * kPieces : 1];    // piece c of row r at c ^ (r & kSwap)
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, lq = lane >> 4;
    const int col = blockIdx.y * 16 + l16, h = blockIdx.x, s = blockIdx.z;   // (a head's workgroups share an L2)
    const int dim = p.dim, vdim = p.vdim, dp = (dim + 15) / 16 * 16;
    const int c0 = p.seq_chunks[s], c1 = p.seq_chunks[s + 1];
    const int64_t n = static_cast<int64_t>(dim) * vdim, pitch = static_cast<int64_t>(p.heads) * n;
    const int64_t m_size = static_cast<int64_t>(dp) * dp, m_pitch = static_cast<int64_t>(p.heads) * m_size;
    float* slot = p.states + (static_cast<int64_t>(p.slots[s]) * p.heads + h) * n;
    float* cs = p.chunk_states + static_cast<int64_t>(h) * n;
    const int row = wave * 16 + lq * 4, k_tiles = dp / 16;
    const bool has_rows = wave * 16 < dp, zero = p.starts[s] == 0;
    const float* mr = p.chunk_trans + h * m_size + static_cast<int64_t>(has_rows ? wave * 16 : 0) * dp;
    // a chunk's matrix and contribution, in flight two chunks ahead (one, where the registers do not hold three matrices)
    constexpr int kAhead = kStaged ? 2 : 1;
    bool ok[4];
    f32x4_t cur, add[kAhead], m4[kAhead][NDT];
    int at[NDT], put[NDT];              // of load k: elements into the wave's rows, and where it goes in LDS
#pragma unroll
    for (int k = 0; k < NDT; ++k) {
        const int kk = min(k, k_tiles - 1), i = kk * kWave + lane, r = i / (dp / 4), c = i - r * (dp / 4);
        at[k] = kStaged ? i * 4 : l16 * dp + lq * 4 + kk * 16;
        put[k] = r * kPieces + (c ^ (r & kSwap));
    }
    // (addresses are held inside instead of loads being skipped: waits can count straight-line loads)
    int64_t from[4];
    auto fetch = [&](int c, f32x4_t& to_add, f32x4_t (&to)[NDT]) {
        c = min(c, c1 - 1);
#pragma unroll
        for (int r = 0; r < 4; ++r) to_add[r] = cs[c * pitch + from[r]];
#pragma unroll
        for (int k = 0; k < NDT; ++k) to[k] = *reinterpret_cast<const f32x4_t*>(mr + c * m_pitch + at[k]);
    };
    auto advance = [&](int c, f32x4_t& my_add, f32x4_t (&mine)[NDT]) {
        float* buf = state[(c - c0) & 1];
        *reinterpret_cast<f32x4_t*>(buf + l16 * kPitch + row) = cur;
        f32x4_t sum[2] = {my_add, f32x4_t{0.0f, 0.0f, 0.0f, 0.0f}};
        if constexpr (kStaged) {
#pragma unroll
            for (int k = 0; k < NDT; ++k) rows[wave][put[k]] = mine[k];
            fetch(c + 2, my_add, mine);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (ok[r]) cs[c * pitch + from[r]] = cur[r];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < NDT; ++k) {
            // (rows beyond dim are zero here, whatever stands in the matrix)
            const f32x4_t s4 = *reinterpret_cast<const f32x4_t*>(buf + l16 * kPitch + k * 16 + lq * 4);
            const f32x4_t m = kStaged ? rows[wave][l16 * kPieces + ((min(k, k_tiles - 1) * 4 + lq) ^ (l16 & kSwap))] : mine[k];
#pragma unroll
            for (int r = 0; r < 4; ++r) sum[r & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(m[r], s4[r], sum[r & 1], 0, 0, 0);
        }
        if constexpr (!kStaged) fetch(c + 1, my_add, mine);
        cur = sum[0] + sum[1];
#pragma unroll
        for (int r = 0; r < 4; ++r) cur[r] = ok[r] ? cur[r] : 0.0f;
    };
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        ok[r] = row + r < dim && col < vdim;
        from[r] = ok[r] ? static_cast<int64_t>(row + r) * vdim + col : 0;
        cur[r] = ok[r] && !zero ? slot[from[r]] : 0.0f;
    }
#pragma unroll
    for (int i = 0; i < kAhead; ++i) fetch(c0 + i, add[i], m4[i]);
    for (int c = c0; c < c1; c += kAhead) {
#pragma unroll
        for (int i = 0; i < kAhead; ++i)
            if (c + i < c1) advance(c + i, add[i], m4[i]);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
        if (ok[r]) slot[from[r]] = cur[r];
}

// ---- decoding: one new token per sequence ----
// A thread holds VEC columns of up to ROWS rows of the state, and sums of every SHARESth of them (2: in the order of twice the threads, so
// that a sequence's sums are the same whatever the launch).  Bound: the states' bytes, read and written once a step, past the caches' order of
// use (us, loads and stores in it / past it: 64 sequences of 64 heads of 128 x 64, 268 MB, 62.5 / 51.2, 8 of them 11.3 / 8.9, 128 112 / 97; the delta
// rule, 16 heads of 128 x 128, 23 sequences 15.2 / 13.1, 64 27.3 / 26.3, 128 71 / 52; a single sequence is the same; either alone gives a third).
// Asking for a thread's channels and taps together, beside the state or in front of it, spills (one sequence of the delta rule 9.2 / 9.8-10.3).
template <typename Elem, bool DELTA, int VEC, int ROWS, int SHARES>
__global__ __launch_bounds__(1024) void recur_step_kernel(RecurProblem p, int groups) {
    typedef typename Elem::storage S;
    typedef float vec_t __attribute__((ext_vector_type(VEC)));
    extern __shared__ __attribute__((aligned(16))) float lds[];
    __shared__ float red[2][16];
    const int dim = p.dim, vdim = p.vdim, threads = blockDim.x, waves = threads / kWave;
    const int cgs = vdim / VEC, sums = groups * SHARES;     // groups <= threads / cgs
    float* lo = lds;                           // [sums][vdim]
    float* lv = lo + sums * vdim;              // [vdim]
    float* lqv = lv + vdim;                    // [dim] q
    float* lk = lqv + dim;                     // [dim] k
    const int tid = threadIdx.x, h = blockIdx.x, s = blockIdx.y, share = p.heads / p.kv_heads, g = h / share;
    const int grp = tid / cgs, c = (tid - grp * cgs) * VEC;
    const int pos = p.starts[s], slot = p.slots[s];
    float* st = p.states + (static_cast<int64_t>(slot) * p.heads + h) * dim * vdim;
    vec_t x[ROWS];
#pragma unroll
    for (int u = 0; u < ROWS; ++u) {
        const int d = grp + u * groups;
        if (grp < groups && d < dim && pos > 0) x[u] = __builtin_nontemporal_load(reinterpret_cast<const vec_t*>(st + d * vdim + c));
        else x[u] = static_cast<vec_t>(0.0f);
    }
    const f32x2_t rate = decay_and_beta<Elem>(p, s, h);
    const float decay = exp2_fast(rate[0]), beta = rate[1];

    const int64_t row = static_cast<int64_t>(s) * p.stride;
    const int channels = 2 * p.kv_heads * dim + p.heads * vdim;
    S* ring = static_cast<S*>(p.ring) + static_cast<int64_t>(slot) * p.taps * channels;
    float q_sum = 0.0f, k_sum = 0.0f;
    for (int i = tid; i < 2 * dim + vdim; i += threads) {
        const bool is_q = i < dim, is_k = !is_q && i < 2 * dim;
        const int at = is_q ? g * dim + i : is_k ? g * dim + i - dim : h * vdim + i - 2 * dim;
        const int channel = is_q ? at : is_k ? p.kv_heads * dim + at : 2 * p.kv_heads * dim + at;
        const S now = static_cast<const S*>(is_q ? p.q : is_k ? p.k : p.v)[row + at];
        const float* w = p.conv_w + static_cast<int64_t>(channel) * p.taps;
        float y = p.conv_b != nullptr ? p.conv_b[channel] : 0.0f;
        for (int back = min(p.taps - 1, pos); back > 0; --back)
            y = fmaf(w[p.taps - 1 - back], Elem::load(ring[static_cast<int64_t>((pos - back) % p.taps) * channels + channel]), y);
        y = silu(fmaf(w[p.taps - 1], Elem::load(now), y));
        // the projection's own row of the ring is read by nobody in this step
        if (!(is_q || is_k) || h % share == 0) ring[static_cast<int64_t>(pos % p.taps) * channels + channel] = now;
        if (is_q) {
            lqv[i] = y;
            q_sum = fmaf(y, y, q_sum);
        } else if (is_k) {
            lk[i - dim] = y;
            k_sum = fmaf(y, y, k_sum);
        } else {
            lv[i - 2 * dim] = Elem::load(Elem::store(y));
        }
    }
    float q_scale = p.q_scale, k_scale = 1.0f;
    if (p.unit_eps > 0.0f) {
        q_sum = wave_sum(q_sum);
        k_sum = wave_sum(k_sum);
        if ((tid & 63) == 0) {
            red[0][tid >> 6] = q_sum;
            red[1][tid >> 6] = k_sum;
        }
    }
    __syncthreads();
    if (p.unit_eps > 0.0f) {
        q_sum = k_sum = 0.0f;
        for (int w = 0; w < waves; ++w) {
            q_sum += red[0][w];
            k_sum += red[1][w];
        }
        q_scale /= sqrtf(q_sum + p.unit_eps);
        k_scale /= sqrtf(k_sum + p.unit_eps);
    }
    vec_t u_new = static_cast<vec_t>(0.0f);
    if (grp < groups) {
#pragma unroll
        for (int j = 0; j < VEC; ++j) u_new[j] = lv[c + j];
    }
    if (DELTA) {
        vec_t sk[SHARES];
#pragma unroll
        for (int i = 0; i < SHARES; ++i) sk[i] = static_cast<vec_t>(0.0f);
#pragma unroll
        for (int u = 0; u < ROWS; ++u) {
            const int d = grp + u * groups;
            if (grp < groups && d < dim) {
                x[u] *= decay;
                sk[u % SHARES] += x[u] * (lk[d] * k_scale);
            }
        }
        if (grp < groups) {
#pragma unroll
            for (int i = 0; i < SHARES; ++i) *reinterpret_cast<vec_t*>(lo + (grp + i * groups) * vdim + c) = sk[i];
        }
        __syncthreads();
        if (grp < groups) {
            for (int w = 0; w < sums; ++w) u_new -= *reinterpret_cast<const vec_t*>(lo + w * vdim + c);
        }
        __syncthreads();
    }
    u_new *= beta;
    vec_t o[SHARES];
#pragma unroll
    for (int i = 0; i < SHARES; ++i) o[i] = static_cast<vec_t>(0.0f);
#pragma unroll
    for (int u = 0; u < ROWS; ++u) {
        const int d = grp + u * groups;
        if (grp < groups && d < dim) {
            if (!DELTA) x[u] *= decay;
            x[u] += u_new * (lk[d] * k_scale);
            o[u % SHARES] += x[u] * (lqv[d] * q_scale);
            __builtin_nontemporal_store(x[u], reinterpret_cast<vec_t*>(st + d * vdim + c));
        }
    }
    if (grp < groups) {
#pragma unroll
        for (int i = 0; i < SHARES; ++i) *reinterpret_cast<vec_t*>(lo + (grp + i * groups) * vdim + c) = o[i];
    }
    __syncthreads();
    float sum = 0.0f;
    for (int v = tid; v < vdim; v += threads) {
        float y = p.skip != nullptr ? p.skip[h] * lv[v] : 0.0f;
        for (int w = 0; w < sums; ++w) y += lo[w * vdim + v];
        lo[v] = y;                              // (column v is this thread's alone)
        sum = fmaf(y, y, sum);
    }
    float scale = 1.0f;
    if (DELTA) {
        sum = wave_sum(sum);
        if ((tid & 63) == 0) red[0][tid >> 6] = sum;      // (the unit vectors' sums were read before the last barriers)
        __syncthreads();
        sum = 0.0f;
        for (int w = 0; w < waves; ++w) sum += red[0][w];
        scale = 1.0f / sqrtf(sum / static_cast<float>(vdim) + p.eps);
    }
    for (int v = tid; v < vdim; v += threads) {
        float y = lo[v];
        if (DELTA) y *= scale * p.norm_w[v] * silu(Elem::load(static_cast<const S*>(p.gate)[row + h * vdim + v]));
        static_cast<S*>(p.out)[(static_cast<int64_t>(s) * p.heads + h) * vdim + v] = Elem::store(y);
    }
}

// ---- launches ----
template <typename Elem>
int launch_conv(const RecurProblem& p, hipStream_t s) {
    int head_lanes = 1;
    while (head_lanes * 4 < round_up(p.dim, 16)) head_lanes *= 2;
    auto units = [&](int tokens) { return 2 * ceil_div(p.kv_heads, kWave / head_lanes) + ceil_div(p.heads * p.vdim, kConvPiece) + ceil_div(tokens * p.heads, kWave); };
    auto grid = [&](int tokens) {
        return dim3(static_cast<unsigned>(p.n_chunks), static_cast<unsigned>(p.chunk_tokens / tokens), static_cast<unsigned>(ceil_div(units(tokens), 4)));
    };
    auto aligned = [](const void* ptr) { return reinterpret_cast<uintptr_t>(ptr) % (4 * sizeof(typename Elem::storage)) == 0; };
    const bool vec = p.dim % 4 == 0 && p.vdim % 4 == 0 && p.stride % 4 == 0 && aligned(p.q) && aligned(p.k) && aligned(p.v);
    // Where the waves of 16 tokens are few, four of them: the way of one token's channels is what a short prompt waits for, and the rows read
    // twice lie in L2 (us, 16 / 4 tokens a wave, heads of 128: 320 tokens 10.0 / 6.3, 1024 10.4 / 9.6, 3200 19.3 / 18.6, 8192 35.9 / 38.4; the whole
    // prefill of 24 heads of 64 x 64, 3505 tokens, 3066 waves of 16, 80.2 / 74.9, 7500, 6566, 114.6 / 117.8, 16 x 512, 7168, 97.7 / 101.3).
    const bool few = int64_t{p.n_chunks} * (p.chunk_tokens / kBlock) * units(kBlock) <= 6144;
    if (p.taps > 4) launch((recur_conv_kernel<Elem, kMaxTaps, false, kBlock>), grid(kBlock), dim3(256), 0, s, p, head_lanes);
    else if (vec && few) launch((recur_conv_kernel<Elem, 4, true, 4>), grid(4), dim3(256), 0, s, p, head_lanes);
    else if (vec) launch((recur_conv_kernel<Elem, 4, true, kBlock>), grid(kBlock), dim3(256), 0, s, p, head_lanes);
    else launch((recur_conv_kernel<Elem, 4, false, kBlock>), grid(kBlock), dim3(256), 0, s, p, head_lanes);
    return launch_status();
}

template <typename Elem, int NDT, bool DELTA, bool OUTPUT, int THREADS>
int launch_chunks(const RecurProblem& p, int tiles, int waves, int group, hipStream_t s) {
    const size_t parts = sizeof(uint16_t) * 2 * 3 * kBlock * (NDT * 16 + 8), whole = sizeof(float) * 2 * kBlock * (NDT * 16 + 4);
    constexpr bool kParts = chunk_parts(THREADS, NDT);
    const size_t keys = kParts ? parts : whole, queries = kParts && DELTA ? parts : whole;
    const size_t lds = keys + (OUTPUT ? queries : 0) + (DELTA && OUTPUT ? sizeof(float) * 2 * THREADS / kWave * kBlock : 0);
    const int rc = allow_lds(reinterpret_cast<const void*>(recur_chunk_kernel<Elem, NDT, DELTA, OUTPUT, THREADS>), lds);
    if (rc != 0) return rc;
    launch((recur_chunk_kernel<Elem, NDT, DELTA, OUTPUT, THREADS>),
           dim3(static_cast<unsigned>(p.n_chunks), static_cast<unsigned>(p.heads / group), static_cast<unsigned>(group > 1 ? 1 : ceil_div(tiles, waves))),
           dim3(static_cast<unsigned>(waves * kWave)), lds, s, p, group);
    return launch_status();
}

template <typename Elem, int NDT, bool DELTA, bool OUTPUT>
int size_chunks(const RecurProblem& p, hipStream_t s) {
    const int v_tiles = static_cast<int>(ceil_div(p.vdim, 16));
    const int tiles = v_tiles + (DELTA && !OUTPUT ? static_cast<int>(ceil_div(p.dim, 16)) : 0);
    // (a head's norm needs all of its columns in one workgroup; eight waves move the operands)
    if (DELTA && OUTPUT && tiles > 8) return launch_chunks<Elem, NDT, DELTA, OUTPUT, DELTA && OUTPUT ? 1024 : 512>(p, tiles, tiles, 1, s);
    if (!DELTA) {
        int group = std::max(1, 8 / v_tiles);         // heads that fill eight waves
        while (p.heads / p.kv_heads % group != 0) --group;
        if (group > 1) return launch_chunks<Elem, NDT, DELTA, OUTPUT, 512>(p, tiles, 8, group, s);
    }
    return launch_chunks<Elem, NDT, DELTA, OUTPUT, 512>(p, tiles, 8, 1, s);
}

template <typename Elem, bool DELTA, bool OUTPUT>
int dispatch_chunks(const RecurProblem& p, hipStream_t s) {
    if (p.dim <= 32) return size_chunks<Elem, 2, DELTA, OUTPUT>(p, s);
    if (p.dim <= 64) return size_chunks<Elem, 4, DELTA, OUTPUT>(p, s);
    if (p.dim <= 128) return size_chunks<Elem, 8, DELTA, OUTPUT>(p, s);
    return size_chunks<Elem, 16, DELTA, OUTPUT>(p, s);
}

template <bool DELTA>
int launch_scan(const RecurProblem& p, hipStream_t s) {
    const unsigned heads = static_cast<unsigned>(p.heads), seqs = static_cast<unsigned>(p.n_seqs);
    if (!DELTA) {
        launch(recur_scan_kernel, dim3(static_cast<unsigned>(ceil_div(p.dim * p.vdim, 256)), heads, seqs), dim3(256), 0, s, p);
        return launch_status();
    }
    const dim3 grid(heads, static_cast<unsigned>(ceil_div(p.vdim, 16)), seqs);
    if (p.dim <= 32) launch(recur_matrix_scan_kernel<2>, grid, dim3(2 * kWave), 0, s, p);
    else if (p.dim <= 64) launch(recur_matrix_scan_kernel<4>, grid, dim3(4 * kWave), 0, s, p);
    else if (p.dim <= 128) launch(recur_matrix_scan_kernel<8>, grid, dim3(8 * kWave), 0, s, p);
    else launch(recur_matrix_scan_kernel<16>, grid, dim3(16 * kWave), 0, s, p);
    return launch_status();
}

template <typename Elem, bool DELTA>
int prefill(const RecurProblem& p, hipStream_t s) {
    int rc = launch_conv<Elem>(p, s);
    if (rc != 0) return rc;
    int per_wave = kBlockHeads;
    while (p.heads / p.kv_heads % per_wave != 0) --per_wave;
    launch(recur_block_kernel<DELTA>, dim3(static_cast<unsigned>(p.n_chunks), static_cast<unsigned>(p.chunk_tokens / kBlock),
                                           static_cast<unsigned>(ceil_div(p.heads / per_wave, 4))), dim3(256), 0, s, p, per_wave);
    rc = launch_status();
    if (rc != 0) return rc;
    if (p.chunk_states != nullptr) {
        rc = dispatch_chunks<Elem, DELTA, false>(p, s);
        if (rc == 0) rc = launch_scan<DELTA>(p, s);
        if (rc != 0) return rc;
    }
    return dispatch_chunks<Elem, DELTA, true>(p, s);
}

template <typename Elem, bool DELTA, int VEC, int ROWS>
int launch_step(const RecurProblem& p, hipStream_t s) {
    const int cgs = p.vdim / VEC;
    // A workgroup that has a CU to itself is shorter with twice the waves and half the rows to each; more of them get in each other's way (us, 256 /
    // 512 threads: delta rule of 16 heads of 128 x 128, one sequence 9.2 / 8.3, 8 10.3 / 9.4, 16 11.8 / 11.4, 64 26.5 / 29.6; 64 heads of 128 x 64, one
    // 6.4 / 6.2, 4 7.2 / 6.8, 16 13.5 / 16.7; 1024 threads are slower everywhere), and so does a small state, whose sums over the waves are what it
    // takes (8 heads of 32 x 32, delta rule 7.2 / 8.0, of 64 x 64 7.2 / 7.5, 80 x 80 7.6 / 7.5; additive 32 x 32 5.0 / 5.4, 48 x 5 8.4 / 9.1).
    // Sums are taken in one order either way, so a sequence's state does not depend on how many others decode beside it: two sums to a thread cost
    // nothing but for the delta rule with values of 64 (64 heads, 16 sequences 16.3 / 16.9, 64 61.2 / 60.6).
    const int few = 256 / cgs;                               // groups of rows that 256 threads make
    const bool enough = few > 0 && ceil_div(p.dim, few) <= ROWS, large = p.dim * p.vdim >= 6400;
    const bool twice = enough && large && static_cast<int64_t>(p.heads) * p.n_seqs <= 256;
    int threads = enough && !twice ? 256 : 512;
    while (!enough && threads < 1024 && (threads / cgs == 0 || ceil_div(p.dim, threads / cgs) > ROWS)) threads *= 2;
    const int groups = !enough ? threads / cgs : twice ? 2 * few : few, shares = enough && large && !twice ? 2 : 1;
    const size_t lds = sizeof(float) * (static_cast<size_t>(groups) * shares * p.vdim + p.vdim + 2 * p.dim);
    const dim3 grid(static_cast<unsigned>(p.heads), static_cast<unsigned>(p.n_seqs)), block(static_cast<unsigned>(threads));
    if (shares == 2) launch((recur_step_kernel<Elem, DELTA, VEC, ROWS, 2>), grid, block, lds, s, p, groups);
    else launch((recur_step_kernel<Elem, DELTA, VEC, ROWS, 1>), grid, block, lds, s, p, groups);
    return launch_status();
}

template <typename Elem, bool DELTA>
int step(const RecurProblem& p, hipStream_t s) {
    return p.vdim % 4 == 0 ? launch_step<Elem, DELTA, 4, 16>(p, s) : launch_step<Elem, DELTA, 1, 64>(p, s);
}

}  // namespace

bool recur_supported(int heads, int kv_heads, int dim, int vdim, int taps) {
    return heads > 0 && heads <= 65535 && kv_heads > 0 && heads % kv_heads == 0 && dim > 0 && dim <= 256 && vdim > 0 && vdim <= 256 &&
           taps > 0 && taps <= kMaxTaps;
}

int launch_recur_prefill(const RecurProblem& p, hipStream_t s) {
    if (p.dtype == EM_DTYPE_BF16) return p.beta_in ? prefill<BF16Elem, true>(p, s) : prefill<BF16Elem, false>(p, s);
    return p.beta_in ? prefill<F32Elem, true>(p, s) : prefill<F32Elem, false>(p, s);
}

int launch_recur_step(const RecurProblem& p, hipStream_t s) {
    if (p.dtype == EM_DTYPE_BF16) return p.beta_in ? step<BF16Elem, true>(p, s) : step<BF16Elem, false>(p, s);
    return p.beta_in ? step<F32Elem, true>(p, s) : step<F32Elem, false>(p, s);
}

}  // namespace em
