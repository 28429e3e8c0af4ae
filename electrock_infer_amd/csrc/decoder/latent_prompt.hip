// Latent attention for long portions of a prompt, bf16: keys and values of every head are written out once by two
// matrix products over the latents of the context (keys [K, heads * dim], values transposed [heads * vdim, K]) and a
// tiled softmax attention runs on them.
//
// A workgroup takes 128 queries of one head, 32 per wave, or half as many where that leaves CUs without work.  Per tile of 64
// keys a wave computes S^T = K Q^T: a lane then holds, for one query, keys (lane / 16) * 4 + 0..3 of every 16.  Since a sum
// over keys may run in any order as long as both operands agree, these registers, rounded to bf16, are the second operand of
// O^T = V^T P^T as they are: the values only have to lie in LDS in the matching key order.  Nothing of the probabilities goes
// through LDS, the running maximum and sum of a query live in one register of its four lanes, and a lane's results are four
// neighbouring outputs.
#include "decoder.h"
#include "mma.h"

namespace em {
namespace {

constexpr int kTileKeys = 64;
constexpr float kLog2e = 1.4426950408889634f;

// DKT: 32-element steps of dim + rot; DVT: 16-element tiles of vdim; QT: 16-query tiles of a wave
template <int DKT, int DVT, int QT>
__global__ __launch_bounds__(256, 2) void latent_prompt_kernel(LatentPromptProblem p) {
    typedef Mma<BF16Elem> M;
    constexpr int kRowsPerWave = 16 * QT, kRows = 4 * kRowsPerWave;
    constexpr int LPK = DKT * 32 + 8, LPV = kTileKeys + 8;
    constexpr int kFetchK = kTileKeys * DKT * 4 / 256, kFetchV = DVT * 16 * (kTileKeys / 8) / 256;
    __shared__ __attribute__((aligned(16))) uint16_t Ks[kTileKeys * LPK];
    __shared__ __attribute__((aligned(16))) uint16_t Vs[DVT * 16 * LPV];
    const int h = blockIdx.x, seq = blockIdx.z;
    const int row0 = p.q_begin[seq], nq = p.q_begin[seq + 1] - row0;
    const int t0 = (static_cast<int>(gridDim.y) - 1 - static_cast<int>(blockIdx.y)) * kRows;  // long rows start first
    if (t0 >= nq) return;
    const int start = p.starts[seq];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, lq = lane >> 4;
    const int D = p.dim + p.rot;
    const int64_t k0 = p.k_begin[seq];
    const int n_tiles = (start + min(t0 + kRows, nq) + kTileKeys - 1) / kTileKeys;
    const int first_pos = start + t0 + wave * kRowsPerWave;      // of this wave's first query

    typename M::frag fq[QT][DKT];
#pragma unroll
    for (int j = 0; j < QT; ++j) {
        const int t = t0 + wave * kRowsPerWave + j * 16 + l16;
        const uint16_t* q = p.q + (row0 + static_cast<int64_t>(min(t, nq - 1))) * p.q_stride + h * D;
#pragma unroll
        for (int k = 0; k < DKT; ++k) {
            const int c = k * 32 + lq * 8;
            fq[j][k] = c < D ? M::load(q + c) : M::zero();
        }
    }

    typename M::frag rk[kFetchK], rv[kFetchV];
    auto fetch = [&](int tile) {
        const int64_t key0 = k0 + static_cast<int64_t>(tile) * kTileKeys;
#pragma unroll
        for (int i = 0; i < kFetchK; ++i) {
            const int e = tid + i * 256, key = e / (DKT * 4), c = (e % (DKT * 4)) * 8;
            rk[i] = M::zero();
            if (c < p.dim) rk[i] = M::load(p.k + (key0 + key) * p.k_stride + h * p.dim + c);
            else if (c < D) rk[i] = M::load(p.k_rot + (key0 + key) * p.k_rot_stride + (c - p.dim));
        }
#pragma unroll
        for (int i = 0; i < kFetchV; ++i) {
            const int e = tid + i * 256, d = e / (kTileKeys / 8), c = (e % (kTileKeys / 8)) * 8;
            rv[i] = d < p.vdim ? M::load(p.vt + (static_cast<int64_t>(h) * p.vdim + d) * p.v_stride + key0 + c) : M::zero();
        }
    };

    f32x4_t o[DVT][QT];
#pragma unroll
    for (int d = 0; d < DVT; ++d)
#pragma unroll
        for (int j = 0; j < QT; ++j) o[d][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    float m[QT], l[QT];   // m in units of log2; l: this lane's share
#pragma unroll
    for (int j = 0; j < QT; ++j) {
        m[j] = -INFINITY;
        l[j] = 0.0f;
    }
    const float c2 = p.scale * kLog2e;

    fetch(0);
    for (int tile = 0; tile < n_tiles; ++tile) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kFetchK; ++i) {
            const int e = tid + i * 256;
            store_frag<BF16Elem>(Ks + (e / (DKT * 4)) * LPK + (e % (DKT * 4)) * 8, rk[i]);
        }
#pragma unroll
        for (int i = 0; i < kFetchV; ++i) {
            // keys 8c .. 8c + 7 of a row: two groups of four, each at (group of four in its 16) * 8 + (16 in its 32) * 4
            const int e = tid + i * 256, d = e / (kTileKeys / 8), c = (e % (kTileKeys / 8)) * 8;
            const int in32 = c & 31, at = (c & 32) + ((in32 & 15) / 4) * 8 + (in32 / 16) * 4;
            u32x2_t w[2];
            __builtin_memcpy(w, &rv[i], 16);
            *reinterpret_cast<u32x2_t*>(Vs + d * LPV + at) = w[0];
            *reinterpret_cast<u32x2_t*>(Vs + d * LPV + at + 8) = w[1];
        }
        __syncthreads();
        if (tile + 1 < n_tiles) fetch(tile + 1);
        if (tile * kTileKeys > first_pos + kRowsPerWave - 1) continue;   // no key of this tile for this wave's queries

        f32x4_t s[4][QT];
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
            for (int j = 0; j < QT; ++j) s[n][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < DKT; ++k)
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                const typename M::frag fk = M::load(Ks + (n * 16 + l16) * LPK + k * 32 + lq * 8);
#pragma unroll
                for (int j = 0; j < QT; ++j) s[n][j] = M::mac(fk, fq[j][k], s[n][j]);
            }
        if (tile * kTileKeys + kTileKeys - 1 > first_pos) {
#pragma unroll
            for (int n = 0; n < 4; ++n)
#pragma unroll
                for (int j = 0; j < QT; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (tile * kTileKeys + n * 16 + lq * 4 + r > first_pos + j * 16 + l16) s[n][j][r] = -INFINITY;
        }
        typename M::frag fp[2][QT];   // [32-key step][query tile]
        float alpha[QT];
        bool same = true;
#pragma unroll
        for (int j = 0; j < QT; ++j) {
            float mx = -INFINITY;
#pragma unroll
            for (int n = 0; n < 4; ++n)
#pragma unroll
                for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[n][j][r]);
            mx = column_max(mx);
            // the scale may be negative or zero only in a configuration error: scores are ordered by s * scale, scale > 0
            const float mn = fmaxf(m[j], mx * c2);
            const float base = mn == -INFINITY ? 0.0f : mn;
            alpha[j] = __builtin_amdgcn_exp2f(m[j] - base);
            m[j] = mn;
            float sum = 0.0f;
#pragma unroll
            for (int n = 0; n < 4; ++n)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float e = __builtin_amdgcn_exp2f(fmaf(s[n][j][r], c2, -base));
                    sum += e;
                    fp[n >> 1][j][(n & 1) * 4 + r] = static_cast<__bf16>(e);
                }
            l[j] = l[j] * alpha[j] + sum;
            same = same && alpha[j] == 1.0f;
        }
        if (!__all(same)) {
#pragma unroll
            for (int d = 0; d < DVT; ++d)
#pragma unroll
                for (int j = 0; j < QT; ++j) o[d][j] *= alpha[j];
        }
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int d = 0; d < DVT; ++d) {
                const typename M::frag fv = M::load(Vs + (d * 16 + l16) * LPV + k * 32 + lq * 8);
#pragma unroll
                for (int j = 0; j < QT; ++j) o[d][j] = M::mac(fv, fp[k][j], o[d][j]);
            }
    }
    const float sk = p.sink[h] * kLog2e;
#pragma unroll
    for (int j = 0; j < QT; ++j) {
        l[j] = column_sum(l[j]);
        const float top = fmaxf(m[j], sk), w = __builtin_amdgcn_exp2f(m[j] - top);
        const float inv = w / (l[j] * w + __builtin_amdgcn_exp2f(sk - top));
        const int t = t0 + wave * kRowsPerWave + j * 16 + l16;
        if (t >= nq) continue;
        uint16_t* out = p.out + ((row0 + static_cast<int64_t>(t)) * p.heads + h) * p.vdim;
#pragma unroll
        for (int d = 0; d < DVT; ++d) {
            const int c = d * 16 + lq * 4;
            if (c < p.vdim) {
                const u32x2_t w2 = {pack_bf16(o[d][j][0] * inv, o[d][j][1] * inv), pack_bf16(o[d][j][2] * inv, o[d][j][3] * inv)};
                *reinterpret_cast<u32x2_t*>(out + c) = w2;
            }
        }
    }
}

template <int DKT, int DVT, int QT>
int launch_tiles(const LatentPromptProblem& p, int n_seqs, int max_q, hipStream_t s) {
    const dim3 grid(static_cast<unsigned>(p.heads), static_cast<unsigned>(ceil_div(max_q, 64 * QT)), static_cast<unsigned>(n_seqs));
    launch((latent_prompt_kernel<DKT, DVT, QT>), grid, dim3(256), 0, s, p);
    return launch_status();
}

// Below two workgroups of 128 queries to a CU, workgroups of 64: a workgroup's time is a chain of tiles, which is shorter with
// half the products and exponentials to a tile, and CUs without work take the other half (us, 128 / 64 queries, heads of
// 128 + 64: 48 workgroups, 300 tokens behind 1000, 53.5 / 35.2; 128, one prompt of 1024 42.8 / 29.1; 256, 2048 80 / 59 and
// 4 x 512 25.7 / 24.0; 384, 3072 123 / 88; 512, 4 x 1024 55.8 / 57.1, 4096 163 / 152, behind 4000 328 / 385; 1024, 8192
// 397 / 520; a little below 512, portions that end early in their last 128 queries lose: 480, 15 x 200, heads of 128 + 32 21.5 /
// 24.2).  Keys of up to 128 elements under values of more than 64 gain little from it, and only while the workgroups of 64 have a
// CU each (96 + 32, values of 128: 128, 1000 behind 1000 56.6 / 51.4; 256, 2 x 1000 behind 3000 107 / 126).  A query's sums keep
// their order either way.  (Eight waves, every other tile each four of them, are faster where workgroups of 64 are few, 300 tokens behind 1000
// 35.5 / 29.2, one prompt of 1000 28.6 / 23.7, but add up in an order that would then depend on the other portions; eight that share every tile's
// keys and value columns in the same order wait for each other twice a tile: 35.8, 28.6.)
template <int DKT, int DVT>
constexpr int64_t few_workgroups() { return DKT <= 4 && DVT > 4 ? 160 : 448; }

template <int DKT, int DVT>
int launch_prompt(const LatentPromptProblem& p, int n_seqs, int max_q, hipStream_t s) {
    if (ceil_div(max_q, 128) * p.heads * n_seqs < few_workgroups<DKT, DVT>()) return launch_tiles<DKT, DVT, 1>(p, n_seqs, max_q, s);
    return launch_tiles<DKT, DVT, 2>(p, n_seqs, max_q, s);
}

template <int DVT>
int dispatch_prompt(const LatentPromptProblem& p, int n_seqs, int max_q, hipStream_t s) {
    const int D = p.dim + p.rot;
    if (D <= 64) return launch_prompt<2, DVT>(p, n_seqs, max_q, s);
    if (D <= 96) return launch_prompt<3, DVT>(p, n_seqs, max_q, s);
    if (D <= 128) return launch_prompt<4, DVT>(p, n_seqs, max_q, s);
    if (D <= 192) return launch_prompt<6, DVT>(p, n_seqs, max_q, s);
    return launch_prompt<8, DVT>(p, n_seqs, max_q, s);
}

}  // namespace

// 16-byte pieces of a query, a key and a row of transposed values; registers bound the head sizes
bool latent_prompt_supported(int dim, int rot, int vdim) {
    return dim > 0 && dim % 8 == 0 && rot >= 0 && rot % 8 == 0 && dim + rot <= 256 && vdim > 0 && vdim % 4 == 0 && vdim <= 128;
}

int launch_latent_prompt(const LatentPromptProblem& p, int n_seqs, int max_q, hipStream_t s) {
    return p.vdim <= 64 ? dispatch_prompt<4>(p, n_seqs, max_q, s) : dispatch_prompt<8>(p, n_seqs, max_q, s);
}

}  // namespace em
