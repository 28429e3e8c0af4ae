// out[T, N] = act(x[T, K] w[N, K]^T) for decode batches and short prompts (up to several hundred rows), bf16 on the matrix units.
//
// A workgroup makes BM token rows x BN weight rows, a wave 16 x 16 pieces of it.  Both operands go from memory straight to LDS,
// 128 bytes of a row per step, in a ring of STAGES stages of which all but the one that is multiplied are in flight.
//
// Short prompts.  Bound: what a CU takes in.  Rows that L2 holds arrive at up to 125 bytes per ns and CU, whatever the width of the pieces,
// rows from beyond at 61 with all CUs, and the products and LDS reads of a step beside the copies cost another quarter (a step of 128 x
// 128 x 64, us: copies alone 0.26, products alone 0.23, all with operands in L2 0.36, weights from memory 0.45-0.52),
// so a tile is as large as still leaves every CU one, and K is split where the results may stay partial sums.  us, this / the
// library's product (and the kernel of its activation), weights from memory: 300 tokens, 6144 x 2048 squared ReLU 16.7 / 17.7 + 4.2,
// 2048 x 6144 parts 18.1 / 26.9, 2048 x 2048 parts 8.5 / 11.5, 4096 x 12288 parts 45.9 / 66.1, 2048 x 512 5.1 / 7.0; and a call
// costs the host 3 us instead of 20.
//
// Decode batches.  Bound: the weights' stream.  One tile of tokens, weights past the caches' order of use (non-temporal), and the
// ring keeps 54-72 KB per workgroup (120 in tiles of 64 x 128) in flight without a register, while the kernel of skinny_gemm.hip asks for a step's rows, waits and
// multiplies.  us, this / that one, weights from memory: 12288 x 4096, 23 tokens 20.1 / 25.5, one 18.9 / 22.8; 4096 x 12288 parts, 64 tokens
// 21.0 / 26.3, one 17.4 / 20.2; 2048 x 6144 parts, 64 tokens 9.4 / 12.7; gated 2 x 4096 x 2048, 64 tokens 10.9 / 14.5; 32000 x 4096
// float32, 64 tokens 43.0 / 53.0 (6.1 TB/s).  That one shares K out over a workgroup's waves and stays ahead where the rows are few and the
// results whole (3072 x 2048, one token 7.7 / 5.7).
//
// The sum of a result runs over K from a place that depends on its tile of columns (tiles side by side ask for different parts of their
// rows at a time), and on nothing else: tokens that are alike have the same results wherever they stand.  Tiles that share weight rows a
// little behind each other too, so that the first brings them into L2, would be 2 to 5 % of a few products (us, 300 x 2048 x 6144 parts 17.4 / 17.8,
// 1000 x 3072 x 2048 20.0 / 21.0, 1000 x 12288 x 4096 111.6 / 115) and lose as much of others (300 x 2048 x 2048 parts 8.2 / 7.7).
#include "decoder.h"
#include "mma.h"
#include "../lds_copy.h"

#include <type_traits>

namespace em {
namespace {

constexpr int kStepK = 64;               // elements of a row per stage: 128 bytes
constexpr int kXcds = 8;

template <int BM, int BN, int WAVES, int STAGES>
struct TileGeo {
    static constexpr int kXBytes = BM * kStepK * 2, kWBytes = BN * kStepK * 2, kStageBytes = kXBytes + kWBytes;
    static constexpr int kLdsBytes = STAGES * kStageBytes;
    // of a wave and stage; a copy is eight rows (where the tokens' do not go round, some are copied twice: every wave counts the same)
    static constexpr int kXPieces = BM / 8, kXCopies = (kXPieces + WAVES - 1) / WAVES, kWCopies = BN / 8 / WAVES, kCopies = kXCopies + kWCopies;
    static_assert(BM % 16 == 0 && BN % (8 * WAVES) == 0, "a copy is eight rows");
    static_assert((STAGES - 1) * kCopies < 64, "vmcnt counts to 63");
};

// at most min(stages, MOST) stages of this wave's copies still in flight
template <int COPIES, int MOST>
__device__ __forceinline__ void wait_stages(int stages) {
    if constexpr (MOST == 0) wait_dma<0>();
    else if (stages >= MOST) wait_dma<MOST * COPIES>();
    else wait_stages<COPIES, MOST - 1>(stages);
}

// `x_stride`, `w_stride`: elements from row to row.  ACT: 0 none, 1 squared ReLU, 2 silu(first half) * second half of w
// [2 N, K].  ONCE: one tile of tokens, so that the weights are read once.
template <int BM, int BN, int WAVES, int WM, int STAGES, int ACT, bool F32OUT, bool ONCE>
__global__ __launch_bounds__(WAVES * kWave, 2) void tile_gemm_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
                                                                  void* __restrict__ out, int64_t x_stride, int64_t w_stride, int T, int N, int K,
                                                                  int m_tiles, int n_tiles) {
    typedef TileGeo<BM, BN, WAVES, STAGES> G;
    typedef Mma<BF16Elem> M;
    constexpr int WN = WAVES / WM, MF = BM / 16 / WM, NF = BN / 16 / WN;      // fragments of a wave
    constexpr int kOutCols = ACT == 2 ? BN / 2 : BN;
    constexpr bool kMixed = ACT == 2 && NF % 2 != 0;             // a fragment holds eight columns of both halves, else two take turns
    constexpr int kPair = ACT == 2 && !kMixed ? 2 : 1;
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, lq = lane >> 4;
    const int wm = wave % WM, wn = wave / WM;
    // an XCD takes neighbouring tiles of one range of K, those of one column first: its L2 reads a weight row once, and the token rows
    // of few ranges
    const int splits = gridDim.y, tiles = m_tiles * n_tiles, all = tiles * splits, per_xcd = (all + kXcds - 1) / kXcds;
    const int id = blockIdx.y * gridDim.x + blockIdx.x, local = id / kXcds, item = id % kXcds * per_xcd + local;
    if (local >= per_xcd || item >= all) return;
    const int split = item / tiles, tile = item - split * tiles;
    const int nt = tile / m_tiles, mt = tile - nt * m_tiles, m0 = mt * BM, n0 = nt * kOutCols, steps = K / kStepK;
    const int s0 = static_cast<int>(static_cast<int64_t>(steps) * split / splits);
    const int nk = static_cast<int>(static_cast<int64_t>(steps) * (split + 1) / splits) - s0;

    // Copies of a stage: 16-byte piece c of LDS holds piece q ^ (u & 7) of the two-row group u = c / 16 (q = row & 1, piece).
    const uint16_t* src[G::kCopies];
#pragma unroll
    for (int i = 0; i < G::kCopies; ++i) {
        const bool is_x = i < G::kXCopies;
        const int c = (is_x ? (i * WAVES + wave) % G::kXPieces : (i - G::kXCopies) * WAVES + wave) * kWave + lane;
        const int u = c >> 4, q = (c & 15) ^ (u & 7), r = u * 2 + (q >> 3), piece = (q & 7) * 8;
        if (is_x) {
            src[i] = x + min(m0 + r, T - 1) * x_stride;
        } else {
            const int f = r / 16, e = r % 16;        // (rows beyond the last are read twice and not stored)
            const int64_t col = kMixed      ? min(n0 + f * 8 + e % 8, N - 1) + (e / 8) * static_cast<int64_t>(N)
                                : ACT == 2 ? min(n0 + f / 2 * 16 + e, N - 1) + (f & 1) * static_cast<int64_t>(N)
                                           : static_cast<int64_t>(min(n0 + r, N - 1));
            src[i] = w + col * w_stride;
        }
        src[i] += static_cast<int64_t>(s0) * kStepK + piece;
    }
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem)));
    const int rot = nt * 5 % nk;
    auto place = [&](int step) {         // elements into the range of K
        const int k = step + rot;
        return (k >= nk ? k - nk : k) * kStepK;
    };
    auto copy = [&](int i, int at, int slot) {
        const uint32_t to = lds0 + slot * G::kStageBytes + (i < G::kXCopies ? (i * WAVES + wave) % G::kXPieces * 1024
                                                                             : G::kXBytes + ((i - G::kXCopies) * WAVES + wave) * 1024);
        if (ONCE && i >= G::kXCopies) dma16_stream(src[i] + at, to);
        else dma16(src[i] + at, to);
    };
    f32x4_t acc[NF][MF];
#pragma unroll
    for (int n = 0; n < NF; ++n)
#pragma unroll
        for (int m = 0; m < MF; ++m) acc[n][m] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    int x_at[2], w_at[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int piece = (h * 4 + lq) ^ ((l16 >> 1) & 7), row = (l16 >> 1) * 256 + ((l16 & 1) * 8 + piece) * 16;
        x_at[h] = wm * MF * 2048 + row;
        w_at[h] = G::kXBytes + wn * NF * 2048 + row;
    }
    M::frag fx[2][MF], fw[2][NF];
    constexpr int kReads = NF + MF, kProducts = NF * MF;
    auto read_one = [&](int slot, int h, int r) {
        const uint8_t* s = smem + slot * G::kStageBytes;
        if (r < NF) fw[h][r] = *reinterpret_cast<const M::frag*>(s + w_at[h] + r * 2048);
        else fx[h][r - NF] = *reinterpret_cast<const M::frag*>(s + x_at[h] + (r - NF) * 2048);
    };
    // The products of half a stage.  Between them, in this order whatever the compiler would like: the reads of the half behind it and
    // (COPIES) the copies of the stage `at` into slot `to`.  Back to back either would hold the wave's products up.
    auto half = [&](auto copies, int h, int from, int at, int to) {
#pragma unroll
        for (int j = 0; j < kProducts; ++j) {
            const int n = j / MF, m = n % 2 == 0 ? j % MF : MF - 1 - j % MF;      // (neighbours share an operand)
#pragma unroll
            for (int i = (j * kReads + kProducts - 1) / kProducts; i < ((j + 1) * kReads + kProducts - 1) / kProducts; ++i) read_one(from, 1 - h, i);
            acc[n][m] = M::mac(fw[h][n], fx[h][m], acc[n][m]);
            if constexpr (decltype(copies)::value) {
#pragma unroll
                for (int i = j * G::kCopies / kProducts; i < (j + 1) * G::kCopies / kProducts; ++i) copy(i, at, to);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    for (int s = 0; s < STAGES && s < nk; ++s)
#pragma unroll
        for (int i = 0; i < G::kCopies; ++i) copy(i, place(s), s);
    wait_stages<G::kCopies, STAGES - 1>(nk - 1);
    block_barrier();
#pragma unroll
    for (int i = 0; i < kReads; ++i) read_one(0, 0, i);
    int slot = 0;
    auto advance = [&]() {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");         // this wave has read its own of the stage
        block_barrier();
    };
    constexpr std::true_type kWithCopies{};
    constexpr std::false_type kWithout{};
    int k = 0;
    for (; k + STAGES < nk; ++k) {
        half(kWithout, 0, slot, 0, 0);
        wait_dma<(STAGES - 2) * G::kCopies>();                     // the next stage has landed
        advance();
        const int next = slot + 1 == STAGES ? 0 : slot + 1;
        half(kWithCopies, 1, next, place(k + STAGES), slot);       // (into the slot that is free now)
        slot = next;
    }
    for (; k + 1 < nk; ++k) {
        half(kWithout, 0, slot, 0, 0);
        wait_stages<G::kCopies, STAGES - 2>(nk - 2 - k);
        advance();
        slot = slot + 1 == STAGES ? 0 : slot + 1;
        half(kWithout, 1, slot, 0, 0);
    }
    half(kWithout, 0, slot, 0, 0);
#pragma unroll
    for (int n = 0; n < NF; ++n)
#pragma unroll
        for (int m = 0; m < MF; ++m) acc[n][m] = M::mac(fw[1][n], fx[1][m], acc[n][m]);

    // element i of a fragment: token l16, column lq * 4 + i
#pragma unroll
    for (int m = 0; m < MF; ++m) {
        const int t = m0 + (wm * MF + m) * 16 + l16;
        const int64_t row = (static_cast<int64_t>(split) * T + t) * N;
#pragma unroll
        for (int n = 0; n < NF; n += kPair) {
            const int c = kMixed ? n0 + (wn * NF + n) * 8 + (lq & 1) * 4 : n0 + (wn * NF + n) / kPair * 16 + lq * 4;
            f32x4_t v = acc[n][m];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (ACT == 1) v[i] = fmaxf(v[i], 0.0f) * fmaxf(v[i], 0.0f);
                if (ACT == 2) v[i] = silu(v[i]) * (kMixed ? __shfl_xor(v[i], 32) : acc[n + kPair - 1][m][i]);
            }
            if (t >= T || (kMixed && lq >= 2)) continue;
            if (N % 4 == 0) {
                if (c >= N) continue;
                if (F32OUT) {
                    *reinterpret_cast<f32x4_t*>(static_cast<float*>(out) + row + c) = v;
                } else {
                    *reinterpret_cast<u32x2_t*>(static_cast<uint16_t*>(out) + row + c) = u32x2_t{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
                }
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (c + i >= N) continue;
                    if (F32OUT) static_cast<float*>(out)[row + c + i] = v[i];
                    else static_cast<uint16_t*>(out)[row + c + i] = f32_to_bf16_bits(v[i]);
                }
            }
        }
    }
}

template <int BM, int BN, int WAVES, int WM, int STAGES, int ACT, bool F32OUT>
int launch_one(const TileGemm& g, hipStream_t s) {
    typedef TileGeo<BM, BN, WAVES, STAGES> G;
    constexpr bool kOnce = BM < 64 || WAVES == 3 || BN == 32 || (BM == 64 && WM == 1);       // the forms of decode batches
    const auto kernel = tile_gemm_kernel<BM, BN, WAVES, WM, STAGES, ACT, F32OUT, kOnce>;
    const int rc = allow_lds(reinterpret_cast<const void*>(kernel), G::kLdsBytes);
    if (rc != 0) return rc;
    const int m_tiles = static_cast<int>(ceil_div(g.T, BM)), n_tiles = static_cast<int>(ceil_div(g.N, ACT == 2 ? BN / 2 : BN));
    launch(kernel, dim3(static_cast<unsigned>(round_up(static_cast<int64_t>(m_tiles) * n_tiles, kXcds)), static_cast<unsigned>(g.splits)),
           dim3(WAVES * kWave), G::kLdsBytes, s, g.x, g.w, g.out, g.x_stride, g.w_stride, g.T, g.N, g.K, m_tiles, n_tiles);
    return launch_status();
}

template <int BM, int BN, int WAVES, int WM, int STAGES>
int launch_form(const TileGemm& g, hipStream_t s) {
    if (g.act == 2) return launch_one<BM, BN, WAVES, WM, STAGES, 2, false>(g, s);
    if (g.act == 1) return launch_one<BM, BN, WAVES, WM, STAGES, 1, false>(g, s);
    return g.f32 ? launch_one<BM, BN, WAVES, WM, STAGES, 0, true>(g, s) : launch_one<BM, BN, WAVES, WM, STAGES, 0, false>(g, s);
}

// The forms of a workgroup and what a step of theirs takes (us): where few CUs have one, where all have, and two on every CU (0:
// the ring leaves room for one).  Fitted, with what the rest of a launch takes, to 140 shapes of 65 to 1024 rows, 2048 to 16960
// weight rows and K of 512 to 12288: the form that the estimate picks takes 1.02 of the best one's time on the average; and of decode
// batches to 20 shapes of 1024 to 32000 rows with 1 to 64 tokens (1.01).
struct Form {
    int bm, bn;
    double few, all, two;
};
constexpr Form kPromptForms[] = {{64, 64, 0.219, 0.238, 0.41}, {128, 64, 0.318, 0.352, 0.60}, {64, 128, 0.303, 0.377, 0.0}, {128, 128, 0.452, 0.516, 0.0},
                                 {128, 256, 0.738, 0.843, 0.0}};
constexpr Form kDecodeForms[3][4] = {{{16, 32, 0.143, 0.143, 0.178}, {16, 48, 0.157, 0.157, 0.290}, {16, 64, 0.183, 0.183, 0.288}, {16, 128, 0.317, 0.317, 0.567}},
                                     {{32, 32, 0.156, 0.156, 0.253}, {32, 48, 0.184, 0.193, 0.364}, {32, 64, 0.204, 0.204, 0.363}, {32, 128, 0.340, 0.378, 0.630}},
                                     {{64, 32, 0.208, 0.208, 0.384}, {64, 48, 0.239, 0.240, 0.466}, {64, 64, 0.271, 0.271, 0.493}, {64, 128, 0.430, 0.471, 0.0}}};
// us; bytes per us: stores, weights from memory, further partial sums that the next kernel reads (the whole chip, or one CU a row)
constexpr double kLaunch = 3.0, kStoreRate = 3.3e6, kPromptStream = 5e6, kDecodeStream = 6e6, kAddRate = 5e6, kAddRow = 5.7e4;

double estimate(const Form& f, bool decode, int64_t T, int N, int64_t rows, int K, int splits, int out_bytes) {
    const int64_t groups = ceil_div(T, f.bm) * ceil_div(rows, f.bn) * splits, steps = ceil_div(K / kStepK, splits);
    const double one = f.few + (f.all - f.few) * static_cast<double>(groups < 256 ? groups : 256) / 256.0;
    const int64_t whole = groups / (f.two > 0 ? 512 : 256), rest = groups % (f.two > 0 ? 512 : 256);
    double us = static_cast<double>(whole * steps) * (f.two > 0 ? f.two : one);
    if (rest > 0) us += static_cast<double>(steps) * (rest <= 256 ? one : f.two);
    const double stream = static_cast<double>(rows) * K * 2 / (decode ? kDecodeStream : kPromptStream), stored = static_cast<double>(T) * N * out_bytes * splits;
    const double add = splits == 1 ? 0.0 : decode ? splits * (N * 4.0 / kAddRow + 0.1) : stored * (1.0 - 0.5 / splits) / kAddRate;
    return kLaunch + (us > stream ? us : stream) + (decode ? 0.35 : 0.1) * (us > stream ? stream : us) + stored / kStoreRate + add;
}

struct Plan {
    int form, splits;
    double us;
};
Plan plan(int64_t T, int N, int K, int act, bool f32, int least, int most) {
    Plan best{0, least, 1e30};
    const bool decode = T <= 64;
    const Form* forms = decode ? kDecodeForms[T <= 16 ? 0 : T <= 32 ? 1 : 2] : kPromptForms;
    for (int splits = least; splits <= most; ++splits) {
        if (splits > least && K / kStepK < 2 * splits) break;
        for (int i = 0; i < (decode ? 4 : 5); ++i) {
            const double us = estimate(forms[i], decode, T, N, act == 2 ? 2 * static_cast<int64_t>(N) : N, K, splits, f32 ? 4 : 2);
            if (us < best.us) best = Plan{i, splits, us};
        }
    }
    return best;
}

}  // namespace

bool tile_gemm_supported(int64_t T, int N, int K) {
    return T > 0 && T <= kTileGemmRows && N > 0 && N <= (1 << 28) && T * N <= (int64_t{1} << 40) && K > 0 && K % kStepK == 0;
}

namespace {
// Where a decode batch is faster this way than by the weight-streaming kernel, which shares K out over a workgroup's waves and so
// makes twice as many, smaller pieces, and than by the library (11 sizes of 1024 to 32000 rows, K of 512 to 12288, T of 1 to 64; this /
// the better of the two: 0.74 to 0.90 of its time beyond 8192 rows, 0.90 for partial sums with the norm behind them):
//   * results stay partial sums, unless K leaves no steps to share out (4096 x 512, one token 7.3 / 6.7 us, 64 tokens 8.2 / 8.5) or up
//     to 16 tokens take a few MB (in a step of one token 2048 x 2048 and x 4096 5.6 / 5.0 on the average);
//   * or the rows are a CU's worth of tiles: 6144 (6144 x 4096, T = 17 13.6 / 14.6, one 12.6 / 12.9; 4096 x 4096, T = 17 11.9 / 9.8), which a
//     short K (8192 x 1024, T = 16 9.1 / 8.6) or a gate (its fragments mix both halves: 8192 x 4096, one token 14.9 / 14.3, T = 32 15.7 / 16.4) moves up.
bool decode_pays(int64_t T, int64_t rows, int K, int act, bool parts) {
    if (parts) return K >= 1024 && (T > 16 || rows * K > (int64_t{1} << 23));
    if (act == 2) return (rows >= 10240 && K >= 1024) || (rows >= 8192 && T > 8 && K > 1024) || (rows >= 6144 && T > 32);
    return rows > 8192 || (rows >= 6144 && (T > 32 || (K > 1024 && (T > 4 || rows >= 8192))));
}
// Whole results of more tokens than a short prompt's, for `rows` weight rows (x and weights as the kernels before leave them; this /
// library's time over 12 widths of 72 to 1536 rows, 1030 to 16384 tokens):
//   * K up to 512: 0.5 to 1.0 up to 8192 tokens (T = 16384 1.05 to 1.36, 1536 rows and 3072 tokens 1.10 to 1.19); where the rows are the
//     many, up to 1536 x 2048 0.77 to 0.98 (1280 x 4096 1.13, x 8192 1.38);
//   * K = 1024: 0.7 to 0.9 for a million results or up to 2048 tokens (512 rows, 4096 tokens 1.29; 1024 rows 1.19);
//   * K = 1536, 2048: 0.6 to 0.85 for 128 to 192 rows and 3072 or 4096 tokens, else the library's tiles are as fast (256 to 512 rows, 4096
//     tokens 1.10 to 1.47), and beyond they are faster (K = 4096, 512 rows, 4096 tokens 1.61);
//   * with an activation, whose kernel is saved, 0.4 to 0.95 (384 to 640 rows of K = 2048, 3072 and more tokens 1.0 to 1.25).
bool prompt_pays(int64_t T, int64_t rows, int K, int act) {
    const int64_t results = T * rows;
    if (act != 0) return K <= 512 ? T <= 16384 : K <= 1024 ? T <= 8192 : K <= 2048 && T <= 8192 && (results <= (1 << 20) || rows > 640);
    if (rows > T) return (K <= 512 && results <= 3 << 20) || (K <= 1024 && results <= 2 << 20);
    if (K <= 512) return T <= 8192 && (rows < 1536 || T <= 2048);
    if (K <= 1024) return (T <= 2048 && rows < 1536) || (T <= 8192 && results <= 1 << 20);
    return K <= 2048 && rows > 96 && rows <= 192 && T >= 3072 && T <= 4096;
}

}  // namespace

// Where this is the faster way (and the host's 15 us a call come on top): up to as many rows as the library needs for tiles of
// 256 x 256 that leave no CU without one, which depends on the weights' size.  us, this / library: 2048 x 2048, 1024 rows
// 14.2 / 16.2; 8192 x 2048 500 rows 23.0 / 25.3, 700 31.6 / 28.5; 6144 x 4096 300 rows 28.5 / 29.7, 420 33.6 / 31.8; 12288 x 4096 200 rows
// 37.0 / 40.1, 300 51.3 / 50.3.  An activation saves the kernel behind the library's product (12288 x 4096, 512 rows 58.1 / 51.7 + 6.5); partial sums
// fill the chip where rows and weights are few (4096 x 8192, 512 rows 42.8 / 52.6, 700 60.4 / 54.8; 2048 x 6144, 1024 rows 36.4 / 40.8).
// Over 1024 to 16384 weight rows, K of 512 to 12288 and 65 to 1024 tokens 0.84 of the library's time on the average, 0.71 with an activation,
// 0.87 for partial sums with the norm behind them; single shapes, where the library's tiles happen to fit, up to 1.2 (3072 x 2048, 384
// tokens 1.20; partial sums 1536 x 4096, 896 tokens 1.25).
//   * Beyond 256 tokens no more results than its tiles take in a few rounds (K = 512, 16384 rows, 640 tokens 1.46, 896 1.39; K = 1024, 8192 rows,
//     640 tokens 1.24, 12288 rows, 300 tokens 1.19; with an activation K = 1024, 16384 rows, 640 tokens 1.30), and no square of 3072 and more
//     (4096 x 4096, 65 to 100 tokens 1.2, 300 to 512 1.06 to 1.26).
//   * Rows that are no multiple of four are stored value by value: 2048 tokens, K = 512 511 rows 0.78, 1001 0.94, 1301 1.10; 300 tokens, 4098
//     x 2048 1.18, partial sums of 2050 x 2048 1.36.
//   * No partial sums for more tokens than the estimate was fitted to, or for fewer rows: the end of a layer with a token input takes whole
//     results in one launch (128 rows of K = 1024, 4096 tokens, two ranges and four launches 26.7, library and one launch 19.0).
bool tile_gemm_pays(int64_t T, int N, int K, int act, bool parts) {
    if (!tile_gemm_supported(T, N, K)) return false;
    const int64_t rows = act == 2 ? 2 * static_cast<int64_t>(N) : N;
    if (T <= 64) return decode_pays(T, rows, K, act, parts);
    const int64_t few = T < rows ? T : rows, many = T < rows ? rows : T, size = many * K;
    if (few <= 64 || many < 1024) return false;
    if (N % 4 != 0 && (parts ? T > 128 : T * N > (int64_t{1} << (act == 0 ? 30 : 32)) / K)) return false;
    if (parts && (T > 1024 || N < 1024)) return false;
    if (parts) return K >= 512 && (few <= 512 || (few <= 1024 && many <= 2048 && size <= (int64_t{1} << 24)));
    if (K > many || (K == many && K > 2048) || (T > 1024 && !prompt_pays(T, rows, K, act))) return false;
    if (few > 256 && T <= 1024 && T * rows > (act != 0 ? int64_t{1} << 23 : int64_t{7} << 19)) return false;
    if (act != 0) return few <= (size <= (int64_t{1} << 24) ? 1024 : size <= (int64_t{1} << 26) ? 512 : 96);
    return few <= (size <= (int64_t{1} << 21) ? 1536 : size <= (int64_t{1} << 23) ? 1024 : size <= (int64_t{1} << 24) ? 512 :
                   size <= (int64_t{1} << 25) ? 320 : size <= (int64_t{1} << 26) ? 224 : 96);
}

// (33 to 64 tokens and rows that are about a CU's worth of tiles: two ranges, where the estimate sees no difference.  us with the norm that
// adds them up, 64 tokens, one / two: 6144 x 1024 13.5 / 12.8, 8192 x 1024 14.8 / 14.6, 8192 x 2048 18.4 / 17.4; 33 tokens 12.8 / 11.6,
// 14.0 / 13.1, 17.0 / 15.6; 10240 x 1024, 64 tokens 13.9 / 16.5)
int tile_gemm_splits(int64_t T, int N, int K) { return plan(T, N, K, 0, true, T > 32 && T <= 64 && N <= 8192 ? 2 : 1, 8).splits; }

int launch_tile_gemm(const TileGemm& g, hipStream_t s) {
    const int form = plan(g.T, g.N, g.K, g.act, g.f32, g.splits, g.splits).form;
    if (g.T <= 16) {
        switch (form) {
            case 0: return launch_form<16, 32, 2, 1, 10>(g, s);
            case 1: return launch_form<16, 48, 3, 1, 10>(g, s);
            case 2: return launch_form<16, 64, 4, 1, 8>(g, s);
            default: return launch_form<16, 128, 4, 1, 4>(g, s);
        }
    }
    if (g.T <= 32) {
        switch (form) {
            case 0: return launch_form<32, 32, 4, 2, 10>(g, s);
            case 1: return launch_form<32, 48, 3, 1, 8>(g, s);
            case 2: return launch_form<32, 64, 4, 1, 6>(g, s);
            default: return launch_form<32, 128, 4, 1, 4>(g, s);
        }
    }
    if (g.T <= 64) {
        switch (form) {
            case 0: return launch_form<64, 32, 4, 2, 6>(g, s);
            case 1: return launch_form<64, 48, 3, 1, 5>(g, s);
            case 2: return launch_form<64, 64, 4, 1, 5>(g, s);
            default: return launch_form<64, 128, 4, 1, 6>(g, s);
        }
    }
    switch (form) {
        case 0: return launch_form<64, 64, 4, 2, 4>(g, s);
        case 1: return launch_form<128, 64, 4, 2, 3>(g, s);
        case 2: return launch_form<64, 128, 8, 2, 6>(g, s);
        case 3: return launch_form<128, 128, 8, 2, 5>(g, s);
        default: return launch_form<128, 256, 8, 2, 3>(g, s);
    }
}

}  // namespace em
