// Projection over a middling number of activation rows (prompts of some tens to some thousand positions) on the matrix
// cores, with bf16 weights: the tiled projection of gemm_tiles.h with a quarter of its output tile, for launches whose
// 256 x 256 tiles would leave most CUs idle, and with key slices where even 128 x 128 tiles do.
//
// It reads the activation rows in the staging layout of gemm_tiles.h (bf16 hi + lo in fragment order, written by
// prepare_rows or by the launch that produced them) and the weights as stored, with the same operand roles and the same
// two MFMAs per product.  Work-group: eight waves, 128 weight rows x 128 activation rows.  Wave (kw, wn, wm) owns 64 x 64
// of them over every second 32-wide k step (kw): four waves' tiles cover the output, so each fragment that is read
// from LDS meets four MFMA pairs, and two waves per SIMD that wait at different points still keep the matrix cores fed.
// The two halves of the k steps are added when the tile is finished, through LDS.
//
// Operands reach LDS by the 16-byte global->LDS DMA, one k pair (64) a buffer (weights 16 KB in whole 128-byte lines,
// XOR-swizzled as in gemm_tiles; activations 32 KB), three buffers: a pair's DMAs are issued two pairs before its
// products.  With key slices (gridDim.y) the work-group leaves raw partial dots, and its slice's share of the row sums of
// squares, for gemm_reduce.
//
// What bounds it: with the device full, the L2->LDS traffic (48 KB per k pair and work-group, 13.7 TB/s over the chip): a
// pair takes 0.9 us against 0.45 us of products.  Deeper rings with a stream per wave (four pairs of weights and three of
// activations, or five and two) and fragments read a pair ahead of their products changed that by -10 to +2%, so neither
// is there.  The smallest launches are round trips (7 us for a single pair).  Measured on MI355X (the launches that it
// replaces: gemm_rows 64 rows at a time with its reduces, gemm_tiles with most CUs idle), us with the split pass and the
// reduce: 200 rows 2048 -> 3072 55.7 -> 26.1, 2048 -> 11264 107 -> 37.6, 5632 -> 2048 67.4 -> 28.2;
// 1013 rows 4096 -> 4096 155 -> 71, 14336 -> 4096 496 -> 222.
#pragma once

#include "kernels/gemm_tiles.h"

namespace dlk::mid {

using gemm::bf16x4;
using gemm::bf16x8;
using gemm::f32x4;
using gemm::kTile;
using gemm::f32x2;
typedef f32x2 f32x2_any __attribute__((aligned(4)));
constexpr int kThreads = 512;
constexpr int kWaves = kThreads / kWave;
constexpr int kBN = 128, kBM = 128;          // weight rows x activation rows per work-group
/// Fewest rows: gemm_rows takes up to 64 in one launch (65 rows of 2048 -> 2048: 21.8 us in two, 18.3 here; the token loop
/// over 65 sequences, whose repacked weights gemm_rows reads and this kernel does not, 36.0 -> 29.2 ms for 16 steps at 1B
/// widths, over 256 95.1 -> 42.7; four 8B layers over 65 19.6 -> 15.3, over 256 40.9 -> 27.0).
constexpr int kMinRows = gemm::kMaxRows + 1;
constexpr int kStages = 3;                   // k pairs in LDS
constexpr int kWeightBytes = kBN * 128;      // one k pair of weight fragments
constexpr int kActBytes = kBM / kTile * 4096; // one k pair of activation fragments (two steps of hi, lo)
constexpr int kOutStride = kBN + 4;          // floats per row of the finished tile in LDS (bank spread)
constexpr int kDma = 6;                      // DMA instructions per wave and pair: two of weights, four of activations
static_assert(kStages * (kWeightBytes + kActBytes) <= 160 * 1024 &&
                  (2 * kBM * kOutStride + kBM) * 4 <= kStages * (kWeightBytes + kActBytes), "LDS");

/// 16-row weight tiles (SwiGLU: gate tiles).
__host__ __device__ inline int tiles_of(const dlk_gemv_params& p) {
    return p.epilogue == DLK_EPI_SWIGLU ? p.seg_rows[0] / kTile : gemm::tiles_of(p);
}
__host__ __device__ inline int col_blocks(const dlk_gemv_params& p) {
    const int per = kBN / kTile / (p.epilogue == DLK_EPI_SWIGLU ? 2 : 1);
    return (tiles_of(p) + per - 1) / per;
}
__host__ __device__ inline int row_blocks(const dlk_gemv_params& p) { return (p.M + kBM - 1) / kBM; }

/// Key slices: as many as keep the launch within one work-group per CU, of at least four k pairs each.  Measured on
/// MI355X at 200 rows (us, with the reduce): at most 256 / 192 / 128 work-groups, 2048 -> 2048 and 5632 -> 2048 on average
/// 22.4 / 23.6 / 25.8, QKV 2048 -> 3072 23.1 / 24.2 / 27.3; gate/up of 128 rows (88 work-groups) 34 in one slice, 29 in two.
inline int splits_of(const dlk_gemv_params& p) {
    const int blocks = col_blocks(p) * row_blocks(p);
    return std::max(1, std::min({256 / blocks, gemm::kMaxSplits, p.K / 64 / 4}));
}
inline int64_t split_floats(const dlk_gemv_params& p) { // the layout that gemm_reduce reads
    const int splits = splits_of(p);
    return splits <= 1 ? 0 : static_cast<int64_t>(splits) * p.M * (gemm::tiles_of(p) * kTile + 1);
}

/// Whether this kernel takes the shape (host side): the conditions of the tiled projection without its row count.
inline bool shape_eligible(const dlk_gemv_params& p) {
    auto aligned = [](const void* at, uintptr_t bytes) { return reinterpret_cast<uintptr_t>(at) % bytes == 0; };
    if (!p.w_bf16 || p.epilogue == DLK_EPI_LOGITS || p.K % 64 != 0 || p.M < kMinRows) return false;
    if (p.ldx % 4 != 0 || !aligned(p.x, 16)) return false;
    if (p.apply_norm && p.norm_weight && !aligned(p.norm_weight, 16)) return false;
    for (int s = 0; s < p.nseg; ++s) {
        if (!aligned(p.w[s], 16)) return false;
        if (p.seg_rows[s] % kTile != 0) return false;
    }
    if (p.epilogue == DLK_EPI_SWIGLU && (p.ldy % 4 != 0 || !aligned(p.y, 16))) return false;
    // four head-dim entries of one head per store
    if (p.epilogue == DLK_EPI_QKV && (p.head_dim % 4 != 0 || p.ldy % 4 != 0 || !aligned(p.y, 16) || !aligned(p.k_cache, 16) ||
                                      !aligned(p.v_cache, 16)))
        return false;
    return static_cast<int64_t>(kTile) * p.K * 2 < (int64_t(1) << 31); // 32-bit DMA lane offsets
}

// Weight rows of work-group tile T: its segment and first row.
struct Tile {
    int seg, n0;
    const uint16_t* base;
};
template <bool SWIGLU>
__device__ __forceinline__ Tile locate(const dlk_gemv_params& p, int n_blk, int T, int tiles) {
    if constexpr (SWIGLU) {
        const int f = kTile * min(n_blk * (kBN / kTile / 2) + T % (kBN / kTile / 2), tiles - 1);
        return {0, f, static_cast<const uint16_t*>(p.w[T < kBN / kTile / 2 ? 0 : 1])};
    } else {
        const gemm::TileMap tm = gemm::locate<false>(p, min(n_blk * (kBN / kTile) + T, tiles - 1));
        return {tm.seg, tm.n0, tm.base0};
    }
}

// Waits until at most N DMAs of this wave are in flight and its LDS reads are done (the next barrier hands the buffer that
// they read to the DMAs of another pair).
template <int N>
__device__ __forceinline__ void wait_pair() {
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));
}

template <int EPI, bool NORM>
__global__ __launch_bounds__(kThreads, 2) void gemm_mid(const dlk_gemv_params p) {
    constexpr bool SWIGLU = EPI == DLK_EPI_SWIGLU;
    __shared__ __attribute__((aligned(1024))) char ring[kStages][kWeightBytes + kActBytes];

    const int t = threadIdx.x, lane = t % kWave, q = lane / 16, r = lane % 16;
    const int wave = __builtin_amdgcn_readfirstlane(t / kWave), kw = wave / 4, wn = wave & 1, wm = (wave >> 1) & 1;
    const int K = p.K, nsteps = K / 32, tiles = tiles_of(p);
    // consecutive work-group ids go to the 8 XCDs in turn: each XCD takes a run of the row-block-fastest order of one key
    // slice, so that the work-groups it runs at once share weight and activation blocks in its L2
    const int mb = row_blocks(p), nb = col_blocks(p), splits = gridDim.y;
    const int total = gridDim.x * splits, per = total / 8, rem = total % 8;
    const int id = blockIdx.x + gridDim.x * blockIdx.y, xcd = id % 8;
    const int logical = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + id / 8;
    const int m_blk = logical % mb, n_blk = logical / mb % nb, slice = logical / (mb * nb);
    const int m_first = m_blk * kBM;
    const int pairs = K / 64, pair0 = static_cast<int>(static_cast<int64_t>(pairs) * slice / splits);
    const int npairs = static_cast<int>(static_cast<int64_t>(pairs) * (slice + 1) / splits) - pair0;

    // DMA: wave w fills weight tile w (two halves of 8 rows x 128 bytes, row R's 16-byte column g at slot g ^ (R >> 1))
    // and activation tile w (4 KB: two k steps of hi and lo)
    const Tile mine = locate<SWIGLU>(p, n_blk, wave, tiles);
    const char* wbase = reinterpret_cast<const char*>(mine.base + static_cast<int64_t>(mine.n0) * K) + 128 * pair0;
    uint32_t woff[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int R = 8 * h + lane / 8;
        woff[h] = static_cast<uint32_t>(R) * K * 2 + 16 * ((lane % 8) ^ (R >> 1));
    }
    const char* xbase = static_cast<const char*>(p.stage) +
                        (static_cast<int64_t>(m_first / kTile + wave) * nsteps + 2 * pair0) * 2048;
    auto issue = [&](int pair, int buf) {
        const uint32_t w = lds_offset(ring[buf]) + wave * 2048, x = lds_offset(ring[buf]) + kWeightBytes + wave * 4096;
#pragma unroll
        for (int h = 0; h < 2; ++h) dma16(wbase + 128 * static_cast<int64_t>(pair), woff[h], w + 1024 * h);
#pragma unroll
        for (int h = 0; h < 4; ++h) dma16(xbase + 4096 * static_cast<int64_t>(pair) + 1024 * h, 16 * lane, x + 1024 * h);
    };

    f32x4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // a wave's weight tiles: generic four consecutive ones; SwiGLU two gate tiles, then the up tiles of their features
    auto slot = [&](int i) { return SWIGLU ? (i < 2 ? 2 * wn + i : 4 + 2 * wn + i - 2) : 4 * wn + i; };
    const uint32_t wfrag = (r / 8) * 1024 + (r % 8) * 128 + 16 * ((4 * kw + q) ^ (r >> 1));
    auto compute = [&](const char* buf) {
        bf16x8 a[4], bh[4], bl[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = *reinterpret_cast<const bf16x8*>(buf + slot(i) * 2048 + wfrag);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const char* frag = buf + kWeightBytes + (4 * wm + j) * 4096 + kw * 2048 + 16 * lane;
            bh[j] = *reinterpret_cast<const bf16x8*>(frag);
            bl[j] = *reinterpret_cast<const bf16x8*>(frag + 1024);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], bh[j], acc[i][j], 0, 0, 0);
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], bl[j], acc[i][j], 0, 0, 0);
            }
    };

    // Buffer b holds pair c (b = c % 3).  At step c the DMAs of pair c + 2 go into the buffer of pair c - 1, which every
    // wave finished before the last barrier; the wait before the next one leaves only them in flight, so pair c + 1
    // has landed.  Issues past the end repeat the last pair into a buffer that nobody reads again.
    issue(0, 0);
    issue(min(1, npairs - 1), 1);
    wait_vm<kDma>();
    tiles::ring_barrier();
    int buf = 0;
    for (int c = 0; c < npairs; ++c) {
        issue(min(c + 2, npairs - 1), buf == 0 ? 2 : buf - 1);
        compute(ring[buf]);
        wait_pair<kDma>();
        tiles::ring_barrier();
        buf = buf == 2 ? 0 : buf + 1;
    }
    wait_vm<0>();
    gemv::lds_barrier(); // the last DMAs have landed: the ring is free

    // The waves' tiles go to LDS as [k half][activation row][weight row], and every thread then finishes four consecutive
    // outputs of every fourth (SwiGLU: eighth) row (even k steps plus odd ones): whole 512-byte row pieces per 32
    // threads.  What the epilogue reads (norm factors, residual, rotation) is requested before.
    constexpr int OUTS = SWIGLU ? kBN / 2 : kBN; // outputs of the work-group per row
    constexpr int STRIDE = kThreads / (OUTS / 4), PASSES = kBM / STRIDE;
    float(*out)[kBM][kOutStride] = reinterpret_cast<float(*)[kBM][kOutStride]>(&ring[0][0]);
    float* inv_s = reinterpret_cast<float*>(&ring[0][0]) + 2 * kBM * kOutStride;
    const int rows = min(kBM, p.M - m_first);
    const int col = 4 * (t % (OUTS / 4)), T = col / kTile, row0 = t / (OUTS / 4); // this thread's outputs of its rows
    const int tile = n_blk * (OUTS / kTile) + T;
    const Tile tm = locate<SWIGLU>(p, n_blk, T, tiles);
    const int n = tm.n0 + col % kTile; // first weight row (feature) of the outputs
    const int64_t width = static_cast<int64_t>(gemm::tiles_of(p)) * kTile; // of a partial row
    const bool finish = splits == 1;
    const bool vec = p.ldy % 4 == 0 && reinterpret_cast<uintptr_t>(p.y) % 16 == 0 &&
                     (EPI != DLK_EPI_RESIDUAL || (p.ldres % 4 == 0 && reinterpret_cast<uintptr_t>(p.residual) % 16 == 0));
    f32x4 residual[PASSES];
    if constexpr (EPI == DLK_EPI_RESIDUAL) {
        if (finish && vec)
#pragma unroll
            for (int i = 0; i < PASSES; ++i)
                residual[i] = *reinterpret_cast<const f32x4*>(
                    p.residual + static_cast<int64_t>(min(m_first + row0 + i * STRIDE, p.M - 1)) * p.ldres + n);
    }
    f32x2 cosine[PASSES], sine[PASSES];
    uint32_t batch[PASSES];
    int64_t position[PASSES];
    if constexpr (EPI == DLK_EPI_QKV) {
        if (finish) {
            const int64_t first = *p.position;
            const uint32_t length = static_cast<uint32_t>(p.length);
#pragma unroll
            for (int i = 0; i < PASSES; ++i) {
                const uint32_t mg = static_cast<uint32_t>(p.m_base + min(m_first + row0 + i * STRIDE, p.M - 1));
                batch[i] = mg / length;
                position[i] = first + (mg - batch[i] * length);
                const int64_t at = position[i] * (p.head_dim / 2) + n % p.head_dim / 2;
                cosine[i] = *reinterpret_cast<const f32x2_any*>(p.cosine + at);
                sine[i] = *reinterpret_cast<const f32x2_any*>(p.sine + at);
            }
        }
    }
    const bool norm = NORM && p.apply_norm;
    if (norm && finish && t < kBM) inv_s[t] = tiles::stage_inv(p, min(m_first + t, p.M - 1));
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            *reinterpret_cast<f32x4*>(&out[kw][64 * wm + 16 * j + r][kTile * slot(i) + 4 * q]) = acc[i][j];
    gemv::lds_barrier();

    const float* hidden = tm.seg == 0 ? p.lora_hidden[0] : tm.seg == 2 ? p.lora_hidden[2] : nullptr;
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
        const int ml = row0 + i * STRIDE, m = m_first + ml;
        // SwiGLU with stage_out also writes the rows past M (copies of the staged rows there), as prepare_rows does
        if (tile >= tiles || (ml >= rows && !(SWIGLU && p.stage_out))) break;
        f32x4 v = *reinterpret_cast<const f32x4*>(&out[0][ml][col]) + *reinterpret_cast<const f32x4*>(&out[1][ml][col]);
        if (!finish) {
            // raw partial dots [slice][m][tile row]; SwiGLU tiles pair gate and up rows (gemm_reduce)
            if (SWIGLU && ml >= rows) break;
            float* part = p.split_partial + (static_cast<int64_t>(slice) * p.M + m) * width;
            if constexpr (SWIGLU) {
                const f32x4 up = *reinterpret_cast<const f32x4*>(&out[0][ml][OUTS + col]) +
                                 *reinterpret_cast<const f32x4*>(&out[1][ml][OUTS + col]);
                part += 2 * n; // (n / 8) * 16 + 2 (n % 8)
                *reinterpret_cast<f32x4*>(part) = f32x4{v[0], up[0], v[1], up[1]};
                *reinterpret_cast<f32x4*>(part + 4) = f32x4{v[2], up[2], v[3], up[3]};
            } else {
                *reinterpret_cast<f32x4*>(part + tile * kTile + col % kTile) = v;
            }
            continue;
        }
        const float scale = (norm ? inv_s[ml] : 1.0f) * p.acc_scale;
        if constexpr (SWIGLU) {
            const f32x4 up = *reinterpret_cast<const f32x4*>(&out[0][ml][OUTS + col]) +
                             *reinterpret_cast<const f32x4*>(&out[1][ml][OUTS + col]);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = gemv::silu(v[e] * scale) * (up[e] * scale);
            if (p.stage_out) {
                // the next launch's staging layout, split as prepare_rows would split the rows (see gemm_tiles)
                const bf16x4 h = __builtin_convertvector(v, bf16x4);
                const bf16x4 l = __builtin_convertvector(v - __builtin_convertvector(h, f32x4), bf16x4);
                char* at = static_cast<char*>(p.stage_out) + (static_cast<int64_t>(m / 16) * (p.seg_rows[0] / 32) + n / 32) * 2048 +
                           ((m % 16) + 16 * ((n % 32) / 8)) * 16 + (n % 8) * 2;
                *reinterpret_cast<bf16x4*>(at) = h;
                *reinterpret_cast<bf16x4*>(at + 1024) = l;
            } else {
                *reinterpret_cast<f32x4*>(p.y + static_cast<int64_t>(m) * p.ldy + n) = v;
            }
        } else if constexpr (EPI == DLK_EPI_QKV) {
            v *= scale;
            const int64_t mg = p.m_base + m;
            if (hidden) {
                // unmerged LoRA: + scale * up[n .. n + 4, :] . hidden[m, :]
                const void* up = tm.seg == 0 ? p.lora_up[0] : p.lora_up[2];
                const float* h = hidden + mg * gemv::lora_stride(p);
                float d[4];
                gemm::lora_pair(p, up, h, n, d[0], d[1]);
                gemm::lora_pair(p, up, h, n + 2, d[2], d[3]);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] += d[e] * p.lora_scale;
            }
            if (tm.seg < 2) {
                // interleaved pairs (src/ops/contraction.cpp:44-49)
                const f32x2 c = cosine[i], s = sine[i];
                v = f32x4{v[0] * c.x - v[1] * s.x, v[0] * s.x + v[1] * c.x, v[2] * c.y - v[3] * s.y, v[2] * s.y + v[3] * c.y};
            }
            if (tm.seg == 0) {
                *reinterpret_cast<f32x4*>(p.y + mg * p.ldy + n) = v;
            } else {
                const int64_t at = ((static_cast<int64_t>(batch[i]) * p.kv_heads + n / p.head_dim) * p.cache_capacity + position[i]) *
                                       p.head_dim + n % p.head_dim;
                void* cache = tm.seg == 1 ? p.k_cache : p.v_cache;
                if (p.cache_bf16)
                    *reinterpret_cast<uint2*>(static_cast<uint16_t*>(cache) + at) =
                        make_uint2(f32_to_bf16(v[0]) | (static_cast<uint32_t>(f32_to_bf16(v[1])) << 16),
                                   f32_to_bf16(v[2]) | (static_cast<uint32_t>(f32_to_bf16(v[3])) << 16));
                else
                    *reinterpret_cast<f32x4*>(static_cast<float*>(cache) + at) = v;
            }
        } else {
            v *= scale;
            const int at = n + (EPI == DLK_EPI_STORE ? gemv::seg_column(p, tm.seg) : 0);
            float* y = p.y + static_cast<int64_t>(m) * p.ldy + at;
            if (EPI == DLK_EPI_STORE && p.bias) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    v[e] += p.bias_bf16 ? bf16_to_f32(static_cast<const uint16_t*>(p.bias)[at + e])
                                        : static_cast<const float*>(p.bias)[at + e];
            }
            if (vec) {
                if constexpr (EPI == DLK_EPI_RESIDUAL) v += residual[i];
                *reinterpret_cast<f32x4*>(y) = v;
            } else {
                const float* res = EPI == DLK_EPI_RESIDUAL ? p.residual + static_cast<int64_t>(m) * p.ldres + n : nullptr;
#pragma unroll
                for (int e = 0; e < 4; ++e) y[e] = EPI == DLK_EPI_RESIDUAL ? v[e] + res[e] : v[e];
            }
        }
    }
    if (splits > 1) {
        // the first column block leaves its slice's share of the row squares
        if (NORM && n_blk == 0 && t < rows) {
            const float* squares = tiles::stage_squares(p);
            float sum = 0.0f;
            for (int c = slice; c < tiles::prep_chunks(K); c += splits) sum += squares[static_cast<int64_t>(c) * p.M + m_first + t];
            p.split_partial[splits * p.M * width + static_cast<int64_t>(slice) * p.M + m_first + t] = sum;
        }
        return;
    }
    if constexpr (EPI == DLK_EPI_STORE || EPI == DLK_EPI_RESIDUAL) {
        if (p.bump_position && id == 0 && t == 0) *p.bump_position += p.bump_count;
    }
}

/// The kernel of a launch; null if none.
template <int EPI>
const void* resolve(const dlk_gemv_params& p) {
    if (gemv::norm_variant(EPI, p.apply_norm != 0)) {
        if constexpr (EPI != DLK_EPI_RESIDUAL) return reinterpret_cast<const void*>(&gemm_mid<EPI, true>);
        return nullptr;
    }
    if constexpr (EPI == DLK_EPI_STORE || EPI == DLK_EPI_RESIDUAL) return reinterpret_cast<const void*>(&gemm_mid<EPI, false>);
    return nullptr;
}

} // namespace dlk::mid

const void* dlk_mid_kernel_store(const dlk_gemv_params& p);
const void* dlk_mid_kernel_residual(const dlk_gemv_params& p);
const void* dlk_mid_kernel_qkv(const dlk_gemv_params& p);
const void* dlk_mid_kernel_swiglu(const dlk_gemv_params& p);
