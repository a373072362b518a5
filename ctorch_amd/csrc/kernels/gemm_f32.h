// Projection over several activation rows on the f32 matrix cores, with the epilogues of the GEMV (see dlk_gemv_params in
// kernels.h): f32 weights, and bf16 weights of the shapes that no bf16 matrix-core kernel takes with whole f32 activations.
//
// One v_mfma_f32_16x16x4_f32 computes D[16 weight rows][16 activation rows] += W[16][4] * X[16][4]^T in f32: lane l
// supplies one weight of row l%16 and one activation of row l%16 at k slot l/16, and receives D[rows 4(l/16) .. +4]
// [l%16].  The k slots of four products are dealt so that a lane's operands are four consecutive k (k slot l/16 of
// product j is k 4(l/16) + j), so the fragments of 16 k are one 16-byte LDS read per tile.
//
// Work-group: four waves, WN x WM, each owning TN x TM tiles of 16 x 16.  Both operands are staged in LDS as f32,
// 32 k at a time, double buffered, the next chunk's loads in flight (in registers) while one is used.  A product rounds
// its sum after every k, so one accumulator over a long K would lose what the GEMV's 64 short sums keep (K = 4096:
// 1.1e-6 against 64-bit results, the GEMV 1.1e-7): each 16 k start from zero and are added up in f64 (the vector ALU
// has time for it beside the products), which leaves the same 8e-8 at every K.  The RMSNorm is
// fused: the staged rows are x * g, the sums of squares accumulate while staging, and the norm factor scales the
// finished dots.  A lane ends with four consecutive outputs of one activation row.
//
// What bounds it: many rows, the matrix cores (96 of 153 TFLOP/s, which a library product of 8192 x 8192 reaches, at
// 2000 x 4096 -> 16000); the small models' few hundred k per projection, the chunk round trips.  The GEMV, which took
// these launches before, streams the weights again for every one to four rows: 2040 rows of the tiny model (d 256,
// SwiGLU 688) were 510 launches a projection.  Measured on MI355X: 2000 x 4096 -> 16000 83.3 -> 2.7 ms, 500 x 2048 ->
// 8191 2742 -> 217 us, 12 x 4096 -> 16000 498 -> 45 us; a layer of the tiny model over those rows 11.1 -> 0.066 ms.
#pragma once

#include "kernels/gemm_rows.h"

namespace dlk::gemm32 {

using gemm::f32x4;
using gemm::kTile;
using gemv::u32x4;
typedef double f64x4 __attribute__((ext_vector_type(4)));
constexpr int kThreads = 256;
constexpr int kWaveChunk = 32;           // k per wave and staged chunk

/// Work-group shapes: weight rows x activation rows.  In the last one the four waves share one tile and split the k.
enum Shape { k128x128 = 0, k64x64, k64x32, k32x16 };
constexpr int shape_rows(int shape) { return shape == k128x128 ? 128 : shape == k32x16 ? 32 : 64; }
constexpr int shape_acts(int shape) { return shape == k128x128 ? 128 : shape == k64x64 ? 64 : shape == k64x32 ? 32 : 16; }

__host__ __device__ inline int segment_tiles(int rows) { return (rows + kTile - 1) / kTile; }
/// 16-row weight tiles of a launch (a segment's last tile may be partial; SwiGLU: tiles of the gate matrix).
__host__ __device__ inline int tiles_of(const dlk_gemv_params& p) {
    int t = segment_tiles(p.seg_rows[0]);
    if (p.epilogue == DLK_EPI_SWIGLU) return t;
    if (p.nseg > 1) t += segment_tiles(p.seg_rows[1]);
    if (p.nseg > 2) t += segment_tiles(p.seg_rows[2]);
    return t;
}
/// Work-groups over the weight rows (SwiGLU: half of a work-group's weight rows are gate rows, half up rows).
__host__ __device__ inline int col_blocks(const dlk_gemv_params& p, int rows) {
    const int per = rows / kTile / (p.epilogue == DLK_EPI_SWIGLU ? 2 : 1);
    return (tiles_of(p) + per - 1) / per;
}

/// Whether this kernel takes the launch (host side; bf16 weights: one that the kernels which split the activations into
/// two bf16 parts leave, see gemv.hip).
/// f32 weights: from the third launch that the GEMV would need, which takes one to four activation rows at a time (K >
/// 3072: one) and streams the weights again for each.
/// bf16 weights: over 65 rows and more, any width, K in whole pairs of k steps.  The activations stay whole as in the
/// GEMV (7.8e-8 against 64-bit results; the GEMV 0.7e-7 to 1.0e-7, two bf16 parts 2.5e-6), and the weights become f32 while
/// they are staged.  Measured on MI355X against the GEMV, us: 65 x 320 -> 640 97 -> 8.5, 100 x 4096 -> 8191 1113 -> 122,
/// 333 x 2048 -> 32001 3538 -> 532, 2000 x 4096 -> 15999 40617 -> 2612 (gemm_mid's two parts: 12, 55, 115, 553).
/// Fewer rows, other K and several segments that are no multiple of 16 were not measured and stay with the GEMV.
inline bool eligible(const dlk_gemv_params& p) {
    if (p.epilogue == DLK_EPI_LOGITS || p.K % (p.w_bf16 ? 64 : 4) != 0 || p.ldx % 4 != 0) return false;
    if (p.M <= (p.w_bf16 ? gemm::kMaxRows : 2 * gemv::plan_of(p.K, false, p.epilogue).mt_max)) return false;
    if (p.w_bf16)
        for (int s = 0; s < p.nseg; ++s)
            if (p.nseg == 1 ? p.seg_rows[s] < kTile : p.seg_rows[s] % kTile != 0) return false;
    auto aligned = [](const void* q, uintptr_t bytes) { return reinterpret_cast<uintptr_t>(q) % bytes == 0; };
    if (!aligned(p.x, 16)) return false;
    for (int s = 0; s < p.nseg; ++s)
        if (!aligned(p.w[s], 16) || p.seg_rows[s] <= 0) return false;
    if (p.apply_norm && p.norm_weight && !aligned(p.norm_weight, p.norm_bf16 ? 8 : 16)) return false;
    // rotated pairs and cache rows are stored two entries at a time
    if (p.epilogue == DLK_EPI_QKV && (p.ldy % 2 != 0 || !aligned(p.y, 8) || !aligned(p.k_cache, 8) || !aligned(p.v_cache, 8)))
        return false;
    return true;
}

inline int64_t blocks_of(const dlk_gemv_params& p, int shape) {
    return static_cast<int64_t>(col_blocks(p, shape_rows(shape))) * ((p.M + shape_acts(shape) - 1) / shape_acts(shape));
}

/// The largest work-group shape that gives each CU a few work-groups to hide one's loads behind another's products.
/// Measured on MI355X, us (128x128 / 64x64 / 64x32 / 32x16; work-groups in brackets), rows x k -> outputs:
/// 2000 x 4096 -> 16000: 2718 (2000) / 2912 / 3124 / 3805;  500 x 2048 -> 8191: 216 (256) / 217 (1024) / 234 / 293;
/// 300 x 2048 -> 16000: 345 (375) / 243 (1250) / 265 / 308;  2040 x 256 -> 1376: 30.1 (176) / 24.2 (704) / 25.5 / 34.9;
/// 150 x 2048 -> 16000: 189 / 150 (750) / 137 (1250) / 162;  300 x 4096 -> 4000: 367 / 214 (315) / 182 (630) / 176.
/// 2040 x 688 -> 256 (64x32: 256) 16.9 against 17.8, and with the norm's sums in every column block 256 -> 384 (384) 14.1
/// against 16.8.  With fewer work-groups than that a launch is a chain of chunk round trips, and waves that split the k make the
/// chain four times shorter: 510 x 688 -> 256: 64.9 / 22.4 / 16.4 (64) / 7.7 (256);  34 x 256 -> 1376: 25.7 / 10.7 / 7.8 /
/// 4.7;  9 x 4096 -> 250: 356 / 116 / 79 / 25.
inline int shape_of(const dlk_gemv_params& p) {
    if (blocks_of(p, k128x128) >= 1024) return k128x128;
    if (blocks_of(p, k64x64) >= 512) return k64x64;
    if (blocks_of(p, k64x32) >= 256) return k64x32;
    return k32x16;
}

// A tile of 16 weight rows: its segment, first row, rows of the segment.
struct Tile {
    int seg, n0, rows;
    const void* base;
};
__device__ __forceinline__ Tile locate(const dlk_gemv_params& p, int tile) {
    const int t0 = segment_tiles(p.seg_rows[0]), t1 = p.nseg > 1 ? segment_tiles(p.seg_rows[1]) : 0;
    if (tile < t0 || p.nseg == 1) return {0, tile * kTile, p.seg_rows[0], p.w[0]};
    if (tile < t0 + t1 || p.nseg == 2)
        return {1, (tile - t0) * kTile, p.seg_rows[1], p.w[1]};
    return {2, (tile - t0 - t1) * kTile, p.seg_rows[2], p.w[2]};
}

// WT: float, or uint16_t for bf16 weights.
template <typename WT, int EPI, bool NORM, int WN, int WM, int WK, int TN, int TM>
__global__ __launch_bounds__(kThreads) void gemm_f32(const dlk_gemv_params p) {
    constexpr bool SWIGLU = EPI == DLK_EPI_SWIGLU;
    constexpr int BN = kTile * WN * TN, BM = kTile * WM * TM;
    constexpr int kChunk = kWaveChunk * WK;          // k per staged chunk
    // floats per staged row: 32 bytes past a multiple of 128, whose 16-row fragment reads do not conflict
    constexpr int kStride = kChunk + 8;
    constexpr int kPieces = kChunk / 4;              // 16-byte pieces per staged row
    constexpr int kRowsPerPass = kThreads / kPieces;
    constexpr int VALUES = 16 / sizeof(WT);          // weights per 16-byte piece
    constexpr int kWeightPieces = kChunk / VALUES, kWeightRowsPerPass = kThreads / kWeightPieces;
    constexpr int WLOADS = BN / kWeightRowsPerPass, XLOADS = (BM + kRowsPerPass - 1) / kRowsPerPass;
    constexpr int FT = BN / kTile / 2; // SwiGLU: gate tiles of a work-group
    static_assert(WN * WM * WK * kWave == kThreads && BN % kWeightRowsPerPass == 0 && (!SWIGLU || TN % 2 == 0), "shape");
    __shared__ __attribute__((aligned(16))) float ws[2][BN][kStride];
    __shared__ __attribute__((aligned(16))) float xs[2][BM][kStride];

    const int t = threadIdx.x, lane = t % kWave, q = lane / 16, r = lane % 16;
    const int wave = __builtin_amdgcn_readfirstlane(t / kWave), wk = wave / (WN * WM);
    const int wn = wave % WN, wm = wave / WN % WM;
    const int K = p.K, chunks = (K + kChunk - 1) / kChunk, tiles = tiles_of(p);

    // consecutive work-group ids go to the 8 XCDs in turn: each XCD takes a run of the row-block-fastest order, so that
    // the work-groups it runs at once share weight blocks in its L2
    const int mb = (p.M + BM - 1) / BM;
    const int total = gridDim.x, per = total / 8, rem = total % 8;
    const int xcd = blockIdx.x % 8, idx = blockIdx.x / 8;
    const int logical = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + idx;
    const int n_blk = logical / mb, m0 = logical % mb * BM;
    const int tile0 = n_blk * (SWIGLU ? FT : BN / kTile);

    // staging: thread t takes one 16-byte piece of rows t / kPieces, + kRowsPerPass, ...; rows past the end repeat the
    // last
    const int piece = t % kPieces, row = t / kPieces, weight_piece = t % kWeightPieces, weight_row = t / kWeightPieces;
    const WT* wp[WLOADS];
#pragma unroll
    for (int i = 0; i < WLOADS; ++i) {
        const int b = weight_row + i * kWeightRowsPerPass; // weight row of the work-group
        if constexpr (SWIGLU) {
            const bool up = b >= FT * kTile;
            const int n = min(tile0 * kTile + (up ? b - FT * kTile : b), p.seg_rows[0] - 1);
            wp[i] = static_cast<const WT*>(up ? p.w[1] : p.w[0]) + static_cast<int64_t>(n) * K;
        } else {
            const Tile tile = locate(p, min(tile0 + b / kTile, tiles - 1));
            wp[i] = static_cast<const WT*>(tile.base) + static_cast<int64_t>(min(tile.n0 + b % kTile, tile.rows - 1)) * K;
        }
    }
    const float* xp[XLOADS];
#pragma unroll
    for (int i = 0; i < XLOADS; ++i)
        xp[i] = p.x + static_cast<int64_t>(min(m0 + row + i * kRowsPerPass, p.M - 1)) * p.ldx;
    const bool affine = NORM && p.apply_norm && p.norm_weight;

    u32x4 wr[WLOADS];
    f32x4 xr[XLOADS], g = {1.f, 1.f, 1.f, 1.f};
    auto load = [&](int chunk) {
        const int k = min(chunk * kChunk + 4 * piece, K - 4);
#pragma unroll
        for (int i = 0; i < XLOADS; ++i) xr[i] = *reinterpret_cast<const f32x4*>(xp[i] + k);
        if (affine) {
            if (p.norm_bf16) {
                const uint2 w = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(p.norm_weight) + k);
                g = f32x4{bf16_lo(w.x), bf16_hi(w.x), bf16_lo(w.y), bf16_hi(w.y)};
            } else {
                g = *reinterpret_cast<const f32x4*>(static_cast<const float*>(p.norm_weight) + k);
            }
        }
#pragma unroll
        for (int i = 0; i < WLOADS; ++i)
            wr[i] = *reinterpret_cast<const u32x4*>(wp[i] + min(chunk * kChunk + VALUES * weight_piece, K - VALUES));
    };
    float squares[XLOADS] = {};
    auto stage = [&](int chunk, int buf) {
        const bool live = chunk * kChunk + 4 * piece < K; // pieces past K are zeros in both operands
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < XLOADS; ++i) {
            f32x4 v = live ? xr[i] : zero;
            if constexpr (NORM) {
                squares[i] += (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]);
                if (affine && live) v = v * g;
            }
            if (BM % kRowsPerPass == 0 || row + i * kRowsPerPass < BM)
                *reinterpret_cast<f32x4*>(&xs[buf][row + i * kRowsPerPass][4 * piece]) = v;
        }
#pragma unroll
        for (int i = 0; i < WLOADS; ++i) {
            float* to = &ws[buf][weight_row + i * kWeightRowsPerPass][VALUES * weight_piece];
            const u32x4 w = chunk * kChunk + VALUES * weight_piece < K ? wr[i] : u32x4{0u, 0u, 0u, 0u};
            if constexpr (VALUES == 4) {
                *reinterpret_cast<u32x4*>(to) = w;
            } else {
                *reinterpret_cast<f32x4*>(to) = f32x4{bf16_lo(w.x), bf16_hi(w.x), bf16_lo(w.y), bf16_hi(w.y)};
                *reinterpret_cast<f32x4*>(to + 4) = f32x4{bf16_lo(w.z), bf16_hi(w.z), bf16_lo(w.w), bf16_hi(w.w)};
            }
        }
    };

    // a wave's weight tiles: generic TN consecutive ones; SwiGLU TN / 2 gate tiles, then the up tiles of the same
    // features
    auto slot = [&](int i) { return SWIGLU ? (i < TN / 2 ? wn * (TN / 2) + i : FT + wn * (TN / 2) + i - TN / 2) : wn * TN + i; };
    f64x4 acc[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) acc[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};

    load(0);
    for (int c = 0; c < chunks; ++c) {
        const int buf = c & 1;
        stage(c, buf);
        gemv::lds_barrier(); // chunk c published; every wave is done with the buffer that chunk c + 1 takes
        if (c + 1 < chunks) load(c + 1);
#pragma unroll
        for (int s = wk * (kWaveChunk / 16); s < (wk + 1) * (kWaveChunk / 16); ++s) {
            f32x4 a[TN], b[TM];
#pragma unroll
            for (int j = 0; j < TM; ++j)
                b[j] = *reinterpret_cast<const f32x4*>(&xs[buf][(wm * TM + j) * kTile + r][16 * s + 4 * q]);
#pragma unroll
            for (int i = 0; i < TN; ++i)
                a[i] = *reinterpret_cast<const f32x4*>(&ws[buf][slot(i) * kTile + r][16 * s + 4 * q]);
#pragma unroll
            for (int i = 0; i < TN; ++i) {
                f32x4 d[TM] = {};
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int j = 0; j < TM; ++j)
                        d[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][e], b[j][e], d[j], 0, 0, 0);
#pragma unroll
                for (int j = 0; j < TM; ++j) acc[i][j] += __builtin_convertvector(d[j], f64x4);
            }
        }
    }

    float inv[TM];
#pragma unroll
    for (int j = 0; j < TM; ++j) inv[j] = 1.0f;
    if (NORM && p.apply_norm) {
        // the pieces of a row sit in consecutive lanes; the factors go where the staged rows were
        float* inv_s = &xs[0][0][0];
        gemv::lds_barrier();
#pragma unroll
        for (int i = 0; i < XLOADS; ++i) {
            float v = squares[i];
#pragma unroll
            for (int lanes = 1; lanes < kPieces; lanes *= 2) v += __shfl_xor(v, lanes, kWave);
            const int b = row + i * kRowsPerPass;
            if (piece == 0 && b < BM) inv_s[b] = rsqrtf(v / static_cast<float>(K) + p.epsilon);
        }
        gemv::lds_barrier();
#pragma unroll
        for (int j = 0; j < TM; ++j) inv[j] = inv_s[(wm * TM + j) * kTile + r];
    }

    if constexpr (WK > 1) {
        // the waves' shares of the k, added in wave order by the first, which finishes the tile
        static_assert(WN == 1 && WM == 1 && sizeof(ws) >= (WK - 1) * TN * TM * 4 * kWave * sizeof(double), "merge");
        double* part = reinterpret_cast<double*>(&ws[0][0][0]);
        gemv::lds_barrier();
        if (wk > 0) {
#pragma unroll
            for (int i = 0; i < TN * TM * 4; ++i)
                part[((wk - 1) * TN * TM * 4 + i) * kWave + lane] = acc[i / 4 / TM][i / 4 % TM][i % 4];
        }
        gemv::lds_barrier();
        if (wk > 0) return;
#pragma unroll
        for (int w = 0; w < WK - 1; ++w)
#pragma unroll
            for (int i = 0; i < TN * TM * 4; ++i)
                acc[i / 4 / TM][i / 4 % TM][i % 4] += part[(w * TN * TM * 4 + i) * kWave + lane];
    }

    // the finished dots, rounded once
    auto dot = [&](int i, int j, int e, float scale) { return static_cast<float>(acc[i][j][e]) * scale; };

    // 16-byte stores where every row of the outputs is aligned for them
    const bool vec = p.ldy % 4 == 0 && reinterpret_cast<uintptr_t>(p.y) % 16 == 0 &&
                     (EPI != DLK_EPI_RESIDUAL || (p.ldres % 4 == 0 && reinterpret_cast<uintptr_t>(p.residual) % 16 == 0));
    const int64_t first_pos = EPI == DLK_EPI_QKV ? *p.position : 0;
#pragma unroll
    for (int j = 0; j < TM; ++j) {
        const int m = m0 + (wm * TM + j) * kTile + r;
        if (m >= p.M) continue;
        const float scale = inv[j] * p.acc_scale;
        if constexpr (SWIGLU) {
#pragma unroll
            for (int i = 0; i < TN / 2; ++i) {
                const int f = (tile0 + wn * (TN / 2) + i) * kTile + 4 * q;
                float o[4];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    o[e] = gemv::silu(dot(i, j, e, scale)) * dot(i + TN / 2, j, e, scale);
                float* y = p.y + static_cast<int64_t>(m) * p.ldy + f;
                if (vec && f + 4 <= p.seg_rows[0]) {
                    *reinterpret_cast<float4*>(y) = make_float4(o[0], o[1], o[2], o[3]);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (f + e < p.seg_rows[0]) y[e] = o[e];
                }
            }
        } else {
            const int64_t mg = p.m_base + m;
            const int64_t batch = EPI == DLK_EPI_QKV ? mg / p.length : 0;
            const int64_t pos = EPI == DLK_EPI_QKV ? first_pos + mg % p.length : 0;
#pragma unroll
            for (int i = 0; i < TN; ++i) {
                const int tile = tile0 + wn * TN + i;
                if (tile >= tiles) continue;
                const Tile tm = locate(p, tile);
                const int n = tm.n0 + 4 * q;
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = dot(i, j, e, scale);
                if constexpr (EPI == DLK_EPI_STORE || EPI == DLK_EPI_RESIDUAL) {
                    const int col = n + (EPI == DLK_EPI_STORE ? gemv::seg_column(p, tm.seg) : 0);
                    float* y = p.y + static_cast<int64_t>(m) * p.ldy + col;
                    const float* res = EPI == DLK_EPI_RESIDUAL ? p.residual + static_cast<int64_t>(m) * p.ldres + n : nullptr;
                    if (EPI == DLK_EPI_STORE && p.bias) {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (n + e < tm.rows)
                                v[e] += p.bias_bf16 ? bf16_to_f32(static_cast<const uint16_t*>(p.bias)[col + e])
                                                    : static_cast<const float*>(p.bias)[col + e];
                    }
                    if (vec && col % 4 == 0 && n + 4 <= tm.rows) {
                        float4 out = make_float4(v[0], v[1], v[2], v[3]);
                        if constexpr (EPI == DLK_EPI_RESIDUAL) {
                            const float4 a = *reinterpret_cast<const float4*>(res);
                            out.x += a.x; out.y += a.y; out.z += a.z; out.w += a.w;
                        }
                        *reinterpret_cast<float4*>(y) = out;
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (n + e < tm.rows) y[e] = EPI == DLK_EPI_RESIDUAL ? v[e] + res[e] : v[e];
                    }
                } else if constexpr (EPI == DLK_EPI_QKV) {
                    const int hd = p.head_dim;
                    const float* hidden = tm.seg == 0 ? p.lora_hidden[0] : tm.seg == 2 ? p.lora_hidden[2] : nullptr;
                    if (hidden) {
                        // unmerged LoRA: + scale * up[n, :] . hidden[m, :] (rows past the segment repeat its last)
                        const WT* up = static_cast<const WT*>(tm.seg == 0 ? p.lora_up[0] : p.lora_up[2]);
                        const float* h = hidden + mg * gemv::lora_stride(p);
                        float d[4] = {0.f, 0.f, 0.f, 0.f};
                        for (int k = 0; k < p.lora_rank; ++k) {
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                const WT value = up[static_cast<int64_t>(min(n + e, tm.rows - 1)) * p.lora_rank + k];
                                if constexpr (sizeof(WT) == 4) d[e] += value * h[k];
                                else d[e] += bf16_to_f32(value) * h[k];
                            }
                        }
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] += d[e] * p.lora_scale;
                    }
#pragma unroll
                    for (int e = 0; e < 4; e += 2) {
                        if (n + e >= tm.rows) continue; // segments are whole pairs
                        const int d = (n + e) % hd, head = (n + e) / hd;
                        float even = v[e], odd = v[e + 1];
                        if (tm.seg < 2) {
                            // even: x_e c - x_o s ; odd: x_e s + x_o c (interleaved pairs, src/ops/contraction.cpp:44-49)
                            const float c = p.cosine[pos * (hd / 2) + d / 2], s = p.sine[pos * (hd / 2) + d / 2];
                            const float x = even;
                            even = x * c - odd * s;
                            odd = x * s + odd * c;
                        }
                        if (tm.seg == 0) {
                            *reinterpret_cast<float2*>(p.y + mg * p.ldy + n + e) = make_float2(even, odd);
                            continue;
                        }
                        const int64_t index = ((batch * p.kv_heads + head) * p.cache_capacity + pos) * hd + d;
                        void* cache = tm.seg == 1 ? p.k_cache : p.v_cache;
                        if (p.cache_bf16)
                            *reinterpret_cast<uint32_t*>(static_cast<uint16_t*>(cache) + index) =
                                f32_to_bf16(even) | (static_cast<uint32_t>(f32_to_bf16(odd)) << 16);
                        else
                            *reinterpret_cast<float2*>(static_cast<float*>(cache) + index) = make_float2(even, odd);
                    }
                }
            }
        }
    }
    if constexpr (EPI == DLK_EPI_STORE || EPI == DLK_EPI_RESIDUAL) {
        if (p.bump_position && blockIdx.x == 0 && t == 0) *p.bump_position += p.bump_count;
    }
}

template <typename WT, int EPI, bool NORM>
const void* shape_kernel(int shape) {
    switch (shape) {
    case k128x128: return reinterpret_cast<const void*>(&gemm_f32<WT, EPI, NORM, 2, 2, 1, 4, 4>);
    case k64x64: return reinterpret_cast<const void*>(&gemm_f32<WT, EPI, NORM, 2, 2, 1, 2, 2>);
    case k64x32: return reinterpret_cast<const void*>(&gemm_f32<WT, EPI, NORM, 2, 2, 1, 2, 1>);
    case k32x16: return reinterpret_cast<const void*>(&gemm_f32<WT, EPI, NORM, 1, 1, 4, 2, 1>);
    default: return nullptr;
    }
}

template <int EPI, bool NORM>
const void* weight_kernel(const dlk_gemv_params& p, int shape) {
    return p.w_bf16 ? shape_kernel<uint16_t, EPI, NORM>(shape) : shape_kernel<float, EPI, NORM>(shape);
}

/// The kernel of a launch for a work-group shape; null if none.
template <int EPI>
const void* resolve(const dlk_gemv_params& p, int shape) {
    if (gemv::norm_variant(EPI, p.apply_norm != 0)) {
        if constexpr (EPI != DLK_EPI_RESIDUAL) return weight_kernel<EPI, true>(p, shape);
        return nullptr;
    }
    if constexpr (EPI == DLK_EPI_STORE || EPI == DLK_EPI_RESIDUAL) return weight_kernel<EPI, false>(p, shape);
    return nullptr;
}

} // namespace dlk::gemm32

const void* dlk_gemm_f32_kernel_store(const dlk_gemv_params& p, int shape);
const void* dlk_gemm_f32_kernel_residual(const dlk_gemv_params& p, int shape);
const void* dlk_gemm_f32_kernel_qkv(const dlk_gemv_params& p, int shape);
const void* dlk_gemm_f32_kernel_swiglu(const dlk_gemv_params& p, int shape);
