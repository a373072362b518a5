// Grouped-query attention over any number of query rows (see dlk_attention_params in kernels.h): one or several new
// positions, causal or not, with or without a keep mask, head sizes 16 to 128.  (One position at head sizes 64 and 128
// takes attention_matrix.hip, causal prefill chunks at those sizes attention_prefill.hip.)
//
// All products run on the f32 matrix cores, so nothing is rounded that the inputs do not round: with
// v_mfma_f32_16x16x4_f32, S^T[16 keys][16 rows] = K Q^T (lane l supplies K[key l%16] and Q[row l%16] at four consecutive
// head-dim entries, 4 (l/16) .. +4 of each 16, one per product) and O^T[16 d][16 rows] += V^T P^T.  The scores come out
// with lane l holding keys 4 (l/16) .. +4 of row l%16, which is the B operand of the second product when its k slot
// l/16 of product j stands for key 4 (l/16) + j, so the probabilities never leave their lane; maximum, sum and rescale
// factor of a row sit in the lanes of its column.
//
// Grid (key split, query-row block, b * KV + kv head).  The G query heads of a KV head at every new position are its
// rows, position-major.  A work-group of four waves serves 16 WR of them: WR waves take 16 rows each, and the 4 / WR
// waves of a row tile share the keys of each staged tile (merged in LDS at the end), so that a few rows still use all
// four.  Key tiles are loaded with 16-byte loads (the next tile in flight, in registers, while one is used) and staged in
// LDS as f32.  With one split the work-group writes the normalised output; otherwise it writes (o, max, sum) partials
// that attention_combine merges in a second launch (the kernel boundary orders them: no device-scope fence, whose L2
// write-back across the XCDs costs microseconds per work-group).
//
// What bounds it: many rows, the f32 matrix cores (153 TFLOP/s); few rows, the round trips of the K/V tiles.
// Measured on MI355X (the kernel before it ran the products on the vector ALU, one key or head-dim column per lane):
// 4 sequences x 7 positions over 1508 f32 keys, 32 / 8 heads of 64: 135.5 -> 11.6 us + 4.7 for the merge; 4 x 500
// positions bidirectional over a padded batch: 455 -> 85 us (the products alone take 38; exponentials, masks and staging
// as much vector work again, and the two barriers of a tile keep them from overlapping fully); causal byte prompts of
// 4 x 510 positions, 8 / 2 heads of 32: 84 -> 15 us; one position of that model: 5.7 -> 5.0 us (4.6 up to 128 keys; each
// further tile is a round trip of 1.7 us).
#include "kernels/device_common.h"

#include <algorithm>
#include <mutex>
#include <type_traits>

namespace dlk {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef f32x4 f32x4_any __attribute__((aligned(4))); // callers' rows: any float alignment
typedef uint32_t u32_any __attribute__((aligned(1)));  // four mask bytes

/// Keys per staged tile: few rows over small heads are a chain of tile round trips, so they take longer tiles.
constexpr int tile_keys(int hd, int wr) { return hd == 16 || (hd == 32 && wr < 4) ? 128 : 64; }

// work-group barrier that orders LDS traffic only: the next tile's loads stay in flight
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <typename KT, int HD, int WR>
__global__ __launch_bounds__(kThreads) void attention_rows(const dlk_attention_params p, int G) {
    constexpr int WK = kWaves / WR;                   // waves that share a row tile's keys
    constexpr int T = tile_keys(HD, WR);
    constexpr int GROUPS = T / 16 / WK;               // 16-key groups of a tile per wave
    constexpr int KS = HD + 8, VS = HD + 4;           // LDS row strides (floats): conflict-free fragment reads
    constexpr int VALUES = 16 / sizeof(KT);           // K/V values per 16-byte piece
    constexpr int PIECES = HD / VALUES;               // pieces per K/V row
    constexpr int LOADS = T * PIECES / kThreads;
    constexpr int DT = HD / 16;                       // 16-wide head-dim tiles
    static_assert(T % (16 * WK) == 0 && T * PIECES % kThreads == 0, "tile");
    __shared__ __attribute__((aligned(16))) float k_tile[T][KS];
    __shared__ __attribute__((aligned(16))) float v_tile[T][VS];
    __shared__ int odd_values[kWaves]; // masked launches: whether the tile's V holds an infinity or NaN

    const int t = threadIdx.x, lane = t % kWave, q = lane / 16, r = lane % 16;
    const int wave = __builtin_amdgcn_readfirstlane(t / kWave), wr = wave / WK, wk = wave % WK;
    // Consecutive work-group ids go to the 8 XCDs in turn.  With the (sequence, KV head) pairs a multiple of 8, XCD x takes
    // the splits and row blocks of pairs x, x + 8, ... one pair after the other, so its L2 holds the few pairs it works
    // on and the sequences of a padded batch, whose masks leave them different work, spread over all XCDs (each XCD
    // on a sequence of its own: 4 x 500 positions 111 -> 90 us).  Otherwise each takes a run of the pairs.
    // One work-group a pair has nothing to share: it skips the divisions, a chain of some 300 instructions before its
    // first load.  With those of the query row moved behind the first tile's loads, and the remainders replaced by
    // products: one position of 8 / 2 heads of 32 over 33-160 keys 5.25 -> 4.98 us, the padded batch of 4 x 500 90 -> 85.
    const int per_pair = gridDim.x * gridDim.y;
    int split = 0, row_block = 0, pair = blockIdx.z;
    if (per_pair > 1) {
        const int total = per_pair * gridDim.z;
        const int id = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
        const int xcd = id % 8, idx = id / 8, per = total / 8, rem = total % 8;
        const int logical = gridDim.z % 8 == 0 ? (idx / per_pair * 8 + xcd) * per_pair + idx % per_pair
                                               : (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + idx;
        split = logical % gridDim.x;
        row_block = logical / gridDim.x % gridDim.y;
        pair = logical / per_pair;
    }
    const int rows_total = G * p.L, row0 = row_block * 16 * WR;

    const size_t head_base = static_cast<size_t>(pair) * p.capacity;
    const KT* kbase = static_cast<const KT*>(p.k) + head_base * HD;
    const KT* vbase = static_cast<const KT*>(p.v) + head_base * HD;
    const int64_t k_begin = static_cast<int64_t>(split) * p.chunk;

    const int64_t first = p.position ? *p.position : p.first_host;

    u32x4 k_next[LOADS], v_next[LOADS];
    uint32_t keep_next[GROUPS]; // four mask bytes each
    const unsigned char* keep = nullptr; // this lane's mask row
    // load_tile loads the tile's rows and this lane's mask entries; those from `end` on repeat the one before it and are
    // dropped when the tile is used (the mask comes first: loads complete in order, and it would wait for the rows)
    auto load_rows = [&](int64_t tile0, int last) {
        const KT* kt = kbase + tile0 * HD;
        const KT* vt = vbase + tile0 * HD;
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int at = t + i * kThreads;
            const uint32_t offset = min(at / PIECES, last) * HD + at % PIECES * VALUES;
            k_next[i] = *reinterpret_cast<const u32x4*>(kt + offset);
            v_next[i] = *reinterpret_cast<const u32x4*>(vt + offset);
        }
    };
    auto last_of = [&](int64_t tile0, int64_t end) { // of the tile's rows, uniform
        return static_cast<int>(min<int64_t>(end - tile0, T)) - 1;
    };
    auto load_tile = [&](int64_t tile0, int64_t end) {
        const int last = last_of(tile0, end);
        if (keep) {
            const int64_t stride = p.mask_stride[3];
            const unsigned char* entries = keep + tile0 * stride;
            if (stride == 1 && last == T - 1) {
#pragma unroll
                for (int g = 0; g < GROUPS; ++g)
                    keep_next[g] = *reinterpret_cast<const u32_any*>(entries + 16 * (wk + WK * g) + 4 * q);
            } else {
#pragma unroll
                for (int g = 0; g < GROUPS; ++g) {
                    uint32_t four = 0;
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        four |= static_cast<uint32_t>(entries[min(16 * (wk + WK * g) + 4 * q + j, last) * stride]) << (8 * j);
                    keep_next[g] = four;
                }
            }
        }
        load_rows(tile0, last);
    };
    // the first tile is requested before the device length arrives, and before the divisions below where no mask entry
    // has to come first, within the storage: what lies past the length is dropped
    const int64_t stored = min(p.capacity, k_begin + p.chunk);
    if (k_begin < stored && !p.keep_mask) load_rows(k_begin, last_of(k_begin, stored));

    // this lane's query row (rows past the end repeat the last; their results are never written)
    const int b = p.B == 1 ? 0 : pair / p.KV, kvh = pair - b * p.KV;
    auto position_of = [&](int row) { return p.L == 1 ? 0 : row / G; };
    const int row = min(row0 + 16 * wr + r, rows_total - 1);
    const int l = position_of(row), h = kvh * G + row - l * G;
    if (p.keep_mask) {
        keep = p.keep_mask + b * p.mask_stride[0] + h * p.mask_stride[1] + l * p.mask_stride[2];
        if (k_begin < stored) load_tile(k_begin, stored);
    }

    const int64_t m_row = static_cast<int64_t>(b) * p.L + l;
    f32x4 qf[DT];
#pragma unroll
    for (int s = 0; s < DT; ++s) {
        const float* src = p.q + (p.q_row ? b * p.q_batch + l * p.q_row + h * p.q_head
                                          : m_row * p.ldq + static_cast<int64_t>(h) * HD) + 16 * s + 4 * q;
        qf[s] = *reinterpret_cast<const f32x4_any*>(src) * (p.scale * 1.4426950408889634f); // scores in base 2
    }
    // keys this lane's row sees, its wave's first and last row (wave_full: without a mask, every row of the wave sees
    // the keys below it), and the work-group's last row
    const int64_t S = first + p.L;
    const int64_t split_end = min(S, k_begin + p.chunk);
    const int64_t limit = p.causal ? min(split_end, first + l + 1) : split_end;
    const int first_row = min(row0 + 16 * wr, rows_total - 1);
    const int last_row = min(row0 + 16 * wr + 15, rows_total - 1), last_block_row = min(row0 + 16 * WR - 1, rows_total - 1);
    const int64_t wave_full = p.causal ? min(split_end, first + position_of(first_row) + 1) : split_end;
    const int64_t wave_end = row0 + 16 * wr >= rows_total ? 0 // no row for this wave
                             : p.causal                   ? min(split_end, first + position_of(last_row) + 1)
                                                          : split_end;
    const int64_t k_end = p.causal ? min(split_end, first + position_of(last_block_row) + 1) : split_end;

    auto stage_tile = [&](int64_t tile0) {
        const int staged = static_cast<int>(min<int64_t>(k_end - tile0, T)); // live keys of the tile
        if (keep) {
            bool odd = false;
#pragma unroll
            for (int i = 0; i < LOADS; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    odd |= (v_next[i][e] & 0x7f800000u) == 0x7f800000u;
                    if constexpr (sizeof(KT) == 2) odd |= (v_next[i][e] & 0x7f80u) == 0x7f80u;
                }
            const bool any = __ballot(odd) != 0;
            if (lane == 0) odd_values[wave] = any;
        }
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int at = t + i * kThreads, key = at / PIECES, d = at % PIECES * VALUES;
            const bool live = key < staged;
            const u32x4 zero = {0u, 0u, 0u, 0u};
            const u32x4 kv = live ? k_next[i] : zero, vv = live ? v_next[i] : zero;
            if constexpr (sizeof(KT) == 4) {
                *reinterpret_cast<u32x4*>(&k_tile[key][d]) = kv;
                *reinterpret_cast<u32x4*>(&v_tile[key][d]) = vv;
            } else {
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    const uint32_t k0 = half ? kv.z : kv.x, k1 = half ? kv.w : kv.y;
                    const uint32_t v0 = half ? vv.z : vv.x, v1 = half ? vv.w : vv.y;
                    *reinterpret_cast<f32x4*>(&k_tile[key][d + 4 * half]) = f32x4{bf16_lo(k0), bf16_hi(k0), bf16_lo(k1), bf16_hi(k1)};
                    *reinterpret_cast<f32x4*>(&v_tile[key][d + 4 * half]) = f32x4{bf16_lo(v0), bf16_hi(v0), bf16_lo(v1), bf16_hi(v1)};
                }
            }
        }
    };

    float m_run = -INFINITY, l_run = 0.0f; // l_run: this lane's keys only
    f32x4 o[DT];
#pragma unroll
    for (int d = 0; d < DT; ++d) o[d] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (int64_t tile0 = k_begin; tile0 < k_end; tile0 += T) {
        lds_barrier(); // every wave is done with the previous tile
        stage_tile(tile0);
        // Tiles that reach past some row's keys, or have a mask: which of this lane's keys its row sees, four bits per
        // group
        uint32_t live = 0xffffffffu;
        const bool partial = keep || tile0 + T > wave_full;
        if (partial) {
            const int rem = static_cast<int>(min<int64_t>(limit - tile0, T)); // keys of the tile below the limit
            live = 0;
#pragma unroll
            for (int g = 0; g < GROUPS; ++g) {
                uint32_t four = (1u << min(max(rem - 16 * (wk + WK * g) - 4 * q, 0), 4)) - 1;
                if (keep) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (!(keep_next[g] & (0xffu << (8 * j)))) four &= ~(1u << j);
                }
                live |= four << (4 * g);
            }
        }
        lds_barrier();
        if (tile0 + T < k_end) load_tile(tile0 + T, k_end);
        // nothing for this wave: its rows end before the tile, or the mask drops every key of its groups (whose zero
        // probabilities still carry an infinity or NaN of V into the sums, as the reference's product does)
        if (tile0 >= wave_end) continue;
        if (partial && __ballot(live != 0) == 0 &&
            !(keep && (odd_values[0] | odd_values[1] | odd_values[2] | odd_values[3])))
            continue;

        f32x4 s[GROUPS];
        float tile_max = -INFINITY;
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) s[g] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int d = 0; d < DT; ++d) {
            f32x4 a[GROUPS];
#pragma unroll
            for (int g = 0; g < GROUPS; ++g)
                a[g] = *reinterpret_cast<const f32x4*>(&k_tile[16 * (wk + WK * g) + r][16 * d + 4 * q]);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int g = 0; g < GROUPS; ++g)
                    s[g] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[g][e], qf[d][e], s[g], 0, 0, 0);
        }
        if (partial) {
#pragma unroll
            for (int g = 0; g < GROUPS; ++g)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (!(live >> (4 * g + j) & 1)) s[g][j] = -INFINITY;
        }
#pragma unroll
        for (int g = 0; g < GROUPS; ++g)
#pragma unroll
            for (int j = 0; j < 4; ++j) tile_max = fmaxf(tile_max, s[g][j]);
        tile_max = fmaxf(tile_max, __shfl_xor(tile_max, 16, kWave));
        tile_max = fmaxf(tile_max, __shfl_xor(tile_max, 32, kWave));
        const float m_new = fmaxf(m_run, tile_max);
        // a row that has seen no key yet keeps -inf, and nothing of its sums
        const float m_safe = m_new == -INFINITY ? 0.0f : m_new;
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_safe);
        l_run *= alpha;
#pragma unroll
        for (int d = 0; d < DT; ++d) o[d] *= alpha;
        m_run = m_new;
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float e = __builtin_amdgcn_exp2f(s[g][j] - m_safe); // 0 for the dropped keys
                s[g][j] = e;
                l_run += e;
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int d = 0; d < DT; ++d)
                    o[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(v_tile[16 * (wk + WK * g) + 4 * q + j][16 * d + r], s[g][j],
                                                                o[d], 0, 0, 0);
        }
    }
    l_run += __shfl_xor(l_run, 16, kWave);
    l_run += __shfl_xor(l_run, 32, kWave);

    if constexpr (WK > 1) {
        // merge the waves of a row tile, in wave order
        constexpr int FLOATS = 4 * DT + 2; // per lane
        static_assert(WR * (WK - 1) * FLOATS * kWave <= T * KS, "merge");
        float* part = &k_tile[0][0];
        lds_barrier();
        if (wk > 0) {
            float* mine = part + (wr * (WK - 1) + wk - 1) * FLOATS * kWave + lane;
#pragma unroll
            for (int i = 0; i < 4 * DT; ++i) mine[i * kWave] = o[i / 4][i % 4];
            mine[4 * DT * kWave] = m_run;
            mine[(4 * DT + 1) * kWave] = l_run;
        }
        lds_barrier();
        if (wk > 0) return;
        float mx = m_run;
#pragma unroll
        for (int w = 0; w < WK - 1; ++w) mx = fmaxf(mx, part[((wr * (WK - 1) + w) * FLOATS + 4 * DT) * kWave + lane]);
        const float safe = mx == -INFINITY ? 0.0f : mx;
        const float own = __builtin_amdgcn_exp2f(m_run - safe);
        l_run *= own;
#pragma unroll
        for (int d = 0; d < DT; ++d) o[d] *= own;
#pragma unroll
        for (int w = 0; w < WK - 1; ++w) {
            const float* theirs = part + (wr * (WK - 1) + w) * FLOATS * kWave + lane;
            const float mw = theirs[4 * DT * kWave];
            const float f = __builtin_amdgcn_exp2f(mw - safe);
            l_run += f * theirs[(4 * DT + 1) * kWave];
#pragma unroll
            for (int i = 0; i < 4 * DT; ++i) o[i / 4][i % 4] += f * theirs[i * kWave];
        }
        m_run = mx;
    }

    if (row0 + 16 * wr + r >= rows_total) return;
    if (p.splits == 1) {
        // a masked row that kept no key: NaN, as the reference's softmax over an all -inf row
        const float inv = l_run > 0.0f ? 1.0f / l_run : p.keep_mask ? __builtin_nanf("") : 0.0f;
        float* out = p.out + m_row * p.ldo + static_cast<int64_t>(h) * HD + 4 * q;
#pragma unroll
        for (int d = 0; d < DT; ++d) *reinterpret_cast<f32x4_any*>(out + 16 * d) = o[d] * inv;
    } else {
        const int64_t slot = ((static_cast<int64_t>(b) * p.H + h) * p.L + l) * p.splits + split;
#pragma unroll
        for (int d = 0; d < DT; ++d) *reinterpret_cast<f32x4_any*>(p.partial_o + slot * HD + 16 * d + 4 * q) = o[d];
        if (q == 0) {
            p.partial_ml[slot * 2] = m_run;
            p.partial_ml[slot * 2 + 1] = l_run;
        }
    }
}

// One work-group per (b, h, l) row merges its split partials: the global maximum first, then each thread takes
// one head-dim column and every (512 / HD)-th split, and the column groups add up in LDS in a fixed order.  A
// thread loads four of its splits at a time (the last group clamped to a valid split and discarded), so their
// loads are in flight together; dead splits are dropped by selection, never by a branch around the loads.
constexpr int kCombineThreads = 512;

// BASE2: attention_rows' partials, whose maxima are in base 2.
template <int HD, bool BASE2>
__global__ __launch_bounds__(kCombineThreads) void attention_combine(const dlk_attention_params p) {
    constexpr int GROUPS = kCombineThreads / HD;
    constexpr int WAVES = kCombineThreads / kWave;
    constexpr int U = 4; // splits per thread in flight
    __shared__ float wave_max_s[WAVES];
    __shared__ float acc_s[GROUPS][HD];
    __shared__ float total_s[GROUPS];
    const int64_t prow = blockIdx.x; // (b * H + h) * L + l
    const int t = threadIdx.x, lane = t % kWave;
    const int64_t l = prow % p.L, h = (prow / p.L) % p.H, b = prow / (static_cast<int64_t>(p.L) * p.H);
    const float* ml = p.partial_ml + prow * p.splits * 2;
    float maximum = -INFINITY;
    for (int s = t; s < p.splits; s += kCombineThreads)
        if (ml[2 * s + 1] > 0.0f) maximum = fmaxf(maximum, ml[2 * s]);
    maximum = wave_max(maximum);
    if (lane == 0) wave_max_s[t / kWave] = maximum;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < WAVES; ++w) maximum = fmaxf(maximum, wave_max_s[w]);
    const int d = t % HD, group = t / HD;
    float acc = 0.0f, total = 0.0f;
    for (int s0 = group; s0 < p.splits; s0 += U * GROUPS) {
        float ms[U], ls[U], o[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int s = min(s0 + u * GROUPS, p.splits - 1);
            ms[u] = ml[2 * s];
            ls[u] = ml[2 * s + 1];
            o[u] = p.partial_o[(prow * p.splits + s) * HD + d];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            // a split without keys has weight 0.  attention_rows writes its partials all the same (BASE2), and what its
            // zero probabilities made of an infinity or NaN of V stays in the sum; the other kernels leave the row
            // unwritten, so it is selected away (0 * a stale NaN or Inf must not enter)
            const bool in = s0 + u * GROUPS < p.splits;
            const bool live = BASE2 ? in : in && ls[u] > 0.0f && ms[u] != -INFINITY;
            const float w = !live   ? 0.0f
                            : BASE2 ? __builtin_amdgcn_exp2f(ms[u] - (maximum == -INFINITY ? 0.0f : maximum))
                                    : expf(ms[u] - maximum);
            total += live ? w * ls[u] : 0.0f;
            acc += live ? w * o[u] : 0.0f;
        }
    }
    acc_s[group][d] = acc;
    if (d == 0) total_s[group] = total;
    __syncthreads();
    if (group == 0) {
        float sum = 0.0f, weight = 0.0f;
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) {
            sum += acc_s[g][d];
            weight += total_s[g];
        }
        const float inv = weight > 0.0f ? 1.0f / weight : p.keep_mask ? __builtin_nanf("") : 0.0f;
        p.out[(b * p.L + l) * p.ldo + h * HD + d] = sum * inv;
    }
}

// ------------------------------------------------------------------------------------------ small heads
// Head sizes below 16 (the reference's tiny test decoders: tests/c_api.c:31 builds one with head size 2).  Not a hot
// path: one wave per (query row, key split); lane = key within each 64-key step, the scores and the weighted V
// columns reduced over the wave, online softmax across the steps.  Writes the output, or (o, max, sum) partials
// for attention_combine when the keys are split.
template <typename KT, int HD>
__global__ __launch_bounds__(kWave) void attention_small(const dlk_attention_params p) {
    const int lane = threadIdx.x;
    const int64_t prow = blockIdx.x; // (b * H + h) * L + l
    const int split = blockIdx.y;
    const int l = static_cast<int>(prow % p.L), h = static_cast<int>((prow / p.L) % p.H);
    const int b = static_cast<int>(prow / (static_cast<int64_t>(p.L) * p.H));
    const int kvh = h / (p.H / p.KV);
    const int64_t first = p.position ? *p.position : p.first_host;
    const int64_t S = first + p.L;
    const int64_t visible = p.causal ? min(S, first + l + 1) : S;
    const int64_t k_begin = static_cast<int64_t>(split) * p.chunk;
    const int64_t k_end = min(visible, k_begin + p.chunk);
    const float* qrow = p.q + (static_cast<int64_t>(b) * p.L + l) * p.ldq + static_cast<int64_t>(h) * HD;
    float q[HD];
#pragma unroll
    for (int d = 0; d < HD; ++d) q[d] = qrow[d] * p.scale;
    const size_t head = (static_cast<size_t>(b) * p.KV + kvh) * p.capacity;
    const KT* kbase = static_cast<const KT*>(p.k) + head * HD;
    const KT* vbase = static_cast<const KT*>(p.v) + head * HD;
    auto value = [](const KT* row, int d) {
        if constexpr (sizeof(KT) == 2) return bf16_to_f32(reinterpret_cast<const uint16_t*>(row)[d]);
        else return static_cast<float>(row[d]);
    };
    float m = -INFINITY, total = 0.0f, o[HD];
#pragma unroll
    for (int d = 0; d < HD; ++d) o[d] = 0.0f;
    const unsigned char* keep =
        p.keep_mask ? p.keep_mask + b * p.mask_stride[0] + h * p.mask_stride[1] + l * p.mask_stride[2] : nullptr;
    for (int64_t k0 = k_begin; k0 < k_end; k0 += kWave) {
        const int64_t key = k0 + lane;
        // a live key the mask keeps (without a mask every step holds one, so m_new is finite)
        const bool live = key < k_end && (!keep || keep[key * p.mask_stride[3]]);
        float s = -INFINITY;
        if (live) {
            s = 0.0f;
#pragma unroll
            for (int d = 0; d < HD; ++d) s += q[d] * value(kbase + key * HD, d);
        }
        const float m_new = fmaxf(m, wave_max(s));
        const float alpha = m == -INFINITY ? 0.0f : expf(m - m_new);
        const float pr = live ? expf(s - m_new) : 0.0f;
        total = total * alpha + wave_sum(pr);
#pragma unroll
        for (int d = 0; d < HD; ++d) o[d] = o[d] * alpha + wave_sum(live ? pr * value(vbase + key * HD, d) : 0.0f);
        m = m_new;
    }
    if (lane != 0) return;
    if (p.splits == 1) {
        float* out = p.out + (static_cast<int64_t>(b) * p.L + l) * p.ldo + static_cast<int64_t>(h) * HD;
#pragma unroll
        for (int d = 0; d < HD; ++d) out[d] = total > 0.0f ? o[d] / total : keep ? __builtin_nanf("") : 0.0f;
    } else {
        const int64_t slot = prow * p.splits + split;
#pragma unroll
        for (int d = 0; d < HD; ++d) p.partial_o[slot * HD + d] = o[d];
        p.partial_ml[slot * 2] = m;
        p.partial_ml[slot * 2 + 1] = total;
    }
}

template <typename KT, int HD>
int launch_small(const dlk_attention_params& p, hipStream_t stream) {
    const int64_t rows = static_cast<int64_t>(p.B) * p.H * p.L;
    hipLaunchKernelGGL((attention_small<KT, HD>), dim3(static_cast<unsigned>(rows), p.splits), dim3(kWave), 0, stream,
                       p);
    int status = static_cast<int>(hipGetLastError());
    if (status != 0 || p.splits == 1 || p.partials_only) return status;
    hipLaunchKernelGGL((attention_combine<HD, false>), dim3(static_cast<unsigned>(rows)), dim3(kCombineThreads), 0, stream, p);
    return static_cast<int>(hipGetLastError());
}

template <int HD, bool BASE2 = false>
int launch_combine(const dlk_attention_params& p, hipStream_t stream) {
    const int64_t combine_rows = static_cast<int64_t>(p.B) * p.H * p.L;
    hipLaunchKernelGGL((attention_combine<HD, BASE2>), dim3(static_cast<unsigned>(combine_rows)), dim3(kCombineThreads), 0, stream, p);
    return static_cast<int>(hipGetLastError());
}

// Row tiles per work-group: the fewest that hold the rows of a KV head, and the waves left over share the keys.
int row_tiles(const dlk_attention_params& p) {
    const int rows = p.H / p.KV * p.L;
    if (rows <= 32) return rows <= 16 ? 1 : 2;
    // four row tiles that leave a CU with less than two work-groups: two, so that one's products run under another's
    // staging and softmax (4 x 510 causal positions, 8 / 2 heads of 32: 18.5 us at 256 work-groups, 15.2 at 512, 16.8 at
    // 1024 of one row tile; 4 x 500 positions of 32 / 8 heads of 64: 111 at 1024, 120 at 2048)
    return static_cast<int64_t>((rows + 63) / 64) * p.splits * p.B * p.KV < 512 ? 2 : 4;
}

template <typename KT, int HD>
int launch(const dlk_attention_params& p, hipStream_t stream) {
    const int group = p.H / p.KV, rows = group * p.L, wr = row_tiles(p);
    const dim3 grid(p.splits, (rows + 16 * wr - 1) / (16 * wr), p.B * p.KV);
    const dim3 threads(kThreads);
    if (wr == 1) hipLaunchKernelGGL((attention_rows<KT, HD, 1>), grid, threads, 0, stream, p, group);
    else if (wr == 2) hipLaunchKernelGGL((attention_rows<KT, HD, 2>), grid, threads, 0, stream, p, group);
    else hipLaunchKernelGGL((attention_rows<KT, HD, 4>), grid, threads, 0, stream, p, group);
    const int status = static_cast<int>(hipGetLastError());
    if (status != 0 || p.splits == 1 || p.partials_only) return status;
    return launch_combine<HD, true>(p, stream);
}

} // namespace
} // namespace dlk

// Key-split partials of the allocation-free attention entry: a fixed array in device memory, one copy per GPU the
// library runs on, held until the process ends.  Host code never passes the array's name to a kernel (on the host
// it is only a stand-in for the symbol): dlk_attention_scratch resolves each device's own address once, with that
// device current, and the launches take that address.
static __device__ __align__(256) float scratch[DLK_ATTENTION_SCRATCH_FLOATS];

extern "C" int dlk_attention_scratch(int device, float** address) {
    constexpr int kDevicesMax = 64;
    static std::mutex mutex;
    static float* addresses[kDevicesMax] = {};
    if (!address || device < 0 || device >= kDevicesMax) return static_cast<int>(hipErrorInvalidValue);
    std::lock_guard<std::mutex> lock(mutex);
    if (!addresses[device]) {
        int current = 0;
        hipError_t status = hipGetDevice(&current);
        if (status != hipSuccess) return static_cast<int>(status);
        if (current != device && (status = hipSetDevice(device)) != hipSuccess) return static_cast<int>(status);
        void* found = nullptr;
        status = hipGetSymbolAddress(&found, HIP_SYMBOL(scratch));
        if (current != device) {
            const hipError_t restored = hipSetDevice(current);
            if (status == hipSuccess) status = restored;
        }
        if (status != hipSuccess) return static_cast<int>(status);
        if (!found) return static_cast<int>(hipErrorInvalidSymbol);
        addresses[device] = static_cast<float*>(found);
    }
    *address = addresses[device];
    return 0;
}

extern "C" const char* dlk_attention_kernel(const dlk_attention_params* p) {
    if (dlk_attention_matrix_eligible(p)) return "matrix";
    if (dlk_attention_prefill_eligible(p)) return "prefill";
    if (p->hd < 16) return "small";
    const int tiles = dlk::row_tiles(*p);
    return tiles == 1 ? "rows 1" : tiles == 2 ? "rows 2" : "rows 4";
}

extern "C" int dlk_attention_takes_strides(const dlk_attention_params* p) {
    return p->hd >= 16 && !dlk_attention_matrix_eligible(p) && !dlk_attention_prefill_eligible(p);
}

extern "C" int dlk_attention(const dlk_attention_params* params, dlh_stream stream_handle) {
    hipStream_t stream = reinterpret_cast<hipStream_t>(stream_handle);
    const dlk_attention_params& p = *params;
    if (p.B <= 0 || p.L <= 0 || p.KV <= 0 || p.H % p.KV != 0 || p.splits <= 0 || p.chunk <= 0 ||
        (p.splits > 1 && (!p.partial_o || !p.partial_ml)) || (p.splits > 1 && p.chunk % 64 != 0))
        return static_cast<int>(hipErrorInvalidValue);
    if (p.q_row && !dlk_attention_takes_strides(&p)) return static_cast<int>(hipErrorInvalidValue);
    // a keep mask is applied by the general and small-head kernels, which serve non-causal attention
    if (p.keep_mask && (p.causal || p.qkv_partial || p.stage_out || p.kv_split)) return static_cast<int>(hipErrorInvalidValue);
    // the QKV projection's partials are finished only by the matrix kernel
    if (p.qkv_partial && (p.stage_out || !dlk_attention_matrix_eligible(&p))) return static_cast<int>(hipErrorInvalidValue);
    // the staged output exists only on the prefill kernel
    if (p.stage_out) {
        if (!dlk_attention_prefill_eligible(&p) || (p.H * p.hd) % 32 != 0 ||
            reinterpret_cast<uintptr_t>(p.stage_out) % 16 != 0)
            return static_cast<int>(hipErrorInvalidValue);
        return dlk_attention_prefill(&p, stream_handle);
    }
    // one position on the matrix cores, then the merge of its key splits
    if (dlk_attention_matrix_eligible(&p)) {
        const int status = dlk_attention_matrix_decode(&p, stream_handle);
        if (status != 0 || p.splits == 1 || p.partials_only) return status;
        return p.hd == 64 ? dlk::launch_combine<64>(p, stream) : dlk::launch_combine<128>(p, stream);
    }
    if (dlk_attention_prefill_eligible(&p)) return dlk_attention_prefill(&p, stream_handle);
    if (p.hd < 16) {
        switch (p.hd) {
        case 2: return p.kv_bf16 ? dlk::launch_small<uint16_t, 2>(p, stream) : dlk::launch_small<float, 2>(p, stream);
        case 4: return p.kv_bf16 ? dlk::launch_small<uint16_t, 4>(p, stream) : dlk::launch_small<float, 4>(p, stream);
        case 8: return p.kv_bf16 ? dlk::launch_small<uint16_t, 8>(p, stream) : dlk::launch_small<float, 8>(p, stream);
        default: return static_cast<int>(hipErrorInvalidValue);
        }
    }
    if (p.kv_bf16) {
        switch (p.hd) {
        case 16: return dlk::launch<uint16_t, 16>(p, stream);
        case 32: return dlk::launch<uint16_t, 32>(p, stream);
        case 64: return dlk::launch<uint16_t, 64>(p, stream);
        case 128: return dlk::launch<uint16_t, 128>(p, stream);
        default: return static_cast<int>(hipErrorInvalidValue);
        }
    }
    switch (p.hd) {
    case 16: return dlk::launch<float, 16>(p, stream);
    case 32: return dlk::launch<float, 32>(p, stream);
    case 64: return dlk::launch<float, 64>(p, stream);
    case 128: return dlk::launch<float, 128>(p, stream);
    default: return static_cast<int>(hipErrorInvalidValue);
    }
}
