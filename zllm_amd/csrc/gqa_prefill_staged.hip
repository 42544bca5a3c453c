// Chunked-prefill GQA attention over Q8g64 rows of head_dim 128 that are converted once a call instead of once a row tile: what it computes
// is gqa_prefill_q8 (gqa_prefill.hip), for calls of full-size row tiles whose workspace has the room (gqa_prefill_staged_tiles).
//
// gqa_stage_q8 writes K and V of the call into the workspace as f16 integers (exact), in the order in which the matrix instructions take
// them, with the f32 scales beside them.  gqa_prefill_staged then moves tiles straight from memory to LDS: no registers, conversions,
// addresses or LDS stores in its loop, where gqa_prefill_q8 spends a fifth of its vector instructions on them, and every row tile does.
// 2,048 rows behind 50,000 keys (64 / 8 heads): 4,500 -> 3,840 us a pass, appends included (3,735 on the fastest card met; the kernel 3,710, the
// staging 69).  Distance from 64 bits as before (2-norm, scores of deviation 1):
// 1.43e-4 there, 1,000 rows behind 20,000 (32 / 8) 1.51e-4 -> 1.50e-4, 333 behind 3,000 (24 / 8) 1.4e-6 -> 1.2e-6.
//
// What bounds the loop: the vector ALU (68 % of a SIMD's cycles) beside the matrix cores (44 %), and the power of both: of its 2.4 GHz the
// device holds 2.0 to 2.1, so that instructions and LDS bytes count even where they are hidden.  Hence
//   32x32x16 tiles: a wave owns 32 pairs and the vector ALU runs beside the matrix cores (with 16x16x32 tiles it hardly does).
//   Scales come to a lane as two words a tile and are multiplied as lane reads of the row of sixteen (row_lane): read from LDS element by
//       element they were half of its traffic (16 of 32 reads a tile and wave; 4,105 -> 3,850 us, built without any scales 20 % less).
//   A tile is sixteen slots of one matrix instruction and the vector instructions that do not wait for it: the keys of the next tile
//       under the exponentials, the values under the packing and the scaling of the next scores (4,586 -> 4,105 us against scores,
//       softmax and values one after the other; three workgroups of four such waves on a compute unit, in parts, 4,424).
#include <type_traits>

#include "gqa_prefill_x32.hpp"

namespace zllm {

namespace {

constexpr int kD = 128;
constexpr int kTile = kStep * kD * 2; // bytes of one 32-token tile as f16
constexpr int kGroups = kD / 64;
constexpr int kScales = kGroups * kStep * 4; // bytes of a tile's f32 scales, [token][group]
constexpr int kWaves = 8; // of 32 pairs each
constexpr int kBufs = 6; // three passes of two tiles: one attended, one complete or on its way, one requested
// A staged tile: K | V | K scales | V scales | the (biased) exponents of the largest V scale of its first 1, 2 ... 32 tokens.  K and V lie as the matrix instructions take
// them, 1 KiB a fragment, 16 bytes a lane: K fragment ks holds columns 16 ks + 8 h .. + 8 of token c (lane 32 h + c), V fragment 2 t + kk
// column 32 t + c of tokens 16 kk + 4 h .. + 4 and eight further.
constexpr int kKsAt = 2 * kTile, kVsAt = 2 * kTile + kScales, kTopAt = 2 * kTile + 2 * kScales;
constexpr int kBlock = kTopAt + 128;
constexpr float kLoThresholdHalves = 24.0f; // see kLoThreshold: a half's walk is short, as those of the kernels whose reference lags are (16)
constexpr int kBlocksBehind = 8; // a part's requests run up to seven tiles past its last

// One tile of one KV head a workgroup; bound by the memory it reads and writes.
template <int SDT> __global__ __launch_bounds__(256) void gqa_stage_q8(GqaPrefillParams p)
{
    const unsigned int tid = threadIdx.x;
    const unsigned int tile = blockIdx.x, kvh = blockIdx.y;
    const unsigned int t0 = (p.staged_first + tile) * kStep, end = p.position + p.rows;
    unsigned char* const block = p.staged + ((size_t)kvh * p.staged_tiles + tile) * kBlock;
    __shared__ unsigned long long rows[kStep];
    if (tid < kStep) {
        // tokens past the end are the last one again, with scales of zero
        rows[tid] = paged_row(p.table, min(t0 + tid, end - 1u), p.block_tokens, 0u) * p.num_kv_heads + kvh;
    }
    __syncthreads();
    if (tid < 128u) { // K: 32 columns of a token
        const unsigned int token = tid >> 2, quarter = tid & 3u;
        const unsigned char* const from = p.k_plane + rows[token] * kD + quarter * 32u;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const u32x4 codes = *(const u32x4*)(from + 16 * ks);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                u32x4 out;
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    unsigned int a, b;
                    codes4_to_f16(codes[2 * h + e], a, b);
                    out[2 * e] = a;
                    out[2 * e + 1] = b;
                }
                *(u32x4*)(block + (2u * quarter + ks) * 1024u + h * 512u + token * 16u) = out;
            }
        }
    } else { // V: four columns of eight tokens
        const unsigned int at = tid - 128u, quad = at & 31u, kk = at >> 6, h = (at >> 5) & 1u;
        const unsigned int first = 16u * kk + 4u * h;
        unsigned int w[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            w[j] = *(const unsigned int*)(p.v_plane + rows[first + (j & 3) + (j >> 2) * 8] * kD + quad * 4u);
        }
        u32x4 out[4];
#pragma unroll
        for (int n = 0; n < 2; ++n) { // four tokens of four columns, transposed
            const unsigned int a = __builtin_amdgcn_perm(w[4 * n + 1], w[4 * n], 0x05010400u), b = __builtin_amdgcn_perm(w[4 * n + 3], w[4 * n + 2], 0x05010400u);
            const unsigned int c = __builtin_amdgcn_perm(w[4 * n + 1], w[4 * n], 0x07030602u), d = __builtin_amdgcn_perm(w[4 * n + 3], w[4 * n + 2], 0x07030602u);
            const unsigned int columns[4] = {__builtin_amdgcn_perm(b, a, 0x05040100u), __builtin_amdgcn_perm(b, a, 0x07060302u),
                                             __builtin_amdgcn_perm(d, c, 0x05040100u), __builtin_amdgcn_perm(d, c, 0x07060302u)};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                unsigned int lo, hi;
                codes4_to_f16(columns[e], lo, hi);
                out[e][2 * n] = lo;
                out[e][2 * n + 1] = hi;
            }
        }
        unsigned char* const to = block + kTile + (2u * (quad >> 3) + kk) * 1024u + h * 512u + (quad & 7u) * 64u;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            *(u32x4*)(to + e * 16) = out[e];
        }
    }
    if (tid < 2u * kGroups * kStep) { // a scale each: [plane][token][group], two waves
        const unsigned int token = (tid / kGroups) & 31u, group = tid % kGroups;
        const bool of_v = tid >= kGroups * kStep;
        float scale = 0.0f;
        if (t0 + token < end) {
            const size_t at = rows[token] * kGroups + group;
            const unsigned char* const plane = of_v ? p.v_scales : p.k_scales;
            if constexpr (SDT == 2) {
                scale = ((const float*)plane)[at];
            } else {
                scale = scale_bits_to_f32<SDT>(((const unsigned short*)plane)[at]);
            }
        }
        // K scales carry the score scale (and log2 e unless a soft cap needs natural units): the loop does not multiply again
        const float fold = of_v ? 1.0f : p.softcap > 0.0f ? p.score_scale : p.score_scale * kLog2e;
        ((float*)(block + kKsAt))[tid] = scale * fold;
        if (of_v) { // the second wave
            unsigned int top = __float_as_uint(fmaxf(scale, 0.0f));
            top = max(top, (unsigned int)__shfl_xor((int)top, 1));
#pragma unroll
            for (int d = kGroups; d < 64; d <<= 1) {
                const unsigned int before = (unsigned int)__shfl_up((int)top, d);
                top = max(top, (tid & 63u) >= (unsigned int)d ? before : 0u);
            }
            if (group == 0u) { // clamped away from the ends of the f32 range
                ((unsigned int*)(block + kTopAt))[token] = min(max((top >> 23) & 0xffu, 2u), 252u);
            }
        }
    }
}

// SOFTCAP: 0 none, 1 caps below 256, 2 larger ones (see gqa_prefill_f16)
// HALVES 1: eight waves of 32 pairs, a wave attends both tiles of a pass.  HALVES 2: four waves of 32 pairs for even tiles and four for odd ones,
// which meet once, at the end: first chunks, whose last row tiles walk longest.  Their reference lags (kSlack): with the maximum itself 2,048 rows of
// 32 / 8 heads 101 -> 97 us (the kernel it stands in for: 111).  Distance from 64 bits there (2-norm) 2.4e-5 in that kernel, 2.8e-6 here.
template <int SOFTCAP, int HALVES> __global__ __launch_bounds__(64 * kWaves, 2) void gqa_prefill_staged(GqaPrefillParams p)
{
    struct Lds {
        unsigned char k[kBufs][kTile];
        unsigned char v[kBufs][kTile];
        float scales[kBufs][2][kStep][kGroups]; // of K and V
    };
    constexpr int kSide = kWaves / HALVES; // waves of a half
    constexpr unsigned int kPairs = 32 * kSide;
    struct Meeting { // of the halves, over the tiles
        float acc[kD / 8][kSide][64][4];
        float stats[3][kSide][64];
    };
    __shared__ __align__(1024) union {
        Lds lds;
        Meeting meeting;
    } shared;
    Lds& lds = shared.lds;

    const unsigned int tid = threadIdx.x;
    const unsigned int lane = tid & 63u;
    const unsigned int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned int m = lane & 15u;
    const unsigned int c = lane & 31u; // the lane's column: a pair
    const unsigned int h = lane >> 5;
    // row tiles with the longest range first, the KV head as the fast index (see gqa_prefill_q8)
    const unsigned int kvh = blockIdx.x % p.num_kv_heads;
    const unsigned int half = HALVES == 1 ? 0u : wave / kSide, side = HALVES == 1 ? wave : wave % kSide;
    const unsigned int rows_per_wg = max(1u, kPairs / p.group);
    const unsigned int row0 = (gridDim.x / p.num_kv_heads - 1u - blockIdx.x / p.num_kv_heads) * rows_per_wg;
    const unsigned int cols_used = rows_per_wg * p.group;
    const unsigned int col = side * 32u + c;
    const unsigned int col_row = row0 + col / p.group;
    const unsigned int col_head = kvh * p.group + col % p.group;
    const bool col_valid = col < cols_used && col_row < p.rows;
    const unsigned int last_row = min(row0 + rows_per_wg, p.rows) - 1u;

    Frag qf[kD / 16];
    {
        const size_t q_at = ((size_t)col_row * p.num_heads + col_head) * kD + h * 8u;
#pragma unroll
        for (int ks = 0; ks < kD / 16; ++ks) {
            qf[ks].u = u32x4{0u, 0u, 0u, 0u};
            if (col_valid) {
                qf[ks].u = *(const u32x4*)((const unsigned short*)p.q + q_at + ks * 16);
            }
        }
    }
    const unsigned int t_end = p.position + last_row + 1u;
    unsigned int t_begin = 0;
    if (p.window != 0) {
        const unsigned int first_pos = p.position + row0 + 1u;
        t_begin = first_pos > p.window ? first_pos - p.window : 0u;
    }
    t_begin &= ~31u;
    const SplitRange part = split_range(p, t_begin, t_end);
    if (!part.live) {
        if (col_valid && h == 0u && half == 0u) {
            store_empty_record(p, col_row, col_head);
        }
        return;
    }
    const unsigned int steps = (part.end - part.begin + kStep - 1) / kStep;

    // ---- staging.  Pass n of the loop attends tiles 2 n and 2 n + 1 and multiplies the keys of the HALVES tiles ahead of them: their K are loaded
    // beside the V of the first two, a fragment of each a wave, and a piece of the scales (the waves' pieces repeat).  Requests run past the range
    // into what follows in the workspace (kBlocksBehind); nothing of that is attended.
    const unsigned char* const staged = p.staged + ((size_t)kvh * p.staged_tiles + (part.begin / kStep - p.staged_first)) * kBlock;
    const unsigned int lds_base = (unsigned int)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)&lds;
    const unsigned int lane16 = lane * 16u, lane4 = lane * 4u;
    const unsigned int wave_lds = lds_base + wave * 1024u;
    const bool scales_of_v = (wave & 2u) != 0u;
    const unsigned int scales_tile = (wave & 1u) + (scales_of_v ? 0u : (unsigned int)HALVES); // of the pass: HALVES more for K
    const unsigned int scales_from = scales_tile * kBlock + kKsAt + (scales_of_v ? kScales : 0u);
    const unsigned int scales_lds = lds_base + offsetof(Lds, scales) + (scales_of_v ? kScales : 0u);
    auto load_pass = [&](auto which, const unsigned char* at) __attribute__((always_inline)) { // tiles from `at` on
        constexpr int set = decltype(which)::value;
        constexpr unsigned int k_at = offsetof(Lds, k), v_at = offsetof(Lds, v);
        const unsigned char* const from = at + wave * 1024u;
        load_to_lds<true, k_at + (2 * set + HALVES) % kBufs * kTile>(from + HALVES * kBlock, lane16, wave_lds);
        load_to_lds<true, v_at + 2 * set * kTile>(from + kTile, lane16, wave_lds);
        load_to_lds<true, k_at + (2 * set + 1 + HALVES) % kBufs * kTile>(from + (1 + HALVES) * kBlock, lane16, wave_lds);
        load_to_lds<true, v_at + (2 * set + 1) * kTile>(from + kBlock + kTile, lane16, wave_lds);
        const unsigned int buf = set == 2 && scales_tile >= 2u ? scales_tile - 2u : 2u * set + scales_tile;
        load_to_lds<false, 0>(at + scales_from, lane4, scales_lds + buf * (2 * kScales));
    };
#pragma unroll
    for (int n = 0; n < HALVES; ++n) { // the first keys
        load_to_lds<true, offsetof(Lds, k)>(staged + n * kBlock + wave * 1024u, lane16, wave_lds + n * kTile);
        load_to_lds<false, offsetof(Lds, scales)>(staged + n * kBlock + kKsAt, lane4, lds_base + n * (2 * kScales));
    }
    load_pass(std::integral_constant<int, 0>{}, staged);
    load_pass(std::integral_constant<int, 1>{}, staged + 2 * kBlock);

    // The wave's queries as f16 after a multiplication by one power of two that puts their largest magnitude into [2^8, 2^9)
    // (exact for bf16 and f16); the inverse goes into the score factor.
    float q_fac;
    {
        float q_amax = 0.0f;
#pragma unroll
        for (int ks = 0; ks < kD / 16; ++ks) {
            float x[8];
            widen8(qf[ks].u, p.q_dtype, x);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                q_amax = fmaxf(q_amax, fabsf(x[e]));
            }
        }
        q_amax = __uint_as_float(wave_max_u(__float_as_uint(q_amax))); // magnitudes: their bits order as they do
        const unsigned int q_exp = min(max((__float_as_uint(q_amax) >> 23) & 0xffu, 16u), 240u);
        const float q_mul = __uint_as_float((262u - q_exp) << 23); // 2^(127 + 8 - q_exp)
#pragma unroll
        for (int ks = 0; ks < kD / 16; ++ks) {
            float x[8];
            widen8(qf[ks].u, p.q_dtype, x);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                qf[ks].u[e] = pack_f16_hw(x[2 * e] * q_mul, x[2 * e + 1] * q_mul);
            }
        }
        q_fac = ldexpf(1.0f, (int)q_exp - 135);
    }
    const float mult = SOFTCAP ? p.softcap * kLog2e : q_fac; // positive: maxima first, the factor rides in the multiply-add
    const float tanh_arg = SOFTCAP ? q_fac * (2.0f * kLog2e) / p.softcap : 0.0f; // scaled product -> 2 y log2(e), y = score / cap
    const float cap_arg = SOFTCAP ? q_fac * (1.0f / p.softcap) : 0.0f;

    f32x16 acc[kD / 32];
#pragma unroll
    for (int t = 0; t < kD / 32; ++t) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            acc[t][i] = 0.0f;
        }
    }
    float run_max = kNegInf, ref_shift = kPBias;
    [[maybe_unused]] float lane_top = kNegInf; // halves: the largest score the lane has met
    bool two_terms = true; // the tile before carried both terms of its probabilities
    float run_sum[2] = {0.0f, 0.0f}; // of the lane's first and second eight tokens of each step
    unsigned int vis_lo, vis_hi;     // visible tokens [lo, hi) of the column's row
    {
        const unsigned int pos = p.position + col_row;
        vis_hi = col_valid ? pos + 1u : 0u;
        vis_lo = p.window != 0 && pos + 1u > p.window ? pos + 1u - p.window : 0u;
    }
    // the tokens that every column of the wave sees are [max_lo, min_hi)
    const unsigned int wave_min_hi = wave_min_u(vis_hi), wave_max_lo = wave_max_u(vis_lo);

    // a half's tiles lie in the buffer of its number behind the pass's first
    const unsigned int frag_at = lane16 + half * kTile;
    const unsigned int scale_at = (8u * (m >> 2) + 4u * h + (m & 3u)) * kGroups + half * (2u * kStep * kGroups); // lane m of a row of sixteen: element m's token

    f32x16 s; // the tile's scores, up to the query's power of two; multiplied a step ahead
    f32x16 d[kGroups];
    auto multiply_keys = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int g = 0; g < kGroups; ++g) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                d[g][i] = 0.0f;
            }
        }
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
            for (int g = 0; g < kGroups; ++g) {
                Frag kf;
                kf.u = *(const u32x4*)(lds.k[buf] + frag_at + (g * 4 + ks) * 1024);
                d[g] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf.h, qf[g * 4 + ks].h, d[g], 0, 0, 0);
            }
        }
    };
    auto scales_of = [&](int buf, int plane) __attribute__((always_inline)) { return *(const f32x2*)(&lds.scales[buf][plane][0][0] + scale_at); };
    // s = sum_g scale_g d_g, four elements; `settled`: an element of d[1] times something, which the compiler has waited for
    auto scale_scores = [&](const f32x2& scale, int q, float settled) __attribute__((always_inline)) {
        float t[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            t[r] = row_lane(scale[0], 4 * q + r) * d[0][4 * q + r];
        }
        row_lane_fmac4(t[0], t[1], t[2], t[3], scale[1], q, d[1][4 * q], d[1][4 * q + 1], d[1][4 * q + 2], d[1][4 * q + 3], settled);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            s[4 * q + r] = t[r];
        }
    };

    auto attend = [&](int buf, unsigned int t0, float v_shift, float acc_fix, bool window_moved) __attribute__((always_inline)) {
        const int next = (buf + HALVES) % kBufs;
        constexpr int kAhead = 3, kRing = kAhead + 1;
        Frag frag[kRing];
        auto request = [&](int n) __attribute__((always_inline)) { // of slot n
            if (n < 8) {
                frag[n % kRing].u = *(const u32x4*)(lds.k[next] + frag_at + ((n & 1) * 4 + n / 2) * 1024);
            } else if (n < 16) {
                const int j = n - 8, t = (j >> 2) * 2 + (j & 1), kk = (j >> 1) & 1;
                frag[n % kRing].u = *(const u32x4*)(lds.v[buf] + frag_at + (2 * t + kk) * 1024);
            }
        };
#pragma unroll
        for (int n = 0; n < kAhead; ++n) {
            request(n);
        }
        // ---- online softmax of the lane's column ----
        if constexpr (SOFTCAP == 1) { // see gqa_prefill_f16
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const float e2y = __builtin_amdgcn_exp2f(s[i] * tanh_arg);
                s[i] = fmaf(-2.0f, __builtin_amdgcn_rcpf(e2y + 1.0f), 1.0f);
            }
        } else if constexpr (SOFTCAP == 2) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                s[i] = soft_tanh(s[i] * cap_arg);
            }
        }
        if (t0 + kStep > wave_min_hi || t0 < wave_max_lo) { // only steps at an edge of some column need the per-token masks
            unsigned int first = t0 + 4u * h;
            asm volatile("" : "+v"(first)); // or sixteen additions leave the branch
            // What the tile's last rows do not see counts as zero, or an infinite V scale there would meet their probabilities of zero: every wave
            // clears the same scales and reads them behind its own writes.
            if (t0 + kStep > part.end && first + 8u * (m >> 2) + (m & 3u) >= part.end) {
                *(f32x2*)(&lds.scales[buf][1][0][0] + scale_at) = f32x2{0.0f, 0.0f};
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const unsigned int token = first + 8u * (i >> 2) + (i & 3);
                s[i] = (token >= vis_lo && token < vis_hi) ? s[i] : kNegInf;
            }
        }
        float lane_max = fmaxf(s[0], s[8]), upper = fmaxf(s[1], s[9]); // two chains
#pragma unroll
        for (int i = 2; i < 8; i += 2) {
            lane_max = fmaxf(fmaxf(lane_max, s[i]), s[i + 8]);
            upper = fmaxf(fmaxf(upper, s[i + 1]), s[i + 9]);
        }
        lane_max = fmaxf(lane_max, upper) * mult;
        bool behind = false, move;
        if constexpr (HALVES == 1) {
            move = __any(lane_max > run_max);
        } else { // first chunks: the reference lags while the tiles carry both terms (see kSlack)
            lane_max = lane_top = fmaxf(lane_top, lane_max);
            behind = __any(lane_top > run_max);
            move = two_terms ? __any(lane_top - run_max > kSlack) : behind;
        }
        if (move || window_moved) {
            behind = false;
            const float new_max = fmaxf(run_max, halves_max(lane_max));
            const float safe_max = new_max == kNegInf ? 0.0f : new_max;
            const float alpha = __builtin_amdgcn_exp2f(run_max - safe_max) * acc_fix;
            ref_shift = v_shift - safe_max;
            run_sum[0] *= alpha;
            run_sum[1] *= alpha;
            run_max = new_max;
            if (__any(alpha != 1.0f)) {
#pragma unroll
                for (int t = 0; t < kD / 32; ++t) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        acc[t][i] *= alpha;
                    }
                }
            }
        }
        PREFILL_PHASE_FENCE();
        // ---- sixteen slots, one matrix instruction each: the next tile's keys (0..7) under this tile's exponentials, then this tile's
        // values (8..15) under the packing of the second group's probabilities and the scaling of the next scores.  What a slot reads
        // from LDS is requested kAhead slots before.
        float pr[16];
        float part_sum[2][2] = {{0.0f, 0.0f}, {0.0f, 0.0f}};
        float settled = 0.0f;
        Frag ph[2][2]; // [group][tokens 16 kk ..]
        const f32x2 v_scale = scales_of(buf, 1), k_scale = scales_of(next, 0);
        auto pack = [&](int g, int q) __attribute__((always_inline)) { // elements 4 q .. + 4
            const float x0 = row_lane(v_scale[g], 4 * q) * pr[4 * q], x1 = row_lane(v_scale[g], 4 * q + 1) * pr[4 * q + 1];
            const float x2 = row_lane(v_scale[g], 4 * q + 2) * pr[4 * q + 2], x3 = row_lane(v_scale[g], 4 * q + 3) * pr[4 * q + 3];
            ph[g][q >> 1].u[(q & 1) * 2] = pack_f16_hw(x0, x1);
            ph[g][q >> 1].u[(q & 1) * 2 + 1] = pack_f16_hw(x2, x3);
        };
#pragma unroll
        for (int g = 0; g < kGroups; ++g) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                d[g][i] = 0.0f;
            }
        }
        __builtin_amdgcn_s_setprio(1); // a wave among its slots goes before one at its softmax: 3,925 -> 3,852 us
#pragma unroll
        for (int n = 0; n < 16; ++n) {
            request(n + kAhead);
            if (n < 8) {
                d[n & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(frag[n % kRing].h, qf[(n & 1) * 4 + n / 2].h, d[n & 1], 0, 0, 0);
#pragma unroll
                for (int e = 2 * n; e < 2 * n + 2; ++e) {
                    pr[e] = __builtin_amdgcn_exp2f(fmaf(s[e], mult, ref_shift));
                    part_sum[e >> 3][e & 1] += pr[e];
                }
            } else {
                const int j = n - 8, g = j >> 2, t = g * 2 + (j & 1), kk = (j >> 1) & 1;
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(frag[n % kRing].h, ph[g][kk].h, acc[t], 0, 0, 0);
            }
            if (n == 3 || n == 5 || n == 7) {
                pack(0, (n - 3) / 2);
            }
            if (n == 8) {
                pack(0, 3);
            }
            if (n >= 8 && n < 12) {
                pack(1, n - 8);
            }
            if (n == 12) {
                settled = d[1][0] * mult;
                asm volatile("" : "+v"(settled));
            }
            if (n >= 12) {
                scale_scores(k_scale, n - 12, settled);
            }
            PREFILL_PHASE_FENCE();
        }
        __builtin_amdgcn_s_setprio(0);
        bool heavy = false;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float eight = part_sum[e][0] + part_sum[e][1];
            run_sum[e] += eight;
            heavy = heavy || (HALVES == 1 && eight * kLoThreshold > run_sum[e]);
        }
        if constexpr (HALVES == 2) { // the two sums of a half are those of a quarter of the row's tokens, as in the kernels whose reference lags
            const float most = fmaxf(part_sum[0][0] + part_sum[0][1], part_sum[1][0] + part_sum[1][1]);
            heavy = most * kLoThresholdHalves > run_sum[0] + run_sum[1];
        }
        two_terms = __any(heavy);
        const bool lo_pass = two_terms || behind;
        if (lo_pass) { // what f16 has dropped of the probabilities
#pragma unroll
            for (int g = 0; g < kGroups; ++g) {
                Frag pl[2];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float x0 = row_lane(v_scale[g], 4 * q) * pr[4 * q], x1 = row_lane(v_scale[g], 4 * q + 1) * pr[4 * q + 1];
                    const float x2 = row_lane(v_scale[g], 4 * q + 2) * pr[4 * q + 2], x3 = row_lane(v_scale[g], 4 * q + 3) * pr[4 * q + 3];
                    const f16x2 h0 = __builtin_bit_cast(f16x2, pack_f16_hw(x0, x1)), h1 = __builtin_bit_cast(f16x2, pack_f16_hw(x2, x3));
                    pl[q >> 1].u[(q & 1) * 2] = pack_f16_hw(x0 - (float)h0[0], x1 - (float)h0[1]);
                    pl[q >> 1].u[(q & 1) * 2 + 1] = pack_f16_hw(x2 - (float)h1[0], x3 - (float)h1[1]);
                }
#pragma unroll
                for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
                    for (int t = 2 * g; t < 2 * g + 2; ++t) {
                        Frag vf;
                        vf.u = *(const u32x4*)(lds.v[buf] + frag_at + (2 * t + kk) * 1024);
                        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf.h, pl[kk].h, acc[t], 0, 0, 0);
                    }
                }
            }
        }
    };

    // ---- main loop ----
    unsigned int wv = 2u; // (biased) exponent of the largest V scale up to the tile being attended
    float v_shift = kPBias + 125.0f;
    // the exponents come by scalar loads, two tiles ahead
    const unsigned char* pass_at = staged;
    auto load_top = [&](unsigned int tile) __attribute__((always_inline)) -> unsigned int { // `tile` tiles past the pass's first
        return *(scalar_words_t)(uintptr_t)(pass_at + tile * kBlock + kTopAt + (kStep - 1) * 4);
    };
    const unsigned int last_top = *(scalar_words_t)(uintptr_t)(staged + (steps - 1u) * kBlock + kTopAt + (part.end - part.begin - (steps - 1u) * kStep - 1u) * 4u); // of what its rows see
    unsigned int top_now = load_top(half), top_next = load_top(half + 1u * HALVES);
    auto attend_tile = [&](unsigned int step, int buf) __attribute__((always_inline)) {
        const unsigned int wv_now = max(wv, step + 1u == steps ? last_top : top_now);
        top_now = top_next;
        top_next = load_top(HALVES == 1 ? 2u + (buf & 1) : half + 4u);
        const bool window_moved = wv_now != wv; // rare: a V scale above everything met so far
        float acc_fix = 1.0f;
        if (window_moved) {
            acc_fix = ldexpf(1.0f, (int)wv - (int)wv_now);
            wv = wv_now;
            v_shift = kPBias + (float)(127 - (int)wv);
        }
        attend(buf, part.begin + step * kStep, v_shift, acc_fix, window_moved);
    };
    // A pass first waits for its loads (a wave for its own, the barrier for the others'), which also says that nobody reads what the pass
    // before it has attended: those are the buffers of the pass requested next.
    auto wait_pass = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(5) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    auto pass_of = [&](unsigned int step, auto which) __attribute__((always_inline)) {
        constexpr int set = decltype(which)::value;
        wait_pass();
        load_pass(std::integral_constant<int, (set + 2) % 3>{}, pass_at + 4 * kBlock);
        if constexpr (HALVES == 1) {
            attend_tile(step, 2 * set);
            if (step + 1u < steps) {
                attend_tile(step + 1u, 2 * set + 1);
            }
        } else if (step + half < steps) {
            attend_tile(step + half, 2 * set);
        }
        pass_at += 2 * kBlock;
    };
    if constexpr (HALVES == 1) {
        wait_pass();
    } else { // the first keys of both halves are behind the loads of two passes
        asm volatile("s_waitcnt vmcnt(10)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    }
    multiply_keys(0);
    {
        float settled = d[1][0] * mult;
        asm volatile("" : "+v"(settled));
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            scale_scores(scales_of(0, 0), q, settled);
        }
    }
    for (unsigned int step = 0;;) {
        pass_of(step, std::integral_constant<int, 0>{});
        if ((step += 2u) >= steps) {
            break;
        }
        pass_of(step, std::integral_constant<int, 1>{});
        if ((step += 2u) >= steps) {
            break;
        }
        pass_of(step, std::integral_constant<int, 2>{});
        if ((step += 2u) >= steps) {
            break;
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // what was requested past the range lands before the LDS is given back

    float total = halves_sum(run_sum[0] + run_sum[1]);
    if constexpr (HALVES == 2) {
        Meeting& meeting = shared.meeting;
        __syncthreads(); // the tiles are read no more
        if (half == 1u) {
            meeting.stats[0][side][lane] = run_max;
            meeting.stats[1][side][lane] = total;
            meeting.stats[2][side][lane] = v_shift;
#pragma unroll
            for (int n = 0; n < kD / 8; ++n) {
                *(f32x4*)meeting.acc[n][side][lane] = f32x4{acc[n / 4][n % 4 * 4], acc[n / 4][n % 4 * 4 + 1], acc[n / 4][n % 4 * 4 + 2], acc[n / 4][n % 4 * 4 + 3]};
            }
        }
        __syncthreads();
        if (half == 1u) {
            return;
        }
        // to the larger reference and the larger window (a half whose sum is zero may have seen nothing)
        const float other_max = meeting.stats[0][side][lane], other_total = meeting.stats[1][side][lane], other_shift = meeting.stats[2][side][lane];
        const float common = fmaxf(run_max, other_max), shift = fminf(v_shift, other_shift);
        const float own_fac = run_max == kNegInf ? 0.0f : __builtin_amdgcn_exp2f((run_max - common) + (shift - v_shift));
        const float other_fac = other_max == kNegInf ? 0.0f : __builtin_amdgcn_exp2f((other_max - common) + (shift - other_shift));
        total = total * own_fac + other_total * other_fac;
#pragma unroll
        for (int n = 0; n < kD / 8; ++n) {
            const f32x4 other = *(const f32x4*)meeting.acc[n][side][lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                acc[n / 4][n % 4 * 4 + e] = acc[n / 4][n % 4 * 4 + e] * own_fac + other[e] * other_fac;
            }
        }
        run_max = common;
        v_shift = shift;
    }
    if (!col_valid) {
        return;
    }
    store_column<kD>(p, col_row, col_head, h, run_max, total, acc, v_shift);
}

} // namespace

uint64_t gqa_prefill_staged_bytes(unsigned int tiles, unsigned int num_kv_heads)
{
    return ((uint64_t)tiles * num_kv_heads + kBlocksBehind) * kBlock;
}

hipError_t launch_gqa_prefill_staged(const GqaPrefillParams& p, int scale_dtype, hipStream_t stream)
{
    const dim3 tiles(p.staged_tiles, p.num_kv_heads);
    if (scale_dtype == 0) {
        gqa_stage_q8<0><<<tiles, dim3(256), 0, stream>>>(p);
    } else if (scale_dtype == 1) {
        gqa_stage_q8<1><<<tiles, dim3(256), 0, stream>>>(p);
    } else {
        gqa_stage_q8<2><<<tiles, dim3(256), 0, stream>>>(p);
    }
    auto launch = [&](auto softcap, auto halves) {
        constexpr unsigned int kPairs = 32 * kWaves / decltype(halves)::value;
        const unsigned int rows_per_wg = p.group >= kPairs ? 1u : kPairs / p.group;
        const dim3 grid((p.rows + rows_per_wg - 1) / rows_per_wg * p.num_kv_heads, 1, p.max_chunks > 1u ? p.max_chunks : 1u);
        gqa_prefill_staged<decltype(softcap)::value, decltype(halves)::value><<<grid, dim3(64 * kWaves), 0, stream>>>(p);
    };
    auto launch_halves = [&](auto halves) {
        if (!(p.softcap > 0.0f)) {
            launch(std::integral_constant<int, 0>{}, halves);
        } else if (p.softcap < 256.0f) {
            launch(std::integral_constant<int, 1>{}, halves);
        } else {
            launch(std::integral_constant<int, 2>{}, halves);
        }
    };
    p.staged_halves ? launch_halves(std::integral_constant<int, 2>{}) : launch_halves(std::integral_constant<int, 1>{});
    return hipGetLastError();
}

} // namespace zllm
