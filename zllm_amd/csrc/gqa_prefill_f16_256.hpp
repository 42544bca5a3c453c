// Chunked-prefill GQA attention over f16 rows at head_dim 256: the long walks of gqa_prefill_tiles (gqa_prefill.hip, kHalvesKeys), over pages that it can
// address by scalars (sixteen tokens at least, see prefill_scalar_pages).
//
// A workgroup is 128 (row, head-in-group) pairs, as there: the models of this head dimension have few query heads a KV head, and tiles of 256
// would leave half the device idle.  Its eight waves are four of 32 pairs for even 32-token tiles and four for odd ones, each half with
// a softmax of its own, and the halves meet once, at the end, in LDS.  So 32x32x16 tiles (a fragment feeds 32 pairs), two waves a SIMD
// and no exchange in the loop, where gqa_prefill_tiles has eight waves of 16 pairs.
// 2,048 rows behind 6,144 keys (16 / 8 heads, soft cap 50), a full layer and one of window 1,024 together: 437 -> 387 us a pass, appends
// included (382 to 394 by the card).  Distance from 64 bits (2-norm) there 1.55e-4 -> 1.44e-4 and 6.6e-5 -> 3.4e-5, 64 rows behind 30,000 6.0e-5 -> 2.2e-5.
//
// What bounds the loop: both waves of a SIMD run the matrix instructions and the vector ALU one after the other and hide little of one behind the
// other's (44 % and 50 % of the cycles in the full layer); what hides is what stands between a wave's own matrix instructions: with the exponentials
// of a tile's second sixteen tokens under the first sixteen's products 407 -> 391, and without spills in the loop (fresh_lane) 391 -> 387.  Tried: the odd half half a pass behind
// (spills in the loop, 457), raised priority for either phase (level), 64 pairs a wave and one wave a SIMD (70 spills).
#pragma once

#include "gqa_prefill_x32.hpp"

namespace zllm {

namespace {

namespace halves256 {

constexpr int kD = 256;
constexpr int kRow = kD * 2;         // bytes of one token of one KV head
constexpr int kWaves = 4;            // of 32 pairs each, in each half
constexpr int kPairs = 32 * kWaves;
constexpr int kHalves = 2;
constexpr int kPass = kHalves * kStep; // tokens
// A tile in LDS: sixteen pairs of rows of 1 KiB, what one load of 64 x 16 bytes fills, 1,056 bytes apart.  Token 16 k + 8 e + 4 h + q is row h of
// pair 8 k + 2 q + e, and row 1 has its neighbouring 16-byte chunks exchanged: the sixteen rows of a 16-byte read and the four rows x
// 64 bytes of a transposed one meet every bank once, and every address is one lane register plus a constant.
constexpr int kPairStride = 2 * kRow + 32;
constexpr int kTile = 16 * kPairStride;
constexpr int kHalfRun = 16;         // a wave's requests of a pass lie in one run of sixteen tokens
constexpr int kLoads = 4;            // loads a wave issues per plane and pass

// P is carried as f16 hi, and lo while eight probabilities of a lane weigh more than an eighth of the lane's sum: a lane sums a quarter of the
// row's tokens, sixteen of each second tile, as in gqa_prefill_tiles.  With a sixteenth 403 -> 413 us.
constexpr float kLoShare = 8.0f;

struct Lds {
    unsigned char tile[2][kHalves][2][kTile]; // [buffer][half][K, V]
};
struct Meeting { // of the halves, over the tiles
    float acc[kD / 32 * 4][kWaves][64][4];
    float stats[2][kWaves][64];
};
union Shared {
    Lds lds;
    Meeting meeting;
};

// One workgroup of 512 threads: keys [part.begin, part.end) of a row tile whose visible range ends at t_end.
// SOFTCAP: 0 none, 1 caps below 256, 2 larger ones (see gqa_prefill_f16)
template <int SOFTCAP> __device__ __forceinline__ void attend_part(const GqaPrefillParams& p, Shared& shared, const SplitRange& part, unsigned int t_end)
{
    Lds& lds = shared.lds;

    const unsigned int tid = threadIdx.x;
    const unsigned int lane = tid & 63u;
    const unsigned int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned int half = wave / kWaves, quarter = wave % kWaves;
    const unsigned int m = lane & 15u;
    const unsigned int c = lane & 31u; // the lane's column: a pair
    const unsigned int h = lane >> 5;
    // row tiles with the longest range first, the KV head as the fast index (see gqa_prefill_q8)
    const unsigned int kvh = blockIdx.x % p.num_kv_heads;
    const unsigned int rows_per_wg = max(1u, (unsigned int)kPairs / p.group);
    const unsigned int row0 = (gridDim.x / p.num_kv_heads - 1u - blockIdx.x / p.num_kv_heads) * rows_per_wg;
    const unsigned int cols_used = rows_per_wg * p.group;
    const unsigned int col = quarter * 32u + c;
    const unsigned int col_row = row0 + col / p.group;
    const unsigned int col_head = kvh * p.group + col % p.group;
    const bool col_valid = col < cols_used && col_row < p.rows;
    const unsigned int last_row = min(row0 + rows_per_wg, p.rows) - 1u;

    // ---- given ranges, then the query's rows, are requested before anything waits ----
    unsigned int own_end = 0, own_start = 0;
    if (p.visible_ends != nullptr) {
        const unsigned int own_row = min(col_row, last_row);
        own_end = min(p.visible_ends[own_row], p.position + p.rows);
        if (p.visible_starts != nullptr) {
            own_start = p.visible_starts[own_row];
        }
    }
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
    const unsigned int passes = (part.end - part.begin + kPass - 1) / kPass;

    // ---- staging.  Wave (half, quarter) requests pairs 4 quarter .. + 4 of its half's tile: tokens 8 e + 4 (lane / 32) + q of a run of
    // sixteen, for q = 2 (quarter % 2) .. + 2.  What is read past the range is its last row again.
    const unsigned int k_row = p.num_kv_heads * kRow;
    const unsigned int last_token = max(t_end, 1u) - 1u;
    const unsigned int q0 = 2u * (quarter & 1u);
    const unsigned int lane_at = (c ^ h) * 16u + kvh * kRow + 4u * h * k_row;
    const unsigned int lds_base = (unsigned int)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)&lds;
    const unsigned int lds_to = lds_base + half * (2 * kTile) + 4u * quarter * kPairStride;
    auto first_of = [&](unsigned int t0) __attribute__((always_inline)) -> unsigned int { // of the wave's run, inside the range
        const unsigned int t = t0 + half * kStep + (quarter >> 1) * kHalfRun;
        return t > last_token ? last_token & ~(unsigned int)(kHalfRun - 1) : t;
    };
    auto load_entry = [&](unsigned int t0) __attribute__((always_inline)) -> unsigned int {
        return ((scalar_words_t)(uintptr_t)p.table)[first_of(t0) >> p.block_shift];
    };
    auto load_pass = [&](int buf, unsigned int t0, unsigned int page) __attribute__((always_inline)) {
        const unsigned int t = first_of(t0), left = last_token - t;
        const unsigned long long at = (((unsigned long long)page << p.block_shift) + (t & (p.block_tokens - 1u))) * k_row;
        const unsigned int to = lds_to + (unsigned int)buf * (kHalves * 2 * kTile);
        const unsigned char* const kp = p.k_plane + at;
        const unsigned char* const vp = p.v_plane + at;
        const bool whole = left >= kHalfRun - 1u;
#pragma unroll
        for (int u = 0; u < kLoads; ++u) { // pair 4 quarter + u: q = q0 + u / 2, e = u % 2
            const unsigned int token = 8u * (u & 1) + q0 + (u >> 1);
            unsigned int from = lane_at + token * k_row;
            if (!whole) {
                const unsigned int l = fresh_lane(), lh = l >> 5;
                from = ((l & 31u) ^ lh) * 16u + kvh * kRow + min(token + 4u * lh, left) * k_row;
            }
            load_to_lds<true, 0>(kp, from, to + u * kPairStride);
            load_to_lds<true, kTile>(vp, from, to + u * kPairStride);
        }
    };
    unsigned int page = load_entry(part.begin);
    load_pass(0, part.begin, page);
    page = load_entry(part.begin + kPass);

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
    // what turns the accumulated product into a score in base-2 units (or, under a soft cap, into natural units first)
    const float score_mult = (SOFTCAP ? p.score_scale : p.score_scale * kLog2e) * q_fac;
    const float mult = SOFTCAP ? p.softcap * kLog2e : score_mult; // positive: maxima first, the factor rides in the multiply-add
    const float tanh_arg = SOFTCAP ? score_mult * (2.0f * kLog2e) / p.softcap : 0.0f; // product -> 2 y log2(e), y = score / cap
    const float cap_arg = SOFTCAP ? score_mult * (1.0f / p.softcap) : 0.0f;

    f32x16 acc[kD / 32];
#pragma unroll
    for (int t = 0; t < kD / 32; ++t) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            acc[t][i] = 0.0f;
        }
    }
    float run_max = kNegInf, ref_shift = kPBias;
    float run_sum = 0.0f; // of the lane's tokens, a quarter of the row's
    float lane_top = kNegInf; // the largest score the lane has met
    bool two_terms = true;    // the step before carried both terms of its probabilities (see kSlack)
    unsigned int vis_lo, vis_hi; // visible tokens [lo, hi) of the column's row
    {
        const unsigned int pos = p.position + col_row;
        unsigned int hi = pos + 1u;
        unsigned int lo = p.window != 0 && hi > p.window ? hi - p.window : 0u;
        if (p.visible_starts != nullptr) { // the row's range as given
            hi = own_end;
            lo = min(own_start, hi);
        } else if (p.visible_ends != nullptr) { // a row may read past itself, up to the end of the chunk
            hi = min(max(hi, own_end), p.position + p.rows);
        }
        vis_hi = col_valid ? hi : 0u;
        vis_lo = lo;
    }
    // the tokens that every column of the wave sees are [max_lo, min_hi); outside [min_lo, max_hi) nobody sees any
    const unsigned int wave_min_hi = wave_min_u(vis_hi), wave_max_lo = wave_max_u(vis_lo);
    const unsigned int wave_max_hi = wave_max_u(vis_hi), wave_min_lo = wave_min_u(col_valid ? vis_lo : 0xffffffffu);

    // lane parts of the LDS addresses: K rows of token c, V rows 4 h + m / 4 of a run of eight
    const unsigned int k_lane = (8u * (c >> 4) + 2u * (c & 3u) + ((c >> 3) & 1u)) * kPairStride + ((c >> 2) & 1u) * kRow + ((h ^ ((c >> 2) & 1u)) * 16u);
    const unsigned int v_lane = 2u * (m >> 2) * kPairStride + h * kRow + (((lane >> 4) & 1u) * 2u + (((m & 3u) >> 1) ^ h)) * 16u + (m & 1u) * 8u;

    auto attend = [&](int buf, unsigned int t0) __attribute__((always_inline)) {
        const unsigned char* kt = lds.tile[buf][0][0] + half * (2 * kTile) + k_lane;
        const unsigned char* vt = lds.tile[buf][0][1] + half * (2 * kTile) + v_lane;
        // ---- S^T = K . Q'.  A lane holds tokens 8 (i / 4) + 4 h + i % 4 of its column in element i ----
        f32x16 s;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            s[i] = 0.0f;
        }
        // (fragments are requested four slots ahead and in pairs: left to itself the compiler requests two, waits for both, and so on)
        constexpr int kRing = 4;
        Frag kf[kRing];
#pragma unroll
        for (int ks = 0; ks < kRing; ++ks) {
            kf[ks].u = *(const u32x4*)(kt + ks * 32);
        }
        PREFILL_PHASE_FENCE();
#pragma unroll
        for (int ks = 0; ks < kD / 16; ++ks) {
            s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[ks % kRing].h, qf[ks].h, s, 0, 0, 0);
            if (ks % 2 == 1 && ks + kRing <= kD / 16 + 1) {
#pragma unroll
                for (int n = ks + kRing - 1; n < ks + kRing + 1 && n < kD / 16; ++n) {
                    kf[n % kRing].u = *(const u32x4*)(kt + n * 32);
                }
            }
            PREFILL_PHASE_FENCE();
        }
        union VFrag {
            s16x4 s[2];
            f16x8 h;
        };
        // tokens 16 kk + 4 h .. + 4 and 16 kk + 8 + 4 h .. + 4 of dims 32 t ..: the order in which a lane holds its scores
        auto load_v = [&](VFrag& vf, int t, int kk) __attribute__((always_inline)) {
#pragma unroll
            for (int r8 = 0; r8 < 2; ++r8) {
                const unsigned char* at = vt + (8 * kk + r8) * kPairStride + t * 64;
                vf.s[r8] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(at));
            }
        };
        VFrag vf[2][2]; // [parity][output tile of a pair]
        load_v(vf[0][0], 0, 0); // before the softmax
        load_v(vf[0][1], 1, 0);
        PREFILL_PHASE_FENCE();
        // ---- online softmax of the lane's column ----
        if constexpr (SOFTCAP == 1) {
            // tanh(y) = 1 - 2 / (e^(2y) + 1): the form cancels for tiny y, and its absolute error, a few units of 2^-24, is
            // multiplied by the cap (3e-6 of a score under a cap of 50)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const float e2y = __builtin_amdgcn_exp2f(s[i] * tanh_arg);
                s[i] = fmaf(-2.0f, __builtin_amdgcn_rcpf(e2y + 1.0f), 1.0f);
            }
        } else if constexpr (SOFTCAP == 2) { // keeps the limit of an ever larger cap
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                s[i] = soft_tanh(s[i] * cap_arg);
            }
        }
        if (t0 + kStep > wave_min_hi || t0 < wave_max_lo) { // only steps at an edge of some column need the per-token masks
            const unsigned int first = t0 + (fresh_lane() >> 5) * 4u;
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
        lane_max = fmaxf(lane_max, upper);
        lane_top = fmaxf(lane_top, lane_max * mult);
        bool behind = __any(lane_top > run_max); // some score passed its column's reference, which stays
        if (two_terms ? __any(lane_top - run_max > kSlack) : behind) {
            behind = false;
            const float new_max = fmaxf(run_max, halves_max(lane_top));
            const float safe_max = new_max == kNegInf ? 0.0f : new_max;
            const float alpha = __builtin_amdgcn_exp2f(run_max - safe_max);
            ref_shift = kPBias - safe_max;
            run_sum *= alpha;
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
        // ---- O^T += V^T . P: f16 hi, with the second half's exponentials under the products of the first, then on heavy steps lo, one turn of a
        // loop each (as branches around the products the two forms cost sixty registers of copies) ----
        float eight[2] = {0.0f, 0.0f};
        auto weigh = [&](int i) __attribute__((always_inline)) {
            s[i] = __builtin_amdgcn_exp2f(fmaf(s[i], mult, ref_shift));
            eight[i >> 3] += s[i];
        };
        PREFILL_PHASE_FENCE();
        for (bool hi = true;; hi = false) {
            Frag ph[2];
            if (hi) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    weigh(2 * e);
                    weigh(2 * e + 1);
                    ph[0].u[e] = pack_f16_hw(s[2 * e], s[2 * e + 1]);
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const f16x2 dropped = __builtin_bit_cast(f16x2, pack_f16_hw(s[2 * e], s[2 * e + 1]));
                    ph[e >> 2].u[e & 3] = pack_f16_hw(s[2 * e] - (float)dropped[0], s[2 * e + 1] - (float)dropped[1]);
                }
            }
#pragma unroll
            for (int n = 0; n < kD / 32; ++n) { // output tiles 2 (n % 4) .. + 2, tokens 16 (n / 4) .. + 16
                if (n < kD / 32 - 1) { // the fragments after these travel while these multiply
                    load_v(vf[(n + 1) & 1][0], (n + 1) % 4 * 2, (n + 1) / 4);
                    load_v(vf[(n + 1) & 1][1], (n + 1) % 4 * 2 + 1, (n + 1) / 4);
                }
                acc[n % 4 * 2] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[n & 1][0].h, ph[n / 4].h, acc[n % 4 * 2], 0, 0, 0);
                acc[n % 4 * 2 + 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[n & 1][1].h, ph[n / 4].h, acc[n % 4 * 2 + 1], 0, 0, 0);
                if (hi && n < 4) {
                    weigh(8 + 2 * n);
                    weigh(8 + 2 * n + 1);
                    ph[1].u[n] = pack_f16_hw(s[8 + 2 * n], s[8 + 2 * n + 1]);
                }
                PREFILL_PHASE_FENCE(); // or every fragment is requested at once, into registers that are not there
            }
            if (!hi) {
                break;
            }
            run_sum += eight[0] + eight[1];
            two_terms = __any(fmaxf(eight[0], eight[1]) * kLoShare > run_sum);
            if (!two_terms && !behind) {
                break;
            }
            load_v(vf[0][0], 0, 0);
            load_v(vf[0][1], 1, 0);
        }
    };

    // ---- main loop.  A pass first waits for its tiles (a wave for its own loads, the barrier for the others'), which also says that nobody
    // reads those of the pass before: their buffers are the ones requested next.
    auto pass_of = [&](unsigned int pass, int buf) __attribute__((always_inline)) {
        const unsigned int t0 = part.begin + pass * kPass;
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        load_pass(buf ^ 1, t0 + kPass, page);
        page = load_entry(t0 + 2u * kPass);
        const unsigned int own = t0 + half * kStep;
        // a tile of packed segments walks the union of its rows' ranges, a wave only what some row of its own sees of the part
        if (own < part.end && own < wave_max_hi && own + kStep > wave_min_lo) {
            attend(buf, own);
        }
    };
    for (unsigned int pass = 0; pass < passes;) {
        pass_of(pass, 0);
        if (++pass >= passes) {
            break;
        }
        pass_of(pass, 1);
        ++pass;
    }
    // what was requested past the range lands, and the tiles are read no more: the halves meet over them
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    Meeting& meeting = shared.meeting;
    float total = halves_sum(run_sum);
    if (half == 1u) {
        meeting.stats[0][quarter][lane] = run_max;
        meeting.stats[1][quarter][lane] = total;
#pragma unroll
        for (int t = 0; t < kD / 32; ++t) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                *(f32x4*)meeting.acc[4 * t + q][quarter][lane] = f32x4{acc[t][4 * q], acc[t][4 * q + 1], acc[t][4 * q + 2], acc[t][4 * q + 3]};
            }
        }
    }
    __syncthreads();
    if (half == 1u) {
        return;
    }
    const float other_max = meeting.stats[0][quarter][lane], other_total = meeting.stats[1][quarter][lane];
    const float common = fmaxf(run_max, other_max);
    // a half that has seen nothing of the column has a sum of zero and accumulators of zero
    const float own_fac = run_max == kNegInf ? 0.0f : __builtin_amdgcn_exp2f(run_max - common);
    const float other_fac = other_max == kNegInf ? 0.0f : __builtin_amdgcn_exp2f(other_max - common);
    total = total * own_fac + other_total * other_fac;
#pragma unroll
    for (int t = 0; t < kD / 32; ++t) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const f32x4 other = *(const f32x4*)meeting.acc[4 * t + q][quarter][lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                acc[t][4 * q + e] = acc[t][4 * q + e] * own_fac + other[e] * other_fac;
            }
        }
    }
    if (!col_valid) {
        return;
    }
    store_column<kD>(p, col_row, col_head, h, common, total, acc, kPBias);
}

} // namespace halves256

} // namespace

} // namespace zllm
