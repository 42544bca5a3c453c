// Chunked-prefill GQA attention over f16 rows at head_dim 128 in tiles of 128 (row, head-in-group) pairs: calls of more than two
// rounds of such tiles that full-size ones would leave a last round of unfilled, and packed segments (gqa_prefill_takes_f16).  What it
// computes is gqa_prefill_tiles (gqa_prefill.hip); how differs.
//
// What bounds such a launch is the chain of instructions a wave runs for a 32-token tile, not the matrix cores, memory or LDS: a
// wave alone on its SIMD takes as long per tile (1,740 cycles, 512 of them matrix work) as one of three.  So the chain is kept short and
// the waves many:
//   32x32x16 matrix tiles: a wave owns 32 pairs, a lane sixteen scores of one pair, so the maximum, the sum and the tests of a
//       step are made once for 32 pairs (twice with 16x16x32 tiles), and every K and V^T fragment read from LDS feeds twice the
//       work of a 16-pair wave (LDS busy cycles 6.5 M -> 3.5 M on 4,100 rows of 16 heads in nine segments).
//   The rows go from global memory straight to LDS (no staging registers) two tiles ahead in a ring of three: 48 KB of tiles
//       and at most 168 registers let three workgroups of four waves live on a compute unit, where eight waves of 16 pairs
//       around four staged tiles were alone on it.
//       Five registers are spilled, all outside the loop.
//   The exponentials of a tile's second sixteen tokens stand between the matrix instructions of the first sixteen: what a wave places between its
//       own hides, the other waves' hardly does.  Nine segments (appends included) 75.1 -> 73.0 us, a first chunk of 2,300 rows 122 -> 119.
// 16 / 4 heads, 4,100 rows in one segment: 285 -> 232 us; in nine segments (16 / 16 heads) 69 -> 66, which are two workgroups a compute
// unit and last as long as the longest walk, 36 tiles of 32 tokens: the longest segment has 21, but a row tile across a boundary walks both its
// neighbours; 32 / 8 heads, 2,300 rows in eleven 48 -> 42, a first chunk of 3,500 rows 263 -> 204.
#include "gqa_prefill_x32.hpp"

namespace zllm {

namespace {

constexpr int kD = 128;
constexpr int kRow = kD * 2;          // bytes of one token of one KV head
constexpr int kTile = kStep * kRow;   // one 32-token tile
constexpr int kWaves = 4;             // of 32 pairs each
constexpr int kPairs = 32 * kWaves;
constexpr int kBufs = 3;              // tile buffers: one attended, two on their way
constexpr int kRun = kStep / kWaves;  // rows of a tile that a wave requests, 4 a load
constexpr int kLoads = kRun / 4;      // loads of 64 x 16 bytes a wave issues per plane and tile
static_assert(kRun <= 8, "prefill_scalar_pages: pages of eight tokens hold a wave's rows");

typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef const __attribute__((address_space(1))) void* global_ptr_t;

// P is carried as f16 hi, and lo while eight probabilities of a lane weigh more than 1 / lo_share of the lane's sum of those (the
// test of the other chunk kernels, twice a lane).  The share is 16 and behind a prefix longer than the chunk 24, where those kernels
// use 8: they cut such calls into other parts, and every part begins with both terms.  Distance from 64 bits (2-norm), tiles of 16-pair
// waves / this kernel, where the standard deviation of the scores is 0.05 and 1: nine segments of 4,100 rows 1.1e-4 / 2.4e-5 and 3.1e-5 /
// 2.9e-7, a first chunk of 2,300 rows (32 / 8 heads) 3.9e-5 / 2.2e-5 and 1.6e-6 / 2.9e-7, 2,300 rows at 9,000 1.80e-4 / 1.74e-4 and 5.6e-5 / 2.6e-5
// (with 16 1.83e-4).  A test of the single largest probability against its row passes near-even rows over: 1.5e-4 on the nine segments.
constexpr float kLoShare = 16.0f, kLoShareBehind = 24.0f;

// 64 x 16 bytes from global memory to 1 KiB of LDS: lane l's bytes land at `to` + 16 l.  The compiler counts these loads and
// waits for all of them before the first transposed LDS read that follows, which it cannot tell from a read of the tile being
// filled, so what a step requests has its scores and its softmax to arrive in.  (Hidden from it in inline assembly, with two
// tiles in flight throughout, the kernel takes the same time; with a ring of two, 85 us instead of 62 on the nine segments.)
__device__ __forceinline__ void load_to_lds(const unsigned char* from, unsigned char* to)
{
    __builtin_amdgcn_global_load_lds((global_ptr_t)from, (lds_ptr_t)to, 16, 0, 0);
}

// SOFTCAP: 0 none, 1 caps below 256 (see below), 2 larger ones.  The rows a wave requests of a tile lie in one page
// (prefill_scalar_pages), and their address is scalar but for the lane's constant part.
template <int SOFTCAP> __global__ __launch_bounds__(64 * kWaves, 3) void gqa_prefill_f16(GqaPrefillParams p)
{
    struct Lds {
        unsigned char k[kBufs][kTile];
        unsigned char v[kBufs][kTile];
    };
    __shared__ __align__(1024) Lds lds;

    const unsigned int tid = threadIdx.x;
    const unsigned int lane = tid & 63u;
    const unsigned int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned int m = lane & 15u;
    const unsigned int c = lane & 31u; // the lane's column: a pair
    const unsigned int h = lane >> 5;
    // row tiles with the longest range first, the KV head as the fast index (see gqa_prefill_q8)
    const unsigned int kvh = blockIdx.x % p.num_kv_heads;
    const unsigned int rows_per_wg = max(1u, (unsigned int)kPairs / p.group);
    const unsigned int row0 = (gridDim.x / p.num_kv_heads - 1u - blockIdx.x / p.num_kv_heads) * rows_per_wg;
    const unsigned int cols_used = rows_per_wg * p.group;
    const unsigned int col = wave * 32u + c;
    const unsigned int col_row = row0 + col / p.group;
    const unsigned int col_head = kvh * p.group + col % p.group;
    const bool col_valid = col < cols_used && col_row < p.rows;
    const unsigned int last_row = min(row0 + rows_per_wg, p.rows) - 1u;

    // ---- given ranges, then the query's rows, are requested before anything waits ----
    unsigned int own_end = 0, own_start = 0, union_end = 0, union_start = 0xffffffffu;
    if (p.visible_ends != nullptr) {
        const unsigned int lane_row = min(row0 + lane, last_row), own_row = min(col_row, last_row);
        const unsigned int lane_end = p.visible_ends[lane_row], end = p.visible_ends[own_row];
        unsigned int lane_start = 0;
        if (p.visible_starts != nullptr) {
            lane_start = p.visible_starts[lane_row];
            own_start = p.visible_starts[own_row];
        }
        own_end = min(end, p.position + p.rows);
        union_end = min(lane_end, p.position + p.rows);
        union_start = min(lane_start, union_end);
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
    unsigned int t_end = p.position + last_row + 1u;
    unsigned int t_begin = 0;
    if (p.visible_ends != nullptr) { // the union over the rows; a lane has taken one of the first 64
        for (unsigned int r = row0 + 64u + lane; r <= last_row; r += 64u) {
            const unsigned int end = min(p.visible_ends[r], p.position + p.rows);
            union_end = max(union_end, end);
            if (p.visible_starts != nullptr) {
                union_start = min(union_start, min(p.visible_starts[r], end));
            }
        }
        if (p.visible_starts != nullptr) {
            t_end = wave_max_u(union_end);
            t_begin = wave_min_u(union_start);
        } else {
            t_end = max(t_end, wave_max_u(union_end));
        }
    }
    t_begin &= ~31u;
    const SplitRange part = split_range(p, t_begin, t_end);
    if (!part.live) {
        if (col_valid && h == 0u) {
            store_empty_record(p, col_row, col_head);
        }
        return;
    }
    const unsigned int steps = (part.end - part.begin + kStep - 1) / kStep;

    // ---- staging.  A load fills four rows of a tile, lane l its l-th 16 bytes; the swizzle goes into the source chunk.  What is
    // read past the range is its last row again, and the first one where every range of the tile ends at 0.
    const unsigned int k_row = p.num_kv_heads * kRow;
    const unsigned int last_token = max(t_end, 1u) - 1u;
    const unsigned int lane_row = lane >> 4;
    unsigned int lane_col[kLoads], lane_at[kLoads];
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
        lane_col[u] = (m ^ swizzle(wave * kRun + u * 4u + lane_row)) * 16u + kvh * kRow;
        lane_at[u] = lane_col[u] + (u * 4u + lane_row) * k_row;
    }
    auto first_of = [&](unsigned int t0) __attribute__((always_inline)) -> unsigned int { // of the wave's rows, inside the range
        const unsigned int t = t0 + wave * kRun;
        return t > last_token ? last_token & ~(unsigned int)(kRun - 1) : t;
    };
    auto load_entry = [&](unsigned int t0) __attribute__((always_inline)) -> unsigned int {
        return ((scalar_words_t)(uintptr_t)p.table)[first_of(t0) >> p.block_shift];
    };
    auto load_tile = [&](int buf, unsigned int t0, unsigned int page) __attribute__((always_inline)) {
        unsigned char* const k_to = lds.k[buf] + wave * (kLoads * 1024u);
        unsigned char* const v_to = lds.v[buf] + wave * (kLoads * 1024u);
        const unsigned int t = first_of(t0), left = last_token - t;
        const unsigned long long at = (((unsigned long long)page << p.block_shift) + (t & (p.block_tokens - 1u))) * k_row;
        const unsigned char* const kp = p.k_plane + at;
        const unsigned char* const vp = p.v_plane + at;
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            unsigned int from = lane_at[u];
            if (left < kRun - 1u) {
                from = lane_col[u] + min(u * 4u + lane_row, left) * k_row;
            }
            load_to_lds(kp + from, k_to + u * 1024u);
            load_to_lds(vp + from, v_to + u * 1024u);
        }
    };
    // the first tiles travel while the query is made ready
    unsigned int page = load_entry(part.begin);
#pragma unroll
    for (int n = 0; n < kBufs - 1; ++n) {
        load_tile(n, part.begin + n * kStep, page);
        page = load_entry(part.begin + (n + 1) * kStep);
    }

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
    float run_sum[2] = {0.0f, 0.0f}; // of the lane's first and second eight tokens of each step
    const float lo_share = p.position > p.rows ? kLoShareBehind : kLoShare;
    float lane_top = kNegInf; // the largest score the lane has met
    bool two_terms = true;    // the step before carried both terms of its probabilities (see kSlack)
    unsigned int vis_lo, vis_hi; // visible tokens [lo, hi) of the column's row
    {
        const unsigned int pos = p.position + col_row;
        unsigned int hi = pos + 1u;
        unsigned int lo = 0;
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

    // LDS offsets of the lane's fragments as finished sums (formed in the loop they cost an addition a read).
    // K: chunk 2 ks + h of row c.  V: chunk 4 t + 2 (lane / 16 % 2) + (m & 3) / 2 of rows 4 h + m / 4 and eight further.
    unsigned int qk_at[8], pv_at[2][4];
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
        qk_at[ks] = c * kRow + (((2u * ks + h) ^ swizzle(c)) << 4);
        asm volatile("" : "+v"(qk_at[ks]));
    }
#pragma unroll
    for (int r8 = 0; r8 < 2; ++r8) {
        const unsigned int tr_row = 8u * r8 + 4u * h + (m >> 2);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            pv_at[r8][t] = tr_row * kRow + (((4u * t + ((lane >> 4) & 1u) * 2u + ((m & 3u) >> 1)) ^ swizzle(tr_row)) << 4) + (m & 1u) * 8u;
            asm volatile("" : "+v"(pv_at[r8][t]));
        }
    }

    auto attend = [&](int buf, unsigned int t0) __attribute__((always_inline)) {
        const unsigned char* kt = lds.k[buf];
        const unsigned char* vt = lds.v[buf];
        // ---- S^T = K . Q'.  A lane holds tokens 8 (i / 4) + 4 h + i % 4 of its column in element i ----
        f32x16 s;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            s[i] = 0.0f;
        }
#pragma unroll
        for (int ks = 0; ks < kD / 16; ++ks) {
            Frag kf;
            kf.u = *(const u32x4*)(kt + qk_at[ks]);
            s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf.h, qf[ks].h, s, 0, 0, 0);
        }
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
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const unsigned int token = t0 + 8u * (i >> 2) + 4u * h + (i & 3);
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
        // ---- O^T += V^T . P: f16 hi, with the second half's exponentials under the products of the first, then on heavy steps lo, one turn of a
        // loop each (as branches around the products the two forms cost sixty registers of copies) ----
        float part_sum[2][2] = {{0.0f, 0.0f}, {0.0f, 0.0f}};
        auto weigh = [&](int i) __attribute__((always_inline)) {
            s[i] = __builtin_amdgcn_exp2f(fmaf(s[i], mult, ref_shift));
            part_sum[i >> 3][i & 1] += s[i];
        };
        PREFILL_PHASE_FENCE();
        union VFrag {
            s16x4 s[2];
            f16x8 h;
        };
        // tokens 16 kk + 4 h .. + 4 and 16 kk + 8 + 4 h .. + 4 of dims 32 t ..: the order in which a lane holds its scores
        auto load_v = [&](VFrag& vf, int t, int kk) __attribute__((always_inline)) {
#pragma unroll
            for (int r8 = 0; r8 < 2; ++r8) {
                const unsigned char* at = vt + pv_at[r8][t] + kk * 16 * kRow;
                vf.s[r8] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(at));
            }
        };
        for (bool hi = true;; hi = false) {
            constexpr int kRing = 2; // a third fragment spills in the loop
            VFrag vf[kRing];
#pragma unroll
            for (int n = 0; n < kRing; ++n) {
                load_v(vf[n], n % 4, n / 4);
            }
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
            for (int n = 0; n < 8; ++n) { // output tile n % 4, tokens 16 (n / 4) .. + 16
                acc[n % 4] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[n % kRing].h, ph[n / 4].h, acc[n % 4], 0, 0, 0);
                if (n + kRing < 8) { // the fragments after these travel while these multiply
                    load_v(vf[n % kRing], (n + kRing) % 4, (n + kRing) / 4);
                }
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
            bool heavy = false;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const float eight = part_sum[e][0] + part_sum[e][1];
                run_sum[e] += eight;
                heavy = heavy || eight * lo_share > run_sum[e];
            }
            two_terms = __any(heavy);
            if (!two_terms && !behind) {
                break;
            }
        }
    };

    // ---- main loop.  A step first waits for its tile (a wave for its own loads, the barrier for the others'), which also says
    // that nobody reads the tile of the step before: that is the buffer of the tile requested next.  Loads are issued
    // unconditionally, so the count that may stay in flight is a constant; past the range they repeat its last row.
    auto step_of = [&](unsigned int step, int buf) __attribute__((always_inline)) {
        const unsigned int t0 = part.begin + step * kStep;
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((kBufs - 2) * kLoads * 2) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        load_tile((buf + kBufs - 1) % kBufs, t0 + (kBufs - 1) * kStep, page);
        page = load_entry(t0 + kBufs * kStep);
        // a tile of packed segments walks the union of its rows' ranges, a wave only what some row of its own sees
        if (t0 < wave_max_hi && t0 + kStep > wave_min_lo) {
            attend(buf, t0);
        }
    };
    for (unsigned int step = 0; step < steps;) {
#pragma unroll
        for (int buf = 0; buf < kBufs; ++buf) {
            step_of(step, buf);
            if (++step >= steps) {
                break;
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // what was requested past the range lands before the LDS is given back

    // ---- normalise and store ----
    const float total = halves_sum(run_sum[0] + run_sum[1]);
    if (!col_valid) {
        return;
    }
    store_column<kD>(p, col_row, col_head, h, run_max, total, acc, kPBias);
}

} // namespace

hipError_t launch_gqa_prefill_f16(const GqaPrefillParams& p, hipStream_t stream)
{
    const unsigned int rows_per_wg = p.group >= (unsigned int)kPairs ? 1u : (unsigned int)kPairs / p.group;
    const dim3 grid((p.rows + rows_per_wg - 1) / rows_per_wg * p.num_kv_heads, 1, p.max_chunks > 1u ? p.max_chunks : 1u);
    const dim3 block(64 * kWaves);
    if (!(p.softcap > 0.0f)) {
        gqa_prefill_f16<0><<<grid, block, 0, stream>>>(p);
    } else if (p.softcap < 256.0f) {
        gqa_prefill_f16<1><<<grid, block, 0, stream>>>(p);
    } else {
        gqa_prefill_f16<2><<<grid, block, 0, stream>>>(p);
    }
    return hipGetLastError();
}

} // namespace zllm
