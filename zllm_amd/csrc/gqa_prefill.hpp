// What the chunked-prefill kernels share: constants, fragments, KV splits, query loads.
#pragma once

#include "common.hpp"
#include "kernels.hpp"

namespace zllm {

namespace {

// Fences for the instruction scheduler between the phases of a step (they keep the early LDS requests early).
#define PREFILL_PHASE_FENCE() __builtin_amdgcn_sched_barrier(0)

constexpr float kLog2e = 1.4426950408889634f;
constexpr int kStep = 32;                 // tokens per step
constexpr float kPBias = 8.0f;            // probabilities are carried as p * 2^8: f16 stays normal down to p = 2^-22
// P' is carried as f16 hi + lo (22 significant bits) while the probabilities a lane holds of a step weigh more than 1 /
// kLoThreshold of its running sum.  A lane sums a quarter of the tokens; where they weigh about the same each is < 1 / 32 of its
// row's sum below that, and the hi term's rounding (2^-12 relative, random sign) moves the normalised output by < 2^-12 / 32 of |v|
// (where a lane holds most of its row's sum, by < 2^-12 / 8).  Kernels whose reference lags (kSlack) take twice the share: their
// ranges are short, and both terms for the first 512 keys of a walk are what the lag pays with.  Distance from 64 bits (2-norm) with 8
// / 16, scores of deviation 1: 1,000 rows of 32 / 8 heads 6.9e-7 / 2.4e-7, of deviation 0.05 2.6e-5 / 2.1e-7; 2,000 rows 4.8e-5 / 2.0e-5, 4,000
// of 16 / 4 7.1e-5 / 4.7e-5.  41.4 / 41.2 us, 90.1 / 91.5, 155 / 162.
constexpr float kLoThreshold = 8.0f, kLoThresholdLag = 16.0f;
// The softmax reference of a column is its running maximum: the probability of the maximum, and of every key that ties with it,
// is a one, which f16 holds.  It moves in some column of a wave on most of the first hundred steps, and every move reduces across
// the lanes and rescales the accumulators.  Where the registers are there (one column tile of head_dim 128, kLag) it stays while
// no score passes it by more than 2^kSlack and the steps carry both terms: a probability is then at most 2^kSlack, and p' = p *
// v_scale * 2^(kPBias - window) below 2^15 (f16 ends at 2^16).  The step after one that needed only the hi term moves every
// reference up to its maximum, and a step that meets one behind carries both terms, so no rounded probability is measured
// against anything else.  1,000 rows of 32 / 8 heads 42.4 -> 40.5 us, 2,048 of 16 / 4 71.8 -> 68.7, 1,000 f16 rows of 32 / 8 34.9 -> 33.3.
// With two column tiles it spills (2,048 rows at 50,000 4.52 -> 5.27 ms), at head_dim 64 the two votes a step cost long chunks more than
// short ones gain (1,000 rows 39.4 -> 37.2, 2,048 at 30,000 1,056 -> 1,098), at 256 it is level.
// The difference is compared, which is exact: from 2^25 on f32 rounds a maximum plus six to eight more.
constexpr float kSlack = 6.0f;

typedef short s16x4 __attribute__((ext_vector_type(4)));

union Frag {
    u32x4 u;
    f16x8 h;
};

__device__ __forceinline__ float soft_tanh(float x)
{
    const float x2 = x * x;
    const float poly = x * (1.0f + x2 * (-1.0f / 3.0f + x2 * (2.0f / 15.0f + x2 * (-17.0f / 315.0f))));
    const float e = __builtin_amdgcn_exp2f(fminf(fabsf(x) * (2.0f * kLog2e), 80.0f));
    const float big = copysignf(1.0f - __fdividef(2.0f, e + 1.0f), x);
    return fabsf(x) < 0.1f ? poly : big;
}

// ---- KV splits of a chunk -------------------------------------------------------------------------------------
// A chunk with few row tiles (a short chunk over a long prefix) leaves most CUs without a workgroup while each
// workgroup walks the whole prefix.  With p.max_chunks > 1 workgroup z of a row tile attends part z of the tile's
// visible range [t_begin, t_end) -- equal 32-aligned parts of at most p.chunk_tokens, as the decode kernels cut a
// sequence -- and writes un-normalised records (sum of p v, running maximum, sum of p) that gqa_decode_merge combines;
// parts beyond the tile's own count write empty records (maximum -inf, sum 0).
struct SplitRange {
    unsigned int begin, end;
    bool live;
};
__device__ __forceinline__ SplitRange split_range(const GqaPrefillParams& p, unsigned int t_begin, unsigned int t_end)
{
    SplitRange r = {t_begin, t_end, true};
    if (p.max_chunks > 1u) {
        const unsigned int parts = max(1u, min(p.max_chunks, (t_end - t_begin + p.chunk_tokens - 1u) / p.chunk_tokens)); // none is live in an empty range
        const unsigned int span = (((t_end - t_begin + parts - 1u) / parts) + 31u) & ~31u;
        const unsigned long long begin = (unsigned long long)t_begin + (unsigned long long)blockIdx.z * span;
        r.live = blockIdx.z < parts && begin < t_end;
        r.begin = r.live ? (unsigned int)begin : t_begin;
        r.end = r.live ? (unsigned int)min((unsigned long long)t_end, begin + span) : t_begin;
    }
    return r;
}

// Eight consecutive query elements (16-byte aligned: the query is, and head_dim is a multiple of 64).  One element at a
// time, a lane sends 32 to 128 two-byte loads before the first step: 1,000 rows of 32 / 8 heads 54.6 -> 49.1 us, a sliding
// layer of 2,048 rows (16 / 8 heads of 256, window 1,024) 108.9 -> 86.3 us.
__device__ __forceinline__ void widen8(const u32x4& raw, int dtype, float (&x)[8])
{
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        x[2 * e] = dtype == 1 ? __uint_as_float(raw[e] << 16) : f16_bits_to_f32((unsigned short)(raw[e] & 0xffffu));
        x[2 * e + 1] = dtype == 1 ? __uint_as_float(raw[e] & 0xffff0000u) : f16_bits_to_f32((unsigned short)(raw[e] >> 16));
    }
}

__device__ __forceinline__ void store_empty_record(const GqaPrefillParams& p, unsigned int row, unsigned int head)
{
    const size_t rec = ((size_t)row * p.max_chunks + blockIdx.z) * p.num_heads + head;
    p.stats[rec * 2] = kNegInf;
    p.stats[rec * 2 + 1] = 0.0f;
}

} // namespace

} // namespace zllm
