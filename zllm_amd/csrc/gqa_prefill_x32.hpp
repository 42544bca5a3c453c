// What the chunk kernels of 32-pair waves (gqa_prefill_f16.hip, gqa_prefill_staged.hip) share: a 32x32x16 matrix tile holds 32 tokens of 32
// (row, head-in-group) pairs, lane l column l % 32 and tokens 8 (i / 4) + 4 (l / 32) + i % 4 in element i of its sixteen.
#pragma once

#include "gqa_prefill.hpp"

namespace zllm {

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef const __attribute__((address_space(4))) unsigned int* scalar_words_t;

// Chunk swizzle of rows of sixteen chunks.  A 16-byte read takes sixteen rows of one chunk at a time, a transposed 8-byte read four rows
// of four chunks: row bits 0 and 1 go into chunk bits 3 and 2, row bits 2 and 3 into chunk bits 0 and 1, and both meet every bank once
// (the conflict counter reads 0).
__device__ __forceinline__ unsigned int swizzle(unsigned int row)
{
    return ((row & 1u) << 3) | ((row & 2u) << 1) | ((row >> 2) & 3u);
}

// The lane number again, for places off the main path: what is formed from it there takes no register of the loop around them
__device__ __forceinline__ unsigned int fresh_lane()
{
    unsigned int lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    asm volatile("" : "+v"(lane));
    return lane;
}

// Reduction over a wave inside the vector ALU: rows of sixteen lanes by rotation, then across the rows
template <class Op> __device__ __forceinline__ unsigned int wave_reduce(unsigned int v, Op op)
{
    v = op(v, (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xf, 0xf, false)); // row_ror:8
    v = op(v, (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x124, 0xf, 0xf, false)); // row_ror:4
    v = op(v, (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x122, 0xf, 0xf, false)); // row_ror:2
    v = op(v, (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x121, 0xf, 0xf, false)); // row_ror:1
    const u32x2_swap a = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    v = op(a.x, a.y);
    const u32x2_swap b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return __builtin_amdgcn_readfirstlane(op(b.x, b.y));
}

__device__ __forceinline__ unsigned int wave_min_u(unsigned int v)
{
    return wave_reduce(v, [](unsigned int x, unsigned int y) { return min(x, y); });
}

__device__ __forceinline__ unsigned int wave_max_u(unsigned int v)
{
    return wave_reduce(v, [](unsigned int x, unsigned int y) { return max(x, y); });
}

__device__ __forceinline__ float halves_sum(float v) // lanes l and l ^ 32, the two halves of a column
{
    const u32x2_swap b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(b.x) + __uint_as_float(b.y);
}

__device__ __forceinline__ float halves_max(float v)
{
    const u32x2_swap b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(b.x), __uint_as_float(b.y));
}

// Lane i of the lane's row of sixteen (`i` a constant after unrolling).  As the factor of a multiplication or a multiply-add it rides in
// that instruction.
__device__ __forceinline__ float row_lane(float v, int i)
{
    const int x = (int)__float_as_uint(v);
#define ROW_LANE(n) case n: return __uint_as_float((unsigned int)__builtin_amdgcn_mov_dpp(x, 0x150 + n, 0xf, 0xf, true));
    switch (i) {
        ROW_LANE(0) ROW_LANE(1) ROW_LANE(2) ROW_LANE(3) ROW_LANE(4) ROW_LANE(5) ROW_LANE(6) ROW_LANE(7)
        ROW_LANE(8) ROW_LANE(9) ROW_LANE(10) ROW_LANE(11) ROW_LANE(12) ROW_LANE(13) ROW_LANE(14)
    default: return __uint_as_float((unsigned int)__builtin_amdgcn_mov_dpp(x, 0x15f, 0xf, 0xf, true));
    }
#undef ROW_LANE
}

// to[0 .. 4) += row_lane(v, 4 q ..) * x[0 .. 4) in four instructions: the compiler would spend another four on moving the lanes first.  It
// does not see the lane reads (a register just written by the vector ALU needs two wait states before them) nor that `x` may come
// from a matrix instruction, so the block begins with the wait states and `settled` is a value the compiler has formed from x's tuple.
__device__ __forceinline__ void row_lane_fmac4(float& t0, float& t1, float& t2, float& t3, float v, int q, float x0, float x1, float x2, float x3, float settled)
{
#define ROW_FMAC(n, a, b, c, d) \
    case n: \
        asm volatile("s_nop 1\n\t" \
                     "v_fmac_f32_dpp %0, %4, %5 row_newbcast:" #a " row_mask:0xf bank_mask:0xf\n\t" \
                     "v_fmac_f32_dpp %1, %4, %6 row_newbcast:" #b " row_mask:0xf bank_mask:0xf\n\t" \
                     "v_fmac_f32_dpp %2, %4, %7 row_newbcast:" #c " row_mask:0xf bank_mask:0xf\n\t" \
                     "v_fmac_f32_dpp %3, %4, %8 row_newbcast:" #d " row_mask:0xf bank_mask:0xf" \
                     : "+v"(t0), "+v"(t1), "+v"(t2), "+v"(t3) \
                     : "v"(v), "v"(x0), "v"(x1), "v"(x2), "v"(x3), "v"(settled)); \
        break;
    switch (q) {
        ROW_FMAC(0, 0, 1, 2, 3)
        ROW_FMAC(1, 4, 5, 6, 7)
        ROW_FMAC(2, 8, 9, 10, 11)
        ROW_FMAC(3, 12, 13, 14, 15)
    }
#undef ROW_FMAC
}

// 64 x 16 bytes (WIDE) or 64 x 4 from `from` + the lane's offset to LDS at `to` + AT + 16 or 4 times the lane.  In assembly, because the
// compiler would wait for all of these loads before every LDS read that follows.
template <bool WIDE, unsigned int AT> __device__ __forceinline__ void load_to_lds(const unsigned char* from, unsigned int lane_at, unsigned int to)
{
    if constexpr (WIDE) {
        asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3" ::"s"(to), "n"(AT), "v"(lane_at), "s"(from) : "memory", "scc");
    } else {
        asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %2, %3" ::"s"(to), "n"(AT), "v"(lane_at), "s"(from) : "memory", "scc");
    }
}

// A finished column: `acc` and `total` carry 2^v_shift.  Split calls leave records in true units, others the normalised row.
template <int D>
__device__ __forceinline__ void store_column(const GqaPrefillParams& p, unsigned int row, unsigned int head, unsigned int h, float run_max, float total,
                                             const f32x16 (&acc)[D / 32], float v_shift)
{
    const bool live = total > 0.0f && total < __builtin_inff();
    if (p.max_chunks > 1u) { // without the bias of the probabilities and the V window
        const size_t rec = ((size_t)row * p.max_chunks + blockIdx.z) * p.num_heads + head;
        const int down = -(int)v_shift;
        const float fa = ldexpf(1.0f, down / 2), fb = ldexpf(1.0f, down - down / 2); // two factors: 2^down alone may leave f32's range
        if (h == 0u) {
            p.stats[rec * 2] = live ? run_max : kNegInf;
            p.stats[rec * 2 + 1] = live ? total * fa * fb : 0.0f;
        }
        float* out = p.partial + rec * (size_t)D + 4u * h;
#pragma unroll
        for (int t = 0; t < D / 32; ++t) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                *(f32x4*)(out + t * 32 + q * 8) = f32x4{acc[t][4 * q], acc[t][4 * q + 1], acc[t][4 * q + 2], acc[t][4 * q + 3]} * fa * fb;
            }
        }
        return;
    }
    const float inv = live ? 1.0f / total : 0.0f; // accumulators and sum carry the same power of two
    const size_t base = ((size_t)row * p.num_heads + head) * D + 4u * h;
#pragma unroll
    for (int t = 0; t < D / 32; ++t) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            f32x4 v = f32x4{acc[t][4 * q], acc[t][4 * q + 1], acc[t][4 * q + 2], acc[t][4 * q + 3]} * inv;
            if (inv == 0.0f) {
                v = f32x4{0.f, 0.f, 0.f, 0.f};
            }
            const size_t at = base + t * 32 + q * 8;
            if (p.gate != nullptr) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[e] = gated(v[e], p.gate, p.gate_cols, p.gate_dtype, row, head * D + 4u * h + t * 32 + q * 8 + e);
                }
            }
            if (p.out_dtype == 0) {
                *(f32x4*)((float*)p.out + at) = v;
            } else {
                unsigned short* o = (unsigned short*)p.out + at;
                u32x2 packed;
                if (p.out_dtype == 1) {
                    packed = u32x2{pack_bf16_rne(v[0], v[1]), pack_bf16_rne(v[2], v[3])};
                } else {
                    packed = u32x2{(unsigned int)f32_to_f16_bits(v[0]) | ((unsigned int)f32_to_f16_bits(v[1]) << 16),
                                   (unsigned int)f32_to_f16_bits(v[2]) | ((unsigned int)f32_to_f16_bits(v[3]) << 16)};
                }
                *(u32x2*)o = packed;
            }
        }
    }
}

} // namespace

} // namespace zllm
