// Split-KV attention of chunked MLA prefill (512 latent + 64 rope columns) over latents that are converted once a call: what it computes is
// mla_partial_ws (mla_decode.hip), for calls whose workspace asks for it (plan_mla_staged, plan_mla_call in api.hip).
//
// mla_stage writes every 32-token tile of the call into the workspace as it is to lie in LDS: the codes as f16 integers (exact), the rope
// columns as the matrix instructions take them, the group scales in f32 for the scores and in f16 over the tile's exponent window for the
// values.  mla_partial_staged moves such tiles straight from memory to LDS.
//
// 512 rows of 128 heads behind 16,384 keys: 2,830 to 2,890 -> 2,340 to 2,400 us a call, by the card (1,010 to 1,060 TFLOP/s in the kernel), 1,000 rows of 16 heads behind 2,000 keys
// 378 -> 167 (a workgroup there is eight rows, where mla_partial_ws is one).  Distance from 64 bits (2-norm), 64 rows of 24 heads behind 30,000
// keys 1.0e-4 -> 7.5e-5, 200 of 32 (192 / 256) behind 3,000 2.2e-4 -> 1.8e-4.
//
// What shapes it: 32x32x16 tiles, under which the vector ALU runs (under 16x16x32 it hardly does), and a fragment feeds 32 pairs.  32 pairs are
// 256 accumulators and 128 query registers a lane: one wave a SIMD, with 512.  A wave alone hides nothing behind another one, so its
// instructions stand in slots of one matrix instruction and what does not wait for it.  Per tile and wave: 68 matrix instructions (2,180
// cycles of 4,400, 1,060 TFLOP/s at the 2.1 GHz that the power leaves), 340 of the vector ALU, 128 LDS reads.  Built without the 128
// scale instructions it is 7 % faster, without the tile loads and the barrier 6 %, without the value reads 4 %: no one of them bounds it.
#include <type_traits>

#include "gqa_prefill_x32.hpp"
#include "mla_rows.hpp"

namespace zllm {

namespace {

constexpr int kLatent = 512, kRope = 64, kRowElems = kLatent + kRope;
constexpr int kGroups = kLatent / 64;
constexpr int kPShift = 4;  // probabilities are carried as p * 2^4, at most 2^12 (see mla_partial_ws)
constexpr int kWaves = 4;   // of 32 (row, head) pairs each
constexpr int kPairs = 32 * kWaves;
// A tile.  Codes: token rows of 1,024 bytes, 16 apart, in the order of code_slot: the sixteen rows of a 16-byte read and the four rows x 64
// bytes of a transposed one then meet every bank once, and every address is one lane register plus a constant.  Rope: 1 KiB a fragment
// of 16 columns, 16 bytes a lane.  Scales for the scores: f32 [group][lane] (lane m of a row of sixteen has that of the token of element m);
// for the values: f16 [group][half][element of the half].
constexpr int kRowStride = kLatent * 2 + 16;
constexpr int kRopeAt = kStep * kRowStride;
constexpr int kScaleAt = kRopeAt + kStep * kRope * 2;
constexpr int kScale16At = kScaleAt + 64 * kGroups * 4;
constexpr int kTile = kScale16At + kStep * kGroups * 2;
static_assert(kTile % 1024 == 0, "tiles are moved in whole wave loads");
constexpr int kLoads = kTile / 1024;
constexpr int kWindowAt = kTile; // exponent windows of the tile's first 1, 2 ... 32 tokens, read by scalar loads
constexpr int kBlock = kTile + 128;
constexpr int kBufs = 3;
constexpr int kBlocksBehind = 4; // a part's requests run up to three tiles past its last

__device__ __forceinline__ unsigned int code_slot(unsigned int token)
{
    return (token & 16u) + 4u * (token & 3u) + ((token >> 2) & 3u);
}

union MlaFrag {
    u32x4 u;
    f16x8 h;
    bf16x8 b;
    s16x4 s[2];
};

// One tile a workgroup; bound by the memory it reads and writes
__global__ __launch_bounds__(256) void mla_stage(MlaDecodeParams p)
{
    const unsigned int tid = threadIdx.x;
    const unsigned int tile = blockIdx.x, seq = blockIdx.y;
    const unsigned int end = p.ctx_lens[seq], t0 = tile * kStep;
    if (t0 >= end) {
        return;
    }
    unsigned char* const block = p.staged + ((size_t)seq * p.staged_tiles + tile) * kBlock;
    const unsigned int token = tid >> 3, part = tid & 7u; // a scale group of a token
    // tokens past the end are the last one again, with scales of zero
    const unsigned int* const table = p.tables != nullptr ? p.tables + (size_t)seq * p.table_stride : nullptr;
    const size_t row = paged_row(table, min(t0 + token, end - 1u), p.block_tokens, 0u);
    const unsigned char* const from = (const unsigned char*)p.latent_codes + row * kLatent + part * 64u;
    u32x4 codes[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        codes[i] = *(const u32x4*)(from + 16 * i);
    }
    const u32x4 rope = *(const u32x4*)((const unsigned char*)p.rope_cache + row * (kRope * 2) + part * 16u);
    const float scale = t0 + token < end ? bf16_bits_to_f32(p.latent_scales[row * kGroups + part]) : 0.0f;
    // An infinite scale or a NaN makes the scores of its token NaN, and with them whatever sees the token.  Nothing else: it counts as zero for the
    // values and the windows, where rows of the workgroup that do not see it would meet it with a probability of zero.
    const float value_scale = fabsf(scale) < __builtin_inff() ? scale : 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            u32x4 out;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                unsigned int lo, hi;
                codes4_to_f16(codes[i][2 * n + e], lo, hi);
                out[2 * e] = lo;
                out[2 * e + 1] = hi;
            }
            *(u32x4*)(block + code_slot(token) * kRowStride + part * 128u + (2 * i + n) * 16) = out;
        }
    }
    *(u32x4*)(block + kRopeAt + (part >> 1) * 1024u + (part & 1u) * 512u + token * 16u) = rope;
    __shared__ unsigned int tops[kStep];
    unsigned int token_top = __float_as_uint(fmaxf(value_scale, 0.0f));
#pragma unroll
    for (int d = 1; d < kGroups; d <<= 1) {
        token_top = max(token_top, (unsigned int)__shfl_xor((int)token_top, d));
    }
    if (part == 0u) {
        tops[token] = token_top;
    }
    __syncthreads();
    unsigned int top = tops[tid & 31u]; // of the tokens up to this one
#pragma unroll
    for (int d = 1; d < kStep; d <<= 1) {
        const unsigned int before = (unsigned int)__shfl_up((int)top, d, kStep);
        top = max(top, (tid & 31u) >= (unsigned int)d ? before : 0u);
    }
    const int up_to = min(max((int)((top >> 23) & 0xffu) - 133, -96), 112); // as in mla_partial_ws
    const int window = __builtin_amdgcn_readlane(up_to, 31);
    const unsigned int element = 4u * (token >> 3) + (token & 3u), half = (token >> 2) & 1u;
#pragma unroll
    for (unsigned int row = 0; row < 2; ++row) { // both rows of sixteen lanes of the half
        ((float*)(block + kScaleAt))[part * 64u + 32u * half + 16u * row + element] = value_scale == scale ? scale : __builtin_nanf("");
    }
    ((_Float16*)(block + kScale16At))[part * 32u + half * 16u + element] = (_Float16)(value_scale * __uint_as_float((unsigned int)(127 - kPShift - window) << 23));
    if (tid < (unsigned int)kStep) {
        ((int*)(block + kWindowAt))[tid] = up_to;
    }
}

__device__ __forceinline__ unsigned int pk_mul_f16(unsigned int x, unsigned int y)
{
    return __builtin_bit_cast(unsigned int, __builtin_bit_cast(f16x2, x) * __builtin_bit_cast(f16x2, y));
}

// sum += both f16 halves of `w`
__device__ __forceinline__ void add_halves(float& sum, unsigned int w)
{
    asm("v_fma_mix_f32 %0, %1, 1.0, %0 op_sel_hi:[1,0,0]\n\tv_fma_mix_f32 %0, %1, 1.0, %0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "+v"(sum) : "v"(w));
}

__global__ __launch_bounds__(64 * kWaves, 1) void mla_partial_staged(MlaDecodeParams p)
{
    __shared__ __align__(1024) unsigned char lds[kBufs * kTile + kWaves * 4096]; // tiles, then every wave's rope queries, 16 bytes a lane

    const unsigned int tid = threadIdx.x;
    const unsigned int lane = tid & 63u;
    const unsigned int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned int m = lane & 15u;
    const unsigned int c = lane & 31u; // the lane's column: a (row, head) pair
    const unsigned int h = lane >> 5;
    // row tiles of a sequence, the last rows first: they see the most keys
    const unsigned int heads_here = min(p.heads, (unsigned int)kPairs);
    const unsigned int rows_per_wg = (unsigned int)kPairs / heads_here;
    const unsigned int tiles_of_rows = (p.query_rows + rows_per_wg - 1u) / rows_per_wg;
    const unsigned int item = gridDim.z - 1u - blockIdx.z;
    const unsigned int seq = item / tiles_of_rows, row0 = item % tiles_of_rows * rows_per_wg;
    const unsigned int col = wave * 32u + c;
    const unsigned int col_row = row0 + col / heads_here;
    const unsigned int col_head = blockIdx.y * heads_here + col % heads_here;
    const bool col_valid = col < rows_per_wg * heads_here && col_row < p.query_rows && col_head < p.heads;
    const unsigned int last_row = min(row0 + rows_per_wg, p.query_rows) - 1u;
    const unsigned int ctx = p.ctx_lens[seq];
    auto visible = [&](unsigned int r) __attribute__((always_inline)) {
        const unsigned int behind = p.query_rows - 1u - r; // rows of the chunk after this one
        return ctx > behind ? ctx - behind : 0u;
    };
    // a split's range is its place in units of chunk_tokens for every row: the merges count a row's splits by its own length
    const unsigned int end_of_rows = min(visible(last_row), p.staged_tiles * kStep);
    const unsigned long long begin64 = (unsigned long long)blockIdx.x * p.chunk_tokens;
    const size_t rec = (((size_t)seq * p.query_rows + col_row) * p.max_chunks + blockIdx.x) * p.heads + col_head;
    if (begin64 >= end_of_rows) {
        if (col_valid && h == 0u) {
            p.stats[rec * 2] = kNegInf;
            p.stats[rec * 2 + 1] = 0.0f;
        }
        return;
    }
    const unsigned int begin = (unsigned int)begin64;
    const unsigned int end = (unsigned int)min((unsigned long long)end_of_rows, begin64 + p.chunk_tokens);
    const unsigned int steps = (end - begin + kStep - 1u) / kStep;

    // ---- staging: a tile is 39 wave loads, ten consecutive ones a wave (one of them twice), four from one address
    const unsigned char* staged = p.staged + ((size_t)seq * p.staged_tiles + begin / kStep) * kBlock;
    constexpr int kOwn = (kLoads + kWaves - 1) / kWaves;
    const unsigned int own_at = min(wave * kOwn, (unsigned int)(kLoads - kOwn)) * 1024u;
    const unsigned int lds_base = (unsigned int)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds + own_at;
    const unsigned char* ahead = staged + own_at; // the wave's part of the next tile to request, and where it goes
    unsigned int fill_at = lds_base;
    const unsigned int lane16 = lane * 16u;
    const unsigned int rope_q_at = kBufs * kTile + wave * 4096u;
    auto load_tile = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kOwn; i += 4) {
            asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3" ::"s"(fill_at), "n"(i * 1024), "v"(lane16), "s"(ahead + i * 1024)
                         : "memory", "scc");
#pragma unroll
            for (int k = 1; k < 4 && i + k < kOwn; ++k) { // the offset counts for both addresses
                asm volatile("global_load_lds_dwordx4 %0, %1 offset:%2" ::"v"(lane16), "s"(ahead + i * 1024), "n"(k * 1024) : "memory");
            }
        }
        ahead += kBlock;
        fill_at = fill_at == lds_base + (kBufs - 1u) * kTile ? lds_base : fill_at + kTile;
    };
#pragma unroll
    for (int n = 0; n < 3; ++n) {
        load_tile();
    }

    // ---- queries.  The latent part multiplies f16 codes: a head's row is carried as f16 after taking out the power of two of its largest
    // magnitude (exact for every element within 2^-14 of it); the rope part stays bf16, in the same unit: rope queries 2^60 above the latent
    // ones bound the unit from below, so that it stays finite.
    MlaFrag qf[kRowElems / 16]; // the last four, the rope part, move on to LDS
    float latent_log2;
    {
        const unsigned short* const qa = p.absorbed + (((size_t)seq * p.query_rows + col_row) * p.heads + col_head) * kRowElems + h * 8u;
        float top = 0.0f, rope_top = 0.0f;
#pragma unroll
        for (int ks = 0; ks < kRowElems / 16; ++ks) {
            qf[ks].u = u32x4{0u, 0u, 0u, 0u};
            if (col_valid) {
                qf[ks].u = *(const u32x4*)(qa + ks * 16);
            }
        }
#pragma unroll
        for (int ks = 0; ks < kRowElems / 16; ++ks) {
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const float most = fmaxf(fabsf(__uint_as_float(qf[ks].u[w] << 16)), fabsf(__uint_as_float(qf[ks].u[w] & 0xffff0000u)));
                if (ks < kLatent / 16) {
                    top = fmaxf(top, most);
                } else {
                    rope_top = fmaxf(rope_top, most);
                }
            }
        }
        const unsigned int top_exp = (__float_as_uint(halves_max(top)) >> 23) & 0xffu, rope_exp = (__float_as_uint(halves_max(rope_top)) >> 23) & 0xffu;
        const unsigned int unit = min(max(max(top_exp, rope_exp > 60u ? rope_exp - 60u : 0u), 1u), 253u);
        const float down = __uint_as_float((254u - unit) << 23);
#pragma unroll
        for (int ks = 0; ks < kLatent / 16; ++ks) {
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const unsigned int word = qf[ks].u[w];
                qf[ks].u[w] = pack_f16_hw(__uint_as_float(word << 16) * down, __uint_as_float(word & 0xffff0000u) * down);
            }
        }
#pragma unroll
        for (int ks = kLatent / 16; ks < kRowElems / 16; ++ks) {
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const unsigned int word = qf[ks].u[w];
                qf[ks].u[w] = pack_bf16_trunc(__uint_as_float(word << 16) * down, __uint_as_float(word & 0xffff0000u) * down);
            }
        }
#pragma unroll
        for (int i = 0; i < kRope / 16; ++i) {
            *(u32x4*)(lds + rope_q_at + lane16 + i * 1024) = qf[kLatent / 16 + i].u;
        }
        latent_log2 = p.score_scale * kLog2e * __uint_as_float(unit << 23);
    }

    f32x16 acc[kLatent / 32];
#pragma unroll
    for (int t = 0; t < kLatent / 32; ++t) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            acc[t][i] = 0.0f;
        }
    }
    const unsigned int vis_hi = col_valid ? visible(col_row) : 0xffffffffu;
    const unsigned int wave_min_hi = wave_min_u(vis_hi);
    float run_max = kNegInf, run_sum = 0.0f;
    float neg_ref_shifted = (float)kPShift; // minus the reference of the scores, plus the shift: log2(p * 2^kPShift)
    float acc_fix = 1.0f;                   // what the accumulators are to be multiplied by before the next tile's values

    // lane parts of the LDS addresses
    const unsigned int k_lane = code_slot(c) * kRowStride + h * 16u;
    const unsigned int v_lane = (4u * (m >> 2) + h) * kRowStride + ((lane >> 4) & 1u) * 32u + (m & 3u) * 8u;

    f32x16 s;    // scores of the tile ahead, in units of the query's power of two
    f32x16 d[2]; // products of two groups in turn
    unsigned int pw[8]; // probabilities of the tile being accumulated, times 2^kPShift: elements 2 i and 2 i + 1
    float k_scale[3]; // of group g from its second matrix instruction on

    // A pass of the loop multiplies the keys of tile n + 1 (36 slots, a matrix instruction each: the rope part, then the groups) and accumulates
    // the values of tile n (32 slots).  The vector ALU scales the products of the group before under the keys, and takes the softmax of
    // tile n + 1 under the values.  What a slot reads from LDS is requested four slots before.
    constexpr int kKeySlots = kRowElems / 16, kValueSlots = kLatent / 16, kRing = 4;
    MlaFrag kf[kRing], vf[kRing], qr[kRope / 16];
    unsigned int keys_at, values_at; // LDS of tile n + 1 and tile n
    auto request_key = [&](int n, unsigned int at) __attribute__((always_inline)) {
        if (n < kRope / 16) {
            kf[n % kRing].u = *(const u32x4*)(lds + at + lane16 + kRopeAt + n * 1024);
            qr[n].u = *(const u32x4*)(lds + rope_q_at + lane16 + n * 1024);
        } else if (n < kKeySlots) {
            kf[n % kRing].u = *(const u32x4*)(lds + at + k_lane + (n - kRope / 16) * 32);
        }
    };
    auto request_value = [&](int n) __attribute__((always_inline)) {
        const int t = (n >> 2) * 2 + (n & 1), kk = (n >> 1) & 1;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            vf[n % kRing].s[e] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (s16x4 __attribute__((address_space(3)))*)(lds + values_at + v_lane + kk * (16 * kRowStride) + e * (2 * kRowStride) + t * 64));
        }
    };
    // s += scale_g d, four elements, in assembly: the compiler would spend another instruction an element on moving the lane.  It does not see
    // the lane reads either: a scale that the vector ALU had just written would need the two wait states that the group's first block has.
    // Nor that d comes from the matrix cores, eleven wait states before which it is not to be read: see the order of the slots.
    auto scale_products = [&](int g, int q) __attribute__((always_inline)) {
        f32x16& x = d[g & 1];
        float t0 = s[4 * q], t1 = s[4 * q + 1], t2 = s[4 * q + 2], t3 = s[4 * q + 3];
        float& scale = k_scale[g % 3];
#define MLA_FMAC(first, a, b, c, e) \
    asm volatile(first "v_fmac_f32_dpp %0, %4, %5 row_newbcast:" #a " row_mask:0xf bank_mask:0xf\n\t" \
                 "v_fmac_f32_dpp %1, %4, %6 row_newbcast:" #b " row_mask:0xf bank_mask:0xf\n\t" \
                 "v_fmac_f32_dpp %2, %4, %7 row_newbcast:" #c " row_mask:0xf bank_mask:0xf\n\t" \
                 "v_fmac_f32_dpp %3, %4, %8 row_newbcast:" #e " row_mask:0xf bank_mask:0xf" \
                 : "+v"(t0), "+v"(t1), "+v"(t2), "+v"(t3), "+v"(scale) \
                 : "v"(x[4 * q]), "v"(x[4 * q + 1]), "v"(x[4 * q + 2]), "v"(x[4 * q + 3]))
        switch (q) {
        case 0:
            if (g == 0) { // nothing stands between the first group's matrix instructions and this
                MLA_FMAC("s_nop 7\n\t", 0, 1, 2, 3);
            } else {
                MLA_FMAC("s_nop 1\n\t", 0, 1, 2, 3);
            }
            break;
        case 1: MLA_FMAC("", 4, 5, 6, 7); break;
        case 2: MLA_FMAC("", 8, 9, 10, 11); break;
        default: MLA_FMAC("", 12, 13, 14, 15); break;
        }
#undef MLA_FMAC
        s[4 * q] = t0;
        s[4 * q + 1] = t1;
        s[4 * q + 2] = t2;
        s[4 * q + 3] = t3;
    };
    auto load_k_scale = [&](int g) __attribute__((always_inline)) { k_scale[g % 3] = *(const float*)(lds + keys_at + (lane16 >> 2) + kScaleAt + g * 256); };
    // Slots in pairs, so that two fragments are waited for at once.  The products of group g are scaled from the second matrix instruction of
    // group g + 1 to just before the first of group g + 2, which takes their registers.
    auto multiply_keys = [&](bool values_follow) __attribute__((always_inline)) {
        const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int n = 0; n < kKeySlots; ++n) {
            const int g = n / 4 - 1, r = n % 4;
            if (g >= 2 && r == 0) {
                scale_products(g - 2, 3);
                PREFILL_PHASE_FENCE();
            }
            if (g < 0) {
                s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[n % kRing].b, qr[r].b, r == 0 ? zero : s, 0, 0, 0);
            } else {
                d[g & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[n % kRing].h, qf[g * 4 + r].h, r == 0 ? zero : d[g & 1], 0, 0, 0);
            }
            if (g >= 0 && r == 1) {
                load_k_scale(g);
            }
            if (r % 2 == 1) {
#pragma unroll
                for (int k = n + kRing - 1; k < n + kRing + 1; ++k) {
                    if (k < kKeySlots) {
                        request_key(k, keys_at);
                    } else if (values_follow) {
                        request_value(k - kKeySlots);
                    }
                }
            }
            PREFILL_PHASE_FENCE();
            if (g >= 1 && r > 0) {
                scale_products(g - 1, r - 1);
                PREFILL_PHASE_FENCE();
            }
        }
        scale_products(kGroups - 2, 3);
        PREFILL_PHASE_FENCE();
    };
    // The softmax of the tile whose keys are multiplied, in the 32 slots of the values.  The reference of a column is the largest score seen
    // when it last moved, which it does when a score passes it by 2^8, so that p stays below 2^8 (as in mla_partial_ws).
    float lane_max = kNegInf;
    int window = 0, tile_window = 0; // the accumulators are in units of 2^window, the tile's f16 scales in 2^tile_window
    auto softmax_slot = [&](int n, unsigned int t0) __attribute__((always_inline)) {
        if (n < 4) { // the last group
            if (n > 0) {
                scale_products(kGroups - 1, n - 1);
            }
        } else if (n == 4) {
            scale_products(kGroups - 1, 3);
            if (t0 + kStep > wave_min_hi) { // only the last tiles of a row have tokens to mask
                unsigned int first = t0 + 4u * h;
                asm volatile("" : "+v"(first)); // or sixteen additions leave the branch
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    s[i] = first + 8u * (i >> 2) + (i & 3) < vis_hi ? s[i] : kNegInf;
                }
            }
            lane_max = fmaxf(fmaxf(s[0], s[1]), s[2]);
        } else if (n < 8) {
#pragma unroll
            for (int i = 4 * n - 17; i < 4 * n - 13; i += 2) {
                lane_max = fmaxf(fmaxf(lane_max, s[i]), s[i + 1]);
            }
            if (n == 7) {
                lane_max = fmaxf(lane_max, s[15]);
            }
        } else if (n == 8) {
            const float neg_ref = neg_ref_shifted - (float)kPShift;
            const float above = fmaf(lane_max, latent_log2, neg_ref);
            acc_fix = 1.0f;
            if (__any(above > 8.0f || run_max == kNegInf)) {
                const float step_max = halves_max(above);
                float new_max = run_max;
                if (step_max > 8.0f || run_max == kNegInf) {
                    new_max = fmaxf(run_max, step_max - neg_ref);
                }
                const float safe_max = new_max == kNegInf ? 0.0f : new_max;
                acc_fix = __builtin_amdgcn_exp2f(run_max - safe_max); // 0 while nothing has been seen
                run_sum *= acc_fix;
                run_max = new_max;
                neg_ref_shifted = (float)kPShift - safe_max;
            }
        } else if (n < 25) {
            const int e = n - 9;
            s[e] = __builtin_amdgcn_exp2f(fmaf(s[e], latent_log2, neg_ref_shifted));
            if (e & 1) { // the sum takes the probabilities as the values are multiplied by them: numerator and denominator carry the same weights
                const unsigned int w = pack_f16_hw(s[e - 1], s[e]);
                add_halves(run_sum, w);
                s[e - 1] = __uint_as_float(w);
            }
        }
    };
    // the f16 scales of the tile at `at` from its f32 ones, for the window given; none for tokens from `seen` on
    auto write_scales = [&](unsigned int at, int to_window, unsigned int seen) __attribute__((always_inline)) {
        const float into_window = __uint_as_float((unsigned int)(127 - kPShift - to_window) << 23);
        unsigned int l = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); // the lane again: no registers of the loop
        asm volatile("" : "+v"(l));
        const bool live = 8u * ((l >> 2) & 3u) + 4u * ((l >> 4) & 1u) + (l & 3u) < seen;
        const unsigned int from = at + kScaleAt + (l >> 4) * 128u + (l & 15u) * 4u, to = at + kScale16At + l * 2u;
#pragma unroll 1
        for (unsigned int i = 0; i < kGroups / 2; ++i) { // two groups of 32 tokens
            const float scale = *(const float*)(lds + from + i * 512);
            *(_Float16*)(lds + to + i * 128) = (_Float16)(live && scale == scale ? scale * into_window : 0.0f);
        }
    };
    // Behind the softmax: the probabilities as f16, the accumulators and the scales of the values in one window.  A tile 2^k below the accumulators'
    // window brings its probabilities down by it, up to k = 8 (what they lose then counts for nothing beside the rounding of the products).
    // Further below, its scales are written anew from f32, 2^min(k, 16) lower, which leaves the largest normal (every wave writes the same table and
    // reads it behind its own writes), and the probabilities take what is left.  k = 20 (3,000 keys, scores of deviation 1), 2-norm from 64
    // bits: 7.0e-4; all of it on the probabilities 2.5e-3, all on the scales, as mla_partial_ws has it, 2.8e-3; up to k = 12 2.7e-4
    // whichever way.  Written for every tile below the window (by 2, among latents of one size) the table costs 512 rows of 128 heads
    // behind 16,384 keys 3 %.
    auto take_probabilities = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            pw[i] = __float_as_uint(s[2 * i]);
        }
        if (tile_window > window) {
            acc_fix *= __uint_as_float((unsigned int)(127 - min(tile_window - window, 126)) << 23);
            window = tile_window;
        } else if (tile_window < window) {
            int rest = window - tile_window;
            if (rest > 8) {
                rest = min(max(rest - 16, 0), 14);
                write_scales(keys_at, window - rest, kStep);
            }
            const float down = __uint_as_float((unsigned int)(127 - rest) << 23);
            const unsigned int down2 = pack_f16_hw(down, down);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                pw[i] = pk_mul_f16(pw[i], down2);
            }
        }
    };

    // A tile's window is that of its whole, in the last tile that of the tokens which some row of the workgroup sees: neither windows nor values hang
    // on what only later rows see.  (Rows of one workgroup share their windows, as the row tiles of the GQA chunk kernels do.)
    const unsigned int last_tile_at = (steps - 1u) * kBlock, last_seen = min(end_of_rows - (begin + (steps - 1u) * kStep), (unsigned int)kStep);
    const unsigned int last_window_at = last_tile_at + kWindowAt + (last_seen - 1u) * 4u;
    unsigned int window_at = min((unsigned int)kWindowAt + (kStep - 1) * 4u, last_window_at); // of tile n + 1
    auto load_window = [&](unsigned int at) __attribute__((always_inline)) { return *(const __attribute__((address_space(4))) int*)(uintptr_t)(staged + at); };
    const int seen_window = load_window(last_window_at), whole_window = load_window(last_tile_at + kWindowAt + (kStep - 1) * 4);
    auto next_buf = [](unsigned int at) __attribute__((always_inline)) { return at == (kBufs - 1u) * kTile ? 0u : at + kTile; };
    auto wait_tile = [&](auto left) __attribute__((always_inline)) { // a wave for its own loads and reads, the barrier for the others'
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(decltype(left)::value) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    // Values of tile n, and with MORE the softmax of tile n + 1.  Four slots before the end everything of tile n has been read: the wait for
    // tile n + 2 stands there, the request of tile n + 3 into tile n's buffer, and those of the first keys of the pass to come.
    auto accumulate = [&](auto more, unsigned int t0, unsigned int upcoming_at) __attribute__((always_inline)) {
        constexpr bool MORE = decltype(more)::value;
        u32x4 v_scale[2];
        MlaFrag pf[2];
        auto load_v_scale = [&](int pair) __attribute__((always_inline)) { // pair = 2 g + kk
            v_scale[pair & 1] = *(const u32x4*)(lds + values_at + kScale16At + ((lane16 >> 4) & 32u) + (pair >> 1) * 64 + (pair & 1) * 16);
        };
        auto weigh = [&](int pair, int w) __attribute__((always_inline)) { // P'_g = p * scale_g, one packed multiply per two tokens
            pf[pair & 1].u[w] = pk_mul_f16(pw[4 * (pair & 1) + w], v_scale[pair & 1][w]);
        };
        load_v_scale(0);
        load_v_scale(1);
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            weigh(0, w);
        }
        PREFILL_PHASE_FENCE();
#pragma unroll
        for (int n = 0; n < kValueSlots; ++n) {
            const int pair = n >> 1, t = (n >> 2) * 2 + (n & 1);
            if (MORE && n == kValueSlots - 4) {
                wait_tile(std::integral_constant<int, 0>{});
                load_tile();
            }
            acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[n % kRing].h, pf[pair & 1].h, acc[t], 0, 0, 0);
            if ((n & 1) == 1) {
#pragma unroll
                for (int k = n + kRing - 1; k < n + kRing + 1; ++k) {
                    if (k < kValueSlots) {
                        request_value(k);
                    }
                }
            }
            if (MORE && n >= kValueSlots - 4) {
#pragma unroll
                for (int k = 0; k < kRing; ++k) {
                    if (k * 4 / kRing == n - (kValueSlots - 4)) {
                        request_key(k, upcoming_at);
                    }
                }
            }
            if (pair < 15) {
                weigh(pair + 1, 2 * (n & 1));
                weigh(pair + 1, 2 * (n & 1) + 1);
                if ((n & 1) == 1 && pair < 14) {
                    load_v_scale(pair + 2);
                }
            }
            if constexpr (MORE) {
                softmax_slot(n, t0);
            }
            PREFILL_PHASE_FENCE();
        }
    };
    auto fix_accumulators = [&]() __attribute__((always_inline)) {
        if (__any(acc_fix != 1.0f)) {
#pragma unroll
            for (int t = 0; t < kLatent / 32; ++t) {
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    acc[t][i] *= acc_fix;
                }
            }
        }
    };
    auto open_keys = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < kRing; ++n) {
            request_key(n, keys_at);
        }
        PREFILL_PHASE_FENCE();
    };

    // The queries stay in accumulation registers, where the matrix instructions read them: left to itself the compiler keeps them there too,
    // but copies four registers in front of every one (144 instructions a pass).
#pragma unroll
    for (int ks = 0; ks < kLatent / 16; ++ks) {
        asm volatile("" : "+a"(qf[ks].u));
    }

    // tile 0: keys and softmax alone
    window = tile_window = load_window(window_at);
    window_at = min(window_at + kBlock, last_window_at);
    keys_at = 0;
    values_at = 0;
    wait_tile(std::integral_constant<int, 2 * kOwn>{});
    open_keys();
    multiply_keys(false);
#pragma unroll
    for (int n = 0; n < 25; ++n) {
        if (n == 1) {
            asm volatile("s_nop 7" ::: "memory"); // no values between the last group's matrix instructions and its scaling
        }
        softmax_slot(n, begin);
    }
    take_probabilities(); // acc_fix of the first tile multiplies zeros
    tile_window = load_window(window_at);
    wait_tile(std::integral_constant<int, kOwn>{});
    keys_at = kTile;
    open_keys();
    for (unsigned int step = 1; step < steps; ++step) {
        const unsigned int upcoming_at = next_buf(keys_at);
        multiply_keys(true);
        accumulate(std::integral_constant<bool, true>{}, begin + step * kStep, upcoming_at);
        take_probabilities();
        window_at = min(window_at + kBlock, last_window_at);
        tile_window = load_window(window_at);
        fix_accumulators();
        values_at = keys_at;
        keys_at = upcoming_at;
    }
#pragma unroll
    for (int n = 0; n < kRing; ++n) {
        request_value(n);
    }
    if (whole_window != seen_window) { // the last tile's scales are in the window of its whole: as take_probabilities has left the others
        const int rest = window - seen_window;
        write_scales(values_at, rest > 8 ? window - min(max(rest - 16, 0), 14) : seen_window, last_seen);
    }
    accumulate(std::integral_constant<bool, false>{}, 0u, 0u);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // what was requested past the range lands before the LDS is given back

    const float total = halves_sum(run_sum) * (1.0f / (float)(1 << kPShift));
    if (!col_valid) {
        return;
    }
    if (h == 0u) {
        p.stats[rec * 2] = run_max;
        p.stats[rec * 2 + 1] = total;
    }
    const float out_of_window = __uint_as_float((unsigned int)(127 + window) << 23);
    float* const out = p.partial + rec * (size_t)kLatent + 4u * h;
#pragma unroll
    for (int t = 0; t < kLatent / 32; ++t) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            *(f32x4*)(out + t * 32 + q * 8) = f32x4{acc[t][4 * q], acc[t][4 * q + 1], acc[t][4 * q + 2], acc[t][4 * q + 3]} * out_of_window;
        }
    }
}

} // namespace

uint64_t mla_staged_bytes(unsigned int tiles, unsigned int batch)
{
    return ((uint64_t)tiles * batch + kBlocksBehind) * kBlock;
}

hipError_t launch_mla_partial_staged(const MlaDecodeParams& p, hipStream_t stream)
{
    const unsigned int sequences = p.batch / p.query_rows;
    mla_stage<<<dim3(p.staged_tiles, sequences), dim3(256), 0, stream>>>(p);
    const unsigned int heads_here = p.heads < (unsigned int)kPairs ? p.heads : (unsigned int)kPairs;
    const unsigned int rows_per_wg = (unsigned int)kPairs / heads_here;
    const dim3 grid(p.max_chunks, (p.heads + heads_here - 1u) / heads_here, (p.query_rows + rows_per_wg - 1u) / rows_per_wg * sequences);
    mla_partial_staged<<<grid, dim3(64 * kWaves), 0, stream>>>(p);
    return hipGetLastError();
}

} // namespace zllm
