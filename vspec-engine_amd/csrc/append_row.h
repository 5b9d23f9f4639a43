// append_row.h -- block-table append of one chunk of a token-head row of K or V
// (kv_paged_cache.c:292-303 in the reference, with quantise-on-write for int4 pools):
// the items of the append kernels (paged_kv.hip), and the int4 codec, which the int4
// decode's fused append uses as well (decode_mfma_int4.hip).
#pragma once
#include "kv_common.h"

namespace vkv {

struct AppendParams {
    uint8_t* k;
    uint8_t* v;
    uint16_t* ks;
    uint16_t* vs;
    uint32_t* kf;  // int4 clamp flags or null
    const int32_t* block_tables;
    const int32_t* start_pos;
    // packed-token mode (token_item != null): source token b (n_new == 1) goes to
    // position token_pos[b] of block-table row token_item[b]
    const int32_t* token_item;
    const int32_t* token_pos;
    uint32_t n_items;  // block-table rows in packed-token mode
    // rotary embedding of K (rope_cos != null): rows [max_pos][rope_dim / 2]
    const float* rope_cos;
    const float* rope_sin;
    uint32_t rope_dim;
    uint32_t max_pos;
    bool rope_vec;  // the rotary tables' rows may be read 16 bytes at a time
    // query rows [batch][n_new][hq][head_dim] rotated into q_out (q_in != null)
    const float* q_in;
    float* q_out;
    uint32_t hq;
    // with start_pos and token_item null: source token b goes to position ctx_lens[b] - 1
    // (the append of an f32 decode step of many rows; a context of 0 appends nothing)
    const int32_t* ctx_lens;
    const uint8_t* k_new;
    const uint8_t* v_new;
    uint32_t batch;
    uint32_t n_new;
    uint32_t hkv;
    uint32_t head_dim;
    uint32_t block_tokens;
    uint32_t max_blocks;
    uint32_t num_blocks;
};

// Elements per append work item: a whole 32-element quantisation group for int4 pools,
// 8 elements (16 or 32 bytes) otherwise.
constexpr int append_ept(int dt) { return dt == VSPEC_KV_INT4 ? 32 : 8; }

// A clamp-flag update: flag word `word` gets bit `bit` set or cleared.
struct FlagOp {
    uint32_t* word;
    uint32_t bit;
    bool set;
};

__device__ __forceinline__ void apply_flag(const FlagOp& f) {
    if (!f.word) return;
    if (f.set) atomicOr(f.word, f.bit);
    else atomicAnd(f.word, ~f.bit);
}

// int4 codec of one 32-element group: rep = 2nd-largest |x|, scale = rep/8 (1 if rep == 0),
// floored at 1e-6, rounded to fp16 (saturating), codes rint(x/scale) in [-8,7]; element e
// in nibble e%8 of w[e/8].  top: the code of the largest |x|, as a positive value.
struct Int4Group {
    uint32_t w[4];
    uint32_t s16;
    float sc;
    int top;
};
// the largest two |x| seen (a1 >= a2; equal values count twice, NaN not at all), updated with a
__device__ __forceinline__ void int4_top2(float a, float& a1, float& a2) {
    a2 = fminf(a1, fmaxf(a2, a));
    a1 = fmaxf(a1, a);
}
// fp16 bits of a group's scale from its 2nd-largest |x|
__device__ __forceinline__ uint32_t int4_scale_bits(float rep) {
    float scale = rep > 0.f ? rep / 8.0f : 1.0f;
    if (scale < 1e-6f) scale = 1e-6f;
    uint32_t s16 = float_to_half_bits(scale);
    if ((s16 & 0x7fffu) >= 0x7c00u) s16 = 0x7bffu;
    return s16;
}
__device__ __forceinline__ int int4_code(float x, float sc) {
    const float rr = rintf(x / sc);
    return rr > 7.0f ? 7 : (rr >= -8.0f ? (int)rr : -8);
}
// The same code as a two's complement nibble, for many elements of one scale: inv is 1 / sc
// correctly rounded, and two Newton steps with exact remainders (Markstein) give x / sc correctly
// rounded, 5 operations instead of a division's 10 or so.  x is held within 16 scales first: the
// code is the same, nothing overflows, and NaN goes to -8 as above.  Adding 1.5 * 2^23 rounds to
// the nearest even integer, whose low bits are the code's.
__device__ __forceinline__ uint32_t int4_nibble(float x, float sc, float inv) {
    const float lim = 16.0f * sc;
    const float xc = fminf(fmaxf(x, -lim), lim);
    const float q0 = xc * inv;
    const float q1 = fmaf(fmaf(-q0, sc, xc), inv, q0);
    const float q = fmaf(fmaf(-q1, sc, xc), inv, q1);
    return __builtin_bit_cast(uint32_t, fminf(fmaxf(q, -8.0f), 7.0f) + 12582912.0f) & 0xfu;
}
__device__ __forceinline__ Int4Group int4_encode_group(const float (&x)[32]) {
    float a1 = 0.f, a2 = 0.f;
#pragma unroll
    for (int e = 0; e < 32; ++e) int4_top2(fabsf(x[e]), a1, a2);
    Int4Group q;
    q.s16 = int4_scale_bits(a2);
    q.sc = half_bits_to_float(q.s16);
    const float inv = 1.0f / q.sc;
    q.w[0] = q.w[1] = q.w[2] = q.w[3] = 0u;
#pragma unroll
    for (int e = 0; e < 32; ++e) q.w[e / 8] |= int4_nibble(x[e], q.sc, inv) << (4 * (e % 8));
    q.top = (int)int4_nibble(a1, q.sc, inv);
    return q;
}
// sum, sum of squares and largest magnitude of a group's codes
__device__ __forceinline__ void int4_code_sums(const Int4Group& q, int& c1, int& c2, int& cm) {
    c1 = c2 = 0;
    uint32_t m8 = 0;  // nibbles that hold -8
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t w = q.w[i];
#if defined(__HIP_DEVICE_COMPILE__)
        c1 = __builtin_amdgcn_sdot8((int)w, 0x11111111, c1, false);
        c2 = __builtin_amdgcn_sdot8((int)w, (int)w, c2, false);
#else
        for (int e = 0; e < 8; ++e) {
            const int code = (int32_t)(w << (28 - 4 * e)) >> 28;
            c1 += code;
            c2 += code * code;
        }
#endif
        m8 |= w & ~(w << 1) & ~(w << 2) & ~(w << 3) & 0x88888888u;
    }
    cm = m8 ? 8 : q.top;
}

// The clamp flag of a key from its row's sums: s1 = sum x, s2 = sum x^2 (the groups' scaled
// code sums, added pairwise (g0 + g1) + (g2 + g3)) and m = max |x|.
__device__ __forceinline__ bool int4_flag_from_sums(float s1, float s2, float m, uint32_t head_dim) {
    const float mean = s1 / (float)head_dim;
    const float ex2 = s2 / (float)head_dim;
    const float var1 = ex2 - mean * mean;
    const float th1 = fminf(fmaxf(1e-6f, 4.5f * sqrtf(fmaxf(var1, 0.f))), 16.0f);
    return m > th1 * (1.0f - 0.0009765625f) || var1 <= ex2 * 0.0009765625f;
}

// Clamp flag of a key (attention_ref.c:56 clips every key at its std threshold): set when
// some element may reach alpha * std (alpha 4.5, the reference default; threshold capped at
// 16 as in 3-bit mode) of the dequantised row.  Mean and E[x^2] come from the code sums of
// the row's groups, which sit in lanes 2c of an aligned run of 2 * head_dim / 32 lanes (the
// append work items of one row: all of these lanes call this together); the 2^-10 margins
// cover the one-pass variance (the decode kernel's screen test, run once per key here).
__device__ __forceinline__ bool int4_key_flag(const Int4Group& q, uint32_t head_dim) {
    int c1, c2, cm;
    int4_code_sums(q, c1, c2, cm);
    float s1 = q.sc * (float)c1;
    float s2 = (q.sc * q.sc) * (float)c2;
    float m = q.sc * (float)cm;
    for (uint32_t o = 2; o < 2 * (head_dim / 32); o <<= 1) {
        s1 += __shfl_xor(s1, (int)o);
        s2 += __shfl_xor(s2, (int)o);
        m = fmaxf(m, __shfl_xor(m, (int)o));
    }
    return int4_flag_from_sums(s1, s2, m, head_dim);
}

// V code byte nn (0..15) of group c: d = 32c + nn in the low nibble, d = 32c + 16 + nn in
// the high one (int4_v_byte places it).
__device__ __forceinline__ uint32_t int4_v_group_byte(const uint32_t (&w)[4], int nn) {
    const uint32_t lo = (w[nn / 8] >> (4 * (nn % 8))) & 0xfu;
    const uint32_t hi = (w[2 + nn / 8] >> (4 * (nn % 8))) & 0xfu;
    return lo | (hi << 4);
}

// Offset of V code byte nn of group c of token `slot` within its 16-token tile.
__device__ __forceinline__ uint32_t int4_v_tile_byte(uint32_t slot, uint32_t c, uint32_t nn, uint32_t D) {
    const uint32_t tt = slot & 15u, tg = tt >> 2, tr = tt & 3u;
    return (16u * tg + nn) * (D / 8u) + 4u * c + 2u * (tr & 1u) + (tr >> 1);
}

// N elements (a multiple of 8) from element el on, as floats
template <int SRC, int N>
__device__ __forceinline__ void load_elements(const uint8_t* src, size_t el, float (&x)[N]) {
    if constexpr (SRC == VSPEC_KV_F32) {
        const float4* s4 = reinterpret_cast<const float4*>(src + el * 4);
#pragma unroll
        for (int j = 0; j < N / 4; ++j) {
            const float4 w = s4[j];
            x[4 * j] = w.x; x[4 * j + 1] = w.y; x[4 * j + 2] = w.z; x[4 * j + 3] = w.w;
        }
    } else {
        const uint4* s4 = reinterpret_cast<const uint4*>(src + el * 2);
#pragma unroll
        for (int j = 0; j < N / 8; ++j) unpack_f16x8(s4[j], x + 8 * j);
    }
}

// Chunk c of the token-head row of K (which 0) or V (which 1) whose first source element
// is src_el, written at position pos of block-table row `seq`, kv head h.  Positions past
// the table, behind an invalid entry or (with rotary tables) past max_pos are not written.
// ROPE: the launch may carry rotary tables (without it their code and registers go)
template <int DT, int SRC, bool ROPE = true>
__device__ __forceinline__ void append_chunk(const AppendParams& p, uint32_t seq, uint32_t pos, uint32_t h,
                                             uint32_t c, int which, size_t src_el) {
    constexpr int EPT = append_ept(DT);
    const uint32_t lb = pos / p.block_tokens;
    if (lb >= p.max_blocks) return;
    // the source elements are read before the table entry is looked at: both loads are in
    // flight together
    float x[EPT];
    const uint8_t* src = which ? p.v_new : p.k_new;
    load_elements<SRC, EPT>(src, src_el, x);
    const int32_t phys = p.block_tables[(size_t)seq * p.max_blocks + lb];
    if (phys < 0 || (uint32_t)phys >= p.num_blocks) return;
    const uint32_t slot = pos % p.block_tokens;
    const size_t row = ((size_t)phys * p.hkv + h) * p.block_tokens + slot;
    const size_t e0 = (size_t)c * EPT;  // first element of this chunk within the row

    const bool rope = ROPE && p.rope_cos != nullptr;
    if (rope) {
        if (pos >= p.max_pos) return;  // no table row: the token is not written
        if (!which) {
#pragma clang fp contract(off)
            // pairs (i, i + half) of the first rope_dim elements rotate by row `pos`:
            // x1*c - x2*s, x1*s + x2*c, each product and sum rounded separately (no
            // fused multiply-add: hipcc contracts by default)
            const uint32_t half = p.rope_dim / 2;
            const size_t row0 = src_el - e0;  // element 0 of this token-head row
            const float* cr = p.rope_cos + (size_t)pos * half;
            const float* sr = p.rope_sin + (size_t)pos * half;
            if (p.rope_vec && half % EPT == 0) {
                // the chunk lies whole in the first or the second half of the rotated
                // elements, or past them: its partners and table entries are one run each
                if (e0 < p.rope_dim) {
                    const bool first = e0 < half;
                    const uint32_t i0 = first ? (uint32_t)e0 : (uint32_t)e0 - half;
                    float other[EPT], cv[EPT], sv[EPT];
                    load_elements<SRC, EPT>(src, row0 + (first ? e0 + half : e0 - half), other);
                    load_elements<VSPEC_KV_F32, EPT>(reinterpret_cast<const uint8_t*>(cr), i0, cv);
                    load_elements<VSPEC_KV_F32, EPT>(reinterpret_cast<const uint8_t*>(sr), i0, sv);
#pragma unroll
                    for (int e = 0; e < EPT; ++e)
                        x[e] = first ? x[e] * cv[e] - other[e] * sv[e] : other[e] * sv[e] + x[e] * cv[e];
                }
            } else {
#pragma unroll
                for (int e = 0; e < EPT; ++e) {
                    const uint32_t d = (uint32_t)e0 + e;
                    if (d >= p.rope_dim) continue;
                    const uint32_t i = d < half ? d : d - half;
                    const size_t pe = row0 + (d < half ? d + half : d - half);
                    float other;
                    if constexpr (SRC == VSPEC_KV_F32) {
                        other = reinterpret_cast<const float*>(src)[pe];
                    } else {
                        other = half_bits_to_float(reinterpret_cast<const uint16_t*>(src)[pe]);
                    }
                    const float c = cr[i], sn = sr[i];
                    x[e] = d < half ? x[e] * c - other * sn : other * sn + x[e] * c;
                }
            }
        }
    }

    uint8_t* dst = which ? p.v : p.k;
    if constexpr (DT == VSPEC_KV_F32) {
        float4* d4 = reinterpret_cast<float4*>(dst + (row * p.head_dim + e0) * 4);
        d4[0] = make_float4(x[0], x[1], x[2], x[3]);
        d4[1] = make_float4(x[4], x[5], x[6], x[7]);
    } else if constexpr (DT == VSPEC_KV_F16) {
        uint32_t hb[8];
        if (SRC == VSPEC_KV_F16 && !(rope && !which)) {
            // pure copy of the source bits
            const uint4 w = *reinterpret_cast<const uint4*>(src + src_el * 2);
            const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                hb[2 * k] = ws[k] & 0xffffu;
                hb[2 * k + 1] = ws[k] >> 16;
            }
        } else {
#pragma unroll
            for (int k = 0; k < 8; ++k) hb[k] = float_to_half_bits(x[k]);
        }
        if (which) {
            // V in 4-token groups: element (d, slot) at f16_v_index (stride 4 in d)
            uint16_t* vt = reinterpret_cast<uint16_t*>(dst) +
                           f16_v_index((size_t)phys * p.hkv + h, p.block_tokens, p.head_dim, slot, e0);
#pragma unroll
            for (int k = 0; k < 8; ++k) vt[4 * k] = (uint16_t)hb[k];
        } else {
            *reinterpret_cast<uint4*>(dst + (row * p.head_dim + e0) * 2) =
                make_uint4(hb[0] | (hb[1] << 16), hb[2] | (hb[3] << 16), hb[4] | (hb[5] << 16),
                           hb[6] | (hb[7] << 16));
        }
    } else {
        const Int4Group q = int4_encode_group(x);
        if (!which && p.kf) {
            const bool flag = int4_key_flag(q, p.head_dim);
            if (c == 0) {
                const FlagOp op = {p.kf + ((size_t)phys * p.hkv + h) * (p.block_tokens / 16) + slot / 16,
                                   1u << (slot % 16), flag};
                apply_flag(op);
            }
        }
        const size_t bh = (size_t)phys * p.hkv + h;
        if (which) {
            // V tiles: byte n of this group's 16 holds d = 32c + n (low nibble) and
            // d = 32c + 16 + n (high nibble) of this token, at lane chunk (g, n)
            uint8_t* vb = dst + bh * ((size_t)p.block_tokens * p.head_dim / 2) + (size_t)(slot >> 4) * (8u * p.head_dim);
#pragma unroll
            for (int nn = 0; nn < 16; ++nn) vb[int4_v_tile_byte(slot, c, nn, p.head_dim)] = (uint8_t)int4_v_group_byte(q.w, nn);
            p.vs[row * (p.head_dim / 32) + c] = (uint16_t)q.s16;
        } else {
            uint4* d4 = reinterpret_cast<uint4*>(dst + row * (p.head_dim / 2) + e0 / 2);
            *d4 = make_uint4(q.w[0], q.w[1], q.w[2], q.w[3]);
            p.ks[int4_ks_index(bh, p.head_dim / 32, p.block_tokens, slot, c)] = (uint16_t)q.s16;
        }
    }
}

// Work items of one append launch: 2 (K, V) x chunks per row x kv heads x tokens.
template <int DT>
__device__ __forceinline__ uint64_t append_items(const AppendParams& p) {
    return (uint64_t)p.batch * p.n_new * p.hkv * (p.head_dim / append_ept(DT)) * 2;
}

// Where source token b (packed tokens, or sequence b's first token) goes: block-table row
// and position.  False: nowhere.
__device__ __forceinline__ bool append_where(const AppendParams& p, uint32_t b, int32_t& item, int32_t& sp) {
    item = p.token_item ? p.token_item[b] : (int32_t)b;
    if (p.token_item) {
        sp = p.token_pos[b];
    } else if (p.start_pos) {
        sp = p.start_pos[b];
    } else {
        const int32_t cl = p.ctx_lens[b];
        sp = cl > 0 ? cl - 1 : -1;
    }
    return sp >= 0 && item >= 0 && !(p.token_item && (uint32_t)item >= p.n_items);
}

// One work item of the append kernel (any order; no two items write the same bytes):
// item `it` = ((token, kv head, chunk) << 1) | which.  Uniform batch (start_pos), packed
// tokens (token_item / token_pos, items not below n_items skipped) or the decode step's
// token at ctx_lens[b] - 1.
template <int DT, int SRC, bool ROPE = true>
__device__ __forceinline__ void append_item(const AppendParams& p, uint64_t it) {
    constexpr int EPT = append_ept(DT);
    const uint32_t chunks = p.head_dim / EPT;
    const int which = (int)(it & 1);
    uint64_t r = it >> 1;
    const uint32_t c = (uint32_t)(r % chunks);
    r /= chunks;
    const uint32_t h = (uint32_t)(r % p.hkv);
    r /= p.hkv;
    const uint32_t i = (uint32_t)(r % p.n_new);
    const uint32_t b = (uint32_t)(r / p.n_new);

    int32_t item, sp;
    if (!append_where(p, b, item, sp)) return;
    const size_t src_el = (((size_t)b * p.n_new + i) * p.hkv + h) * p.head_dim + (size_t)c * EPT;
    append_chunk<DT, SRC, ROPE>(p, (uint32_t)item, (uint32_t)sp + i, h, c, which, src_el);
}

// ---------------------------------------------------------------------------
// f16 and f32 pools, items by section: K chunks, then V chunks, then query chunks (each
// section a whole number of workgroups).  The K section is one 8-element chunk of one row
// an item, as append_item's; the V section of f16 pools takes a chunk of a whole group of
// 4 tokens where the launch holds the group's tokens, since a group's chunk is 64
// contiguous bytes of the pool while one token's is eight 2-byte pieces.
// ---------------------------------------------------------------------------

// V items of one sequence per chunk and head: groups of 4 positions that n_new tokens may
// meet (uniform batches of f16 pools), else tokens
template <int DT>
__host__ __device__ __forceinline__ uint32_t append_v_units(uint32_t n_new, bool packed) {
    return DT == VSPEC_KV_F16 && !packed ? (n_new + 2) / 4 + 1 : n_new;
}

// One chunk of the 4 tokens of a group (positions pos0 .. pos0 + 3, pos0 a multiple of 4;
// token j's chunk at source element el0 + j * stride).
template <int SRC>
__device__ __forceinline__ void append_v_group(const AppendParams& p, uint32_t seq, uint32_t pos0, uint32_t h, uint32_t c,
                                               size_t el0, size_t stride) {
    const uint32_t lb = pos0 / p.block_tokens;
    if (lb >= p.max_blocks) return;
    uint32_t w[4][4];  // token, pair of elements
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const size_t el = el0 + j * stride;
        if constexpr (SRC == VSPEC_KV_F16) {
            const uint4 s = *reinterpret_cast<const uint4*>(p.v_new + el * 2);
            w[j][0] = s.x; w[j][1] = s.y; w[j][2] = s.z; w[j][3] = s.w;
        } else {
            float x[8];
            load_elements<SRC, 8>(p.v_new, el, x);
#pragma unroll
            for (int e = 0; e < 4; ++e) w[j][e] = float_to_half_bits(x[2 * e]) | (float_to_half_bits(x[2 * e + 1]) << 16);
        }
    }
    const int32_t phys = p.block_tables[(size_t)seq * p.max_blocks + lb];
    if (phys < 0 || (uint32_t)phys >= p.num_blocks) return;
    uint4* d = reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(p.v) +
                                        f16_v_index((size_t)phys * p.hkv + h, p.block_tokens, p.head_dim,
                                                    pos0 % p.block_tokens, 8 * c));
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        // elements 2e and 2e + 1: tokens 0..3 of each
        d[e] = make_uint4((w[0][e] & 0xffffu) | (w[1][e] << 16), (w[2][e] & 0xffffu) | (w[3][e] << 16),
                          (w[0][e] >> 16) | (w[1][e] & 0xffff0000u), (w[2][e] >> 16) | (w[3][e] & 0xffff0000u));
    }
}

// Item `it` of the K section: ((sequence, token), kv head, chunk).
template <int DT, int SRC, bool ROPE>
__device__ __forceinline__ void append_k_item(const AppendParams& p, uint32_t it) {
    const uint32_t chunks = p.head_dim / 8;
    const uint32_t c = it % chunks, r = it / chunks;
    const uint32_t h = r % p.hkv, t = r / p.hkv;
    const uint32_t b = t / p.n_new, i = t % p.n_new;
    int32_t item, sp;
    if (!append_where(p, b, item, sp)) return;
    append_chunk<DT, SRC, ROPE>(p, (uint32_t)item, (uint32_t)sp + i, h, c, 0, ((size_t)t * p.hkv + h) * p.head_dim + 8 * c);
}

// Item `it` of the V section: ((sequence, group or token), kv head, chunk).
template <int DT, int SRC, bool ROPE>
__device__ __forceinline__ void append_v_item(const AppendParams& p, uint32_t it) {
    const uint32_t chunks = p.head_dim / 8;
    const uint32_t c = it % chunks, r = it / chunks;
    const uint32_t h = r % p.hkv, u = r / p.hkv;
    const size_t stride = (size_t)p.hkv * p.head_dim;
    const size_t el_hc = (size_t)h * p.head_dim + 8 * c;
    int32_t item, sp;
    if constexpr (DT == VSPEC_KV_F16) {
        if (!p.token_item) {
            const uint32_t units = append_v_units<DT>(p.n_new, false);
            const uint32_t b = u / units, g = u % units;
            if (!append_where(p, b, item, sp)) return;
            const uint32_t pos0 = ((uint32_t)sp & ~3u) + 4 * g;
            const size_t el_b = (size_t)b * p.n_new * stride + el_hc;
            // tokens of the launch in the group: lo .. hi - 1 of 0..3
            const uint32_t lo = pos0 < (uint32_t)sp ? (uint32_t)sp - pos0 : 0u;
            const uint32_t end = (uint32_t)sp + p.n_new;
            const uint32_t hi = pos0 >= end ? 0u : (end - pos0 < 4u ? end - pos0 : 4u);
            if (lo == 0 && hi == 4 && !(ROPE && p.rope_cos && pos0 + 3 >= p.max_pos)) {
                append_v_group<SRC>(p, (uint32_t)item, pos0, h, c, el_b + (size_t)(pos0 - (uint32_t)sp) * stride, stride);
                return;
            }
            for (uint32_t j = lo; j < hi; ++j) {
                append_chunk<DT, SRC, ROPE>(p, (uint32_t)item, pos0 + j, h, c, 1, el_b + (size_t)(pos0 + j - (uint32_t)sp) * stride);
            }
            return;
        }
        if (!append_where(p, u, item, sp)) return;
        // the packed tokens around u hold its group, in order: its first token's items
        // write the group, the others nothing
        const uint32_t r4 = (uint32_t)sp & 3u;
        if (u >= r4 && u - r4 + 4 <= p.batch) {
            const uint32_t u0 = u - r4;
            bool whole = true;
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j)
                whole = whole && p.token_item[u0 + j] == item && p.token_pos[u0 + j] == sp - (int32_t)r4 + (int32_t)j;
            if (whole) {
                if (r4 == 0) append_v_group<SRC>(p, (uint32_t)item, (uint32_t)sp, h, c, u * stride + el_hc, stride);
                return;
            }
        }
        append_chunk<DT, SRC, ROPE>(p, (uint32_t)item, (uint32_t)sp, h, c, 1, u * stride + el_hc);
    } else {
        const uint32_t b = u / p.n_new, i = u % p.n_new;
        if (!append_where(p, b, item, sp)) return;
        append_chunk<DT, SRC, ROPE>(p, (uint32_t)item, (uint32_t)sp + i, h, c, 1, u * stride + el_hc);
    }
}

// Query section: an item is 4 elements of the first half of the rotated elements and their
// partners, or 4 elements past them, of up to kRopeHeads heads of one token (the table
// entries are read once for them all).  rope_dim / 2 a multiple of 4, rows and tables
// 16-byte aligned.
constexpr uint32_t kRopeHeads = 4;
__host__ __device__ __forceinline__ uint32_t rope_q_chunks(uint32_t head_dim, uint32_t rope_dim) {
    return rope_dim / 8 + (head_dim - rope_dim) / 4;
}
__device__ __forceinline__ void rope_q_item(const AppendParams& p, uint32_t it) {
    const uint32_t chunks = rope_q_chunks(p.head_dim, p.rope_dim);
    const uint32_t c = it % chunks, r = it / chunks;
    const uint32_t hg = (p.hq + kRopeHeads - 1) / kRopeHeads;
    const uint32_t h0 = (r % hg) * kRopeHeads, t = r / hg;
    int32_t item, sp;
    if (!append_where(p, t / p.n_new, item, sp)) return;
    const uint32_t pos = (uint32_t)sp + t % p.n_new;
    if (pos >= p.max_pos) return;
    const uint32_t half = p.rope_dim / 2, d4 = p.head_dim / 4;
    const uint32_t nh = p.hq - h0 < kRopeHeads ? p.hq - h0 : kRopeHeads;
    const float4* in = reinterpret_cast<const float4*>(p.q_in) + ((size_t)t * p.hq + h0) * d4;
    float4* out = reinterpret_cast<float4*>(p.q_out) + ((size_t)t * p.hq + h0) * d4;
    if (c >= half / 4) {  // past the rotated elements
        const uint32_t i = c + half / 4;
        for (uint32_t h = 0; h < nh; ++h) out[h * d4 + i] = in[h * d4 + i];
        return;
    }
    const float4 cv = reinterpret_cast<const float4*>(p.rope_cos + (size_t)pos * half)[c];
    const float4 sv = reinterpret_cast<const float4*>(p.rope_sin + (size_t)pos * half)[c];
    float4 x[kRopeHeads], y[kRopeHeads];
#pragma unroll
    for (uint32_t h = 0; h < kRopeHeads; ++h) {
        const uint32_t hh = h < nh ? h : 0;  // loads stay unconditional
        x[h] = in[hh * d4 + c];
        y[h] = in[hh * d4 + c + half / 4];
    }
#pragma unroll
    for (uint32_t h = 0; h < kRopeHeads; ++h) {
#pragma clang fp contract(off)
        if (h >= nh) break;
        out[h * d4 + c] = make_float4(x[h].x * cv.x - y[h].x * sv.x, x[h].y * cv.y - y[h].y * sv.y,
                                      x[h].z * cv.z - y[h].z * sv.z, x[h].w * cv.w - y[h].w * sv.w);
        out[h * d4 + c + half / 4] = make_float4(x[h].x * sv.x + y[h].x * cv.x, x[h].y * sv.y + y[h].y * cv.y,
                                                 x[h].z * sv.z + y[h].z * cv.z, x[h].w * sv.w + y[h].w * cv.w);
    }
}

}  // namespace vkv
