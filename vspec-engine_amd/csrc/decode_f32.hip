// decode_f32.hip -- single-query GQA decode attention over f32 paged KV on the vector ALUs
// (fp32 products throughout: the matrix cores' f32 form measured no faster), with the
// reference numerics (per-key std clamp, attention_ref.c:50-62).
//
// One workgroup of 4 waves per part of a work item (item_part); wave w takes the part's
// tiles w, w + 4, ...  D/16 lanes hold one key, 16 elements each (chunks of 4 elements
// sub + j * D/16); D/8 lanes hold one token of V, 8 elements each.  The decode step's tokens are
// taken from their source rows by every wave that reads their tiles, whichever row of the batch
// they belong to, so no launch precedes this one.
//
// Bound by the memory rate at full batches (16 x 2049 tokens: 269 MB in 52.7 us with the merge
// launch, 61 us with an append launch ahead and ordinary loads) and by a wave's chain of round
// trips per tile (about 3 us) at small ones.
#include "kv_common.h"

namespace vkv {
namespace {

template <bool ONCE>
__device__ __forceinline__ float4 load_row4(const float* p) {
    if constexpr (!ONCE) return *reinterpret_cast<const float4*>(p);
    const uint4 w = load_stream4(p);
    return make_float4(__builtin_bit_cast(float, w.x), __builtin_bit_cast(float, w.y), __builtin_bit_cast(float, w.z),
                       __builtin_bit_cast(float, w.w));
}

// 4 elements of a new token's row in its source type
__device__ __forceinline__ float4 load_new4(const uint8_t* src, size_t el, int32_t type) {
    if (type == VSPEC_KV_F32) return *reinterpret_cast<const float4*>(src + el * 4);
    const uint2 w = *reinterpret_cast<const uint2*>(src + el * 2);
    return make_float4(half_bits_to_float(w.x & 0xffffu), half_bits_to_float(w.x >> 16), half_bits_to_float(w.y & 0xffffu),
                       half_bits_to_float(w.y >> 16));
}

// Clip a row held by LPK lanes (16 elements each) to +-max(1e-6, alpha*std),
// then to +-input_clip (three_bit_runtime_modules.c:175-203, :138-173).
template <int LPK, int D>
__device__ __forceinline__ void clamp_row(float* x, float alpha, float input_clip) {
    float s = 0.f;
#pragma unroll
    for (int e = 0; e < 16; ++e) s += x[e];
    const float mean = group_sum<LPK>(s) * (1.0f / D);
    float v = 0.f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const float d = x[e] - mean;
        v = fmaf(d, d, v);
    }
    const float var = group_sum<LPK>(v) * (1.0f / D);
    const float th = fminf(fmaxf(1e-6f, alpha * sqrtf(var)), input_clip);
#pragma unroll
    for (int e = 0; e < 16; ++e) x[e] = fminf(fmaxf(x[e], -th), th);
}

// ONCE: each tile is read by one work item; else the gsplit items of a kv head share it in their
// XCD's L2 (25 x 37-2392 tokens, 8 heads per kv head: 54.8 us, 57.5 past the caches).  Read once,
// K goes past the caches, and V too with 64-element heads.  First pass on a pool just written /
// repeated passes on three pools in turn, us, K and V past the caches, K alone, neither:
//   16 x 2049 tokens, D = 128         76 / 55.2   67 / 54.7   68 / 58.9
//   64 x 1025, D = 128               129 / 93.2  118 / 91.3  159 / 100.1
//   13 x 3101-6203, D = 128          130 / 106   159 / 104   171 / 108
//   36 x 649-5195, D = 64             86 / 69.9   79 / 70.7   80 / 71.0
// (the kernel before the item split: 70 / 61.2, 162 / 105.7, 158 / 105.2, 98 / 83.3)
// STEP: the decode step's tokens come with the launch (k_new).
template <int D, int GW, bool ONCE, bool STEP>
__global__ __launch_bounds__(256, 2) void decode_f32(DecodeParams p) {
    constexpr int LPK = D / 16;           // lanes per key
    constexpr int KPP = 64 / LPK;         // keys per K pass
    constexpr int KPASS = kTile / KPP;    // K passes per tile
    constexpr int VLPT = D / 8;           // lanes per token on the V side
    constexpr int VTPP = 64 / VLPT;       // tokens per V pass
    constexpr int VPASS = kTile / VTPP;   // V passes per tile
    static_assert(KPASS >= 1 && VPASS >= 1, "tile geometry");

    __shared__ float p_lds[kWaves][2][kTile][GW];
    __shared__ float comb[kWaves][GW][D + 2];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // The decode step's tokens, row i's in lane i (at most kStepRows rows).  Rows may share
    // blocks, as two rows that verify two tokens of one session do: a tile can hold tokens that
    // other rows' workgroups store while it is read here, so all of them are taken from the
    // source rows.  The two dependent loads run beside those of the item's context and entry.
    const int ctx_cap = (int)(p.max_blocks * p.block_tokens);
    const int step_row = min(lane, (int)p.batch - 1);
    const int step_ctx = STEP ? p.ctx_lens[step_row] : 0;
    int lo, hi;
    size_t part_slot;
    const ItemCursor c = item_part<true>(p, lo, hi, part_slot);
    if (lo >= hi) return;
    const int hk = __builtin_amdgcn_readfirstlane(c.y / (int)p.gsplit);
    const int hq0 = c.y * GW;
    const int tiles_per_block = (int)p.block_tokens / kTile;
    const const_i32* table = as_const(p.block_tables) + (size_t)c.b * p.max_blocks;

    const int kk = lane / LPK;      // key within a K pass
    const int sub = lane % LPK;     // lane within the key
    const int vc = lane % VLPT;     // V chunk
    const int vt = lane / VLPT;     // token within a V pass

    int tile = lo + wave;
    int entry = table[min(tile, hi - 1) / tiles_per_block];
    const int raw_ctx = as_const(p.ctx_lens)[c.b];
    const int ctx = min(max(raw_ctx, 0), ctx_cap);
    // the row's own new token: its position, and the decoded tile whose wave stores it
    const int papp = STEP && raw_ctx >= 1 && raw_ctx <= ctx_cap ? raw_ctx - 1 : -1;
    const int tnew = papp >= 0 ? min(papp / kTile, c.U - 1) : -1;

    // q' = clip(q) * scale * log2(e), in the K-side lane layout
    float qv[GW][16];
#pragma unroll
    for (int h = 0; h < GW; ++h) {
        const float* qrow = p.q + ((size_t)c.b * p.hq + hq0 + h) * D;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float4 w = *reinterpret_cast<const float4*>(qrow + 4 * (sub + j * LPK));
            qv[h][4 * j] = w.x; qv[h][4 * j + 1] = w.y; qv[h][4 * j + 2] = w.z; qv[h][4 * j + 3] = w.w;
        }
    }
    // (behind the query rows, which are waited for first.  What it costs, a step of one tile or two
    // pays: 3 x 40 tokens 7.9 -> 8.3 us, 60 x 20-100 9.6 -> 10.3; one gather per workgroup through
    // LDS instead of one per wave 8.5 and 10.6)
    int step_block = -1, step_slot = 0;
    if constexpr (STEP) {
        const int pos = min(max(step_ctx, 1), ctx_cap) - 1;
        const int e = p.block_tables[(size_t)step_row * p.max_blocks + pos / (int)p.block_tokens];
        const bool is = lane < (int)p.batch && step_ctx >= 1 && step_ctx <= ctx_cap && (uint32_t)e < p.num_blocks;
        step_block = is ? e : -1;
        step_slot = pos % (int)p.block_tokens;
    }
#pragma unroll
    for (int h = 0; h < GW; ++h) {
        clamp_row<LPK, D>(qv[h], p.alpha, p.input_clip);
#pragma unroll
        for (int e = 0; e < 16; ++e) qv[h][e] *= p.qscale;
    }

    float m_run[GW], l_run[GW], acc[GW][8];
#pragma unroll
    for (int h = 0; h < GW; ++h) {
        m_run[h] = -INFINITY;
        l_run[h] = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[h][e] = 0.f;
    }

    const bool v_early = D == 64 || hi - lo <= kWaves;
    int buf = 0;
    for (; tile < hi; tile += kWaves) {
        const int phys = entry;
        const int lblock = tile / tiles_per_block;
        entry = table[min(tile + kWaves, hi - 1) / tiles_per_block];  // the wave's next tile's
        const bool ok = phys >= 0 && (uint32_t)phys < p.num_blocks;  // else the tile is skipped
        const int tok0 = tile * kTile;
        const int slot0 = (tile % tiles_per_block) * kTile;
        const size_t row0 = ((size_t)(ok ? phys : 0) * p.hkv + hk) * p.block_tokens + slot0;
        const float* krow = reinterpret_cast<const float*>(p.k) + row0 * D;
        const float* vrow = reinterpret_cast<const float*>(p.v) + row0 * D;
        const size_t new_el = ((size_t)c.b * p.hkv + hk) * D;
        // (its block may be another one where the context exceeds the bound)
        if (tile == tnew && c.y % (int)p.gsplit == 0) {
            const int e = table[papp / (int)p.block_tokens];
            if (e >= 0 && (uint32_t)e < p.num_blocks && lane < D / 4) {
                const size_t row = ((size_t)e * p.hkv + hk) * p.block_tokens + papp % (int)p.block_tokens;
                *reinterpret_cast<float4*>(const_cast<uint8_t*>(p.k) + (row * D + 4 * lane) * 4) = load_new4(p.k_new, new_el + 4 * lane, p.append_src);
                *reinterpret_cast<float4*>(const_cast<uint8_t*>(p.v) + (row * D + 4 * lane) * 4) = load_new4(p.v_new, new_el + 4 * lane, p.append_src);
            }
        }
        if (!ok) continue;
        // valid slots of this tile: below the context and, with block_used, below its
        // block's used count (a prefix of the block's slots)
        const int lim = p.block_used ? min(ctx - tok0, used_cap(as_const(p.block_used)[(size_t)c.b * p.max_blocks + lblock], slot0))
                                     : ctx - tok0;
        if (lim <= 0) continue;

        // V goes out with K where a wave's chain of round trips, not the memory rate, is what
        // it waits for: one tile per wave (89 x 1-26 tokens 19.2 -> 17.4 us), and 64-element
        // heads (36 x 649-5195 67.0 -> 62.6 us); with 128 and longer parts it only costs
        // registers (16 x 2049 55.7 -> 56.2 us)
        float4 va[VPASS], vb[VPASS];
        auto load_v = [&]() {
#pragma unroll
            for (int vp = 0; vp < VPASS; ++vp) {
                va[vp] = load_row4<ONCE && D == 64>(vrow + (size_t)(vp * VTPP + vt) * D + 8 * vc);
                vb[vp] = load_row4<ONCE && D == 64>(vrow + (size_t)(vp * VTPP + vt) * D + 8 * vc + 4);
            }
        };
        if (v_early) load_v();
        // ---- scores ----
        float s[KPASS][GW], x[KPASS][16];
        const int ts = STEP && tile == papp / kTile ? papp % kTile : -1;  // the row's own token's slot
#pragma unroll
        for (int kp = 0; kp < KPASS; ++kp) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float4 w = load_row4<ONCE>(krow + (size_t)(kp * KPP + kk) * D + 4 * (sub + j * LPK));
                x[kp][4 * j] = w.x; x[kp][4 * j + 1] = w.y; x[kp][4 * j + 2] = w.z; x[kp][4 * j + 3] = w.w;
            }
        }
        auto take_k = [&](const int at, const size_t el) {
#pragma unroll
            for (int kp = 0; kp < KPASS; ++kp) {
                if (kp * KPP + kk != at) continue;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float4 w = load_new4(p.k_new, el + 4 * (sub + j * LPK), p.append_src);
                    x[kp][4 * j] = w.x; x[kp][4 * j + 1] = w.y; x[kp][4 * j + 2] = w.z; x[kp][4 * j + 3] = w.w;
                }
            }
        };
        if (STEP && ts >= 0) take_k(ts, new_el);
        // the rows with another new token in this tile (looked up once the tile is on its way)
        const uint64_t fresh =
            STEP ? __ballot(step_block == phys && step_slot / kTile == slot0 / kTile && (ts < 0 || lane != c.b)) : 0ull;
        for (uint64_t m = fresh; m; m &= m - 1) {
            const int r = __builtin_ctzll(m);
            take_k(__builtin_amdgcn_readlane(step_slot, r) % kTile, ((size_t)r * p.hkv + hk) * D);
        }
#pragma unroll
        for (int kp = 0; kp < KPASS; ++kp) {
            const int slot = kp * KPP + kk;
            clamp_row<LPK, D>(x[kp], p.alpha, p.input_clip);
            const bool valid = slot < lim;
#pragma unroll
            for (int h = 0; h < GW; ++h) {
                float d = 0.f;
#pragma unroll
                for (int e = 0; e < 16; ++e) d = fmaf(qv[h][e], x[kp][e], d);
                d = group_sum<LPK>(d);
                d = fminf(fmaxf(d, -p.logit_clip), p.logit_clip);
                s[kp][h] = valid ? d : -INFINITY;
            }
        }

        // ---- online softmax (rescale only when the max grows by > 2^8) ----
#pragma unroll
        for (int h = 0; h < GW; ++h) {
            float mt = s[0][h];
#pragma unroll
            for (int kp = 1; kp < KPASS; ++kp) mt = fmaxf(mt, s[kp][h]);
            mt = max_across_groups<LPK>(mt);
            // uniform across the wave after the reduction: keep it in an SGPR
            mt = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, mt)));
            if (mt > m_run[h] + 8.0f) {
                const float f = exp2f(m_run[h] - mt);
                l_run[h] *= f;
#pragma unroll
                for (int e = 0; e < 8; ++e) acc[h][e] *= f;
                m_run[h] = mt;
            }
        }
#pragma unroll
        for (int kp = 0; kp < KPASS; ++kp) {
            if (sub < GW) {
                float sv = s[kp][0], mv = m_run[0];
#pragma unroll
                for (int h = 1; h < GW; ++h) {
                    if (sub == h) {
                        sv = s[kp][h];
                        mv = m_run[h];
                    }
                }
                p_lds[wave][buf][kp * KPP + kk][sub] = exp2f(sv - fmaxf(mv, kLowestMax));
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

        // ---- P.V ----
        if (!v_early) load_v();
        const bool tail = lim < kTile;
#pragma unroll
        for (int vp = 0; vp < VPASS; ++vp) {
            const int slot = vp * VTPP + vt;
            float4 a = va[vp], b = vb[vp];
            if (STEP && slot == ts) {
                a = load_new4(p.v_new, new_el + 8 * vc, p.append_src);
                b = load_new4(p.v_new, new_el + 8 * vc + 4, p.append_src);
            }
            for (uint64_t m = fresh; m; m &= m - 1) {
                const int r = __builtin_ctzll(m);
                if (slot != __builtin_amdgcn_readlane(step_slot, r) % kTile) continue;
                a = load_new4(p.v_new, ((size_t)r * p.hkv + hk) * D + 8 * vc, p.append_src);
                b = load_new4(p.v_new, ((size_t)r * p.hkv + hk) * D + 8 * vc + 4, p.append_src);
            }
            float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
            if (tail && slot >= lim) {
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = 0.f;
            }
            float pv[GW];
#pragma unroll
            for (int h = 0; h < GW; ++h) pv[h] = p_lds[wave][buf][slot][h];
#pragma unroll
            for (int h = 0; h < GW; ++h) {
                l_run[h] += pv[h];
#pragma unroll
                for (int e = 0; e < 8; ++e) acc[h][e] = fmaf(pv[h], x[e], acc[h][e]);
            }
        }
        buf ^= 1;
    }

    // ---- reduce the token groups of the V layout (lanes with equal chunk) ----
#pragma unroll
    for (int h = 0; h < GW; ++h) {
#pragma unroll
        for (int off = VLPT; off < 64; off <<= 1) {
            l_run[h] += __shfl_xor(l_run[h], off);
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[h][e] += __shfl_xor(acc[h][e], off);
        }
    }
    if (lane < VLPT) {
#pragma unroll
        for (int h = 0; h < GW; ++h) {
#pragma unroll
            for (int e = 0; e < 8; ++e) comb[wave][h][2 + 8 * vc + e] = acc[h][e];
            if (vc == 0) {
                comb[wave][h][0] = m_run[h];  // (-inf: a wave without tokens)
                comb[wave][h][1] = l_run[h];
            }
        }
    }
    __syncthreads();
    finish_item<D, GW>(p, comb, c, part_slot, hi - lo == c.U);
}

template <int D, int GW, bool STEP>
void launch_decode(const DecodeParams& p, dim3 grid, hipStream_t s) {
    if (p.gsplit == 1) hipLaunchKernelGGL((decode_f32<D, GW, true, STEP>), grid, dim3(kWaves * 64), 0, s, p);
    else hipLaunchKernelGGL((decode_f32<D, GW, false, STEP>), grid, dim3(kWaves * 64), 0, s, p);
}

template <int D, int GW>
void launch(const DecodeParams& p, dim3 grid, hipStream_t s) {
    if (p.k_new) launch_decode<D, GW, true>(p, grid, s);
    else launch_decode<D, GW, false>(p, grid, s);
    if (p.item_parts > 1) {
        hipLaunchKernelGGL((decode_merge_items<D, GW>), dim3(p.hkv * p.gsplit, p.batch), dim3(256), 0, s, p);
    }
}

template <int D>
int launch_gw(uint32_t gw, const DecodeParams& p, dim3 grid, hipStream_t s) {
    switch (gw) {
        case 1: launch<D, 1>(p, grid, s); return 1;
        case 2: launch<D, 2>(p, grid, s); return 1;
        case 3: launch<D, 3>(p, grid, s); return 1;
        case 4: launch<D, 4>(p, grid, s); return 1;
        default: return 0;
    }
}

}  // namespace

int launch_decode_f32(const DecodeParams& p, uint32_t head_dim, uint32_t gw, dim3 grid, hipStream_t stream) {
    if (head_dim == 64) return launch_gw<64>(gw, p, grid, stream);
    if (head_dim == 128) return launch_gw<128>(gw, p, grid, stream);
    return 0;
}

}  // namespace vkv
