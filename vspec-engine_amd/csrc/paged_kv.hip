// paged_kv.hip -- gfx950 kernels and C-ABI for the Vspec paged KV-cache decode path.
//
// Kernels (all wave64):
//   kv_append_rows   block-table append of new K/V to f16 and f32 pools, with rotary k and q
//   kv_append        the same to int4 pools, which quantise on write
//   rope_q_rows, rope_q   the query rows of appends that do not carry them
//   kv_gather_quads, kv_gather   block-table gather into [T][H][D] (raw bytes or dequantised f32)
//   kv_gather_rows   single tokens by page and slot
//   kv_compact       whole-block moves (compaction after eviction)
// and the plan of a decode, whose kernels are in decode_f32.hip, decode_mfma.hip and
// decode_mfma_int4.hip.
//
// The C-ABI is declared in include/vspec_rocm.h.
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <mutex>
#include <vector>

#include "vspec_rocm_paged.h"

// ---------------------------------------------------------------------------
// error reporting
// ---------------------------------------------------------------------------
namespace {
thread_local char g_err[512] = "";

void set_err(const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
}
}  // namespace

extern "C" void vspec_rocm_set_error_(const char* msg) { set_err("%s", msg ? msg : ""); }

#define HIP_CHECK(call, what)                                              \
    do {                                                                   \
        hipError_t e_ = (call);                                            \
        if (e_ != hipSuccess) {                                            \
            set_err("%s: %s", (what), hipGetErrorString(e_));              \
            return 0;                                                      \
        }                                                                  \
    } while (0)

#include "kv_common.h"
#include "append_row.h"

namespace {
using namespace vkv;

// Per-dtype geometry of one row (one token of one kv head).
template <int DT, int D>
struct Row {
    static constexpr int kBytes = DT == VSPEC_KV_F32 ? D * 4 : (DT == VSPEC_KV_F16 ? D * 2 : D / 2);
    static constexpr int kScales = DT == VSPEC_KV_INT4 ? D / 32 : 0;
};

// ---------------------------------------------------------------------------
// append (quantise-on-write for int4)
// ---------------------------------------------------------------------------
// One work item = EPT consecutive elements of one token-head row of K or V: a whole
// 32-element quantisation group for int4 pools, 8 elements (16 or 32 bytes) otherwise.
// int4 is bound by its vector instructions: 8 x 512 tokens (32/8 heads of 128) 10.4 us, 12.6 with
// a full division, rounding and clip per element (int4_nibble).  f16 and f32 pools come here only
// where a launch has more items than kv_append_rows counts in 32 bits.
template <int DT, int SRC, bool ROPE>
__global__ __launch_bounds__(256) void kv_append(AppendParams p) {
    const uint64_t total = append_items<DT>(p);
    for (uint64_t it = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; it < total;
         it += (uint64_t)gridDim.x * blockDim.x) {
        append_item<DT, SRC, ROPE>(p, it);
    }
}

// f16 and f32 pools: the K, V and query sections of append_row.h, 256 items a workgroup.
// Bound by memory: a 4096-token f16 chunk with rotary q and k (32/8 heads of 128) moves
// 170 MB, in 36 us (4.7 TB/s, the rate of a large copy).  One item per lane keeps whole rows
// coalesced (16 lanes a row), sections instead of K and V in alternate lanes keep a wave on
// one path, V goes out in whole 4-token groups, and the rotary tables and partners are read
// 16 bytes at a time, the tables once for 4 query heads.  Before (V in 2-byte pieces, tables
// and partners element by element, q rotated one element a lane by a second launch): 114 us.
template <int DT, int SRC, bool ROPE>
__global__ __launch_bounds__(256) void kv_append_rows(AppendParams p, uint32_t k_wgs, uint32_t v_wgs, uint32_t k_items,
                                                      uint32_t v_items, uint32_t q_items) {
    const uint32_t wg = blockIdx.x;
    if (wg < k_wgs) {
        const uint32_t it = wg * 256 + threadIdx.x;
        if (it < k_items) append_k_item<DT, SRC, ROPE>(p, it);
    } else if (wg < k_wgs + v_wgs) {
        const uint32_t it = (wg - k_wgs) * 256 + threadIdx.x;
        if (it < v_items) append_v_item<DT, SRC, ROPE>(p, it);
    } else {
        const uint32_t it = (wg - k_wgs - v_wgs) * 256 + threadIdx.x;
        if (it < q_items) rope_q_item(p, it);
    }
}

// The query section alone (int4 pools, whose K and V items are whole quantisation groups).
__global__ __launch_bounds__(256) void rope_q_rows(AppendParams p, uint32_t q_items) {
    const uint32_t it = blockIdx.x * 256 + threadIdx.x;
    if (it < q_items) rope_q_item(p, it);
}

// Rotary embedding of the query rows of the appended tokens: q [B][n_new][Hq][D] fp32,
// token (b, i) at position start_pos[b] + i; tokens without a table row are not written.
struct RopeQParams {
    const float* q_in;
    float* q_out;
    const int32_t* start_pos;
    const float* rope_cos;
    const float* rope_sin;
    uint32_t batch, n_new, hq, head_dim, rope_dim, max_pos;
};

__global__ __launch_bounds__(256) void rope_q(RopeQParams p) {
    const uint64_t total = (uint64_t)p.batch * p.n_new * p.hq * p.head_dim;
    for (uint64_t it = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; it < total;
         it += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t d = (uint32_t)(it % p.head_dim);
        const uint64_t row = it / p.head_dim;  // ((b * n_new + i) * hq + h)
        const uint32_t i = (uint32_t)((row / p.hq) % p.n_new);
        const uint32_t b = (uint32_t)(row / ((uint64_t)p.hq * p.n_new));
        const int32_t sp = p.start_pos[b];
        if (sp < 0) continue;
        const uint32_t pos = (uint32_t)sp + i;
        if (pos >= p.max_pos) continue;
        const float* x = p.q_in + row * p.head_dim;
        float y = x[d];
        if (d < p.rope_dim) {
#pragma clang fp contract(off)
            const uint32_t half = p.rope_dim / 2;
            const uint32_t k = d < half ? d : d - half;
            const float c = p.rope_cos[(size_t)pos * half + k], sn = p.rope_sin[(size_t)pos * half + k];
            y = d < half ? x[d] * c - x[d + half] * sn : x[d - half] * sn + x[d] * c;
        }
        p.q_out[row * p.head_dim + d] = y;
    }
}

// ---------------------------------------------------------------------------
// gather / compaction
// ---------------------------------------------------------------------------
struct GatherParams {
    const uint8_t* k;
    const uint8_t* v;
    const uint16_t* ks;
    const uint16_t* vs;
    const int32_t* block_tables;
    const int32_t* ctx_lens;
    const int64_t* out_off;
    uint8_t* ok;
    uint8_t* ov;
    uint16_t* oks;
    uint16_t* ovs;
    uint32_t hkv;
    uint32_t head_dim;
    uint32_t block_tokens;
    uint32_t max_blocks;
    uint32_t num_blocks;
    uint32_t max_ctx;
};

// Raw gather: one thread per 16-byte chunk of a row (int4: 4-byte chunks plus
// the row's scales).  Dequantising gather (OUTF32): one thread per 8 elements.
template <int DT, int OUTF32>
__global__ __launch_bounds__(256) void kv_gather(GatherParams p) {
    const int b = blockIdx.y;
    const int ctx = p.ctx_lens[b];
    const uint32_t D = p.head_dim;
    const uint32_t row_bytes = DT == VSPEC_KV_F32 ? D * 4 : (DT == VSPEC_KV_F16 ? D * 2 : D / 2);
    const uint32_t cpr = OUTF32 ? D / 8 : (DT == VSPEC_KV_INT4 ? row_bytes / 4 : row_bytes / 16);
    const uint64_t total = (uint64_t)p.max_ctx * p.hkv * cpr * 2;
    for (uint64_t it = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; it < total;
         it += (uint64_t)gridDim.x * blockDim.x) {
        const int which = (int)(it & 1);
        uint64_t r = it >> 1;
        const uint32_t c = (uint32_t)(r % cpr);
        r /= cpr;
        const uint32_t h = (uint32_t)(r % p.hkv);
        const uint32_t t = (uint32_t)(r / p.hkv);
        if ((int)t >= ctx) continue;
        const uint32_t lb = t / p.block_tokens;
        if (lb >= p.max_blocks) continue;
        const int32_t phys = p.block_tables[(size_t)b * p.max_blocks + lb];
        if (phys < 0 || (uint32_t)phys >= p.num_blocks) continue;
        const size_t row = ((size_t)phys * p.hkv + h) * p.block_tokens + t % p.block_tokens;
        const size_t orow = ((size_t)p.out_off[b] + t) * p.hkv + h;
        const uint8_t* src = which ? p.v : p.k;
        uint8_t* dst = which ? p.ov : p.ok;
        if (DT == VSPEC_KV_F16 && which) {
            // V in 4-token groups: 8 elements of row `slot`, stride 4
            const uint16_t* vt = reinterpret_cast<const uint16_t*>(src) +
                                 f16_v_index((size_t)phys * p.hkv + h, p.block_tokens, D, t % p.block_tokens, 8 * c);
            uint16_t e16[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) e16[i] = vt[4 * i];
            if (OUTF32) {
                float4* d = reinterpret_cast<float4*>(dst + orow * (size_t)D * 4) + 2 * c;
                d[0] = make_float4(half_bits_to_float(e16[0]), half_bits_to_float(e16[1]),
                                   half_bits_to_float(e16[2]), half_bits_to_float(e16[3]));
                d[1] = make_float4(half_bits_to_float(e16[4]), half_bits_to_float(e16[5]),
                                   half_bits_to_float(e16[6]), half_bits_to_float(e16[7]));
            } else {
                reinterpret_cast<uint4*>(dst + orow * row_bytes)[c] =
                    make_uint4(e16[0] | ((uint32_t)e16[1] << 16), e16[2] | ((uint32_t)e16[3] << 16),
                               e16[4] | ((uint32_t)e16[5] << 16), e16[6] | ((uint32_t)e16[7] << 16));
            }
            continue;
        }
        if constexpr (OUTF32) {
            float x[8];
            if constexpr (DT == VSPEC_KV_F32) {
                const float4* s = reinterpret_cast<const float4*>(src + row * row_bytes) + 2 * c;
                const float4 a = s[0], bb = s[1];
                x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
                x[4] = bb.x; x[5] = bb.y; x[6] = bb.z; x[7] = bb.w;
            } else if constexpr (DT == VSPEC_KV_F16) {
                unpack_f16x8(reinterpret_cast<const uint4*>(src + row * row_bytes)[c], x);
            } else {
                const size_t bh = (size_t)phys * p.hkv + h;
                const uint32_t slot = t % p.block_tokens;
                const uint32_t w = which ? int4_v_canonical_dword(src, bh, p.block_tokens, D, slot, c)
                                         : reinterpret_cast<const uint32_t*>(src + row * row_bytes)[c];
                const float s = half_bits_to_float(
                    which ? p.vs[row * (D / 32) + c / 4] : p.ks[int4_ks_index(bh, D / 32, p.block_tokens, slot, c / 4)]);
#pragma unroll
                for (int i = 0; i < 8; ++i) x[i] = nibble(w, i) * s;
            }
            float4* d = reinterpret_cast<float4*>(dst + orow * (size_t)D * 4) + 2 * c;
            d[0] = make_float4(x[0], x[1], x[2], x[3]);
            d[1] = make_float4(x[4], x[5], x[6], x[7]);
        } else if constexpr (DT == VSPEC_KV_INT4) {
            // output rows are canonical packed codes whatever the pool layout
            const size_t bh = (size_t)phys * p.hkv + h;
            const uint32_t slot = t % p.block_tokens;
            reinterpret_cast<uint32_t*>(dst + orow * row_bytes)[c] =
                which ? int4_v_canonical_dword(src, bh, p.block_tokens, D, slot, c)
                      : reinterpret_cast<const uint32_t*>(src + row * row_bytes)[c];
            if (c < D / 32) {
                uint16_t* od = which ? p.ovs : p.oks;
                od[orow * (D / 32) + c] =
                    which ? p.vs[row * (D / 32) + c] : p.ks[int4_ks_index(bh, D / 32, p.block_tokens, slot, c)];
            }
        } else {
            reinterpret_cast<uint4*>(dst + orow * row_bytes)[c] =
                reinterpret_cast<const uint4*>(src + row * row_bytes)[c];
        }
    }
}

// 16 bytes that this launch does not read again
__device__ __forceinline__ void store_stream4f(void* p, float a, float b, float c, float d) {
    typedef float nt_f32x4 __attribute__((ext_vector_type(4)));
    const nt_f32x4 v = {a, b, c, d};
    __builtin_nontemporal_store(v, reinterpret_cast<nt_f32x4*>(p));
}

// f16 and int4 pools (int4: D = 64 or 128): K (blockIdx.z 0) or V (1) of 4 consecutive tokens
// of one head per lane, the unit in which both pools hold V.  Bound by memory.  f16: a lane
// takes E elements of each token, so that every store of a wave covers whole rows (f32 out: 4
// elements, 16 bytes; raw: 8).  int4 V: lane n of 16 takes the tile chunk that holds d = n,
// 16 + n, ... of the 4 tokens.  Against the row kernel, whose V elements are 2-byte (f16) or
// byte (int4) loads: 8 sequences of 1k-8k tokens, 32/8 heads of 128: f16 to f32 174 -> 81 us
// (5.7 TB/s; 85.5 with ordinary stores); 8 sequences of 0.5k-4k: f16 raw 66 -> 31, int4 raw
// 37 -> 10.5, int4 to f32 69 -> 42 us; 24 short sequences (12-640 tokens) 7.6 us either way.
template <int DT, int OUTF32, int D>
__global__ __launch_bounds__(256) void kv_gather_quads(GatherParams p) {
    const int b = blockIdx.y;
    const uint32_t head_dim = D ? (uint32_t)D : p.head_dim;
    const uint32_t tokens = min((uint32_t)max(p.ctx_lens[b], 0), p.max_ctx);
    constexpr int E = OUTF32 ? 4 : 8;
    const uint32_t lanes = DT == VSPEC_KV_F16 ? head_dim / E : 16u;  // lanes of a quad of one head
    const uint32_t it = blockIdx.x * 256 + threadIdx.x;  // the host keeps this below 2^31
    const uint32_t c = it % lanes, r = it / lanes;
    const uint32_t h = r % p.hkv, quad = r / p.hkv;
    // lanes that have nothing to copy stay for the wave's exchange through LDS below
    bool on = quad < (tokens + 3) / 4;
    const uint32_t t0 = on ? 4 * quad : 0u;
    const uint32_t lb = t0 / p.block_tokens;
    on = on && lb < p.max_blocks;
    const int32_t phys = on ? p.block_tables[(size_t)b * p.max_blocks + lb] : -1;
    on = on && phys >= 0 && (uint32_t)phys < p.num_blocks;
    const uint32_t slot = t0 % p.block_tokens;
    const size_t bh = (size_t)(on ? phys : 0) * p.hkv + h;
    const size_t row = bh * p.block_tokens + slot;
    const size_t orow = ((size_t)p.out_off[b] + t0) * p.hkv + h;  // token j: + j * hkv
    const uint32_t n = on ? min(4u, tokens - t0) : 0u;
    const bool v = blockIdx.z != 0;
    if constexpr (DT == VSPEC_KV_F16) {
        if (!on) return;
        uint32_t w[4][E / 2];  // token, pair of elements
        if (v) {
            const uint16_t* src = reinterpret_cast<const uint16_t*>(p.v) + f16_v_index(bh, p.block_tokens, head_dim, slot, E * c);
#pragma unroll
            for (int e = 0; e < E / 2; ++e) {  // tokens 0..3 of elements 2e and 2e + 1
                const uint4 x = load_stream4(src + 8 * e);
                w[0][e] = (x.x & 0xffffu) | (x.z << 16);
                w[1][e] = (x.x >> 16) | (x.z & 0xffff0000u);
                w[2][e] = (x.y & 0xffffu) | (x.w << 16);
                w[3][e] = (x.y >> 16) | (x.w & 0xffff0000u);
            }
        } else {
            const uint16_t* src = reinterpret_cast<const uint16_t*>(p.k) + row * head_dim + E * c;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if constexpr (E == 4) {
                    const uint2 x = load_stream2(src + (size_t)j * head_dim);
                    w[j][0] = x.x; w[j][1] = x.y;
                } else {
                    const uint4 x = load_stream4(src + (size_t)j * head_dim);
                    w[j][0] = x.x; w[j][1] = x.y; w[j][2] = x.z; w[j][3] = x.w;
                }
            }
        }
        uint8_t* dst = v ? p.ov : p.ok;
        const size_t stride = (size_t)p.hkv * head_dim * (OUTF32 ? 4 : 2);
        uint8_t* o = dst + orow * head_dim * (OUTF32 ? 4 : 2) + 16 * c;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (j >= (int)n) break;
            if constexpr (OUTF32) {
                store_stream4f(o + j * stride, half_bits_to_float(w[j][0] & 0xffffu), half_bits_to_float(w[j][0] >> 16),
                               half_bits_to_float(w[j][1] & 0xffffu), half_bits_to_float(w[j][1] >> 16));
            } else {
                *reinterpret_cast<uint4*>(o + j * stride) = make_uint4(w[j][0], w[j][1], w[j][2], w[j][3]);
            }
        }
    } else {
        constexpr int G = D ? D / 32 : 1;  // groups of a row, dwords of a lane's chunk
        if constexpr (OUTF32) {
            if (!on) return;
            if (v) {
                // the 4 tokens' scales are one run; byte 2 * (j & 1) + (j >> 1) of dword q is
                // token j's d = 32q + c (low nibble) and 32q + 16 + c (high)
                uint32_t w[G];
                const uint32_t* src = reinterpret_cast<const uint32_t*>(p.v + bh * ((size_t)p.block_tokens * D / 2) +
                                                                        (size_t)(slot >> 4) * (8u * D)) + (4 * (slot & 15) + c) * G;
#pragma unroll
                for (int q = 0; q < G; ++q) w[q] = src[q];
                float* o = reinterpret_cast<float*>(p.ov) + orow * D + c;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (j >= (int)n) break;
#pragma unroll
                    for (int q = 0; q < G; ++q) {
                        const float s = half_bits_to_float(p.vs[(row + j) * G + q]);
                        const int byte = 2 * (j & 1) + (j >> 1);
                        o[(size_t)j * p.hkv * D + 32 * q] = nibble(w[q], 2 * byte) * s;
                        o[(size_t)j * p.hkv * D + 32 * q + 16] = nibble(w[q], 2 * byte + 1) * s;
                    }
                }
            } else {
                // lane c: elements 4c .. 4c + 3 (and 64 + 4c .. of a 128-element row)
                const uint16_t* src = reinterpret_cast<const uint16_t*>(p.k + row * (D / 2));
                float* o = reinterpret_cast<float*>(p.ok) + orow * D + 4 * c;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (j >= (int)n) break;
#pragma unroll
                    for (int q = 0; q < D / 64; ++q) {
                        const uint32_t w = src[(size_t)j * (D / 4) + 16 * q + c];
                        const float s = half_bits_to_float(p.ks[int4_ks_index(bh, G, p.block_tokens, slot + j, 2 * q + c / 8)]);
                        *reinterpret_cast<float4*>(o + (size_t)j * p.hkv * D + 64 * q) =
                            make_float4(nibble(w, 0) * s, nibble(w, 1) * s, nibble(w, 2) * s, nibble(w, 3) * s);
                    }
                }
            }
        } else {
            // canonical packed codes: lane c of a quad writes group c % G of token c / G (D = 64:
            // lanes 8..15 idle), 16 bytes
            const uint32_t j = c / G, q = c % G;
            const bool mine = on && c < 4 * G && j < n;
            uint4 out = make_uint4(0u, 0u, 0u, 0u);
            if (v) {
                // the quad's 16 chunks through LDS (a wave's own accesses, in program order),
                // then the 16 bytes of (token, group): low nibbles d = 32q + i, high ones + 16
                __shared__ uint32_t tile[256 / 16][16][G];
                uint32_t(*mine_tile)[G] = tile[threadIdx.x / 16];
                if (on) {
                    const uint32_t* src = reinterpret_cast<const uint32_t*>(p.v + bh * ((size_t)p.block_tokens * D / 2) +
                                                                            (size_t)(slot >> 4) * (8u * D)) + (4 * (slot & 15) + c) * G;
#pragma unroll
                    for (int i = 0; i < G; ++i) mine_tile[c][i] = src[i];
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                const uint32_t byte = 2 * (j & 1) + (j >> 1);
                uint32_t lo[2] = {0u, 0u}, hi[2] = {0u, 0u};
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const uint32_t x = reinterpret_cast<const uint8_t*>(&mine_tile[i][q])[byte & 3];
                    lo[i / 8] |= (x & 0xfu) << (4 * (i % 8));
                    hi[i / 8] |= (x >> 4) << (4 * (i % 8));
                }
                out = make_uint4(lo[0], lo[1], hi[0], hi[1]);
            } else if (mine) {
                out = *reinterpret_cast<const uint4*>(p.k + (row + j) * (D / 2) + 16 * q);
            }
            if (mine) {
                const size_t o = orow + (size_t)j * p.hkv;
                *reinterpret_cast<uint4*>((v ? p.ov : p.ok) + o * (D / 2) + 16 * q) = out;
                (v ? p.ovs : p.oks)[o * G + q] =
                    v ? p.vs[(row + j) * G + q] : p.ks[int4_ks_index(bh, G, p.block_tokens, slot + j, q)];
            }
        }
    }
}

struct GatherRowsParams {
    const uint8_t* k;
    const uint8_t* v;
    const uint16_t* ks;
    const uint16_t* vs;
    const int32_t* pages;
    const int32_t* slots;
    float* ok;
    float* ov;
    uint32_t n;
    uint32_t hkv;
    uint32_t head_dim;
    uint32_t block_tokens;
    uint32_t num_blocks;
};

// Row-list gather to f32: output token i is (pages[i], slots[i]) of every head, [n][H][D].
// One thread per 8 elements of one row of K or V.
template <int DT>
__global__ __launch_bounds__(256) void kv_gather_rows(GatherRowsParams p) {
    const uint32_t D = p.head_dim, P = p.block_tokens;
    const uint32_t cpr = D / 8;
    const uint64_t total = (uint64_t)p.n * p.hkv * cpr * 2;
    for (uint64_t it = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; it < total;
         it += (uint64_t)gridDim.x * blockDim.x) {
        const int which = (int)(it & 1);
        uint64_t r = it >> 1;
        const uint32_t c = (uint32_t)(r % cpr);
        r /= cpr;
        const uint32_t h = (uint32_t)(r % p.hkv);
        const uint32_t i = (uint32_t)(r / p.hkv);
        const int32_t page = p.pages[i], slot = p.slots[i];
        if (page < 0 || (uint32_t)page >= p.num_blocks || slot < 0 || (uint32_t)slot >= P) continue;
        const size_t tile = (size_t)page * p.hkv + h;
        const size_t row = tile * P + slot;
        const uint8_t* src = which ? p.v : p.k;
        float x[8];
        if constexpr (DT == VSPEC_KV_F32) {
            const float4* s4 = reinterpret_cast<const float4*>(src + row * D * 4) + 2 * c;
            const float4 a = s4[0], bb = s4[1];
            x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
            x[4] = bb.x; x[5] = bb.y; x[6] = bb.z; x[7] = bb.w;
        } else if constexpr (DT == VSPEC_KV_F16) {
            if (which) {
                const uint16_t* vt = reinterpret_cast<const uint16_t*>(src) + f16_v_index(tile, P, D, slot, 8 * c);
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = half_bits_to_float(vt[4 * e]);
            } else {
                unpack_f16x8(reinterpret_cast<const uint4*>(src + row * D * 2)[c], x);
            }
        } else {
            const uint32_t w = which ? int4_v_canonical_dword(src, tile, P, D, slot, c)
                                     : reinterpret_cast<const uint32_t*>(src + row * (D / 2))[c];
            const float sc = half_bits_to_float(which ? p.vs[row * (D / 32) + c / 4]
                                                      : p.ks[int4_ks_index(tile, D / 32, P, slot, c / 4)]);
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = nibble(w, e) * sc;
        }
        float4* d = reinterpret_cast<float4*>((which ? p.ov : p.ok) + ((size_t)i * p.hkv + h) * D) + 2 * c;
        d[0] = make_float4(x[0], x[1], x[2], x[3]);
        d[1] = make_float4(x[4], x[5], x[6], x[7]);
    }
}

struct CompactParams {
    uint8_t* k;
    uint8_t* v;
    uint16_t* ks;
    uint16_t* vs;
    uint32_t* kf;            // int4 clamp flags or null
    uint32_t block_flags;    // flag words per physical block
    const int32_t* src;
    const int32_t* dst;
    uint32_t n;
    uint32_t num_blocks;
    uint64_t block_bytes;    // data bytes per physical block (all heads), multiple of 16
    uint64_t block_scales;   // scale entries per physical block (int4)
};

__global__ __launch_bounds__(256) void kv_compact(CompactParams p) {
    const uint32_t i = blockIdx.y;
    const int32_t s = p.src[i], d = p.dst[i];
    if (s < 0 || d < 0 || (uint32_t)s >= p.num_blocks || (uint32_t)d >= p.num_blocks) return;
    const uint64_t n16 = p.block_bytes / 16;
    for (uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; j < 2 * n16;
         j += (uint64_t)gridDim.x * blockDim.x) {
        uint8_t* base = j < n16 ? p.k : p.v;
        const uint64_t jj = j < n16 ? j : j - n16;
        // each byte moves once: streaming (non-temporal) load and store
        const uint4 w = load_stream4(reinterpret_cast<const uint4*>(base + (uint64_t)s * p.block_bytes) + jj);
        nt_u32x4 wv = {w.x, w.y, w.z, w.w};
        __builtin_nontemporal_store(wv, reinterpret_cast<nt_u32x4*>(base + (uint64_t)d * p.block_bytes) + jj);
    }
    if (p.block_scales) {
        for (uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; j < 2 * p.block_scales;
             j += (uint64_t)gridDim.x * blockDim.x) {
            uint16_t* base = j < p.block_scales ? p.ks : p.vs;
            const uint64_t jj = j < p.block_scales ? j : j - p.block_scales;
            base[(uint64_t)d * p.block_scales + jj] = base[(uint64_t)s * p.block_scales + jj];
        }
    }
    if (p.kf) {
        for (uint32_t j = blockIdx.x * blockDim.x + threadIdx.x; j < p.block_flags; j += gridDim.x * blockDim.x)
            p.kf[(uint64_t)d * p.block_flags + j] = p.kf[(uint64_t)s * p.block_flags + j];
    }
}

// ---------------------------------------------------------------------------
// host helpers
// ---------------------------------------------------------------------------
int g_num_cus = 0;

int num_cus() {
    if (g_num_cus > 0) return g_num_cus;
    int dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess &&
        prop.multiProcessorCount > 0) {
        g_num_cus = prop.multiProcessorCount;
    } else {
        g_num_cus = 256;
    }
    return g_num_cus;
}

size_t row_bytes_of(int32_t dtype, uint32_t d) {
    return dtype == VSPEC_KV_F32 ? (size_t)d * 4 : (dtype == VSPEC_KV_F16 ? (size_t)d * 2 : d / 2);
}

// Geometry every kernel accepts; `decode` adds the attention kernels' limits
// (head_dim 64 or 128, block_tokens a multiple of the 16-token tile).
int check_kv(const VspecPagedKV* kv, const char* who, bool decode = false) {
    if (!kv) {
        set_err("%s: null pool", who);
        return 0;
    }
    if (kv->dtype < VSPEC_KV_F32 || kv->dtype > VSPEC_KV_INT4) {
        set_err("%s: bad dtype %d", who, (int)kv->dtype);
        return 0;
    }
    if (kv->num_blocks == 0 || kv->num_kv_heads == 0 || kv->block_tokens == 0 || kv->head_dim == 0) {
        set_err("%s: empty pool geometry", who);
        return 0;
    }
    // block-table entries are int32, and the kernels index (block, kv head) pairs in 32 bits
    if (kv->num_blocks > 0x7fffffffu || (uint64_t)kv->num_blocks * kv->num_kv_heads > 0xffffffffull) {
        set_err("%s: num_blocks must fit int32 and num_blocks x num_kv_heads 32 bits", who);
        return 0;
    }
    const uint32_t quantum = kv->dtype == VSPEC_KV_INT4 ? 32u : 8u;
    if (kv->head_dim % quantum != 0) {
        set_err("%s: head_dim must be a multiple of %u", who, quantum);
        return 0;
    }
    // int4 and f16 pools keep tiles of 16 tokens (f16 V: groups of 4 tokens, f16_v_index)
    if (kv->dtype != VSPEC_KV_F32 && kv->block_tokens % kTile != 0) {
        set_err("%s: %s pools need block_tokens a multiple of %d", who, kv->dtype == VSPEC_KV_INT4 ? "int4" : "f16",
                kTile);
        return 0;
    }
    if (decode && kv->block_tokens % kTile != 0) {
        set_err("%s: block_tokens must be a positive multiple of %d", who, kTile);
        return 0;
    }
    if (decode && kv->head_dim != 64 && kv->head_dim != 128) {
        set_err("%s: head_dim must be 64 or 128", who);
        return 0;
    }
    if (!kv->k_data || !kv->v_data) {
        set_err("%s: null pool data", who);
        return 0;
    }
    if (kv->dtype == VSPEC_KV_INT4 && (!kv->k_scales || !kv->v_scales)) {
        set_err("%s: int4 pool without scales", who);
        return 0;
    }
    // the int4 decode builds buffer descriptors whose base field holds address bits 0..47
    // (device addresses of user allocations lie below 2^47)
    const uintptr_t hi = ((uintptr_t)kv->k_data | (uintptr_t)kv->v_data | (uintptr_t)kv->k_scales |
                          (uintptr_t)kv->v_scales | (uintptr_t)kv->k_flags) >> 47;
    if (hi != 0) {
        set_err("%s: pool address at or above 2^47", who);
        return 0;
    }
    return 1;
}

// Grow-only library workspace per device (used when the caller passes none); the mutex
// keeps host threads that decode on one device from growing it at the same time (its
// contents are shared: concurrent decodes need workspaces of their own).  A buffer that
// is outgrown is retired, not freed: a HIP graph captured from an earlier decode still
// holds its address, and replays must find it allocated.  Retired buffers are freed by
// vspec_rocm_release_retired_workspaces() or at process exit.
struct Workspace {
    void* ptr = nullptr;
    size_t bytes = 0;
};
Workspace g_ws[64];
std::vector<void*> g_retired[64];
std::mutex g_ws_mu;

void* library_workspace(size_t bytes) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return nullptr;
    std::lock_guard<std::mutex> lock(g_ws_mu);
    Workspace& w = g_ws[dev];
    if (w.bytes >= bytes) return w.ptr;
    void* fresh = nullptr;
    if (hipMalloc(&fresh, bytes) != hipSuccess) return nullptr;
    if (w.ptr) g_retired[dev].push_back(w.ptr);
    w.ptr = fresh;
    w.bytes = bytes;
    return w.ptr;
}

// ---- the no-allocation decode step's device scratch ----
// Partial states of vspec_rocm_paged_decode_step_noalloc live in this file-scope array,
// one copy per device for the life of the process.  Host code never uses its name as an
// address: the per-device address comes from hipGetSymbolAddress on the entry point's
// first call on that device.
constexpr size_t kScratchBytes = (size_t)6 << 20;  // partial (max, sum, acc) slots
static __device__ __align__(256) uint8_t scratch[kScratchBytes];
void* g_scratch_ptr[64];
bool g_scratch_ready[64];

uint8_t* scratch_address(int dev) {
    std::lock_guard<std::mutex> lock(g_ws_mu);
    if (!g_scratch_ready[dev]) {
        void* ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) {
            set_err("paged_decode_step_noalloc: hipGetSymbolAddress(scratch) failed: %s", hipGetErrorString(e));
            return nullptr;
        }
        g_scratch_ptr[dev] = ptr;
        g_scratch_ready[dev] = true;
    }
    return (uint8_t*)g_scratch_ptr[dev];
}

constexpr uint32_t kDefaultOldPermille = 700;
constexpr uint32_t kDefaultOldPermilleInt4 = 500;

// workgroups per CU of the balanced MFMA split: VSPEC_ROCM_DECODE_WGS_PER_CU (1..8) when
// set, else 0 (the plan decides)
uint32_t decode_wgs_per_cu_env() {
    static const uint32_t v = [] {
        const char* e = getenv("VSPEC_ROCM_DECODE_WGS_PER_CU");
        const long x = e ? strtol(e, nullptr, 10) : 0;
        return x >= 1 && x <= 8 ? (uint32_t)x : 0u;
    }();
    return v;
}

// Share of the first-half workgroup of each pair sharing a CU under the balanced split,
// in 1/1000 (VSPEC_ROCM_DECODE_OLD_PERMILLE for f16 pools, ..._INT4 for int4 pools,
// 500..900).  Read on every call.  int4 keeps equal shares by default: measured per
// workgroup at the north-star shape, the first-half workgroups end at ~65 us and their
// partners at ~86 us (the CU's wave arbiter favours the older waves), yet unequal shares
// are slower there (80.6 us at 500, 88.3 at 600, 98.7 at 700: work items then span two
// workgroups, and each extra item costs its set-up and a merge launch; with the current
// kernel 74.8 us at 500, 84.1 / 83.0 / 81.9 at 530 / 560 / 600, and equal at 16k tokens).
uint32_t decode_old_permille(uint32_t dtype) {
    const bool i4 = dtype == VSPEC_KV_INT4;
    const char* e = getenv(i4 ? "VSPEC_ROCM_DECODE_OLD_PERMILLE_INT4" : "VSPEC_ROCM_DECODE_OLD_PERMILLE");
    const long x = e ? strtol(e, nullptr, 10) : 0;
    return x >= 500 && x <= 900 ? (uint32_t)x : i4 ? kDefaultOldPermilleInt4 : kDefaultOldPermille;
}

// Least tiles per workgroup of the balanced split: VSPEC_ROCM_DECODE_MIN_TILES_PER_WG
// (1..256) when set, else 16 for batches of at most 8 work items and 1 otherwise.  With
// 8 work items (one sequence, 8 kv heads) and a grid of 2 workgroups per CU, a 1k-4k
// context leaves 1-4 tiles per workgroup and 64 partials per work item for its last
// workgroup to merge (eight rounds of loads); 16 tiles per workgroup cut the int4 step at
// B=1 from 30 to 21 us and the f16 one from 23 to 21 us.  At 16 work items the same floor
// loses (f16 at 1k: 21 -> 26 us), and from 16k tokens on it makes no difference.  Read
// on every call.
uint32_t decode_min_tiles_per_wg(uint64_t items) {
    const char* e = getenv("VSPEC_ROCM_DECODE_MIN_TILES_PER_WG");
    const long x = e ? strtol(e, nullptr, 10) : 0;
    if (x >= 1 && x <= 256) return (uint32_t)x;
    return items <= 8 ? 16u : 1u;
}

// An explicitly set knob of the balanced split (the functions around here) selects it.
bool balanced_split_env() {
    for (const char* k : {"VSPEC_ROCM_DECODE_WGS_PER_CU", "VSPEC_ROCM_DECODE_OLD_PERMILLE", "VSPEC_ROCM_DECODE_OLD_PERMILLE_INT4",
                          "VSPEC_ROCM_DECODE_MIN_TILES_PER_WG", "VSPEC_ROCM_DECODE_SEGMENT_COST",
                          "VSPEC_ROCM_DECODE_SEGMENT_COST_INT4"}) {
        if (getenv(k)) return true;
    }
    return false;
}

// Parts of a work item under the item split (kv_common.h item_part), or 0 for the balanced
// split of all items' tiles.  Read on every call: VSPEC_ROCM_DECODE_ITEM_PARTS 0 never, 1..64
// that many (as far as the workspace holds them).
//
// Else the cheaper one by a cost model in us, fitted to both splits over 30 shapes (1-128
// sequences of 19-16k tokens): `slots` workgroups run at a time; with k of them running, a
// part of n tiles takes n * hypot(lat, k * bw), lat being a tile's share of one workgroup's
// dependent round trips and bw its share of the memory rate (f16) or of the issue rate
// (int4); a set-up `pro` is paid once, a merge launch with more than one part.  The balanced
// split pays more set-up (its pass over the contexts, several items per workgroup one after
// the other, a merge launch that redoes the split) and no last round of few workgroups.
// Measured, balanced -> item split, f16: 1 x 21 tokens 38.4 -> 7.4 us, 1 x 4097 22.1 -> 15.1,
// 16 x 2049 36.2 -> 27.8, 61 x 102 30.8 -> 11.7, 64 x 1025 50.4 -> 45.3, 64 x 4097 168.5 -> 166.1,
// 65 x 4097 187 -> 218 (not taken); int4: 1 x 4097 17.9 -> 15.1, 16 x 2049 22.2 -> 18.5, 64 x 1025
// 22.8 -> 21.8, 100 x 2000 68.1 -> 59.9, 65 x 4097 74 -> 89 (not taken).  A batch whose
// contexts may differ takes the item split only up to 72 tiles a part, since the launch ends
// with its longest part (64 sequences of 128-8192 tokens, 2 parts of up to 256 tiles: 162.5
// -> 183.8 us).  The parts never need more workspace than the balanced split's plan.
struct SplitCost {
    double lat, bw, pro, bal_tile, bal;
};
uint32_t plan_item_parts(const VspecPagedAttnDesc* d, uint64_t items, uint64_t tiles, uint64_t slots, uint64_t max_wgs,
                         bool same) {
    if (d->batch > 65535u || items / d->batch * 64 > 0x7fffffu) return 0;
    const uint64_t most = max_wgs / items > 1 ? max_wgs / items : 1;
    const char* e = getenv("VSPEC_ROCM_DECODE_ITEM_PARTS");
    if (e && *e) {
        const long x = strtol(e, nullptr, 10);
        return x <= 0 ? 0u : (uint32_t)((uint64_t)x < most ? (x < 64 ? x : 64) : (most < 64 ? most : 64));
    }
    if (balanced_split_env()) return 0;
    const bool i4 = d->kv.dtype == VSPEC_KV_INT4;
    const double size = d->kv.head_dim / 128.0;
    const SplitCost c = i4 ? SplitCost{0.15, 2.6e-4 * (1 + size) / 2, 7.0, 4.2e-4 * (1 + size) / 2, 19.0}
                           : SplitCost{0.215, 1.26e-3 * size, 6.5, 1.26e-3 * size, 22.0};
    const double busy = sqrt(c.lat * c.lat + (double)(slots * slots) * c.bw * c.bw);
    double best = (double)(items * tiles) * c.bal_tile * (same ? 1.0 : 0.75) + c.bal;
    uint32_t parts = 0;
    for (const uint32_t p : {1u, 2u, 3u, 4u, 6u, 8u, 12u, 16u, 24u, 32u, 48u, 64u}) {
        if (p > 1 && (p > most || (uint64_t)p * 4 > tiles + 3)) break;
        const uint64_t n = (tiles + p - 1) / p;
        if (!same && n > 72) continue;
        const double full = (double)(items * p / slots), rem = (double)(items * p % slots);
        const double t = (double)n * (full * busy + (rem > 0 ? sqrt(c.lat * c.lat + rem * rem * c.bw * c.bw) : 0.0)) + c.pro +
                         (p > 1 ? 5.0 + 0.12 * p : 0.0);
        if (t < best) {
            best = t;
            parts = p;
        }
    }
    return parts;
}

// Balanced split of ragged f16 batches: every work item also costs this many tiles
// (VSPEC_ROCM_DECODE_SEGMENT_COST, 0..64; 0: tiles only), the set-up of its q operands and
// the merge of its waves' states in each workgroup that holds part of it.  Measured on C4
// (64 sequences, contexts U[128, 8192]): workgroups ran ~2 us longer per work item they
// started, so those holding many short items ended the launch; decode step with a cost of
// 0 / 2 / 4 / 8 / 12 / 16 / 24 / 32 tiles: 183.1 / 179.1 / 177.6 / 175.3 / 172.6 / 174.1 /
// 176.6 / 180.0 us (another seed of the same distribution: 226.1 at 0, 197.0 at 16).  Read on
// every call.
constexpr uint32_t kDefaultSegmentCost = 12;
uint32_t decode_segment_cost() {
    const char* e = getenv("VSPEC_ROCM_DECODE_SEGMENT_COST");
    const long x = e ? strtol(e, nullptr, 10) : -1;
    return x >= 0 && x <= 64 ? (uint32_t)x : kDefaultSegmentCost;
}

// The same for int4 pools (VSPEC_ROCM_DECODE_SEGMENT_COST_INT4, 0..64), whose work items
// cost more set-up against their tiles (q operands, three barriers, the merge of the waves'
// states): decode step at the C4 shape with int4 KV (64 sequences, contexts U[128, 8192])
// with a cost of 0 / 8 / 16 / 24 / 32 / 40 / 48 / 64 tiles: 128.8 / 105.4 / 86.7 / 81.4 /
// 79.2 / 78.6 / 78.0 / 81.6 us; two other seeds 124.6 -> 86.3 (40) and 104.7 -> 86.8 (32,
// 48); C5 decode 53.8 -> 50.8 (32) / 51.2 (48).  Read on every call.
constexpr uint32_t kDefaultSegmentCostInt4 = 40;
uint32_t decode_segment_cost_int4() {
    const char* e = getenv("VSPEC_ROCM_DECODE_SEGMENT_COST_INT4");
    const long x = e ? strtol(e, nullptr, 10) : -1;
    return x >= 0 && x <= 64 ? (uint32_t)x : kDefaultSegmentCostInt4;
}

// int4 clamp flags are read by the decode only when the balanced split gives each workgroup
// at least this many tiles (VSPEC_ROCM_DECODE_FLAG_MIN_TILES, 0..4096); shorter shares read
// no flags and screen every tile.  Measured (fused step, µs): C3 (32 tiles per workgroup)
// 23.1 with flags against 23.9 screening; B = 8 at 4k 23.2 against 24.0; B = 1-4 equal;
// B = 16 at 6k 38.6 against 40.7.  Read on every call.
constexpr uint32_t kDefaultFlagMinTiles = 16;
uint32_t decode_flag_min_tiles() {
    const char* e = getenv("VSPEC_ROCM_DECODE_FLAG_MIN_TILES");
    const long x = e ? strtol(e, nullptr, 10) : -1;
    return x >= 0 && x <= 4096 ? (uint32_t)x : kDefaultFlagMinTiles;
}

struct DecodePlan {
    bool merge;  // split MFMA kernels: some work item may span two workgroups (merge launch)
    uint32_t part_tiles;  // item split: least tiles per part, for the first near_parts of them
    uint32_t near_parts;
    uint32_t far_tiles;  // least tiles per part with more parts
    uint32_t item_parts;  // item split (kv_common.h): parts of a work item, 0: ranges of all items' tiles
    uint32_t gw;
    uint32_t gsplit;
    size_t ws_bytes;
    // MFMA kernels (f16 / int4 pools): tiles of all work items split over grid_x workgroups
    bool split;
    uint32_t grid_x;
    uint32_t chunk_tiles;
    uint64_t split_tiles;  // tiles the balanced split spreads over grid_x (upper bound)
    uint32_t min_tiles;    // least tiles per workgroup of the balanced split
    uint32_t max_tiles;
    uint32_t old_permille;  // pair share of the first-half workgroups (500: equal shares)
    uint32_t uniform_tiles; // tiles per work item when every context is known to be the same
};

// Parts of a work item of f32 pools (always the item split).  Where the host knows every
// context to be the same, by the same kind of model: a part of n tiles takes n * hypot(0.8, k *
// 16 KB / 5.9 TB/s) us with k workgroups running.  Else an item's parts follow from its own
// context, not from the host's bound: enough workgroups of at least 8 tiles to fill the card
// once, and where that cuts an item in fewer than 4, up to three times as many of at least 16
// tiles, so that the longest context's parts do not outlast the others.  Once / three times, us, at
// 64, 86, 104, 128, 144 and 280 items (4 heads of 128):
//   500-4000 tokens    41/46  54/62  64/64    73/77    84/81    208/144
//   2000-4000          44/49  59/68  70/76    80/86    93/96    218/162
//   100-1600           25/25  30/27  33/35    36/39    41/42    87/64
//   120-7700           61/59  89/78  117/99   118/111  144/122  361/209
// (64-element heads alike; from 86 items on three times was slower than the kernel before the item
// split, 500-4000 tokens in heads of 64: 49 us against 38, 39 once).  *ws_parts: what the workspace is sized
// for.  It never falls as the bound on the contexts rises and does not depend on `same`, so that
// a workspace for the longest contexts serves every shorter one of as many sequences (not every
// smaller batch: fewer items are cut into more parts).  Neither rule goes past three rounds of
// workgroups, which is what is reserved.
// Measured at 1 / 2 / 4 / 8 / 16 / 32 parts: 1 x 4097 tokens (8 items) 227 / 122 / 69 / 42 / 29 / 24
// us, 16 x 2049 (128) 126 / 75 / 56 / 65, 36 x 649-5195 (144, D = 64) 189 / 107 / 76 / 64, 64 x 1025
// (512) 95 / 107.
uint32_t plan_f32_parts(uint64_t items, uint64_t tiles, uint32_t head_dim, uint64_t slots, bool same, uint32_t* ws_parts,
                        DecodePlan* pl) {
    uint64_t most = (3 * slots + items - 1) / items;
    if (most > 4 * slots / items) most = 4 * slots / items;
    if (most > (tiles + 3) / 4) most = (tiles + 3) / 4;
    if (most > 128) most = 128;
    if (most < 1) most = 1;
    *ws_parts = (uint32_t)most;
    const char* e = getenv("VSPEC_ROCM_DECODE_ITEM_PARTS");
    const long x = e ? strtol(e, nullptr, 10) : 0;
    if (x > 0) return (uint32_t)((uint64_t)x < most ? (uint64_t)x : most);
    if (!same) {
        pl->part_tiles = 8;
        if (items * 4 > slots) pl->far_tiles = 16;
        pl->near_parts = (uint32_t)(slots / items > 1 ? slots / items : 1);
        const uint64_t far_parts = items * 4 > slots ? (3 * slots / items > 1 ? 3 * slots / items : 1) : 1;
        const uint64_t near = (tiles + 7) / 8 < pl->near_parts ? (tiles + 7) / 8 : pl->near_parts;
        const uint64_t far = (tiles + 15) / 16 < far_parts ? (tiles + 15) / 16 : far_parts;
        const uint64_t p = near > far ? near : far;
        return (uint32_t)(p < most ? p : most);
    }
    const double lat = 0.8, bw = 2.75e-3 * head_dim / 128.0;
    const double busy = sqrt(lat * lat + (double)(slots * slots) * bw * bw);
    double best = 0;
    uint32_t parts = 0;
    for (const uint32_t p : {1u, 2u, 3u, 4u, 6u, 8u, 12u, 16u, 24u, 32u, 48u, 64u, 96u, 128u}) {
        if (p > most) break;
        const double full = (double)(items * p / slots), rem = (double)(items * p % slots);
        const double t = (double)((tiles + p - 1) / p) * (full * busy + (rem > 0 ? sqrt(lat * lat + rem * rem * bw * bw) : 0.0)) +
                         (p > 1 ? 5.0 + 0.12 * p : 0.0);
        if (!parts || t < best) {
            best = t;
            parts = p;
        }
    }
    return parts;
}

// With every context known to be the same (min_ctx_len == the context bound), the split
// of the MFMA kernels (kv_common.h work_split with equal shares, as for any batch whose
// contexts are equal) is known on the host: returns whether some range boundary falls
// strictly inside a work item.  Without that knowledge a merge launch is always needed.
// Tiles per work item when every context is known to be the same (min_ctx_len at least
// the bound), as the kernels' item_tiles computes them; 0 otherwise.
uint32_t uniform_item_tiles(const VspecPagedAttnDesc* d, const DecodePlan* pl, uint64_t ctx_bound) {
    if (!d->min_ctx_len || d->min_ctx_len < ctx_bound) return 0;
    const uint64_t ctx = ctx_bound < (uint64_t)d->max_blocks_per_seq * d->kv.block_tokens
                             ? ctx_bound : (uint64_t)d->max_blocks_per_seq * d->kv.block_tokens;
    uint64_t U = (ctx + kTile - 1) / kTile;
    if (U > pl->max_tiles) U = pl->max_tiles;
    if (U < 1) U = 1;
    return (uint32_t)U;
}

bool uniform_split_has_partials(const VspecPagedAttnDesc* d, const DecodePlan* pl, uint64_t ctx_bound) {
    const uint64_t U = uniform_item_tiles(d, pl, ctx_bound);
    if (!U) return true;
    const uint64_t items = (uint64_t)d->batch * d->kv.num_kv_heads * pl->gsplit;
    const uint64_t T = items * U;
    if (pl->chunk_tiles) return pl->chunk_tiles % U != 0 && T > pl->chunk_tiles;
    uint64_t G = pl->grid_x < T ? pl->grid_x : T;
    if (pl->min_tiles > 1) {
        const uint64_t cap = T / pl->min_tiles > 1 ? T / pl->min_tiles : 1;
        if (cap < G) G = cap;
    }
    // the int4 kernel's unequal pair shares (the kernels' split_shape: contexts are equal
    // here, so the f16 kernel keeps equal shares)
    const uint64_t wa = pl->old_permille;
    if (d->kv.dtype == VSPEC_KV_INT4 && wa != 500 && G == pl->grid_x && G % 2 == 0 && T >= 64 * G &&
        (1000 - wa) * T >= 500 * G) {
        const uint64_t half = G / 2;
        for (uint64_t g = 1; g < G; ++g) {
            const uint64_t c = wa * (g < half ? g : half) + (1000 - wa) * (g > half ? g - half : 0);
            if ((c * T / (1000 * half)) % U != 0) return true;
        }
        return false;
    }
    for (uint64_t g = 1; g < G; ++g) {
        if ((g * T / G) % U != 0) return true;
    }
    return false;
}

// most_heads: query heads that one work item may hold, 8 or 4
int plan_decode(const VspecPagedAttnDesc* d, DecodePlan* pl, uint32_t most_heads = 8) {
    pl->merge = true;
    const uint32_t hkv = d->kv.num_kv_heads;
    if (d->num_q_heads == 0 || d->num_q_heads % hkv != 0) {
        set_err("paged_decode: num_q_heads must be a positive multiple of num_kv_heads");
        return 0;
    }
    const uint32_t g = d->num_q_heads / hkv;
    if (g <= 4) {
        pl->gw = g;
        pl->gsplit = 1;
    } else if (g % 8 == 0 && d->kv.dtype == VSPEC_KV_F16 && most_heads >= 8) {
        // f16: the score MFMA's 16 columns hold 8 heads as well as 4, so that a tile is read
        // and multiplied once for all of them (64 x 4097 tokens, 32/4 heads: 172 us with two
        // items of 4 heads, 142 with the two on one XCD, 89.5 with one of 8)
        pl->gw = 8;
        pl->gsplit = g / 8;
    } else if (g % 4 == 0) {
        pl->gw = 4;
        pl->gsplit = g / 4;
    } else {
        set_err("paged_decode: GQA group %u unsupported (need <= 4 or a multiple of 4)", g);
        return 0;
    }
    // the host's bound on ctx_lens; 0 stands for the block table's capacity
    const uint64_t ctx_bound = d->max_ctx_len ? (uint64_t)d->max_ctx_len
                                              : (uint64_t)d->max_blocks_per_seq * d->kv.block_tokens;
    if (ctx_bound > (uint64_t)INT32_MAX) {
        set_err("paged_decode: context bound beyond 2^31 tokens");
        return 0;
    }
    const uint32_t max_tiles = (uint32_t)((ctx_bound + kTile - 1) / kTile);
    pl->split = d->kv.dtype != VSPEC_KV_F32;
    pl->item_parts = 0;
    pl->chunk_tiles = 0;
    pl->part_tiles = 4;  // one for each wave
    pl->near_parts = 0x7fffffffu;
    pl->far_tiles = 0x40000000u;
    if (pl->split) {
        // every workgroup streams an equal share of all work items' tiles
        pl->min_tiles = decode_min_tiles_per_wg((uint64_t)d->batch * hkv * pl->gsplit);
        const uint64_t bound = (uint64_t)d->batch * hkv * pl->gsplit * (max_tiles ? max_tiles : 1);
        if (bound > (uint64_t)INT32_MAX) {
            set_err("paged_decode: batch * work items * tiles exceeds 2^31");
            return 0;
        }
        uint64_t grid;
        if (d->partition_tokens) {
            if (d->partition_tokens % kTile) {
                set_err("paged_decode: partition_tokens must be a multiple of %d", kTile);
                return 0;
            }
            pl->chunk_tiles = d->partition_tokens / kTile;
            grid = (bound + pl->chunk_tiles - 1) / pl->chunk_tiles;
        } else {
            // two workgroups per CU; small f16 batches (under 64 tiles per workgroup at two
            // per CU) take one, which halves the cross-workgroup merges per work item
            // (C2: 41.6 -> 38.9 us; the int4 kernel, bound by vector ALU work, needs both)
            uint32_t wpc = decode_wgs_per_cu_env();
            if (!wpc) wpc = d->kv.dtype == VSPEC_KV_F16 && bound < 128ull * (uint64_t)num_cus() ? 1u : 2u;
            grid = (uint64_t)wpc * (uint64_t)num_cus();
            // the kernel caps its groups at total / min_tiles of the actual split total (tiles,
            // plus the segment cost of every work item of a ragged batch); the grid, from a
            // bound of that total, only trims idle workgroups, so the split does not depend on
            // the host's context bound
            const uint64_t seg = d->kv.dtype == VSPEC_KV_F16    ? decode_segment_cost()
                                 : d->kv.dtype == VSPEC_KV_INT4 ? decode_segment_cost_int4()
                                                                : 0u;
            const uint64_t cost_bound = bound + seg * (uint64_t)d->batch * hkv * pl->gsplit;
            const uint64_t min_tiles = pl->min_tiles;
            if (grid * min_tiles > cost_bound) grid = cost_bound / min_tiles;
        }
        pl->grid_x = (uint32_t)(grid ? grid : 1);
        pl->split_tiles = bound;
        pl->max_tiles = max_tiles;
        // unequal pair shares need the grid of two workgroups per CU (g and g + G/2 share one)
        pl->old_permille = !pl->chunk_tiles && pl->grid_x == 2u * (uint32_t)num_cus()
                               ? decode_old_permille(d->kv.dtype) : 500u;
        pl->merge = uniform_split_has_partials(d, pl, ctx_bound);
        pl->uniform_tiles = uniform_item_tiles(d, pl, ctx_bound);
        // (a partial state of the balanced split's plan per part: 2 slots per workgroup)
        if (!pl->chunk_tiles && d->batch) {
            pl->item_parts = plan_item_parts(d, (uint64_t)d->batch * hkv * pl->gsplit, max_tiles ? max_tiles : 1,
                                             2ull * (uint64_t)num_cus(), 2ull * pl->grid_x, pl->uniform_tiles != 0);
        }
        // the workspace stays even without a merge launch: a context below min_ctx_len (a
        // caller error) then leaves its partial states in valid memory, not its output
        pl->ws_bytes = (size_t)pl->grid_x * 2 * pl->gw * (2 + d->kv.head_dim) * sizeof(float);
        return 1;
    }
    pl->uniform_tiles = 0;
    pl->max_tiles = max_tiles;
    pl->item_parts = 1;
    uint32_t ws_parts = 0;  // the workspace holds this many parts per work item
    if (d->partition_tokens) {
        if (d->partition_tokens % kTile) {
            set_err("paged_decode: partition_tokens must be a multiple of %d", kTile);
            return 0;
        }
        const uint32_t tpp = d->partition_tokens / kTile;
        pl->chunk_tiles = pl->part_tiles = tpp;
        if (max_tiles) pl->item_parts = (max_tiles + tpp - 1) / tpp;
    } else if (d->batch) {
        pl->item_parts = plan_f32_parts((uint64_t)d->batch * hkv * pl->gsplit, max_tiles ? max_tiles : 1, d->kv.head_dim,
                                        2ull * (uint64_t)num_cus(), uniform_item_tiles(d, pl, ctx_bound) != 0, &ws_parts,
                                        pl);
    }
    if (!ws_parts) ws_parts = pl->item_parts;
    pl->ws_bytes = ws_parts > 1
                       ? (size_t)d->batch * d->num_q_heads * ws_parts * (2 + d->kv.head_dim) * sizeof(float)
                       : 0;
    return 1;
}

}  // namespace

// ---------------------------------------------------------------------------
// C-ABI
// ---------------------------------------------------------------------------
extern "C" {

const char* vspec_rocm_last_error(void) { return g_err; }

int vspec_rocm_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

int vspec_rocm_sync(void* stream) {
    HIP_CHECK(hipStreamSynchronize((hipStream_t)stream), "sync");
    return 1;
}

size_t vspec_rocm_kv_pool_bytes(int32_t dtype, uint32_t num_blocks, uint32_t block_tokens,
                                uint32_t num_kv_heads, uint32_t head_dim) {
    const size_t rows = (size_t)num_blocks * num_kv_heads * block_tokens;
    size_t bytes = 2 * rows * row_bytes_of(dtype, head_dim);
    if (dtype == VSPEC_KV_INT4) {
        bytes += 2 * rows * (head_dim / 32) * sizeof(uint16_t);
        bytes += (rows / 16) * sizeof(uint32_t);  // clamp flags
    }
    return bytes;
}

int vspec_rocm_kv_pool_create(VspecPagedKV* kv, int32_t dtype, uint32_t num_blocks,
                              uint32_t block_tokens, uint32_t num_kv_heads, uint32_t head_dim) {
    if (!kv) {
        set_err("kv_pool_create: null descriptor");
        return 0;
    }
    memset(kv, 0, sizeof(*kv));
    kv->dtype = dtype;
    kv->num_blocks = num_blocks;
    kv->block_tokens = block_tokens;
    kv->num_kv_heads = num_kv_heads;
    kv->head_dim = head_dim;
    kv->k_data = kv->v_data = (void*)1;  // placeholders for validation
    kv->k_scales = kv->v_scales = (uint16_t*)1;
    if (!check_kv(kv, "kv_pool_create")) {
        memset(kv, 0, sizeof(*kv));
        return 0;
    }
    kv->k_data = kv->v_data = nullptr;
    kv->k_scales = kv->v_scales = nullptr;
    const size_t rows = (size_t)num_blocks * num_kv_heads * block_tokens;
    const size_t data = rows * row_bytes_of(dtype, head_dim);
    if (hipMalloc(&kv->k_data, data) != hipSuccess || hipMalloc(&kv->v_data, data) != hipSuccess) {
        set_err("kv_pool_create: hipMalloc of %zu bytes failed", 2 * data);
        vspec_rocm_kv_pool_destroy(kv);
        return 0;
    }
    if (dtype == VSPEC_KV_INT4) {
        const size_t sb = rows * (head_dim / 32) * sizeof(uint16_t);
        const size_t fb = (rows / 16) * sizeof(uint32_t);
        if (hipMalloc((void**)&kv->k_scales, sb) != hipSuccess ||
            hipMalloc((void**)&kv->v_scales, sb) != hipSuccess ||
            hipMalloc((void**)&kv->k_flags, fb) != hipSuccess ||
            hipMemset(kv->k_flags, 0, fb) != hipSuccess) {
            set_err("kv_pool_create: hipMalloc of scales or flags failed");
            vspec_rocm_kv_pool_destroy(kv);
            return 0;
        }
    }
    return 1;
}

void vspec_rocm_kv_pool_destroy(VspecPagedKV* kv) {
    if (!kv) return;
    if (kv->k_data) (void)hipFree(kv->k_data);
    if (kv->v_data) (void)hipFree(kv->v_data);
    if (kv->k_scales) (void)hipFree(kv->k_scales);
    if (kv->v_scales) (void)hipFree(kv->v_scales);
    if (kv->k_flags) (void)hipFree(kv->k_flags);
    memset(kv, 0, sizeof(*kv));
}

static int append_launch(const char* who, const VspecPagedKV* kv, AppendParams& p, int32_t src_dtype,
                         void* stream) {
    p.k = (uint8_t*)kv->k_data;
    p.v = (uint8_t*)kv->v_data;
    p.ks = kv->k_scales;
    p.vs = kv->v_scales;
    p.kf = kv->dtype == VSPEC_KV_INT4 ? kv->k_flags : nullptr;
    p.hkv = kv->num_kv_heads;
    p.head_dim = kv->head_dim;
    p.block_tokens = kv->block_tokens;
    p.num_blocks = kv->num_blocks;
    p.rope_vec = p.rope_cos && ((uintptr_t)p.rope_cos | (uintptr_t)p.rope_sin) % 16 == 0;
    hipStream_t s = (hipStream_t)stream;
    const uint64_t tokens = (uint64_t)p.batch * p.n_new;
    // query rows ride along when their halves and the tables split into 16-byte chunks
    const bool q_vec = p.q_in && p.rope_vec && p.rope_dim % 8 == 0 && ((uintptr_t)p.q_in | (uintptr_t)p.q_out) % 16 == 0;
    const uint64_t q_items =
        q_vec ? tokens * ((p.hq + kRopeHeads - 1) / kRopeHeads) * rope_q_chunks(p.head_dim, p.rope_dim) : 0;
    const uint64_t k_items = tokens * p.hkv * (p.head_dim / 8);
    const uint64_t v_items = kv->dtype == VSPEC_KV_F16
                                 ? (uint64_t)p.batch * append_v_units<VSPEC_KV_F16>(p.n_new, p.token_item != nullptr) *
                                       p.hkv * (p.head_dim / 8)
                                 : k_items;
    // the row kernel counts its items in 32 bits
    const bool rows = kv->dtype != VSPEC_KV_INT4 && k_items + v_items + q_items + 768 < 0xffffffffull;
    const bool q_rows = q_items && (rows || q_items + 256 < 0xffffffffull);
    if (rows) {
        const uint32_t kw = (uint32_t)((k_items + 255) / 256), vw = (uint32_t)((v_items + 255) / 256);
        const dim3 grid(kw + vw + (uint32_t)((q_items + 255) / 256));
#define VSPEC_APPEND_(DT, SRC, ROPE)                                                                         \
    hipLaunchKernelGGL((kv_append_rows<DT, SRC, ROPE>), grid, dim3(256), 0, s, p, kw, vw, (uint32_t)k_items, \
                       (uint32_t)v_items, (uint32_t)q_items)
#define VSPEC_APPEND(DT, SRC) \
    if (p.rope_cos) VSPEC_APPEND_(DT, SRC, true); \
    else VSPEC_APPEND_(DT, SRC, false)
        if (src_dtype == VSPEC_KV_F32) {
            if (kv->dtype == VSPEC_KV_F32) { VSPEC_APPEND(VSPEC_KV_F32, VSPEC_KV_F32); }
            else { VSPEC_APPEND(VSPEC_KV_F16, VSPEC_KV_F32); }
        } else {
            if (kv->dtype == VSPEC_KV_F32) { VSPEC_APPEND(VSPEC_KV_F32, VSPEC_KV_F16); }
            else { VSPEC_APPEND(VSPEC_KV_F16, VSPEC_KV_F16); }
        }
#undef VSPEC_APPEND_
    } else {
        const uint32_t ept = kv->dtype == VSPEC_KV_INT4 ? 32 : 8;
        const uint64_t items = tokens * p.hkv * (p.head_dim / ept) * 2;
        uint64_t blocks = (items + 255) / 256;
        if (blocks > 65536) blocks = 65536;
        const dim3 grid((unsigned)blocks);
#define VSPEC_APPEND_(DT, SRC, ROPE) hipLaunchKernelGGL((kv_append<DT, SRC, ROPE>), grid, dim3(256), 0, s, p)
        if (src_dtype == VSPEC_KV_F32) {
            if (kv->dtype == VSPEC_KV_F32) { VSPEC_APPEND(VSPEC_KV_F32, VSPEC_KV_F32); }
            else if (kv->dtype == VSPEC_KV_F16) { VSPEC_APPEND(VSPEC_KV_F16, VSPEC_KV_F32); }
            else { VSPEC_APPEND(VSPEC_KV_INT4, VSPEC_KV_F32); }
        } else {
            if (kv->dtype == VSPEC_KV_F32) { VSPEC_APPEND(VSPEC_KV_F32, VSPEC_KV_F16); }
            else if (kv->dtype == VSPEC_KV_F16) { VSPEC_APPEND(VSPEC_KV_F16, VSPEC_KV_F16); }
            else { VSPEC_APPEND(VSPEC_KV_INT4, VSPEC_KV_F16); }
        }
        if (q_rows) hipLaunchKernelGGL(rope_q_rows, dim3((unsigned)((q_items + 255) / 256)), dim3(256), 0, s, p, (uint32_t)q_items);
#undef VSPEC_APPEND
#undef VSPEC_APPEND_
    }
    if (p.q_in && !q_rows) {
        RopeQParams rq = {p.q_in, p.q_out, p.start_pos, p.rope_cos, p.rope_sin, p.batch, p.n_new, p.hq,
                          p.head_dim, p.rope_dim, p.max_pos};
        uint64_t blocks = (tokens * p.hq * p.head_dim + 255) / 256;
        if (blocks > 65536) blocks = 65536;
        hipLaunchKernelGGL(rope_q, dim3((unsigned)blocks), dim3(256), 0, s, rq);
    }
    HIP_CHECK(hipGetLastError(), who);
    return 1;
}

int vspec_rocm_kv_append(const VspecPagedKV* kv, uint32_t batch, const int32_t* block_tables,
                         uint32_t max_blocks_per_seq, const int32_t* start_pos, uint32_t n_new,
                         const void* k_new, const void* v_new, int32_t src_dtype, void* stream) {
    if (!check_kv(kv, "kv_append")) return 0;
    if (src_dtype != VSPEC_KV_F32 && src_dtype != VSPEC_KV_F16) {
        set_err("kv_append: src_dtype must be f32 or f16");
        return 0;
    }
    if (batch == 0 || n_new == 0) return 1;
    if (!block_tables || !start_pos || !k_new || !v_new || max_blocks_per_seq == 0) {
        set_err("kv_append: null argument");
        return 0;
    }
    AppendParams p = {};
    p.block_tables = block_tables;
    p.start_pos = start_pos;
    p.k_new = (const uint8_t*)k_new;
    p.v_new = (const uint8_t*)v_new;
    p.batch = batch;
    p.n_new = n_new;
    p.max_blocks = max_blocks_per_seq;
    return append_launch("kv_append launch", kv, p, src_dtype, stream);
}

int vspec_rocm_kv_append_rope(const VspecPagedKV* kv, uint32_t batch, const int32_t* block_tables,
                              uint32_t max_blocks_per_seq, const int32_t* start_pos, uint32_t n_new,
                              const void* k_new, const void* v_new, int32_t src_dtype, const float* rope_cos,
                              const float* rope_sin, uint32_t rope_dim, uint32_t max_pos, const float* q_in,
                              float* q_out, uint32_t num_q_heads, void* stream) {
    if (!check_kv(kv, "kv_append_rope")) return 0;
    if (src_dtype != VSPEC_KV_F32 && src_dtype != VSPEC_KV_F16) {
        set_err("kv_append_rope: src_dtype must be f32 or f16");
        return 0;
    }
    if (!rope_cos || !rope_sin || rope_dim == 0 || rope_dim % 2 != 0 || rope_dim > kv->head_dim || max_pos == 0) {
        set_err("kv_append_rope: need cos/sin tables and an even rope_dim <= head_dim");
        return 0;
    }
    if ((q_in == nullptr) != (q_out == nullptr) || (q_in && num_q_heads == 0)) {
        set_err("kv_append_rope: q_in and q_out go together, with num_q_heads > 0");
        return 0;
    }
    if (batch == 0 || n_new == 0) return 1;
    if (!block_tables || !start_pos || !k_new || !v_new || max_blocks_per_seq == 0) {
        set_err("kv_append_rope: null argument");
        return 0;
    }
    AppendParams p = {};
    p.block_tables = block_tables;
    p.start_pos = start_pos;
    p.k_new = (const uint8_t*)k_new;
    p.v_new = (const uint8_t*)v_new;
    p.batch = batch;
    p.n_new = n_new;
    p.max_blocks = max_blocks_per_seq;
    p.rope_cos = rope_cos;
    p.rope_sin = rope_sin;
    p.rope_dim = rope_dim;
    p.max_pos = max_pos;
    p.q_in = q_in;
    p.q_out = q_out;
    p.hq = num_q_heads;
    return append_launch("kv_append_rope launch", kv, p, src_dtype, stream);
}

int vspec_rocm_kv_append_tokens(const VspecPagedKV* kv, uint32_t n_tokens, const int32_t* token_item,
                                const int32_t* token_pos, const int32_t* block_tables, uint32_t n_items,
                                uint32_t max_blocks_per_seq, const void* k_new, const void* v_new,
                                int32_t src_dtype, void* stream) {
    if (!check_kv(kv, "kv_append_tokens")) return 0;
    if (src_dtype != VSPEC_KV_F32 && src_dtype != VSPEC_KV_F16) {
        set_err("kv_append_tokens: src_dtype must be f32 or f16");
        return 0;
    }
    if (n_tokens == 0) return 1;
    if (!token_item || !token_pos || !block_tables || !k_new || !v_new || max_blocks_per_seq == 0 || n_items == 0) {
        set_err("kv_append_tokens: null argument or no block-table rows");
        return 0;
    }
    AppendParams p = {};
    p.block_tables = block_tables;
    p.token_item = token_item;
    p.token_pos = token_pos;
    p.n_items = n_items;
    p.k_new = (const uint8_t*)k_new;
    p.v_new = (const uint8_t*)v_new;
    p.batch = n_tokens;
    p.n_new = 1;
    p.max_blocks = max_blocks_per_seq;
    return append_launch("kv_append_tokens launch", kv, p, src_dtype, stream);
}

int vspec_rocm_kv_gather(const VspecPagedKV* kv, uint32_t batch, const int32_t* block_tables,
                         uint32_t max_blocks_per_seq, const int32_t* ctx_lens,
                         uint32_t max_ctx_len, const int64_t* out_token_offset, int32_t out_mode,
                         void* out_k, void* out_v, uint16_t* out_k_scales,
                         uint16_t* out_v_scales, void* stream) {
    if (!check_kv(kv, "kv_gather")) return 0;
    if (out_mode != VSPEC_GATHER_RAW && out_mode != VSPEC_GATHER_F32) {
        set_err("kv_gather: bad out_mode");
        return 0;
    }
    if (batch == 0 || max_ctx_len == 0) return 1;
    if (!block_tables || !ctx_lens || !out_token_offset || !out_k || !out_v || max_blocks_per_seq == 0) {
        set_err("kv_gather: null argument");
        return 0;
    }
    if (out_mode == VSPEC_GATHER_RAW && kv->dtype == VSPEC_KV_INT4 && (!out_k_scales || !out_v_scales)) {
        set_err("kv_gather: int4 raw gather needs scale outputs");
        return 0;
    }
    GatherParams p = {};
    p.k = (const uint8_t*)kv->k_data;
    p.v = (const uint8_t*)kv->v_data;
    p.ks = kv->k_scales;
    p.vs = kv->v_scales;
    p.block_tables = block_tables;
    p.ctx_lens = ctx_lens;
    p.out_off = out_token_offset;
    p.ok = (uint8_t*)out_k;
    p.ov = (uint8_t*)out_v;
    p.oks = out_k_scales;
    p.ovs = out_v_scales;
    p.hkv = kv->num_kv_heads;
    p.head_dim = kv->head_dim;
    p.block_tokens = kv->block_tokens;
    p.max_blocks = max_blocks_per_seq;
    p.num_blocks = kv->num_blocks;
    p.max_ctx = max_ctx_len;
    const uint32_t D = kv->head_dim;
    const size_t rb = row_bytes_of(kv->dtype, D);
    const uint32_t cpr = out_mode == VSPEC_GATHER_F32 ? D / 8 : (kv->dtype == VSPEC_KV_INT4 ? rb / 4 : rb / 16);
    const uint64_t items = (uint64_t)max_ctx_len * kv->num_kv_heads * cpr * 2;
    uint64_t gx = (items + 255) / 256;
    if (gx > 16384) gx = 16384;
    const dim3 grid((unsigned)gx, batch);
    hipStream_t s = (hipStream_t)stream;
    // 4-token units (not the row kernel): f16 pools, and int4 ones of the usual head sizes
    const bool i4 = kv->dtype == VSPEC_KV_INT4, f32_out = out_mode == VSPEC_GATHER_F32;
    if (kv->dtype == VSPEC_KV_F16 || (i4 && (D == 64 || D == 128))) {
        const uint64_t lanes = i4 ? 16 : D / (f32_out ? 4 : 8);
        const uint64_t wgs = (((uint64_t)max_ctx_len + 3) / 4 * kv->num_kv_heads * lanes + 255) / 256;
        if (wgs <= 0x7fffffffull / 256) {
            const dim3 qgrid((unsigned)wgs, batch, 2);
#define VSPEC_GATHER(DT, DIM)                                                                                  \
    if (f32_out) hipLaunchKernelGGL((kv_gather_quads<DT, 1, DIM>), qgrid, dim3(256), 0, s, p); \
    else hipLaunchKernelGGL((kv_gather_quads<DT, 0, DIM>), qgrid, dim3(256), 0, s, p)
            if (!i4) { VSPEC_GATHER(VSPEC_KV_F16, 0); }
            else if (D == 64) { VSPEC_GATHER(VSPEC_KV_INT4, 64); }
            else { VSPEC_GATHER(VSPEC_KV_INT4, 128); }
#undef VSPEC_GATHER
            HIP_CHECK(hipGetLastError(), "kv_gather launch");
            return 1;
        }
    }
#define VSPEC_GATHER(DT, OF) hipLaunchKernelGGL((kv_gather<DT, OF>), grid, dim3(256), 0, s, p)
    if (out_mode == VSPEC_GATHER_F32) {
        if (kv->dtype == VSPEC_KV_F32) VSPEC_GATHER(VSPEC_KV_F32, 1);
        else if (kv->dtype == VSPEC_KV_F16) VSPEC_GATHER(VSPEC_KV_F16, 1);
        else VSPEC_GATHER(VSPEC_KV_INT4, 1);
    } else {
        if (kv->dtype == VSPEC_KV_F32) VSPEC_GATHER(VSPEC_KV_F32, 0);
        else if (kv->dtype == VSPEC_KV_F16) VSPEC_GATHER(VSPEC_KV_F16, 0);
        else VSPEC_GATHER(VSPEC_KV_INT4, 0);
    }
#undef VSPEC_GATHER
    HIP_CHECK(hipGetLastError(), "kv_gather launch");
    return 1;
}

int vspec_rocm_kv_compact(const VspecPagedKV* kv, uint32_t n, const int32_t* src_blocks,
                          const int32_t* dst_blocks, void* stream) {
    if (!check_kv(kv, "kv_compact")) return 0;
    if (n == 0) return 1;
    if (!src_blocks || !dst_blocks) {
        set_err("kv_compact: null block list");
        return 0;
    }
    CompactParams p = {};
    p.k = (uint8_t*)kv->k_data;
    p.v = (uint8_t*)kv->v_data;
    p.ks = kv->k_scales;
    p.vs = kv->v_scales;
    p.src = src_blocks;
    p.dst = dst_blocks;
    p.n = n;
    p.num_blocks = kv->num_blocks;
    const uint64_t rows = (uint64_t)kv->num_kv_heads * kv->block_tokens;
    p.block_bytes = rows * row_bytes_of(kv->dtype, kv->head_dim);
    p.block_scales = kv->dtype == VSPEC_KV_INT4 ? rows * (kv->head_dim / 32) : 0;
    p.kf = kv->dtype == VSPEC_KV_INT4 ? kv->k_flags : nullptr;
    p.block_flags = (uint32_t)(rows / 16);
    uint64_t gx = (2 * (p.block_bytes / 16) + 255) / 256;
    if (gx > 64) gx = 64;
    if (gx == 0) gx = 1;
    hipLaunchKernelGGL(kv_compact, dim3((unsigned)gx, n), dim3(256), 0, (hipStream_t)stream, p);
    HIP_CHECK(hipGetLastError(), "kv_compact launch");
    return 1;
}

int vspec_rocm_kv_gather_rows(const VspecPagedKV* kv, uint32_t n, const int32_t* pages,
                              const int32_t* slots, float* out_k, float* out_v, void* stream) {
    if (!check_kv(kv, "kv_gather_rows")) return 0;
    if (n == 0) return 1;
    if (!pages || !slots || !out_k || !out_v) {
        set_err("kv_gather_rows: null argument");
        return 0;
    }
    GatherRowsParams p = {};
    p.k = (const uint8_t*)kv->k_data;
    p.v = (const uint8_t*)kv->v_data;
    p.ks = kv->k_scales;
    p.vs = kv->v_scales;
    p.pages = pages;
    p.slots = slots;
    p.ok = out_k;
    p.ov = out_v;
    p.n = n;
    p.hkv = kv->num_kv_heads;
    p.head_dim = kv->head_dim;
    p.block_tokens = kv->block_tokens;
    p.num_blocks = kv->num_blocks;
    const uint64_t items = (uint64_t)n * kv->num_kv_heads * (kv->head_dim / 8) * 2;
    uint64_t gx = (items + 255) / 256;
    if (gx > 16384) gx = 16384;
    hipStream_t s = (hipStream_t)stream;
    if (kv->dtype == VSPEC_KV_F32) hipLaunchKernelGGL(kv_gather_rows<VSPEC_KV_F32>, dim3((unsigned)gx), dim3(256), 0, s, p);
    else if (kv->dtype == VSPEC_KV_F16) hipLaunchKernelGGL(kv_gather_rows<VSPEC_KV_F16>, dim3((unsigned)gx), dim3(256), 0, s, p);
    else hipLaunchKernelGGL(kv_gather_rows<VSPEC_KV_INT4>, dim3((unsigned)gx), dim3(256), 0, s, p);
    HIP_CHECK(hipGetLastError(), "kv_gather_rows launch");
    return 1;
}

size_t vspec_rocm_paged_decode_workspace_bytes(const VspecPagedAttnDesc* desc) {
    DecodePlan pl;
    if (!desc) {
        set_err("paged_decode_workspace_bytes: null descriptor");
        return 0;
    }
    if (!check_kv(&desc->kv, "paged_decode_workspace_bytes", true) || !plan_decode(desc, &pl)) return 0;
    return pl.ws_bytes;
}

}  // extern "C"

namespace {

// Decode attention, with the decode step's append of k_new / v_new when they are given: by the
// decode kernel itself, or for f32 pools and more than kStepRows rows by a launch before it
// (the f32 kernel looks in every tile for the new tokens of all rows, which may share blocks).
// noalloc: the partial states come from the file-scope scratch array
// (no allocation, no library state beyond it); the descriptor's workspace is ignored.
int paged_decode(const VspecPagedAttnDesc* desc, const void* k_new, const void* v_new, int32_t src_dtype,
                 bool noalloc) {
    if (!desc) {
        set_err("paged_decode: null descriptor");
        return 0;
    }
    if (!check_kv(&desc->kv, "paged_decode", true)) return 0;
    if (desc->batch == 0) return 1;
    if (!desc->block_tables || !desc->ctx_lens || !desc->q || !desc->out || desc->max_blocks_per_seq == 0) {
        set_err("paged_decode: null argument");
        return 0;
    }
    if (desc->numerics != VSPEC_NUMERICS_PLAIN && desc->numerics != VSPEC_NUMERICS_3BIT) {
        set_err("paged_decode: bad numerics mode");
        return 0;
    }
    if ((uint64_t)desc->max_ctx_len > (uint64_t)desc->max_blocks_per_seq * desc->kv.block_tokens) {
        set_err("paged_decode: max_ctx_len exceeds the block table");
        return 0;
    }
    DecodePlan pl;
    if (!plan_decode(desc, &pl)) return 0;
    void* ws = nullptr;
    if (noalloc) {
        // a workgroup's two partial states are twice as large with 8 heads to a work item as with
        // 4: plans of many workgroups (VSPEC_ROCM_DECODE_WGS_PER_CU 3 to 5) fit only with 4
        if (pl.ws_bytes > kScratchBytes && pl.gw == 8 && !plan_decode(desc, &pl, 4)) return 0;
        if (pl.ws_bytes > kScratchBytes) {
            set_err("paged_decode_step_noalloc: the plan needs %zu bytes of partial states, more than the "
                    "%zu-byte scratch (use vspec_rocm_paged_decode_step with a workspace)",
                    pl.ws_bytes, kScratchBytes);
            return 0;
        }
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
            set_err("paged_decode_step_noalloc: no current device");
            return 0;
        }
        uint8_t* base = scratch_address(dev);
        if (!base) return 0;
        ws = pl.ws_bytes ? base : nullptr;
    } else if (pl.ws_bytes) {
        if (desc->workspace) {
            if (desc->workspace_bytes < pl.ws_bytes) {
                set_err("paged_decode: workspace too small (%zu < %zu)", desc->workspace_bytes, pl.ws_bytes);
                return 0;
            }
            ws = desc->workspace;
        } else {
            ws = library_workspace(pl.ws_bytes);
            if (!ws) {
                set_err("paged_decode: cannot allocate %zu workspace bytes", pl.ws_bytes);
                return 0;
            }
        }
    }
    const uint32_t D = desc->kv.head_dim;
    float scale = desc->scale > 0.f ? desc->scale : 1.0f / sqrtf((float)D);
    const bool three = desc->numerics == VSPEC_NUMERICS_3BIT;
    if (three) scale = fminf(fmaxf(scale, 1e-4f), 32.0f);

    DecodeParams p = {};
    p.k = (const uint8_t*)desc->kv.k_data;
    p.v = (const uint8_t*)desc->kv.v_data;
    p.ks = desc->kv.k_scales;
    p.vs = desc->kv.v_scales;
    p.kf = desc->kv.dtype == VSPEC_KV_INT4 ? desc->kv.k_flags : nullptr;
    p.read_flags = p.kf && pl.split && pl.split_tiles >= (uint64_t)decode_flag_min_tiles() * pl.grid_x;
    p.block_tables = desc->block_tables;
    p.ctx_lens = desc->ctx_lens;
    p.block_used = desc->block_used;
    p.q = desc->q;
    p.out = desc->out;
    p.part_ml = (float*)ws;
    p.hq = desc->num_q_heads;
    p.hkv = desc->kv.num_kv_heads;
    p.block_tokens = desc->kv.block_tokens;
    p.max_blocks = desc->max_blocks_per_seq;
    p.num_blocks = desc->kv.num_blocks;
    p.gsplit = pl.gsplit;
    p.qscale = scale * kLog2e;
    p.alpha = desc->clamp_alpha > 0.f ? desc->clamp_alpha : 4.5f;
    p.logit_clip = three ? 24.0f * kLog2e : INFINITY;
    p.input_clip = three ? 16.0f : INFINITY;
    p.split_grid = pl.split ? pl.grid_x : 0u;
    p.merge = pl.split && pl.merge;
    p.batch = desc->batch;
    p.max_tiles = pl.max_tiles;
    p.chunk_tiles = pl.chunk_tiles;
    p.append_src = src_dtype;
    p.split_old_permille = pl.split ? pl.old_permille : 500u;
    p.uniform_tiles = pl.split ? pl.uniform_tiles : 0u;
    p.min_tiles = pl.split && !pl.chunk_tiles ? pl.min_tiles : 1u;
    p.item_parts = pl.item_parts;
    p.part_tiles = pl.part_tiles;
    p.near_parts = pl.near_parts;
    p.far_tiles = pl.far_tiles;
    p.seg_cost = !pl.split || pl.chunk_tiles ? 0u
                 : desc->kv.dtype == VSPEC_KV_F16 ? decode_segment_cost()
                 : desc->kv.dtype == VSPEC_KV_INT4 ? decode_segment_cost_int4() : 0u;

    hipStream_t s = (hipStream_t)desc->stream;
    if (k_new && !pl.split && desc->batch > kStepRows) {
        AppendParams a = {};
        a.block_tables = desc->block_tables;
        a.ctx_lens = desc->ctx_lens;
        a.k_new = (const uint8_t*)k_new;
        a.v_new = (const uint8_t*)v_new;
        a.batch = desc->batch;
        a.n_new = 1;
        a.max_blocks = desc->max_blocks_per_seq;
        if (!append_launch("paged_decode_step append launch", &desc->kv, a, src_dtype, s)) return 0;
    } else {
        p.k_new = (const uint8_t*)k_new;
        p.v_new = (const uint8_t*)v_new;
    }
    if (pl.split) {
        // partial slots [grid][2][GW] of (max, sum) then of acc[D]
        p.part_acc = (float*)ws + (size_t)pl.grid_x * 2 * pl.gw * 2;
    }
    if (pl.item_parts) {
        // partial slots [batch][item][part][GW]: acc[D] of all, then (max, sum)
        p.part_acc = (float*)ws;
        p.part_ml = (float*)ws + (size_t)desc->batch * desc->kv.num_kv_heads * pl.gsplit * pl.item_parts * pl.gw * D;
    }
    const dim3 grid = pl.item_parts ? dim3(desc->kv.num_kv_heads * pl.gsplit * pl.item_parts, desc->batch)
                                    : dim3(pl.grid_x);
    int ok = 0;
    switch (desc->kv.dtype) {
        case VSPEC_KV_F32: ok = launch_decode_f32(p, D, pl.gw, grid, s); break;
        case VSPEC_KV_F16:
            ok = D == 64 ? launch_decode_mfma_f16_d64(p, pl.gw, grid, s) : launch_decode_mfma_f16_d128(p, pl.gw, grid, s);
            break;
        default:
            ok = D == 64 ? launch_decode_mfma_int4_d64(p, pl.gw, grid, s) : launch_decode_mfma_int4_d128(p, pl.gw, grid, s);
            break;
    }
    if (!ok) {
        set_err("paged_decode: no kernel for head_dim %u, group %u", D, pl.gw);
        return 0;
    }
    HIP_CHECK(hipGetLastError(), "decode launch");
    return 1;
}

}  // namespace

extern "C" {

int vspec_rocm_paged_decode_attention(const VspecPagedAttnDesc* desc) {
    return paged_decode(desc, nullptr, nullptr, VSPEC_KV_F32, false);
}

static int decode_step(const char* who, const VspecPagedAttnDesc* desc, const void* k_new, const void* v_new,
                       int32_t src_dtype, bool noalloc) {
    const bool empty = desc && desc->batch == 0;  // a no-op, like every other entry point
    if (!empty && (!k_new || !v_new)) {
        set_err("%s: null k_new or v_new", who);
        return 0;
    }
    if (src_dtype != VSPEC_KV_F32 && src_dtype != VSPEC_KV_F16) {
        set_err("%s: src_dtype must be f32 or f16", who);
        return 0;
    }
    return paged_decode(desc, k_new, v_new, src_dtype, noalloc);
}

int vspec_rocm_paged_decode_step(const VspecPagedAttnDesc* desc, const void* k_new, const void* v_new,
                                 int32_t src_dtype) {
    return decode_step("paged_decode_step", desc, k_new, v_new, src_dtype, false);
}

int vspec_rocm_paged_decode_step_noalloc(const VspecPagedAttnDesc* desc, const void* k_new, const void* v_new,
                                         int32_t src_dtype) {
    return decode_step("paged_decode_step_noalloc", desc, k_new, v_new, src_dtype, true);
}

int vspec_rocm_release_retired_workspaces(void) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
        set_err("release_retired_workspaces: no current device");
        return 0;
    }
    std::lock_guard<std::mutex> lock(g_ws_mu);
    int ok = 1;
    for (void* ptr : g_retired[dev]) {
        if (hipFree(ptr) != hipSuccess) ok = 0;
    }
    g_retired[dev].clear();
    if (!ok) set_err("release_retired_workspaces: hipFree failed");
    return ok;
}

}  // extern "C"
