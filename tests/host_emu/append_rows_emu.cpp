// Host comparison of the two append paths of f16 and f32 pools (append_row.h): the section
// items that the row kernel runs (append_k_item, append_v_item, rope_q_item) in a shuffled
// order against the general per-item code (append_item) and the rotary formula, over seeded
// launches.  Built with AddressSanitizer: every index is checked against exact extents.
//
//   append_rows_emu <seed> <launches>      exits 0 when every launch gives the same bytes
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <random>
#include <vector>

#include "append_row.h"

using namespace vkv;

static std::mt19937 rng;
static unsigned below(unsigned n) { return (unsigned)(rng() % n); }

template <class T>
struct Exact {  // heap block of exactly n values
    T* p;
    explicit Exact(size_t n) : p((T*)aligned_alloc(16, n ? (n * sizeof(T) + 15) / 16 * 16 : 16)) {}
    ~Exact() { free(p); }
};

template <int DT, int SRC>
static int launch_once(int id) {
    const unsigned dims[] = {8, 24, 64, 128};
    const unsigned D = dims[below(4)], H = 1 + below(3), Hq = H * (1 + below(5));
    const unsigned P = DT == VSPEC_KV_F16 ? 16 * (1 + below(3)) : 1 + below(40);
    const unsigned nb = 24, max_blocks = 1 + below(6);
    const bool packed = below(3) == 0;
    const unsigned rows = 1 + below(4);  // block-table rows
    AppendParams p = {};
    p.hkv = H; p.head_dim = D; p.block_tokens = P; p.num_blocks = nb; p.max_blocks = max_blocks;
    // distinct blocks, some entries invalid
    std::vector<int32_t> ids(nb);
    for (unsigned i = 0; i < nb; ++i) ids[i] = (int32_t)i;
    std::shuffle(ids.begin(), ids.end(), rng);
    std::vector<int32_t> tables(rows * max_blocks);
    for (size_t i = 0; i < tables.size(); ++i) tables[i] = below(12) == 0 ? (below(2) ? -1 : (int32_t)nb) : ids[i];
    p.block_tables = tables.data();
    std::vector<int32_t> start, item, pos;
    if (packed) {
        // runs of consecutive positions of a row, distinct over the launch, sometimes shuffled
        std::vector<unsigned> at(rows, 0);
        for (unsigned run = 0; run < 5; ++run) {
            const unsigned b = below(rows);
            at[b] += below(5);
            for (unsigned n = 1 + below(11); n--;) {
                item.push_back(below(30) == 0 ? (int32_t)rows : (int32_t)b);
                pos.push_back((int32_t)at[b]++);
            }
        }
        if (below(3) == 0) {
            const size_t i = below((unsigned)item.size()), j = below((unsigned)item.size());
            std::swap(item[i], item[j]);
            std::swap(pos[i], pos[j]);
        }
        p.batch = (uint32_t)item.size(); p.n_new = 1; p.n_items = rows;
        p.token_item = item.data(); p.token_pos = pos.data();
    } else {
        p.batch = rows; p.n_new = 1 + below(below(2) ? 9 : 70);
        for (unsigned b = 0; b < rows; ++b) start.push_back(below(8) == 0 ? -1 : (int32_t)below(P * max_blocks));
        p.start_pos = start.data();
    }
    const size_t tokens = (size_t)p.batch * p.n_new, n = tokens * H * D;
    Exact<uint8_t> k(n * (SRC == VSPEC_KV_F32 ? 4 : 2)), v(n * (SRC == VSPEC_KV_F32 ? 4 : 2));
    std::normal_distribution<float> normal;
    for (size_t i = 0; i < n; ++i) {
        for (uint8_t* d : {k.p, v.p}) {
            const float x = normal(rng) * (below(50) == 0 ? 1e5f : below(50) == 0 ? 1e-7f : 1.f);
            if (SRC == VSPEC_KV_F32) ((float*)d)[i] = x;
            else ((uint16_t*)d)[i] = (uint16_t)float_to_half_bits(x);
        }
    }
    p.k_new = k.p; p.v_new = v.p;
    const bool rope = !packed && below(2) == 0;
    const unsigned rope_dim = rope ? (below(2) ? D : 2 * (1 + below(D / 2))) : 0;
    const unsigned max_pos = rope ? 1 + below(P * max_blocks + 80) : 0;
    Exact<float> cs(max_pos * (rope_dim / 2)), sn(max_pos * (rope_dim / 2));
    const size_t nq = rope ? tokens * Hq * D : 0;
    Exact<float> q(nq), qo(nq), qw(nq);
    if (rope) {
        for (size_t i = 0; i < (size_t)max_pos * (rope_dim / 2); ++i) { cs.p[i] = normal(rng); sn.p[i] = normal(rng); }
        for (size_t i = 0; i < nq; ++i) { q.p[i] = normal(rng); qo.p[i] = qw.p[i] = 7.f; }
        p.rope_cos = cs.p; p.rope_sin = sn.p; p.rope_dim = rope_dim; p.max_pos = max_pos;
        p.q_in = q.p; p.q_out = qo.p; p.hq = Hq;
    }
    const size_t bytes = (size_t)nb * H * P * D * (DT == VSPEC_KV_F32 ? 4 : 2);
    Exact<uint8_t> k0(bytes), v0(bytes), k1(bytes), v1(bytes);
    for (uint8_t* d : {k0.p, v0.p, k1.p, v1.p}) memset(d, 0x5a, bytes);

    p.k = k0.p; p.v = v0.p; p.rope_vec = false;
    for (uint64_t it = 0, e = append_items<DT>(p); it < e; ++it) append_item<DT, SRC>(p, it);

    p.k = k1.p; p.v = v1.p; p.rope_vec = rope;
    const uint32_t k_items = (uint32_t)(tokens * H * (D / 8));
    const uint32_t v_items = p.batch * append_v_units<DT>(p.n_new, packed) * H * (D / 8);
    std::vector<uint32_t> order(k_items + v_items);
    for (uint32_t i = 0; i < order.size(); ++i) order[i] = i;
    std::shuffle(order.begin(), order.end(), rng);
    for (uint32_t it : order) {
        if (it < k_items) append_k_item<DT, SRC, true>(p, it);
        else append_v_item<DT, SRC, true>(p, it - k_items);
    }
    bool ok = !memcmp(k0.p, k1.p, bytes) && !memcmp(v0.p, v1.p, bytes);
    if (rope && rope_dim % 8 == 0) {
        const uint32_t qi = (uint32_t)tokens * ((Hq + kRopeHeads - 1) / kRopeHeads) * rope_q_chunks(D, rope_dim);
        for (uint32_t it = 0; it < qi; ++it) rope_q_item(p, it);
        const unsigned half = rope_dim / 2;
        for (size_t r = 0; r < tokens * Hq; ++r) {
            const size_t t = r / Hq;
            const int32_t sp = start[t / p.n_new];
            const unsigned at = (unsigned)sp + (unsigned)(t % p.n_new);
            if (sp < 0 || at >= max_pos) continue;
            const float *x = q.p + r * D, *c = cs.p + (size_t)at * half, *s = sn.p + (size_t)at * half;
            float* o = qw.p + r * D;
            for (unsigned d = 0; d < D; ++d) {
#pragma clang fp contract(off)
                if (d < half) o[d] = x[d] * c[d] - x[d + half] * s[d];
                else if (d < rope_dim) o[d] = x[d - half] * s[d - half] + x[d] * c[d - half];
                else o[d] = x[d];
            }
        }
        ok = ok && !memcmp(qo.p, qw.p, nq * 4);
    }
    if (!ok) fprintf(stderr, "launch %d differs: DT %d SRC %d D %u P %u H %u packed %d rope_dim %u max_pos %u\n", id, DT, SRC, D, P, H, packed, rope_dim, max_pos);
    return ok ? 0 : 1;
}

int main(int argc, char** argv) {
    if (argc != 3) return 2;
    rng.seed((unsigned)atoi(argv[1]));
    int bad = 0;
    for (int i = 0, n = atoi(argv[2]); i < n; ++i) {
        switch (i % 4) {
            case 0: bad += launch_once<VSPEC_KV_F16, VSPEC_KV_F16>(i); break;
            case 1: bad += launch_once<VSPEC_KV_F16, VSPEC_KV_F32>(i); break;
            case 2: bad += launch_once<VSPEC_KV_F32, VSPEC_KV_F16>(i); break;
            default: bad += launch_once<VSPEC_KV_F32, VSPEC_KV_F32>(i); break;
        }
    }
    return bad ? 1 : 0;
}
