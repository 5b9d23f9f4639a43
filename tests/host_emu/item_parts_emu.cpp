// Host check of the item split's arithmetic (kv_common.h part_range): the parts of an item are
// runs of tiles that follow each other from 0 to U and differ by one tile at most, or all but the
// last have the size that the caller gave.
#include <random>

#include "kv_common.h"

using namespace vkv;

static int check(const DecodeParams& p, uint32_t U) {
    const int n = item_parts_of(p, (int)U);
    int at = 0, least = 0x7fffffff, most = 0;
    for (uint32_t part = 0; part < p.item_parts; ++part) {
        int lo, hi;
        part_range<true>(p, part, U, lo, hi);
        if ((int)part >= n) {
            if (lo < hi) return printf("U %u: part %u of %d is not empty\n", U, part, n), 1;
            continue;
        }
        if (lo != at || hi <= lo) return printf("U %u, %d parts: part %u is [%d, %d) after %d\n", U, n, part, lo, hi, at), 1;
        least = hi - lo < least ? hi - lo : least;
        most = hi - lo > most ? hi - lo : most;
        at = hi;
    }
    if (p.chunk_tiles) {
        if (at != (int)U || n != (int)((U - 1) / p.chunk_tiles + 1) || (n > 1 && most != (int)p.chunk_tiles))
            return printf("U %u, chunks of %u: %d parts, end %d, longest %d\n", U, p.chunk_tiles, n, at, most), 1;
        return 0;
    }
    if (at != (int)U || most - least > 1) return printf("U %u, %d parts: end %d, %d to %d tiles\n", U, n, at, least, most), 1;
    return 0;
}

int main() {
    std::mt19937 rng(1);
    DecodeParams p = {};
    p.far_tiles = 0x40000000u;
    // up to the 2^27 tiles of 2^31 tokens, few and many parts
    for (uint32_t U : {1u, 2u, 3u, 4u, 5u, 63u, 64u, 65u, 4097u, 65536u, 131071u, 131072u, 131073u, 262145u, 1u << 22, (1u << 27) - 1, 1u << 27}) {
        for (uint32_t parts : {1u, 2u, 3u, 5u, 64u, 128u, 32768u, 65537u}) {
            for (uint32_t tiles : {1u, 4u, 8u, 33u}) {
                p.item_parts = parts;
                p.part_tiles = tiles;
                p.near_parts = rng() % 2 ? 0x7fffffffu : 1 + rng() % 100;
                if (check(p, U)) return 1;
            }
        }
    }
    // parts of a given size, of an item up to as long as the longest one
    p.near_parts = 0x7fffffffu;
    for (uint32_t chunk : {1u, 3u, 4u, 32u, 512u, 100000u, 1u << 27}) {
        p.chunk_tiles = p.part_tiles = chunk;
        for (uint32_t most : {1u, 33u, 2064u, 131072u, 262145u}) {
            p.item_parts = (most + chunk - 1) / chunk;
            for (uint32_t U : {1u, 2u, 32u, 33u, 129u, most / 2 + 1, most}) {
                if (U <= most && check(p, U)) return 1;
            }
        }
    }
    return 0;
}
