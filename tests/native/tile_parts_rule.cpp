// Prints what psk::implicit_part_heads and explicit_part_heads
// (phaseshift_amd/csrc/tile_parts.h) answer for the launches on stdin, on 256
// CUs: "i psq bf16 head_dim q_per_kv kv_heads rows" or
// "e psq bf16 head_dim q_per_kv kv_heads split range units".
#include <cstdio>
#include "tile_parts.h"

int main() {
    char kind;
    unsigned psq, bf16;
    psk::TileShape s{};
    while (std::scanf(" %c %u %u %u %u %u", &kind, &psq, &bf16, &s.head_dim, &s.q_per_kv, &s.kv_heads) == 6) {
        s.psq = psq != 0;
        s.bf16 = bf16 != 0;
        unsigned long long a, b;
        unsigned split;
        if (kind == 'i' && std::scanf("%llu", &a) == 1)
            std::printf("%u\n", psk::implicit_part_heads(s, a, 256));
        else if (kind == 'e' && std::scanf("%u %llu %llu", &split, &a, &b) == 3)
            std::printf("%u\n", psk::explicit_part_heads(s, split != 0, a, b, 256));
        else
            return 1;
    }
    return 0;
}
