// Check: psk::used_splits and split_pages (phaseshift_amd/csrc/split_units.h)
// equal 64-bit arithmetic at the ends of their ranges, and the split indexes
// that the combine clamps to used - 1 stay inside a row's partials.
#include <cstdio>
#include <vector>
#include "split_units.h"

int main() {
    const uint64_t top = uint64_t{1} << 32;
    const std::vector<uint32_t> page{1u, 16u, 24u, 65536u, 0x80000000u, 0xFFFFFFFFu};
    const std::vector<uint32_t> splits{1u, 2u, 7u, 64u, 1024u};
    const std::vector<uint32_t> pps{0u, 1u, 3u, 16384u, 0x80000000u, 0xFFFFFFFFu};
    uint64_t bad = 0, skipped = 0, checked = 0;
    for (uint32_t P : page)
        for (uint64_t stride : {uint64_t{1}, uint64_t{5}, uint64_t{65536}, top / P, top - 1}) {
            if (stride == 0) continue;
            const uint64_t cap = (uint64_t)(uint32_t)stride * P;
            std::vector<uint64_t> pos;
            for (uint64_t edge : {uint64_t{0}, (uint64_t)P, cap, top - P, top, top / 2})
                for (int64_t d = -3; d <= 3; ++d) pos.push_back(edge + (uint64_t)d);
            for (uint64_t q : pos) {
                if (q >= top) continue;
                for (uint32_t s : splits)
                    for (uint32_t n : pps) {
                        const uint64_t vis = q + 1u, pc = (vis + P - 1u) / P;
                        uint64_t want = 0;
                        if (vis <= cap && vis + P - 1u < top) {
                            const uint64_t per = n != 0u ? n : (pc + s - 1u) / s;
                            want = (pc + per - 1u) / per;
                            if (want > s) want = s;
                            if (psk::split_pages((uint32_t)pc, s, n) != per) ++bad;
                        }
                        const uint32_t got = psk::used_splits((uint32_t)q, cap, P, s, n);
                        skipped += got == 0u;
                        ++checked;
                        bool ok = got == want;
                        // the combine's lanes read split min(lane, used - 1) of a row that is not skipped
                        for (uint32_t lane : {0u, 1u, 63u, 255u, 1087u})
                            if (got != 0u && (lane < got - 1u ? lane : got - 1u) >= s) ok = false;
                        if (!ok && bad++ < 10)
                            std::printf("pos %llu page %u cap %llu splits %u pps %u: %u, want %llu\n",
                                        (unsigned long long)q, P, (unsigned long long)cap, s, n, got,
                                        (unsigned long long)want);
                    }
            }
        }
    std::printf("checked %llu skipped %llu mismatches %llu\n", (unsigned long long)checked,
                (unsigned long long)skipped, (unsigned long long)bad);
    return bad != 0 || skipped == 0;
}
