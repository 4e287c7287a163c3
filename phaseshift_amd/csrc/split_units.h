// How split-K launches divide one row's pages, for the attention and combine
// kernels alike: both must agree on which splits hold partials. Plain C++
// (constexpr functions are host and device functions in HIP), so the CPU tests
// check these rules at the ends of the 32-bit range.
#pragma once
#include <cstdint>

namespace psk {

// Pages of one split of a row of pc >= 1 pages; pps: pages_per_split, 0 for
// ceil(pc / splits). At least 1.
constexpr uint32_t split_pages(uint32_t pc, uint32_t splits, uint32_t pps) {
    return pps != 0u ? pps : (pc - 1u) / splits + 1u;
}

// Splits that hold pages of a row of pc pages (0 without pages).
constexpr uint32_t splits_of_pages(uint32_t pc, uint32_t splits, uint32_t pps) {
    if (pc == 0u) return 0u;
    const uint32_t used = (pc - 1u) / split_pages(pc, splits, pps) + 1u;
    return used < splits ? used : splits;
}

// The same for a row at position pos under a block table of `capacity`
// tokens: 0 for a row that the kernels skip, because its pos + 1 tokens pass
// the block table or end in the last page below 2^32 (its page count does not
// come out of 32-bit arithmetic). A skipped row has no partials: the combine
// must not read any.
constexpr uint32_t used_splits(uint32_t pos, uint64_t capacity, uint32_t page_tokens, uint32_t splits,
                               uint32_t pps) {
    const uint64_t visible = (uint64_t)pos + 1u;
    if (visible > capacity || visible + page_tokens - 1u > 0xFFFFFFFFull) return 0u;
    return splits_of_pages(((uint32_t)visible + page_tokens - 1u) / page_tokens, splits, pps);
}

}  // namespace psk
