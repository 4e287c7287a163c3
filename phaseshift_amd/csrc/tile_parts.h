// Which tile launches run in two parts: a tile's even and odd 32-token chunks
// on two waves per head, joined in LDS, and how many heads one workgroup
// takes. Plain C++ (the launchers call it, the CPU tests hold it against
// measured times of both kernels).
#pragma once
#include <cstdint>

namespace psk {

// A two-part launch's tiles of up to this many tokens run as one part: joining
// the parts costs 1-2 us, about what splitting 8 chunks gains (FP8, 24/4 heads,
// 6 per workgroup, 128 rows without context 15.1 us, in two parts 16.3; 512
// rows 29.6 and 27.2).
constexpr uint32_t kTwoPartTokens = 256;

struct TileShape {
    uint32_t head_dim;
    uint32_t q_per_kv;
    uint32_t kv_heads;
    bool psq;
    bool bf16;
};

// Heads per workgroup of an unsplit launch of implicit tiles (the prefill
// launchers) of `rows` rows on `cus` CUs, 0 for one part.
//
// Such a launch has only tiles x kv_heads workgroups (units) and no scratch to
// split K over, and its waves are bound by instruction issue: 5-6 one-head
// waves load two of the four SIMDs twice, and up to 256 workgroups leave the
// rest of the chip idle. In two parts 6 heads put 3 waves on every SIMD; where
// the tiles alone do not reach the CUs the heads go to workgroups of 4 or 2.
// Launcher times, one part -> two (us, 24/4 heads of 256; rows + context):
//   FP8   48+0 12.5 -> 9.4 (2 heads)      BF16  128+1024 55.6 -> 42.8 (2)
//   FP8   512+4096 166 -> 111 (4; 6: 122) PSQ4  512+4096 218 -> 172 (4; 6: 192)
//   FP8   700+1024 69.3 -> 55.7 (6; 4: 81) PSQ8 1024+2048 157 -> 129 (6; 4: 207)
//   FP8   2048+2048 262 -> 199 (6)        BF16  2048+0 154 -> 127 (6)
// so the smallest workgroups that stay within one per CU win, then all heads.
// A PSQ workgroup dequantizes for all its heads, so 2 of them pay only on a
// nearly empty chip (8/1 heads of 128, PSQ8 128+1024: 4 heads 33.1, 2 34.9;
// 48+0: 8.9 and 8.3).
//
// Where two parts lose (times one part -> two as above; the lines lie where
// the sign changes in the recorded times that the tests hold):
// - Few heads over a short range: the launch does not know its context, but more
//   than kTwoPartTokens rows always reach past it. Up to 2 heads 128+0 1.03-1.08x
//   slower, 17+0 up to 1.19x (PSQ4, 8/4 heads of 256), the same for 3 (PSQ) and
//   up to 4 (heads of 32 and 64); PSQ with 4 heads loses on 17 rows, and with
//   5, dequantized by workgroups of 4 and 1, on 128+0 (PSQ4 1.05x). PSQ with 4 heads
//   of 256 on 33-256 rows takes pairs, also past a quarter of the CUs (PSQ4 16/4
//   heads: 140+0 17.7 -> 18.6, in fours 19.8; 140+333 32.9 -> 29.6, 31.4;
//   140+2900 150 -> 118, 119): it loses up to 7% without context and gains
//   6-25% from 256 tokens of it, so two parts stay.
// - The 16-wave workgroups of 7-8 heads start slower: 64/8 heads of 128, 260+0
//   FP8 16.6 -> 18.5, BF16 16.3 -> 17.8, PSQ8 290+0 21.3 -> 22.6; level from 400 rows
//   (PSQ, BF16) and 520 (FP8); of 64, FP8 800+0 24.2 -> 25.1, level at 1000.
// - BF16 heads of 128 in groups of 1-2, just below three workgroups per CU (16/8
//   heads, 1500 rows: +0 60.5 -> 57.9, +1000 109 -> 113, +2900 199 -> 214; at 2.65
//   and 3.05 per CU two parts gain 2-9%, and so they do at 2.97 on 4 KV heads, whose
//   3036 rows differ more in length).
// - Beyond one workgroup per CU. PSQ with 1-2 heads dequantizes for half the
//   waves (8/8 heads of 256, 4000+0: PSQ4 522 -> 696; of 128, where a CU holds
//   two, past 2 per CU 249 -> 295). 3-4 heads gain only in BF16 at 256 (16/4
//   heads 2060+2048 392 -> 340; FP8 2048+2048 156 -> 171). 5-6 heads gain at 256 in every
//   format, at 128 in BF16 and FP8 (24/4 heads 4000+0 0.84-0.86x; 5 heads lose
//   2-4% between one and three workgroups per CU), in FP8 at 64 up to two per CU
//   (20/4 heads 2040+0 0.97x, 2060+2048 1.07x) and in BF16 at 32; PSQ at 128
//   (24/8 heads 1024+1024 1.03-1.06x, 4000+0 1.13-1.16x) and BF16 at 64 (24/8
//   heads 1.02-1.11x) lose. 7-8 heads lose (32/4 heads of 128, PSQ 1.04-1.13x).
// 16 waves (7-8 heads) need 128 registers a wave: head_dim <= 128.
constexpr uint32_t implicit_part_heads(const TileShape& s, uint64_t rows, uint64_t cus) {
    const uint32_t q = s.q_per_kv, D = s.head_dim;
    const uint64_t units = (rows + 15u) / 16u * s.kv_heads;
    const bool few = q <= 2u || (s.psq ? q == 3u : q <= 4u && D <= 64u);
    if (rows <= (few ? kTwoPartTokens : s.psq && q == 4u ? 32u : 0u)) return 0u;
    if (q <= 2u && s.bf16 && D == 128u && rows < 2048u && 10u * units > 27u * cus && units <= 3u * cus)
        return 0u;
    if (q <= 2u) return !s.psq || units <= (D == 256u ? cus : 2u * cus) ? 2u : 0u;
    const bool pairs = !s.psq || (q == 4u && D == 256u && rows <= kTwoPartTokens);
    if (units * ((q + 1u) / 2u) <= (pairs ? cus : cus / 4u)) return 2u;
    if (s.psq && q == 5u && rows <= kTwoPartTokens) return 0u;
    if (units * ((q + 3u) / 4u) <= cus) return 4u;
    if (q == 5u || q == 6u) {
        const bool gains = D == 256u || units <= cus ||
                           (!s.psq && (D == 128u ? q == 6u || units > 3u * cus
                                                 : s.bf16 ? D == 32u : units <= 2u * cus));
        return gains ? 6u : 0u;
    }
    if (q <= 4u) return units <= cus || (D == 256u && s.bf16) ? 4u : 0u;
    return units <= cus && D < 256u && rows > (D <= 64u ? 896u : s.psq || s.bf16 ? 384u : 512u) ? 8u : 0u;
}

// The same for explicit tiles (verify blocks) and split launches: 6 for 5-6
// heads, 0 otherwise. range: most tokens a workgroup reads (a split's, or the
// longest visible range); units: workgroups with work.
//
// Whole verify calls repeated on the same buffers, whose K/V the last-level
// cache then holds (us, 24/4 heads of 256, one part -> two): FP8 8 blocks of 16
// rows over 2-16k tokens 56.3 -> 52.5, 32 over 2-8k 165 -> 157; unsplit, 16 of 12
// rows over 256-2000 tokens 79.2 -> 63.1; BF16 61.7 -> 59.4, 221 -> 214. With K/V
// read from HBM (600 MB of other reads before each call; call times with their
// launch) the first gains 63.3 -> 61.4, 32 FP8 blocks over 1.6-6.8k 119.6 -> 110.2
// (cached 116.6 -> 101.4), 17 BF16 blocks of 14 rows over 424-1594 86.8 -> 75.8,
// and of 43 drawn verify calls none is slower by more than 1.3%, what calls of
// the same kernel differ by. Over short ranges the second half
// of the waves only costs its start: 8 blocks over 252 tokens 20.5 -> 22.3, 256
// over 76 63.1 -> 71.6, and ranges up to 320 gain nothing (BF16 1.00-1.02x).
// Other group sizes stay one part: they were not measured in two here.
// Heads below 256 leave room for several one-part workgroups on a CU: two parts
// lose beyond one workgroup per CU (24/4 heads of 128, 128 blocks over 516
// tokens, FP8 37.5 -> 44.5; at 32 past two per CU) and on splits up to 512 tokens
// (16 blocks over 0.3-4k, 368 a split: 1.06-1.12x). PSQ gains from splits past
// 512 tokens (PSQ4 32 blocks 211 -> 199; 272 tokens lose 3 us of 32-41);
// unsplit its 8 one-part waves share the dequantization.
constexpr uint32_t explicit_part_heads(const TileShape& s, bool split, uint64_t range, uint64_t units,
                                       uint64_t cus) {
    if (s.q_per_kv != 5u && s.q_per_kv != 6u) return 0u;
    if (s.psq && !split) return 0u;
    const bool wide = s.head_dim == 256u;
    if (range <= (s.psq || (split && !wide) ? 2u * kTwoPartTokens : kTwoPartTokens + 64u)) return 0u;
    return wide || units <= (s.head_dim == 32u ? 2u * cus : cus) ? 6u : 0u;
}

}  // namespace psk
