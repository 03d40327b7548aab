// dsx_q8_0_rules.hpp -- which kernels take the products of Q8_0 matrices, by sizes alone (host code).
//
// Figures: us, on one MI355X; old: the by-expert kernels below 1.5 picks per expert and the 128-column int8 GEMM from there
// on, before these rules (that GEMM 3 to 12 % slower than it is now).  "same picks": every token names the same experts.
// Taken with the int8 GEMM of that time, 2 to 10 % slower in all tiles than since its scales come in segments (k_q8_0_gemm), but
// for q8_gate_up_columns.
#pragma once
#include <stdint.h>

namespace dsx {

constexpr uint32_t kQ8StreamMembers = 16;   // members of a streaming work item (dsx_stream_kernels.hpp)
// columns of the int8 GEMM's tiles (k_q8_0_gemm), rows of them all
constexpr uint32_t kQgCols = 128, kQgColsMiddle = 64, kQgColsNarrow = 32, kQgRows = 64;

struct Q8Shape {
    uint32_t hidden, inter, n_expert, n_used;
    uint64_t elements() const { return (uint64_t)hidden * inter; }
    // fewer than halves / 2 picks per expert at T tokens
    bool picks_below_halves(uint32_t T, uint32_t halves) const { return 2u * (uint64_t)T * n_used < (uint64_t)n_expert * halves; }
};

// Whether both products of an all-Q8_0 layer run on the streaming kernels: below 1.5 picks per expert, where the
// by-expert kernels are the other path (2048 x 1408, 64 experts, top-6, old / streaming: 4 tokens 75 / 61, 8: 103 / 82;
// 4096 x 1536, 128 experts, top-8: 2: 100 / 89, 16: 359 / 316; 2560 x 1792, 96 experts, top-4: 16: 185 / 163; 1024 x
// 512, 64 experts, top-4: 16: 60 / 43), and to below 4 where the other path is the 32-column GEMM (old / streaming /
// GEMM: 2048 x 1408: 16 tokens 137 / 114 / 122, 24: 147 / 129 / 133, 32: 151 / 133 / 136; 4096 x 1536: 32: 496 / 428 /
// 444, 48: 535 / 469 / 490; 4096 x 1024, 128 experts, top-8: 48: 369 / 320 / 340; 2560 x 1792: 48: 305 / 261 / 293, 64:
// 338 / 287 / 315) -- but not with matrices of up to 2 M elements: a workgroup has too few row tiles to stream (512 x
// 2048, 64 experts, top-4: 24: 58 / 74 / 50, 48: 68 / 87 / 56; 512 x 4096, 32 experts, top-4: 16: 67 / 82 / 58; 1024 x
// 512, 128 experts, top-8: 32: 63 / 70 / 57; 2048 x 768, 128 experts, top-8: 32: 151 / 139 / 133).
inline bool q8_all_streams(const Q8Shape &s, uint32_t T) {
    return T >= 2u && s.picks_below_halves(T, s.elements() > (2ull << 20) ? 8u : 3u);
}

// Whether the device chooses between streaming and the 32-column GEMM (StreamChoice): from 1.5 picks per expert on, for
// more tokens than one item holds.  Where tokens share experts the GEMM reads these fewer times (same picks, old /
// streaming / GEMM / both launched: 3072 x 2048, 64 experts, top-4: 24 tokens 66 / 70 / 55 / 60, 48: 77 / 89 / 62 / 65;
// 2560 x 1792: 64: 79 / 90 / 65 / 71), but the two launches that return at once take 5 us (spread picks, streaming /
// both launched: 3072 x 2048: 48: 262 / 268; 2560 x 1792: 64: 283 / 290).  Layers of under 256 M elements in a kind of
// matrix stream whatever the picks: they would lose more on spread ones (2048 x 1408: 24 tokens 131 / 136, 40: 143 /
// 149) than they do on the same ones (old / streaming 24: 52 / 53, 32: 53 / 55, 40: 60 / 61).
inline bool q8_stream_choice(const Q8Shape &s, uint32_t T) {
    return T > kQ8StreamMembers && !s.picks_below_halves(T, 3u) && s.n_expert * s.elements() >= (256ull << 20);
}

// Columns per work item of the int8 GEMMs of T tokens on n_cu CUs.
//
// Narrow: few members per expert.  An item reads its rows of the weights whatever its members, so that an expert which
// every token names is read T / 32 times: over 256 tokens the middle tile (64: down in 64 columns, gate/up in 128) is
// no slower on spread picks and much faster on the same ones (all-Q8_0 layer, spread / same picks, old; narrow; middle:
// 7168 x 2048, 256 experts, top-8: 256 tokens 2546 / 609; 2397 / 599; 2385 / 471, 512: 2753 / 937; 2613 / 1180; 2564 /
// 769, 768: 3271 / 1283; 2884 / 1780; 2847 / 1138; 5120 x 1536, 160 experts, top-6: 512: 1027 / 446; 987 / 480; 946 /
// 360; 3072 x 2048, 64 experts, top-4: 384: 360 / 194; 354 / 213; 338 / 160; MXFP4 gate/up, 7168 x 2048: 512: 1882 / -;
// 1747 / 612; 1746 / 533).  Up to 2 M elements it stays the faster one (2048 x 768, 128 experts, top-8: 384 tokens 217
// / 127; 190 / 98; 194 / 107).  It ends at 28 picks per expert (4096 x 1536, 128 experts, top-8, 24: narrow 656 /
// middle 633, 32: 773 / 679; 2048 x 1408, 64 experts, top-6, 24: 185 / 184, 36: 238 / 202), at 42 on up to 16 experts
// whose down product makes less than a round of three workgroups per CU, of which an item more or less per expert is a
// large part (4096 x 14336, 8 experts, top-2, 32 picks: old 705, narrow 584, middle 650, wide 610; MXFP4 gate/up: 528,
// 482, 551, 503; but 1024 x 2048, 32 experts, top-4, 32: 110, 92, 88; 512 x 2048, 64 experts, 40: 122, 111, 96).
//
// Middle: to 42 picks per expert, 56 where down makes eight rounds and more of three workgroups per CU (us per layer,
// wide / middle: 7168 x 2048, 256 experts, MXFP4 gate/up, 1000 tokens [31 picks per expert] 2349 / 2143, 1700 [53] 2723
// / 2504, 2100 [66: most experts make two items] 2906 / 2999; all-Q8_0 2048 x 1408, 64 experts: 300 tokens [28] 196 /
// 191, 420 [39] 220 / 214, 512 [48] 234 / 239, 700 [66] 265 / 277: its 2048 workgroups are then four full rounds of the
// wide tile's two per CU, but 2.7 of the middle one's three; 4096 x 1536, 128 experts, 48: 830 / 815; layers of four
// and five rounds would gain at 48 as well: 3072 x 2048, 64 experts, top-4: 468 / 444, 2048 x 768, 128 experts: 253 /
// 247).
inline uint32_t q8_gemm_columns(const Q8Shape &s, uint32_t T, uint32_t n_cu) {
    const uint64_t workgroups = (uint64_t)s.n_expert * (s.hidden / kQgRows);   // down's, a work item per expert
    const uint32_t narrow = s.n_expert <= 16u && workgroups < 3u * n_cu ? 84u : 56u;
    if ((T <= 256u || s.elements() <= (2ull << 20)) && s.picks_below_halves(T, narrow)) return kQgColsNarrow;
    return s.picks_below_halves(T, workgroups >= 24u * n_cu ? 112u : 84u) ? kQgColsMiddle : kQgCols;
}

// The same for gate/up of an all-Q8_0 layer whose down product has `down` columns by the above; down takes no more than
// gate/up.  64 between the narrow tile's end and 60 picks per expert, where experts begin to make two items (us per layer, gate/up
// and down in 128 and 64 or 128 columns, the better of the two / both in 64: 2048 x 1408, 64 experts, top-6: 300 tokens
// [28 picks] 187 / 179, 512 [48] 222 / 212, 600 [56] 243 / 240, 700 [66] 267 / 284; 4096 x 1536, 128, top-8: 400 [25] 617 /
// 605, 768 [48] 804 / 758, 900 [56] 884 / 846, 1200 [75] 1021 / 1198; 3072 x 2048, 64, top-4: 450 [28] 345 / 339, 900 [56] 525 /
// 468, 1100 [69] 604 / 591; 2048 x 768, 128, top-8: 512 [32] 205 / 200, 900 [56] 272 / 259, 1200 [75] 319 / 350; 1024 x 2048,
// 32, top-4: 300 [38] 102 / 92, 600 [75] 144 / 147; 4096 x 14336, 8, top-2: 192 [48] 835 / 664; 7168 x 2048, 256, top-8: 1000 [31]
// 3124 / 2835, 2000 [63] 4352 / 4284).
inline uint32_t q8_gate_up_columns(const Q8Shape &s, uint32_t T, uint32_t down) {
    return down == kQgColsNarrow ? down : s.picks_below_halves(T, 120u) ? kQgColsMiddle : kQgCols;
}

// Whether gate/up's launch in 64 columns takes the list of 128-column items after all (on the device, by the items that the picks make):
// where few experts are hot, 64 columns cut their groups into up to twice as many items.  A round of resident workgroups takes about three
// fifths as long with 64 columns (three rounds beat two of 128, seven lose to four).  us per layer, 128 / 64 columns (items,
// rounds): 4096 x 1536, 128 experts, top-8, 900 tokens on 32 experts (72, 4 / 143, 7) 650 / 688; 3072 x 2048, 64, top-4, 900 tokens on the
// same picks (40, 3 / 75, 5) 364 / 377; 7168 x 2048, 256, top-8, 1000 on 64 experts 1766 / 1828; but 4096 x 1536, 300, same (27, 2 /
// 45, 3) 293 / 256; 2048 x 1408, 64, top-6, 512, same (28, 2 / 56, 3) 163, with older scale loads, / 151.  The number of items is asked
// as well because a few items more can make a round, which is not a full one.  Spread picks keep their 64 columns, Zipf-skewed ones were as
// fast (4096 x 1536, 900 tokens 866 / 870; 2048 x 1408, 512: 220 / 220).  The choice costs passes that keep 64 columns up to 1 % (253 / 255).
constexpr bool q8_takes_wide_items(uint32_t middle, uint32_t wide, uint32_t row_tiles, uint32_t slots) {
    const uint32_t rounds_middle = (middle * row_tiles + slots - 1u) / slots, rounds_wide = (wide * row_tiles + slots - 1u) / slots;
    return 5u * middle >= 7u * wide && 5u * rounds_wide <= 3u * rounds_middle;
}

// Columns per work item of a dense Q8_0 expert of b tokens (dsx_dense_ffn; both products, one list): 32 where the wide
// tile would leave workgroup slots empty in gate/up (two per CU) -- over 128 tokens unless the items, each of which
// reads gate and up whole, come to about a gigabyte of reads, in brackets (us, wide / narrow: 7168 x 2048: 96 tokens
// 162 / 84, 512 [0.5] 203 / 129, 768 [0.75] 203 / 194, 1000 [1.0] 204 / 269, 1900 [1.9] 328 / 514; 7168 x 3072: 512
// [0.75] 297 / 197, 640 [0.94] 299 / 291, 1000 [1.5] 301 / 401; 5120 x 1536: 1500 [0.79] 218 / 194, 1900 [1.0] 222 /
// 256; 7168 x 512: 3000 [0.73] 204 / 181, 4096 [1.0] 230 / 238; 2048 x 1408: 1900 [0.37] 98 / 94; 7168 x 18432: 128
// [1.1] 1366 / 624).
inline uint32_t q8_dense_columns(uint32_t hidden, uint32_t inter, uint32_t b, uint32_t n_cu) {
    const uint64_t wide = (uint64_t)((b + kQgCols - 1u) / kQgCols) * (inter / kQgRows);
    const uint64_t item = 2u * (uint64_t)hidden * inter / 32u * 34u;
    const bool few_reads = b <= kQgCols || (b + kQgColsNarrow - 1u) / kQgColsNarrow * item < 950000000u;
    return wide < 2u * n_cu && few_reads ? kQgColsNarrow : kQgCols;
}

}  // namespace dsx
