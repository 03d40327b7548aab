// dsx_q8_0_rules.hpp -- which kernels take the products of Q8_0 matrices, by sizes alone (host code).
//
// Figures: us, on one MI355X; old: the by-expert kernels below 1.5 picks per expert and the 128-column int8 GEMM from
// there on, with which layers began.  "same picks": every token names the same experts.
#pragma once
#include <stdint.h>

namespace dsx {

constexpr uint32_t kQ8StreamMembers = 16;   // members of a streaming work item (dsx_stream_kernels.hpp)

struct Q8Shape {
    uint32_t hidden, inter, n_expert, n_used;
    uint64_t elements() const { return (uint64_t)hidden * inter; }
    // T tokens make fewer than `per_expert` halves of a pick per expert
    bool picks_below_halves(uint32_t T, uint32_t per_expert) const { return 2u * (uint64_t)T * n_used < (uint64_t)n_expert * per_expert; }
};

// Whether both products of an all-Q8_0 layer run on the streaming kernels: below 1.5 picks per expert, where the by-expert
// kernels are the other path (2048 x 1408, 64 experts, top-6, old / streaming: 4 tokens 75 / 61, 8: 103 / 82; 4096 x 1536, 128
// experts, top-8: 2: 100 / 89, 16: 359 / 316; 2560 x 1792, 96 experts, top-4: 16: 185 / 163; 1024 x 512, 64 experts, top-4: 16: 60 /
// 43), and to below 4 where the other path is the 32-column GEMM (old / streaming / GEMM: 2048 x 1408: 16 tokens 137 / 114 / 122,
// 24: 147 / 129 / 133, 32: 151 / 133 / 136; 4096 x 1536: 32: 496 / 428 / 444, 48: 535 / 469 / 490; 4096 x 1024, 128 experts, top-8:
// 48: 369 / 320 / 340; 2560 x 1792: 48: 305 / 261 / 293, 64: 338 / 287 / 315) -- but not with matrices of up to 2 M elements: a
// workgroup has too few row tiles to stream (512 x 2048, 64 experts, top-4: 24: 58 / 74 / 50, 48: 68 / 87 / 56; 512 x 4096, 32
// experts, top-4: 16: 67 / 82 / 58; 1024 x 512, 128 experts, top-8: 32: 63 / 70 / 57; 2048 x 768, 128 experts, top-8: 32: 151 / 139 / 133).
inline bool q8_all_streams(const Q8Shape &s, uint32_t T) {
    return T >= 2u && s.picks_below_halves(T, s.elements() > (2ull << 20) ? 8u : 3u);
}

// Whether the device chooses between streaming and the 32-column GEMM (StreamChoice): from 1.5 picks per expert on, for more
// tokens than one item holds.  Where tokens share experts the GEMM reads these fewer times (same picks, old / streaming / GEMM /
// both launched: 3072 x 2048, 64 experts, top-4: 24 tokens 66 / 70 / 55 / 60, 48: 77 / 89 / 62 / 65; 2560 x 1792: 64: 79 / 90 /
// 65 / 71), but the two launches that return at once take 5 us (spread picks, streaming / both launched: 3072 x 2048: 48: 262 / 268;
// 2560 x 1792: 64: 283 / 290).  Layers of under 256 M elements in a kind of matrix stream whatever the picks: they would lose more on spread
// ones (2048 x 1408: 24 tokens 131 / 136, 40: 143 / 149) than they do on the same ones (old / streaming 24: 52 / 53, 32: 53 / 55, 40: 60 / 61).
inline bool q8_stream_choice(const Q8Shape &s, uint32_t T) {
    return T > kQ8StreamMembers && !s.picks_below_halves(T, 3u) && s.n_expert * s.elements() >= (256ull << 20);
}

}  // namespace dsx
