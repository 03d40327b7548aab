// dsx_stream_kernels.hpp -- expert products for groups of up to 32 members (MXFP4) or 16 (Q8_0): what these read is
// weights, and they read them as whole row tiles.
//
// A tile of 16 of the engine's rows is one contiguous stretch of 16 n_sb 136 bytes (a super-block of 256 MXFP4
// values, four blocks of 32 Q8_0 values).  A workgroup (8 waves, one per CU: it takes nearly all of the LDS; for some Q8_0
// rows 4 waves, two per CU: with_q8_stream_kernel) streams such stretches through a ring of LDS stages with LDS-direct loads, so that every cache line is requested
// once and 60-120 KB per CU are under way at any time; what differs from the grouped GEMM
// (dsx_gemm_kernels.hpp), which walks 512 rows in step and asks for 136 bytes of each at a time (two
// lines for 1.06 lines' worth, and every step waits for its own loads).
//
// The roles of the operands are swapped for that: the columns stay, the weights pass.  MXFP4: the eight waves
// split k by half super-blocks -- wave w takes half w % 2 of super-blocks w / 2, w / 2 + 4, .. -- and
// hold the columns' operands of their share in registers for as long as the work item (expert, up to
// 16 NCG members) lasts.  Of a tile they each multiply their share, and the eight partial sums per
// result meet in LDS, added in wave order.
//
// The work, (items) x (row tiles), is cut into one contiguous range per workgroup, so that a workgroup
// changes its item only once or twice.
//
// Q8_0: of W waves, wave w takes every W-th group of four blocks.  Against the by-expert kernels and the 128-column int8
// GEMM (whole layers: dsx_q8_0_rules.hpp), us: 2048 x 1408, 64 experts, top-6, gate/up + down: 4 tokens 35 + 26 / 30 + 19, 16: 70 + 49 / 63 + 36; 7168
// x 2048, 256 experts, down, 16 tokens: 413 / 298.  32 and 64 columns per item lost to the int8 GEMM's narrow tile (512
// tokens, down 7168 x 2048, 32 columns: 915 / 870): a stage's products, sums and two barriers then outlast its loads.
//
// MXFP4: bound by the weight stream.  Every line of a group's weights is asked for once per item, whole and by one instruction
// (but the ends of a unit), so the loads of a group that is one item are non-temporal: whole layers, us with ordinary loads /
// with these: 7168 x 2048, 256 experts, top-8: 16 tokens 478 / 421, 100: 1096 / 963; 4096 x 1024, 128 experts, 37 tokens 182 /
// 158; all-Q8_0 2048 x 1408: 4 tokens 65.6 / 59.2, 40: 149 / 131.  The items of one group find each other's lines in the L2
// (non-temporal throughout / there not: 7168 x 2048, every token on the same picks: 100 tokens 272 / 234, 40: 143 / 132; gate/up beside
// a Q8_0 down matrix, same picks, 60: 215 / 200).  The kind of load is chosen once per stage: a branch beside every load delays
// the stage's requests (same picks, 100: 254, 40: 138; 2560 x 2048, 96 experts, 95 tokens 216 / 205; 2048 x 1536, 64, 24: 84.0 / 79.5).  The
// workgroups of one launch end within 5 % of each other at 64 tokens and 10 % at 16.  Measured and not
// taken: the last tenth of the work claimed in chunks through a counter (64 tokens 4 % faster, 200 tokens 2
// to 5 % slower: every chunk loads an item's columns again); a stage read into registers and its place
// requested before the products (16 columns: no change; 32: the registers spill).  Scalar registers run out in
// the instances for long rows (16 / 32 columns: 44 / 68 of them live in lanes of a vector register in gate/up, 29 / 54 in
// down; no memory); what that costs was not measured.
//
// A shared expert of another format runs beside these on the layer's side stream although they take nearly all
// of every CU's LDS: the layer of 256 experts 7168 x 2048 with a Q8_0 shared expert, us before / with the streaming
// kernels: 24 tokens 750 / 674, 64: 1201 / 1061, 128: 1644 / 1274, 400: 1708 / 1457, 512: 1735 / 1486.
#pragma once

#include "dsx_device.hpp"
#include "dsx_gemm_kernels.hpp"
#include "dsx_q8_0_kernels.hpp"

namespace dsx {

constexpr uint32_t kStMaxSb = 28;          // super-blocks per row that the registers hold (16 or 32 columns)
constexpr uint32_t kStQ8MaxSb = 32;        // groups of four Q8_0 blocks per row
constexpr uint32_t stream_part_bytes(uint32_t waves) { return waves * 1024u; }   // the partial sums of one 16 x 16 fragment
// s_dest | s_src | s_ew, one of each per column, in whole cache lines
constexpr uint32_t stream_head_bytes(uint32_t ncg) { return (ncg * 192u + 127u) / 128u * 128u; }
// A stage of gate and one of up in turn share one set of partial sums; else every tile of a stage has its own.
constexpr uint32_t stream_fragments(bool pair, uint32_t rt, uint32_t ncg) { return (pair && rt == 1u ? 1u : pair ? 2u : rt) * ncg; }
constexpr uint32_t kStLds = 160u * 1024u;
constexpr uint32_t kStMaxDepth = 8;

struct StreamParams {
    const uint8_t *w0, *w1;        // [n_expert] experts (gate, up), or down in w0
    const uint8_t *sh_w0, *sh_w1;  // the extra expert with index n_expert, or null
    uint64_t bpe0, bpe1;
    const uint8_t *act;            // staged FP6 rows or Q8_0 rows, act_row_bytes apart: by token (PAIR) or by dest row
    const int32_t *group_count, *group_offset, *members, *work_items, *n_work_items;
    StreamChoice choice;           // a GEMM launch offers the same product
    const float *ew;               // [n_tokens, n_used]   (PAIR)
    float *out;                    // PAIR: mid, else partial rows: f32 [dest rows, n_rows]
    uint32_t n_tokens, n_used, n_expert, n_rows, act_row_bytes;
    uint32_t n_sb;                 // 136-byte pieces of a row: super-blocks (MXFP4), groups of four blocks (Q8_0)
    float clamp, sh_clamp;
    // set by stream_layout
    uint32_t run, pitch, pitch_magic;   // 16-byte pieces of a row, of its place in LDS
    uint32_t loads, stage_bytes, depth;   // 1 KB loads per stage and matrix; stages in the ring
};

// Where a stage's bytes go in LDS: rows of an odd number of 16-byte pieces, so that 16 lanes reading 16
// rows at one offset hit every bank once (a row of n_sb super-blocks is 8.5 n_sb pieces; n_sb odd:
// whole tiles, no padding).  rt: row tiles of a stage -- PAIR: 1, gate and up in turn, or 2, one of each.
inline bool stream_layout(StreamParams &p, bool pair, uint32_t rt, uint32_t ncg, uint32_t waves) {
    const uint32_t tiles = pair ? 1u : rt;   // of one matrix
    const bool even = p.n_sb % 2u == 0u;
    p.run = even ? p.n_sb * 17u / 2u : p.n_sb * 136u;
    p.pitch = even ? p.run | 1u : p.run;
    p.pitch_magic = (uint32_t)((0x100000000ull + p.pitch - 1u) / p.pitch);
    p.loads = ((even ? 16u : 1u) * tiles * p.pitch + 63u) / 64u;
    p.stage_bytes = p.loads * 1024u * (pair ? rt : 1u);
    const uint32_t fixed = stream_head_bytes(ncg) + stream_fragments(pair, rt, ncg) * stream_part_bytes(waves);
    p.depth = std::min<uint32_t>(kStMaxDepth, (kStLds * waves / 8u - fixed) / p.stage_bytes);
    return p.depth >= 2u;
}
inline size_t stream_lds_bytes(const StreamParams &p, bool pair, uint32_t rt, uint32_t ncg, uint32_t waves) {
    return stream_head_bytes(ncg) + (size_t)stream_fragments(pair, rt, ncg) * stream_part_bytes(waves) + (size_t)p.depth * p.stage_bytes;
}

// 1 where a group has no item but `wi`, which `after` follows in the list (`last`: nothing does); uniform.  (Written out, as the
// compiler would keep the truth value in a vector register.)
__device__ __forceinline__ uint32_t only_item(uint32_t wi, uint32_t after, uint32_t last) {
    uint32_t once, start;
    asm volatile("s_xor_b32 %0, %2, %3\n\ts_lshr_b32 %0, %0, 16\n\ts_cselect_b32 %0, 1, %4\n\t"   // (SCC: another expert's)
                 "s_and_b32 %1, %2, 0xffff\n\ts_cselect_b32 %0, 0, %0"
                 : "=&s"(once), "=&s"(start) : "s"(wi), "s"(after), "s"(last) : "scc");
    return once;
}

// ---- what a wave keeps of an item's columns, and how it multiplies a tile with them ------------------

// MXFP4 weights, FP6 planes.  NI: super-blocks per wave (n_sb <= 4 NI); wave w has half w % 2 of super-blocks
// w / 2 + 4 i.
template <int NI, int NCG>
struct StreamMxfp4 {
    static constexpr int kWaves = 8;
    static constexpr bool kRoles = true;   // (below, stream_body)
    static constexpr uint32_t kPart = stream_part_bytes(kWaves) / 4u;
    // operand (super-block sb0 + 4 i, the wave's half) of column n16 of a column group; a super-block past
    // the row's end has zero codes and d = 0
    v8i bh[NI][NCG], bl[NI][NCG];
    float yd[NI][NCG];

    __device__ __forceinline__ void load(const StreamParams &p, const uint32_t *s_src, uint32_t wave, uint32_t g4, uint32_t n16) {
        const uint32_t half = wave & 1u, sb0 = wave >> 1, n_sb = p.n_sb;
#pragma unroll
        for (int cg = 0; cg < NCG; cg++) {
            const uint8_t *row = p.act + (uint64_t)s_src[cg * 16 + (int)n16] * p.act_row_bytes;
#pragma unroll
            for (int i = 0; i < NI; i++) {
                const uint32_t sb = sb0 + 4u * (uint32_t)i;
                const bool live = sb < n_sb;
                const uint8_t *b = row + (live ? sb : 0u) * kStaged6Bytes;
                const uint8_t *hd = b + half * 128u + g4 * 16u, *tl = b + 256u + half * 64u + g4 * 8u;
                const uint4 h0 = *(const uint4 *)hd, h1 = *(const uint4 *)(hd + 64);
                const uint2 t0 = *(const uint2 *)tl, t1 = *(const uint2 *)(tl + 32);
                const float d = *(const float *)(row + n_sb * kStaged6Bytes + (live ? sb : 0u) * 4u);
                bh[i][cg] = live ? v8i{(int)h0.x, (int)h0.y, (int)h0.z, (int)h0.w, (int)t0.x, (int)t0.y, 0, 0} : v8i{0, 0, 0, 0, 0, 0, 0, 0};
                bl[i][cg] = live ? v8i{(int)h1.x, (int)h1.y, (int)h1.z, (int)h1.w, (int)t1.x, (int)t1.y, 0, 0} : v8i{0, 0, 0, 0, 0, 0, 0, 0};
                yd[i][cg] = live ? d : 0.0f;
            }
        }
        // they have arrived when this block ends (a wait left to their first use would sit in the loop
        // over the stages and hold back every stage's loads)
#pragma unroll
        for (int cg = 0; cg < NCG; cg++)
#pragma unroll
            for (int i = 0; i < NI; i++) {
#pragma unroll
                for (int k = 0; k < 6; k++) {
                    int vh = bh[i][cg][k], vl = bl[i][cg][k];
                    asm volatile("" : "+v"(vh), "+v"(vl));
                    bh[i][cg][k] = vh;
                    bl[i][cg][k] = vl;
                }
                asm volatile("" : "+v"(yd[i][cg]));
            }
    }

    // `row`: row n16 of the tile in LDS.  part: the lane's place in the wave's partial sums.
    __device__ __forceinline__ void tile(const uint8_t *row, uint32_t n_sb, uint32_t wave, uint32_t g4, float *part) const {
        const uint32_t half = wave & 1u, sb0 = wave >> 1;
        const uint32_t a_off = half * 64u + g4 * 16u, s_off = 128u + half * 4u + g4;
        v4f acc[NCG];
#pragma unroll
        for (int cg = 0; cg < NCG; cg++) acc[cg] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const uint32_t sb = min(sb0 + 4u * (uint32_t)i, n_sb - 1u);
            const uint8_t *pa = row + a_off + sb * (uint32_t)kSuperBytes;   // (8-byte aligned: an odd super-block of a row)
            const uint2 lo2 = *(const uint2 *)pa, hi2 = *(const uint2 *)(pa + 8);
            const int sc = (int)row[s_off + sb * (uint32_t)kSuperBytes];
            const v8i av = {(int)lo2.x, (int)lo2.y, (int)hi2.x, (int)hi2.y, 0, 0, 0, 0};
#pragma unroll
            for (int cg = 0; cg < NCG; cg++) {
                v4f c = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, bh[i][cg], v4f{0.f, 0.f, 0.f, 0.f}, 4, 2,
                                                                        0, sc, 0, kScaleB6High);
                c = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, bl[i][cg], c, 4, 2, 0, sc, 0, kScaleB6Low);
                acc[cg].x = fmaf(yd[i][cg], c.x, acc[cg].x);
                acc[cg].y = fmaf(yd[i][cg], c.y, acc[cg].y);
                acc[cg].z = fmaf(yd[i][cg], c.z, acc[cg].z);
                acc[cg].w = fmaf(yd[i][cg], c.w, acc[cg].w);
            }
        }
#pragma unroll
        for (int cg = 0; cg < NCG; cg++)
            *(float4 *)(part + (uint32_t)cg * kPart) = make_float4(acc[cg].x, acc[cg].y, acc[cg].z, acc[cg].w);
    }
};

// Q8_0 weights and activations, 16 columns.  NI: groups of four blocks per wave (n_sb <= W NI); wave w has groups
// w + W i.  One v_mfma_i32_16x16x32_i8 is a block of a fragment (Q8Frag).
template <int W, int NI>
struct StreamQ8 {
    static constexpr int kWaves = W;
    static constexpr bool kRoles = false;
    static constexpr uint32_t kPart = stream_part_bytes(kWaves) / 4u;
    long codes[NI][4];   // bytes 8 g4 .. of block b of a group: column n16
    float xs[NI];        // scale of block g4 of the group; a group past the row's end has zero codes and scales

    __device__ __forceinline__ void load(const StreamParams &p, const uint32_t *s_src, uint32_t wave, uint32_t g4, uint32_t n16) {
        const uint32_t n_sb = p.n_sb;
        const uint8_t *row = p.act + (uint64_t)s_src[n16] * p.act_row_bytes;
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const uint32_t sb = wave + (uint32_t)(W * i);
            const bool live = sb < n_sb;
            const uint8_t *b = row + (live ? sb : 0u) * 128u + g4 * 8u;
            const float d = *(const float *)(row + n_sb * 128u + (live ? sb : 0u) * 16u + g4 * 4u);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const long v = *(const long *)(b + 32 * k);
                codes[i][k] = live ? v : 0;
            }
            xs[i] = live ? d : 0.0f;
        }
        // (they have arrived when this block ends, as above)
#pragma unroll
        for (int i = 0; i < NI; i++) {
#pragma unroll
            for (int k = 0; k < 4; k++) {
                long v = codes[i][k];
                asm volatile("" : "+v"(v));
                codes[i][k] = v;
            }
            asm volatile("" : "+v"(xs[i]));
        }
    }

    __device__ __forceinline__ void tile(const uint8_t *row, uint32_t n_sb, uint32_t wave, uint32_t g4, float *part) const {
        long av[NI][4];
        float dw[NI];
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const uint32_t q = wave + (uint32_t)(W * i), sb = min(q, n_sb - 1u);
            const uint8_t *a = row + n_sb * 8u + sb * 128u + g4 * 8u;
#pragma unroll
            for (int k = 0; k < 4; k++) av[i][k] = *(const long *)(a + 32 * k);
            const float d = __half2float(__ushort_as_half(*(const uint16_t *)(row + sb * 8u + g4 * 2u)));
            dw[i] = q < n_sb ? d : 0.0f;   // (an infinite scale must not meet the zero of a group that is not there)
        }
        float acc[4] = {0.f, 0.f, 0.f, 0.f};
        Q8Frag fr[2];
        fr[0].start(av[0], codes[0], dw[0], xs[0]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < NI; i++) {
            if (i + 1 < NI) fr[(i + 1) & 1].start(av[i + 1], codes[i + 1], dw[i + 1], xs[i + 1]);
            fr[i & 1].fold(acc);
            Q8Frag::interleave();
        }
        *(float4 *)part = make_float4(acc[0], acc[1], acc[2], acc[3]);
    }
};

// NCG: 16-column groups; RT: 16-row tiles of a stage (a stage of a short k is then still large beside its two
// barriers).  PAIR: a stage of gate and one of up in turn (RT = 1) or a tile of each per stage (RT = 2).
template <typename COLS, bool PAIR, int NCG, int RT>
__device__ __forceinline__ void stream_body(const StreamParams &p) {
    static_assert(!PAIR || RT <= 2, "one row tile of either matrix");
    constexpr int kW = COLS::kWaves;
    // Between two stages a wave requests the next one or adds up and stores the last one's sums.  MXFP4: the first half of
    // the waves does the one, the second half the other, at the same time and without a load that waits behind a store
    // (vmcnt counts them in order; 7168 x 2048, 256 experts, every wave both / so: 100 tokens 977 / 961 us, Zipf-skewed 200: 1146 / 1117); Q8_0: every wave does its part of both (half each: 2048 x 1408, 40 tokens 124 / 126 us).
    constexpr uint32_t kLoaders = COLS::kRoles ? (uint32_t)kW / 2u : (uint32_t)kW;
    constexpr uint32_t kSummer0 = COLS::kRoles ? kLoaders : 0u;               // the first wave that sums
    constexpr uint32_t kSummers = ((uint32_t)kW - kSummer0) * 64u;            // threads that do
    constexpr bool kTurns = PAIR && RT == 1;
    constexpr uint32_t kTiles = PAIR ? 1u : (uint32_t)RT;   // row tiles of a unit
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    constexpr uint32_t kCols = 16u * NCG;
    constexpr uint32_t kFrags = stream_fragments(PAIR, RT, NCG);   // fragments whose partial sums meet
    uint32_t *s_dest = (uint32_t *)smem, *s_src = s_dest + kCols;
    float *s_ew = (float *)(s_dest + 2u * kCols);
    constexpr uint32_t kHead = stream_head_bytes(NCG);
    float *s_part = (float *)(smem + kHead);
    constexpr uint32_t kStages = kHead + kFrags * stream_part_bytes(kW);   // a multiple of 128

    const uint32_t tid = threadIdx.x, lane = tid & 63u, g4 = lane >> 4, n16 = lane & 15u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t n_sb = p.n_sb;

    // ---- the workgroup's range of units (item, row tile) --------------------------------------
    // ranges next to each other run on one XCD (ids go round the 8 of them): they share items
    const uint32_t G = gridDim.x;
    const uint32_t r = G % 8u == 0u ? (blockIdx.x & 7u) * (G >> 3) + (blockIdx.x >> 3) : blockIdx.x;
    const uint32_t n_items = __builtin_amdgcn_readfirstlane((uint32_t)*p.n_work_items);
    if (p.choice.offered() && !p.choice.streams()) return;   // uniform
    const uint32_t n_ut = p.n_rows / (16u * kTiles);
    const uint64_t total = (uint64_t)n_items * n_ut;
    const uint64_t lo = total * r / G, hi = total * (r + 1u) / G;
    if (lo >= hi) return;   // uniform
    const uint32_t n_stages = (uint32_t)(hi - lo) * (kTurns ? 2u : 1u);
    const uint32_t item0 = (uint32_t)(lo / n_ut), ut0 = (uint32_t)(lo % n_ut);

    // ---- requesting stages ----------------------------------------------------------------------
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)smem) + kStages;
    const bool loader = !COLS::kRoles || wave < kLoaders, summer = !COLS::kRoles || !loader;
    const uint32_t n_loads = PAIR && !kTurns ? 2u * p.loads : p.loads;   // of a stage; the wave's: wave, wave + kLoaders, ..
    const uint32_t my_loads = (n_loads + kLoaders - 1u - wave) / kLoaders;
    const uint32_t unit_bytes = kTiles * 16u * n_sb * (uint32_t)kSuperBytes;
    const uint32_t last_piece = unit_bytes / 16u - 1u;
    uint32_t q_item = item0, q_ut = ut0, q_m = 0, q_slot = 0, q_left = n_stages;   // the next stage to request
    const uint8_t *q_base[2];
    uint32_t q_once;   // whether nobody else reads the item's weights
    auto q_bases = [&]() {
        const uint32_t wi = __builtin_amdgcn_readfirstlane((uint32_t)p.work_items[q_item]), e = wi >> 16;
        // (a group's items follow each other in the list)
        const uint32_t after = __builtin_amdgcn_readfirstlane((uint32_t)p.work_items[min(q_item + 1u, n_items - 1u)]);
        q_once = only_item(wi, after, (n_items - q_item - 2u) >> 31);
        const bool extra = e >= p.n_expert;
        q_base[0] = extra ? p.sh_w0 : p.w0 + (uint64_t)e * p.bpe0;
        q_base[1] = !PAIR ? nullptr : extra ? p.sh_w1 : p.w1 + (uint64_t)e * p.bpe1;
    };
    q_bases();
    auto request = [&]() __attribute__((always_inline)) {
        const uint8_t *src0 = (kTurns && q_m ? q_base[1] : q_base[0]) + (uint64_t)q_ut * unit_bytes;
        const uint8_t *src1 = PAIR && !kTurns ? q_base[1] + (uint64_t)q_ut * unit_bytes : nullptr;
        const uint32_t dst = lds0 + q_slot * p.stage_bytes;
        // (the offsets are the same for every stage, but there are no registers to keep them in)
        auto loads = [&](auto nt) __attribute__((always_inline)) {
            for (uint32_t L = wave; L < n_loads; L += kLoaders) {
                const bool second = PAIR && !kTurns && L >= p.loads;
                const uint32_t s = (second ? L - p.loads : L) * 64u + lane;
                const uint32_t run = __umulhi(s, p.pitch_magic);   // s / pitch
                uint32_t piece = s - run * p.pitch;
                piece = min(piece, p.run - 1u);   // a row's padding repeats its last piece
                // (slots past the last row fetch the unit's last piece: the load stays in the unit)
                lds_dma16<decltype(nt)::value>(dst + L * 1024u, second ? src1 : src0, min(run * p.run + piece, last_piece) * 16u);
            }
        };
        if (q_once) loads(std::true_type{});   // uniform
        else loads(std::false_type{});
        q_left--;
        q_slot = q_slot + 1u == p.depth ? 0u : q_slot + 1u;
        if (kTurns) {
            q_m ^= 1u;
            if (q_m) return;
        }
        if (++q_ut == n_ut) {
            q_ut = 0;
            if (q_left) {
                q_item++;
                q_bases();
            }
        }
    };

    // ---- an item's columns ---------------------------------------------------------------------
    COLS cols;
    uint32_t cnt = 0;
    float clamp = p.clamp;
    auto load_item = [&](uint32_t item) {
        const uint32_t wi = __builtin_amdgcn_readfirstlane((uint32_t)p.work_items[item]);
        const uint32_t e = wi >> 16, start = wi & 0xFFFFu;
        cnt = min(kCols, __builtin_amdgcn_readfirstlane((uint32_t)p.group_count[e]) - start);
        const uint32_t mbase = (uint32_t)p.group_offset[e] + start;
        clamp = e >= p.n_expert ? p.sh_clamp : p.clamp;
        if (tid < kCols) {
            // columns past the end of the group repeat its last member; they are never stored
            const uint32_t m = (uint32_t)p.members[mbase + min(tid, cnt - 1u)];
            const uint32_t dest = gemm_dest_row(m, p.n_tokens, p.n_used);
            s_dest[tid] = dest;
            s_src[tid] = PAIR ? (m >> 16) : dest;
            if (PAIR) s_ew[tid] = (m & 0xFFFFu) >= p.n_used ? 1.0f : p.ew[dest];
        }
        __syncthreads();
        cols.load(p, s_src, wave, g4, n16);
    };

    // the first stage is requested ahead of the look-ups, the others behind them: loads return in order
    if (loader) request();
    load_item(item0);
    if (loader)
        for (uint32_t d = 1; d < p.depth && q_left; d++) request();

    // ---- the stages ----------------------------------------------------------------------------
    // read side: row n16 of a tile
    const uint32_t row_lds = n_sb % 2u == 0u ? p.pitch * 16u : n_sb * (uint32_t)kSuperBytes;
    const uint32_t tile_lds = PAIR ? p.loads * 1024u : 16u * row_lds;
    // partial sums: [fragment][wave][column][row], a column's four row quads rotated by column / 4 so
    // that the lanes' 16-byte writes spread over the banks
    float *part_w = s_part + wave * 256u + n16 * 16u + ((g4 + (n16 >> 2)) & 3u) * 4u;
    uint32_t c_item = item0, c_ut = ut0, slot = 0;
    // a loader that stores: its stores of the last `depth` stages, four bits each, and their sum
    uint32_t n_st = 0, st_hist = 0;

    // Adds up partial sums, wave after wave: a thread's values in the order (column, row tile, row), so that the rows of a
    // unit's tiles, which follow each other in a result row, are stored in whole lines where there is more than one tile
    // (7168 x 2048, 256 experts, 300 tokens, layer: 1186 / 1170 us).
    // gate: the first of two stages in turn, whose sums wait in registers for the second's.
    constexpr uint32_t kOuts = kTiles * NCG * 256u;
    constexpr uint32_t kRounds = (kOuts + kSummers - 1u) / kSummers;
    float gate_sum[kTurns ? kRounds : 1];
    auto finish = [&](bool gate) __attribute__((always_inline)) {
#pragma unroll
        for (uint32_t r = 0; r < kRounds; r++) {
            const uint32_t ow = r * kSummers + (wave - kSummer0) * 64u;   // the wave's first value
            const uint32_t colw = ow / (16u * kTiles);
            if ((kOuts % kSummers != 0u && ow >= kOuts) || colw >= cnt) continue;   // uniform: no member among its columns
            const uint32_t col = colw + lane / (16u * kTiles), tile = g4 % kTiles, col16 = col & 15u;
            const float *f = s_part + (tile * NCG + (col >> 4)) * COLS::kPart + col16 * 16u + ((n16 + (col16 & 12u)) & 15u);
            float a = f[0], b = 0.0f;
#pragma unroll
            for (int w = 1; w < kW; w++) a += f[w * 256];
            if (kTurns) {
                if (gate) {
                    gate_sum[r] = a;
                    continue;
                }
                b = a;
                a = gate_sum[r];
            } else if (PAIR) {
                f += NCG * COLS::kPart;
                b = f[0];
#pragma unroll
                for (int w = 1; w < kW; w++) b += f[w * 256];
            }
            if (kSummer0 == 0u) {
                n_st++;
                st_hist++;
            }
            if (col < cnt) {
                float *dst = p.out + (uint64_t)s_dest[col] * p.n_rows + (c_ut * kTiles + tile) * 16u + n16;
                *dst = PAIR ? swiglu_clamp(a, b, clamp, s_ew[col]) : a;
            }
        }
    };

    uint32_t m = 0;   // which matrix the stage is of (in turn)
#pragma unroll 1
    for (uint32_t j = 0; j < n_stages; j++) {
        // (opaque: told apart at compile time, the two kinds of stage get two copies of everything below)
        if (kTurns) asm volatile("" : "+s"(m));
        // the stage's loads have landed; what this wave sent after them may be under way: the younger
        // stages' loads and the stores of the last `depth` stages (counted exactly: a store more than
        // allowed for would be made up by a load of the next stage, most of a stage's time later)
        if (loader) wait_vm<COLS::kRoles>(min(n_stages - 1u - j, p.depth - 1u) * my_loads + n_st);
        __syncthreads();
        if (kSummer0 == 0u) {
            n_st -= (st_hist >> (4u * p.depth - 4u)) & 15u;
            st_hist <<= 4;
        }
        const uint8_t *st = smem + kStages + slot * p.stage_bytes;
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            cols.tile(st + (uint32_t)rt * tile_lds + n16 * row_lds, n_sb, wave, g4,
                      part_w + (kTurns ? 0u : (uint32_t)rt * NCG) * COLS::kPart);
        }
        __syncthreads();   // the partial sums are there, and nobody reads the stage any more
        slot = slot + 1u == p.depth ? 0u : slot + 1u;
        if (loader && q_left) request();
        const bool gate = kTurns && m == 0u;
        if (summer) finish(gate);
        if (!gate) c_ut++;
        m ^= 1u;
        if (c_ut == n_ut && j + 1u < n_stages) {
            c_ut = 0;
            __syncthreads();   // the old item's destinations have been read
            load_item(++c_item);
        }
    }
}

template <bool PAIR, int NI, int NCG, int RT>
__global__ __launch_bounds__(512, 2) void k_mxfp4_stream(const StreamParams p) {
    stream_body<StreamMxfp4<NI, NCG>, PAIR, NCG, RT>(p);
}

// Items of 16 and of 32 columns are both there: the narrower ones unless they are over a fifth more, as each of them reads its
// weights anew (items of 16 per item of 32, time with these per time with those: 4096 x 1024, 128 experts, 110 tokens: spread
// picks 1.02, 0.85, Zipf-skewed 1.05, 0.87, on 48 experts 1.69, 1.15; 180: spread 1.11, 0.94, Zipf 1.18, 0.95; 5120 x 1536, 160, 220:
// Zipf 1.11, 0.98, on 100 experts 1.23, 1.04, on 60 1.96, 1.37; 2048 x 1536, 64, 100: on 40 1.34, 1.09).
template <bool PAIR, int NI, int RT>
__global__ __launch_bounds__(512, 2) void k_mxfp4_stream_widths(const StreamParams narrow, const StreamParams wide) {
    if (5u * (uint32_t)*narrow.n_work_items <= 6u * (uint32_t)*wide.n_work_items)   // uniform
        stream_body<StreamMxfp4<NI, 1>, PAIR, 1, RT>(narrow);
    else
        stream_body<StreamMxfp4<NI, 2>, PAIR, 2, RT>(wide);
}

template <bool PAIR, int W, int NI, int RT>
__global__ __launch_bounds__(W * 64, 2) void k_q8_0_stream(const StreamParams p) {
    stream_body<StreamQ8<W, NI>, PAIR, 1, RT>(p);
}

}  // namespace dsx
