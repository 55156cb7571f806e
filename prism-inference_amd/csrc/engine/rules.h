/* rules.h - which kernel, how many waves and how many workgroups a call gets,
 * as functions of sizes alone (no HIP). Host plain C++. */
#ifndef PRISM_RULES_H
#define PRISM_RULES_H

#include <algorithm>
#include <cstdint>

#include "prism.h"

namespace prism {

/* Compute units of an MI355X. */
constexpr int CU_COUNT = 256;

/* ---- block chain */

/* The chain of a batch with more than CHAIN_SPLIT_ROUTED (MoE blocks) or
 * CHAIN_SPLIT_DENSE windows (see chain_plan) runs as up to CHAIN_SPLIT
 * independent sub-chains of whole frames, on their own streams
 * (parallel branches of the hipGraph): windows and tokens never interact
 * across frames, and one sub-chain's expert launches overlap another's
 * attention launches and the tails of both. */
constexpr int CHAIN_SPLIT = 2;
constexpr int CHAIN_SPLIT_ROUTED = CU_COUNT * 3 / 4;
constexpr int CHAIN_SPLIT_DENSE = 2 * CU_COUNT;
static_assert(CHAIN_SPLIT >= 1 && CHAIN_SPLIT <= 4, "sub-chain streams");

/* How a forward's blocks are launched. */
struct ChainPlan {
    int split;       /* sub-chains */
    bool one_launch; /* a dense chain: every block in one launch */
    bool pair8;      /* both sub-chains' launches on 8 waves */
    int64_t windows; /* of the batch */
};

/* Sub-chains. A routed block's two launches leave CUs idle in
 * turn (the attention's while its last windows finish, the experts' while
 * they wait for weights), so the frames of a batch go in halves as soon as
 * one half's attention launch no longer fits beside the other's experts for
 * free: 16 blocks, one chain against two: 160 windows 411 and 418 us, 192
 * 442 and 438, 256 578 and 509 (64 experts), 270 641 and 504, 288 684 and
 * 539, 504 859 and 814. With more than 32 experts, whose weights fill most of
 * a small launch's time, not while both launches are one round of 8-wave
 * workgroups (expert_w8): 64 experts, graphs of three frames of 56x75 (210
 * windows) 451 and 480 us, of 36x123 (240) 457 and 482, of two of 81x81 462
 * and 479, of 9 of 24x64 (216) 466 and 483, of 6 of 33x51 (210) 419 and 440
 * (eager, where the second stream costs less, 441 and 437, 446 and 434, 450 and
 * 462, 455 and 455, 409 and 410). A dense block is one launch: its frames stay together
 * while they fit one round of the 4-wave kernels (two workgroups per CU; four
 * blocks, 256 windows 83 and 91 us, d128 512 windows 61 and 74; 540 windows
 * 170 and 150).
 *
 * One launch. A dense chain's windows meet no others in any block, so one launch can take
 * each through all of them with its rows in LDS: no launch, row load or store
 * between the blocks. At d256 while the windows fit one round of workgroups
 * (two 4-wave ones per CU): 12 blocks of 135, 270 and 405 windows 195 -> 151,
 * 267 -> 229 and 339 -> 300 us; of 540 windows, whose second round is nearly
 * empty for all 12 blocks, 393 and 430; of 1,080, 699 and 739. At d128, whose
 * windows are short, always: 4 blocks of 135, 540, 1,080 and 2,160 windows
 * 38 -> 31, 72 -> 57, 104 -> 98 and 182 -> 172 us.
 *
 * 257 windows and more in one launch are 4-wave workgroups, and the launch
 * takes as long as the two that share a CU through all blocks, 272-280 us for
 * 12 blocks, be it a few CUs or all. Two sub-chains of 8-wave launches, a
 * block each, share the work out again at every block, and their time goes by
 * the amount of it, a window whose lower half is padding (attn.hpp's HALF)
 * counting two thirds. One launch against two sub-chains, by windows (of these
 * half): 264 (88) 274 and 228 us, 264 (0) 274 and 263, 300 (100) 272 and 256,
 * 300 (150) 272 and 243, 315 (63) 272 and 263, 336 (0) 282 and 282, 350 (70)
 * 277 and 278, 360 (0) 281 and 301, 385 (77) 283 and 299, 420 (210) 280 and
 * 285. So sub-chains up to 4/3 window per CU, but one launch where the
 * windows past the 256th are all half ones, the last row of the last frame:
 * 258 (129) 217 and 225, 270 (30) 222 and 236.
 *
 * The waves of two sub-chains (chain_attn_w8). The launches of a dense chain's
 * are on 8 together, up to 4/3 window per CU, or on 4 (two of 256 at once: 162
 * us a four-block chain on 8 waves, 134 on 4). A routed sub-chain's go by its
 * own windows, except that with more than 32 experts, 513 to CHAIN_PAIR8_MAX
 * windows in about equal halves and expert launches of more than
 * CHAIN_PAIR8_TILES tiles attention and experts both stay on 8 waves. 64 experts, both on 8, attention on 4,
 * both on 4: 4 frames of 68x120 (2 x 270 windows, 319 tiles) 759, 779 and 804
 * us, of 66x118 (307 tiles) 740, 750 and 782, of 72x120 782, 791 and 831; 22
 * of 24x64 (2 x 264) 771, 780 and 797; 23 804, 819 and 830; but 24 (2 x 288)
 * 819, 827 and 806, 4 of 65x121 (2 x 288, 310 tiles) 774, 759 and 806, 16 of
 * 33x51 (2 x 280, 275 tiles) 795 and 750. With 32 experts (4 of 72x120: 1,034,
 * 983 and 1,004) or 16 (732, 701 and 714) the windows alone decide. */
constexpr int CHAIN_PAIR8_MAX = CU_COUNT * 11 / 5, CHAIN_PAIR8_TILES = CU_COUNT * 7 / 6;
inline ChainPlan chain_plan(const prism_model_desc& d, int batch) {
    const int64_t wx = (d.spatial_w + 7) / 8, frame = wx * ((d.spatial_h + 7) / 8), windows = frame * batch;
    if (d.n_experts > 1) {
        const int64_t tokens = (int64_t)d.spatial_w * d.spatial_h * batch;
        const bool one_round = d.dim == 256 && d.n_experts > 32 && windows <= CU_COUNT &&
                               (tokens + 63) / 64 + d.n_experts / 2 <= CU_COUNT;
        const int split = windows > CHAIN_SPLIT_ROUTED && !one_round ? std::min(CHAIN_SPLIT, batch) : 1;
        const bool pair8 = split > 1 && d.dim == 256 && d.n_experts > 32 && windows > 2 * CU_COUNT &&
                           windows <= CHAIN_PAIR8_MAX && (batch + 1) / 2 * frame <= CU_COUNT * 9 / 8 &&
                           tokens / 128 + d.n_experts > CHAIN_PAIR8_TILES;
        return {split, false, pair8, windows};
    }
    if (d.dim == 128) return {1, true, false, windows};
    if (windows > CHAIN_SPLIT_DENSE) return {std::min(CHAIN_SPLIT, batch), false, false, windows};
    const int64_t half = d.spatial_h % 8 >= 1 && d.spatial_h % 8 <= 4 ? wx : 0; /* a frame */
    if (windows > CU_COUNT + half && 3 * windows - half * batch <= 4 * CU_COUNT && batch > 1)
        return {CHAIN_SPLIT, false, true, windows};
    return {1, true, false, windows};
}

/* Attention: 8 waves (a workgroup per CU at d256)? Windows that fit the CUs as
 * 8-wave workgroups (a head per wave) take those, which shortens each window's
 * serial path; more of them go as 4-wave workgroups, two per CU (three at
 * d128). A d256 8-wave workgroup fills its CU's registers, so window 257
 * starts a second round: routed launches of 270, 405 and 510 windows take
 * 28.6, 32.6 and 35 us on 8 waves, 23.6, 27.5 and 30.7 on 4, and one of 135
 * takes 16.8 us on 8. Two d128 ones share a CU (270 windows 13.0 us either
 * way, 405 16.3 and 16.0). */
inline bool attn_w8(int dim, int64_t windows) { return windows <= (dim == 256 ? CU_COUNT : 2 * CU_COUNT - 1); }

/* The same for a chain's launch of `windows` (chain_plan). */
inline bool chain_attn_w8(const prism_model_desc& d, const ChainPlan& p, int64_t windows) {
    if (p.pair8) return true;
    if (d.dim == 256 && p.split > 1 && d.n_experts == 1) return false;
    return attn_w8(d.dim, windows);
}

/* Experts, 64-token tiles: 8 waves? tiles: the launch's grid, n / 64 and a
 * partial tile per expert; n: its tokens; partial: the experts (0 if dense);
 * p: the chain's plan, NULL for a stage call.
 * Up to a tile per CU 8 waves per tile, which halve each wave's weight
 * stream; more go as 4 waves x 2 tiles per CU. Where nothing runs beside the
 * launch (a stage call, a chain without sub-chains) what counts
 * is the tiles that hold tokens, about half a tile per expert more than
 * n / 64 (the rest of the grid ends at once): stage calls of n / 64 = 246, 16
 * experts (254 tiles) 10.2 us on 8 waves, 11.1 on 4; 250 (258) 16.7 and 14.8;
 * 64 experts 220 (252) 10.8 and 11.4; 236 (268) 17.1 and 15.3; a chain of one
 * 120x128 frame, 64 experts (272) 580 and 542. Beside the other sub-chain's
 * attention a small second round costs less than slower tiles, and the line
 * lies at 5/4 of the grid's tiles per CU: chains with launches of 280 tiles
 * 696 us on 8 waves, 770 on 4; of 296, 745 and 789; of 352, 891 and 855; at
 * the line itself, 320, 816 and 832 on one run, 807 and 789 on another; with
 * more than 32 experts 3/32 further (344: 4 frames of 115x77 819 and 881). d128
 * tiles leave room for two 8-wave workgroups per CU. */
inline bool expert_w8(int dim, int64_t tiles, int64_t n, int partial, const ChainPlan* p) {
    if (dim != 256) return tiles < 2 * CU_COUNT;
    if (p && p->pair8) return true;
    const int64_t beside = CU_COUNT * (partial > 32 ? 27 : 25) / 20;
    return p && p->split > 1 ? tiles <= beside : (n + 63) / 64 + partial / 2 <= CU_COUNT;
}

/* The leading blocks' expert weights are read past the memory-side cache
 * (ctx.h's WEIGHT_CACHE_KEEP) by 8-wave launches, and by 4-wave ones of a chain
 * without sub-chains (64 experts, one frame of 135x240: 842 -> 815 us). Two
 * sub-chains read a block's weights one after the other, and what the first
 * left in that cache is worth more: 8 frames of 68x120 1,277 -> 1,266 us on
 * plain loads, 10 frames 1,543 -> 1,527. */
inline bool expert_wnt(bool leading, bool w8, const ChainPlan& p) { return leading && (w8 || p.split == 1); }

/* ---- projection stages */

/* Workgroups of a projection stage launch (persistent, 64-token tiles in a
 * loop): PROJ_SLOTS, the two per CU that are resident; at d256 up to two
 * rounds of them go a tile to a workgroup, which spreads a partial second
 * round over the CUs. Both d256 launches, 700 tiles: 18.6 us on 512 workgroups,
 * 18.0 on 700; 800: 21.9 and 20.4; 900: 22.5 and 20.9; 1,020: 23.5 and 22.2;
 * but 1,500 32.3 and 34.6; 2,040 42.5 and 45.3. */
constexpr int PROJ_SLOTS = 2 * CU_COUNT;
inline int64_t project_grid(int dim, int64_t tiles) {
    return dim == 256 && tiles <= 2 * PROJ_SLOTS ? tiles : std::min<int64_t>(tiles, PROJ_SLOTS);
}
/* 8 waves: d256 (16 waves per CU instead of 8), but not the down-projection's
 * persistent form, which they slow (2,040 tiles 21.3 us, 4 waves 20.6; up 19.0
 * on either); at d128 4 waves are 4 % faster. */
inline bool project_w8(int dim, bool up, int64_t tiles) { return dim == 256 && (up || tiles <= 2 * PROJ_SLOTS); }

/* ---- codec */

/* workgroups of the persistent codec launches the GPU holds at once */
constexpr int CODEC_DEC3_SLOTS = 3 * CU_COUNT, CODEC_DEC21_SLOTS = 3 * CU_COUNT, CODEC_ENC01_SLOTS = 2 * CU_COUNT,
              CODEC_ENC3_SLOTS = 2 * CU_COUNT;
/* enc2 of up to four blocks per CU runs one workgroup per CU. Two of its
 * workgroups on every CU draw so much that the GPU lowers its clock for
 * hundreds of microseconds after them: behind an encode of 960x540 (510
 * blocks) every launch of a chain ran 4 % slower (16 MoE blocks 421 against
 * 406 us, 2,372 against 2,395 MHz on average), so the frame lost what the
 * encoder had gained: 466 -> 449 us; the 12-block dense model's 236 -> 224,
 * two MoE frames 612 -> 603. The encode itself gains too: 960x540 34.7 -> 33.8,
 * 1280x720 (920 blocks) 54.7 -> 53.4, two of 960x540 (1,020) 56.6 -> 55.5.
 * Above, two workgroups hide each other's waits: three frames (1,530) 85.5
 * against 86.4, 1920x1080 (2,040) 108.1 against 109.4, and the frame's chain
 * is long enough to take no harm (1,052 us either way). */
inline int codec_enc2_slots(int64_t blocks) { return blocks <= 4 * CU_COUNT ? CU_COUNT : 2 * CU_COUNT; }

/* Grid of a persistent codec launch: `slots` workgroups at once, every one
 * the same number of the launch's blocks (or one fewer), so no workgroup is
 * left with a block of its own at the end. */
inline unsigned even_grid(int64_t blocks, int slots) {
    const int64_t each = (blocks + slots - 1) / slots;
    return (unsigned)((blocks + each - 1) / each);
}

}  // namespace prism

#endif
