// The full decode step's launch: constants, and how its workgroups are chosen from the shapes
// alone.  Host code without HIP, so that tests compile it too.
#pragma once
#include <algorithm>
#include <cstdint>

namespace tq4 {
namespace xdl {

constexpr int kStepWaves = 8;  // waves per workgroup at most: two per SIMD of one CU
// What a further segment costs a workgroup (block table, query, rotation, first loads), in tiles of
// each of its waves: a sequence counts this many tiles times the waves per head part more than it has
// when the list is cut.  Measured with one wave, 64 sequences of 512 to 8192 tokens, with 3 / 6 / 10 /
// 14 / 20: 79.7 / 78.1 / 76.3 / 75.3 / 77.3 us; over 130 ragged batches with more waves, 7 / 10 / 14 / 20
// relative: 1.016 / 1.007 / 1 / 1.001 (14 tiles whatever the waves: 16 sequences of 500 to 8000 tokens on
// 1 kv-head, eight waves, 28.3 / 17.5 us, 12 of 94 to 1500 27.8 / 16.9).
constexpr int kSegmentTiles = 14;
// Tiles whose block-table entries a wave keeps in LDS: a stream this long runs without a stop (a
// stop, the block-table read and the refill of the ring, costs about 3 us).
constexpr int kTableTiles = 512;
constexpr int kRotateWaves = 4;   // least waves of a workgroup that rotates (StepPlan::rotates)
constexpr int kMinWaveTiles = 4;  // a wave's stream is whole turns of the 4-slot ring anyway

// How a step is cut into workgroups, from the shapes alone.
struct StepPlan {
    int vw, sw;    // head parts per workgroup, waves per head part
    int nx;        // workgroups along the list of sequences
    int per_seq;   // of them per sequence (0: fewer than one)
    bool whole;    // one workgroup per sequence, which writes the output rows itself
    // Its workgroups rotate a 16-bit query themselves.  Every segment stages all 64 KB of rot_t, 16
    // columns per wave at a time: with one or two waves that is eight or four rounds of load, barrier
    // and arithmetic, and the launch that rotates all rows first is faster, unless one workgroup
    // has a whole sequence's heads and so stages rot_t once for it.  In the kernel / by the launch:
    // 8 heads on 1 kv-head, 64 sequences of 500 to 8000 tokens (two waves): 40.0 / 31.6 us; 5 kv-heads,
    // 256 x 2000 (one wave): 125.8 / 109.8; 6 kv-heads, 64 of 500 to 8000 (two): 73.3 / 67.1; 4 kv-heads
    // (four waves): 48.7 / 48.7; 8 kv-heads, 64 x 4096 (eight): 68.1 / 70.6, AoS (four): 82.8 / 83.5.
    bool rotates;
};
inline int floor_pow2(int64_t x, int most) {
    int p = 1;
    while (p < most && 2 * p <= x)
        p *= 2;
    return p;
}

// What the plan depends on.
struct StepShape {
    int held;         // waves the device holds at once
    int nvh;          // head parts of a sequence
    int batch, max_blocks, block_size, num_splits;
    bool whole_lines; // a head's records are whole 128-byte lines (4-bit SoA)
};
// The table's width stands for the lengths, which only the device knows: under a backend's table of
// its longest context short sequences run in parts too (one of 333 tokens, 2048 blocks: 16.1 us against
// 12.9 under a table of 21, where separate launches take 14.6).
inline StepPlan step_plan(const StepShape &s, bool have_parts) {
    const int held = s.held, nvh = s.nvh;
    const int64_t pairs = (int64_t)nvh * s.batch;  // (sequence, head part) pairs
    const int64_t tiles = ((int64_t)s.max_blocks * s.block_size + 15) / 16;  // of the longest sequence the table can hold
    // eight head parts per workgroup for 4-bit SoA records (whole 128-byte lines), four for the others,
    // whose neighbouring heads share lines: B64 x 4096 with 32 / 8 heads takes 66.0 (8) / 67.2 us
    // (4), AoS 88.8 / 80.4, 3-bit B48 58.8 / 57.5; with two 70.3 to 73.6, 86 to 88 and 66.7
    const int most_vw = s.whole_lines ? kStepWaves : kStepWaves / 2;
    int vw = 1;
    while (vw < most_vw && nvh % (2 * vw) == 0)
        vw *= 2;
    // whole: one wave per pair fills at least 9/10 of every round, so cutting further would only
    // add the merge launch; or sequences so short that a wave has at most kShortTiles tiles, and at
    // most kMergeTiles (about what the merge launch takes) more than it would have in parts.  Beyond
    // kShortTiles ragged lengths lose more than the merge.  Whole / parts: 64 x 700 tokens 18.3 /
    // 21.9 us (70 to 700: 18.0 / 21.9), 100 of 30 to 300 18.1 / 23.1 (11 and 10 tiles in either form);
    // 1 x 1500 17.6 / 15.9 (12 against 4 tiles), 16 x 2000 20.6 / 18.7 (16 against 8).
    constexpr int kShortTiles = 12;
    constexpr int kMergeTiles = 5;
    const int64_t rounds = (pairs + held - 1) / held;
    const bool full = 10 * pairs >= 9 * rounds * held;
    // or the pairs fill more than half of the rounds' waves and the table holds few tiles: at most 124
    // times the share less 32, or 40 with more than one round (the next one's sequences start as the
    // first ones end).  Idle waves leave the others faster, so what parts gain by even stretches has to
    // pay for their further segments and the merge.  Whole / parts for ragged lengths (a 16th to the longest),
    // 32 / 8 heads: 200 sequences (0.78 of a round) of up to 500 tokens 29.1 / 37.0 us, 700 36.2 / 41.4,
    // 1000 51.6 / 50.2, 2000 92.5 / 74.2; 135 (0.53) 500 29.0 / 29.4, 700 35.8 / 31.6; 160 (0.63) 700
    // 35.9 / 35.3; 300 (0.59 of two) 500 46.8 / 49.3, 700 58.9 / 56.4; 400 (0.78 of two) 1000 91.6 / 85.0;
    // 32 / 4 heads, 400 (0.78) 1000 54.7 / 62.2, 520 (0.51 of two) 600 47.5 / 61.5.  Equal lengths gain
    // more (200 x 1000 56.8 / 64.4; 200 x 2000, beyond the line, 102.2 / 114.6).
    const bool few_tiles = 2 * pairs > rounds * held &&
                           (rounds == 1 ? (tiles + 32) * held <= 124 * pairs : tiles <= 40);
    int sw = full ? 1 : floor_pow2(held / pairs, kStepWaves);
    const int64_t wave_tiles = (tiles + sw - 1) / sw;
    const int64_t parts_tiles = std::max<int64_t>(kMinWaveTiles, (pairs * tiles + held - 1) / held);
    if (full || few_tiles || !have_parts || wave_tiles <= std::min<int64_t>(kShortTiles, parts_tiles + kMergeTiles)) {
        vw = std::min(vw, kStepWaves / sw);
        return StepPlan{vw, sw, s.batch, 1, true, vw * sw >= kRotateWaves || vw == nvh};
    }
    // parts: enough waves of a workgroup on one head part that sequences of equal lengths have at most
    // kMostParts parts to merge, as far as eight waves reach (one sequence on 8 kv-heads: 32 parts); more
    // waves than that cut ragged batches coarser (FP8 keys, 24 sequences of 1001 to 6001 tokens: 42.3 us with one wave, 44.6 with two; 64 of 512 to
    // 8192: 78.1 with one, 82.8 with two, 84.4 with four)
    constexpr int kMostParts = 16;
    sw = 1;
    while (sw < kStepWaves && held > pairs * sw * std::min(kMostParts, s.num_splits - 1))
        sw *= 2;
    vw = std::min(vw, kStepWaves / sw);
    const int64_t useful = s.batch * ((tiles + kMinWaveTiles * sw - 1) / (kMinWaveTiles * sw));
    const int nx = (int)std::max<int64_t>(1, std::min<int64_t>(held / (vw * sw) / (nvh / vw), useful));
    return StepPlan{vw, sw, nx, nx / s.batch, false, vw * sw >= kRotateWaves};
}

}  // namespace xdl
}  // namespace tq4
