// How the tiles of a decode step's sequences are cut into workgroups' stretches, worked out by
// every workgroup from seq_lens.  Compiled into decode_step_kernel (step.h), and for the host by
// the tests, which run the same functions over 64 emulated lanes: the wave-wide operations
// (wave_scan, wave_max, __ballot, readlane, readfirstlane), kWave and div_pos come from the file
// that includes this one.
#pragma once
#include <cstdint>

#include "step_plan.h"

namespace tq4 {
namespace xdl {

// What the cut depends on besides the grid.
struct CutArgs {
    const int32_t *seq_lens;
    int batch, num_splits;
    int sw;       // waves per head part (a power of two)
    int per_seq;  // workgroups there are per sequence (0: fewer than one)
};

// Run i of n over `tiles` tiles: [first, first + count), the first tiles % n runs one longer.
struct Run {
    int first, count;
};
__device__ __forceinline__ Run run_of(int tiles, int n, int i) {
    const int q = div_pos(tiles, n), r = tiles - q * n;
    return Run{i * q + min(i, r), q + (i < r ? 1 : 0)};
}

// One workgroup's stretch of the list.  Sequences with tiles count tiles + kSegmentTiles sw; the
// workgroup takes [x cell, (x + 1) cell) of that weight, and of sequence b, whose weight starts
// at `start`, the tiles that fall in it after the first kSegmentTiles sw.
struct Cut {
    int b;           // current sequence (its batch index); >= batch: done
    int len, tiles;
    uint32_t start;  // weight of the sequences before b
    uint32_t cell;   // weight per workgroup
    Run run;         // the workgroup's tiles of sequence b
    int p, n_parts;  // its part and the sequence's parts
};
__device__ __forceinline__ int tiles_of(int len) { return (max(len, 0) + 15) >> 4; }
__device__ __forceinline__ uint32_t weight_of(int tiles, int sw) {
    return tiles > 0 ? (uint32_t)(tiles + kSegmentTiles * sw) : 0u;
}
// Places the stretch in sequence c.b (c.len, c.start set).
__device__ __forceinline__ void place(Cut &c, int x, int sw) {
    c.tiles = tiles_of(c.len);
    const int64_t first = (int64_t)c.start + kSegmentTiles * sw, lo = (int64_t)x * c.cell - first;
    const int t0 = (int)max(lo, (int64_t)0), t1 = (int)min(lo + (int64_t)c.cell, (int64_t)c.tiles);
    c.run = Run{t0, max(t1 - t0, 0)};
    if (c.run.count > 0) {
        const int xf = (int)((uint32_t)first / c.cell), xl = (int)((uint32_t)(first + c.tiles - 1) / c.cell);
        c.p = x - xf;
        c.n_parts = xl - xf + 1;
    }
}
// The next sequence in the stretch with tiles for this workgroup; false when there is none.
__device__ __forceinline__ bool next_segment(Cut &c, const CutArgs &a, int x, bool inside) {
    const uint64_t end = (uint64_t)(x + 1) * c.cell;
    while (c.b < a.batch) {
        if (inside) {  // leave sequence b
            c.start += weight_of(tiles_of(c.len), a.sw);
            if (++c.b >= a.batch || c.start >= end)
                return false;
            c.len = a.seq_lens[c.b];
        }
        inside = true;
        place(c, x, a.sw);
        if (c.run.count > 0)
            return true;
    }
    return false;
}
// The first segment of workgroup x of nx.  `alone` (out): every sequence has workgroups of its own, so
// this one has no further segment.  len_lane: seq_lens[lane], read by the caller.
__device__ __forceinline__ bool first_segment(Cut &c, const CutArgs &a, int nx, int x, int lane, int len_lane,
                                              bool &alone) {
    const int32_t *sl = a.seq_lens;
    uint32_t total = 0, most = 0, w0 = 0, s0 = 0;  // (w0, s0: the first 64 sequences' weights and their scan)
    int l0 = 0;
    for (int c0 = 0; c0 < a.batch; c0 += kWave) {
        const int len = c0 + lane >= a.batch ? 0 : c0 == 0 ? len_lane : sl[c0 + lane];
        const int t = tiles_of(len);
        const uint32_t w = weight_of(t, a.sw), sc = wave_scan(w);
        if (c0 == 0) {
            l0 = len;
            w0 = w;
            s0 = sc;
        }
        total += (uint32_t)__builtin_amdgcn_readlane((int)sc, kWave - 1);
        most = max(most, wave_max((uint32_t)t));
    }
    if (most == 0)
        return false;
    const int least = kMinWaveTiles * a.sw;  // tiles below which a workgroup's waves run dry
    uint32_t cell = max((uint32_t)div_pos((int)(total + nx - 1), nx), (uint32_t)least);
    // at most num_splits parts: a sequence of T tiles touches at most (T - 1) / cell + 2 cells
    if ((uint64_t)cell * (uint32_t)(a.num_splits - 1) < most)
        cell = max(cell, (most + (uint32_t)a.num_splits - 2) / (uint32_t)(a.num_splits - 1));
    alone = false;
    if (a.per_seq > 0) {
        const int k = min(min(a.per_seq, a.num_splits), (int)div_pos((int)most + least - 1, least));
        // (3-bit keys, 48 sequences of 256 tiles on 256 workgroups: 5 each, 52 tiles, take 53.9 us;
        // stretches of 51 take 56.7)
        if ((uint32_t)div_pos((int)most + k - 1, k) <= cell + cell / 16) {
            alone = true;
            c.b = div_pos(x, k);
            if (c.b >= a.batch)
                return false;
            c.len = c.b < kWave ? __builtin_amdgcn_readlane(l0, c.b) : sl[c.b];
            c.tiles = tiles_of(c.len);
            c.p = x - c.b * k;
            c.n_parts = min(k, (int)div_pos(c.tiles + least - 1, least));
            if (c.p >= c.n_parts)
                return false;
            c.run = run_of(c.tiles, c.n_parts, c.p);
            return true;
        }
    }
    c.cell = cell;
    const uint64_t lo64 = (uint64_t)x * cell;
    if (lo64 >= total)
        return false;
    const uint32_t lo = (uint32_t)lo64;
    uint32_t carry = 0;
    for (int c0 = 0; c0 < a.batch; c0 += kWave) {
        int len = l0;
        uint32_t w = w0, sc = s0;
        if (c0 > 0) {
            len = c0 + lane < a.batch ? sl[c0 + lane] : 0;
            w = weight_of(tiles_of(len), a.sw);
            sc = wave_scan(w);
        }
        const uint32_t before = carry + sc - w;
        const uint64_t hit = __ballot(w > 0 && lo >= before && lo < before + w);
        if (hit) {
            const int l = __builtin_ctzll(hit);
            c.b = c0 + l;
            c.len = __builtin_amdgcn_readlane(len, l);
            c.start = (uint32_t)__builtin_amdgcn_readlane((int)before, l);
            return next_segment(c, a, x, false);
        }
        carry += (uint32_t)__builtin_amdgcn_readlane((int)sc, kWave - 1);
    }
    return false;
}

}  // namespace xdl
}  // namespace tq4
