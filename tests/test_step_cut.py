"""How a decode step is cut into workgroups (``step_plan`` in ``tq4_decode.hip``, ``first_segment`` /
``next_segment`` / ``run_of`` in ``step.h``), restated on the CPU with the constants read from the
sources: for any batch, every 16-token tile of every sequence falls to exactly one workgroup
and one of its waves, a sequence's parts are numbered 0 .. n-1 in order with one agreed n, and n
never exceeds the rows there are (``num_kv_splits``).
"""
import random
import re

import pytest

from conftest import ROOT

CSRC = ROOT / "turboquant-cuda-decode_amd" / "csrc"
STEP, HOST = (CSRC / "step.h").read_text(), (CSRC / "tq4_decode.hip").read_text()


def _const(text, name):
    return int(re.search(rf"constexpr int {name} = (\d+);", text).group(1))


SEGMENT, MIN_WAVE, WAVES = (_const(STEP, n) for n in ("kSegmentTiles", "kMinWaveTiles", "kStepWaves"))
SHORT, MERGE, MOST_PARTS = (_const(HOST, n) for n in ("kShortTiles", "kMergeTiles", "kMostParts"))
HELD = 256 * WAVES


def up(a, b):
    return -(-a // b)


def plan(batch, nvh, tiles, splits, most_vw, have_parts=True):
    pairs, vw, sw = nvh * batch, 1, 1
    while vw < most_vw and nvh % (2 * vw) == 0:
        vw *= 2
    rounds = up(pairs, HELD)
    full = 10 * pairs >= 9 * rounds * HELD
    if not full:
        while sw < WAVES and 2 * sw <= HELD // pairs:
            sw *= 2
    in_parts = max(MIN_WAVE, up(pairs * tiles, HELD))
    if full or not have_parts or splits == 1 or up(tiles, sw) <= min(SHORT, in_parts + MERGE):
        return dict(vw=min(vw, WAVES // sw), sw=sw, nx=batch, per_seq=1, whole=True)
    sw = 1
    while sw < WAVES and HELD > pairs * sw * min(MOST_PARTS, splits - 1):
        sw *= 2
    vw = min(vw, WAVES // sw)
    useful = batch * up(tiles, MIN_WAVE * sw)
    nx = max(1, min(HELD // (vw * sw) // (nvh // vw), useful))
    return dict(vw=vw, sw=sw, nx=nx, per_seq=nx // batch, whole=False)


def run_of(tiles, n, i):
    q, r = divmod(tiles, n)
    first = i * q + min(i, r)
    return first, first + q + (i < r)


def segments(lens, splits, p, x):
    """(sequence, first tile, end tile, part, parts) of workgroup x."""
    tiles = [(n + 15) >> 4 for n in lens]
    if p["whole"]:
        return [(x, 0, tiles[x], 0, 1)] if tiles[x] else []
    weights = [t + SEGMENT if t else 0 for t in tiles]
    most, least = max(tiles), MIN_WAVE * p["sw"]
    if most == 0:
        return []
    cell = max(up(sum(weights), p["nx"]), least)
    if cell * (splits - 1) < most:
        cell = max(cell, up(most, splits - 1))
    if len(set(lens)) == 1 and p["per_seq"] > 0:
        k = min(p["per_seq"], splits, up(most, least))
        if up(most, k) <= cell + cell // 16:
            b = x // k
            return [(b, *run_of(most, k, x - b * k), x - b * k, k)] if b < len(lens) else []
    out, start = [], 0
    for b, t in enumerate(tiles):
        first = start + SEGMENT
        lo = x * cell - first
        t0, t1 = max(lo, 0), min(lo + cell, t)
        if t and t1 > t0:
            xf, xl = first // cell, (first + t - 1) // cell
            out.append((b, t0, t1, x - xf, xl - xf + 1))
        start += weights[b]
    return out


@pytest.mark.parametrize("seed", range(8))
def test_every_tile_has_one_wave(seed):
    r = random.Random(seed)
    for _ in range(250):
        batch = r.choice([1, 2, 3, 5, 8, 13, 24, 48, 64, 65, 100, 130, 200, 256, 300, 520])
        nvh, splits = r.choice([1, 2, 3, 4, 5, 6, 8, 12, 16]), r.choice([1, 2, 3, 8, 16, 32, 64, 300])
        longest = r.choice([1, 10, 100, 1000, 8192, 32768])
        if r.random() < 0.3:
            lens = [r.randint(0, longest)] * batch
        else:
            lens = [r.choice([0, 1, 16, 17, r.randint(0, longest), r.randint(0, longest), longest])
                    for _ in range(batch)]
        table = max(1, up(max(lens), 16)) * r.choice([1, 1, 3])
        p = plan(batch, nvh, table, splits, r.choice([4, 8]), r.random() < 0.9)
        assert nvh % p["vw"] == 0 and p["vw"] * p["sw"] <= WAVES
        got = {}
        for x in range(p["nx"]):
            for b, t0, t1, part, parts in segments(lens, splits, p, x):
                assert 0 <= t0 < t1
                got.setdefault(b, []).append((t0, t1, part, parts))
                runs = [run_of(t1 - t0, p["sw"], s) for s in range(p["sw"])]
                assert runs[0][0] == 0 and runs[-1][1] == t1 - t0
                assert all(a[1] == c[0] for a, c in zip(runs, runs[1:]))
        for b, n in enumerate(lens):
            g, tiles = sorted(got.get(b, [])), (n + 15) >> 4
            assert bool(g) == bool(tiles)
            if not tiles:
                continue
            parts = g[0][3]
            assert [q[2] for q in g] == list(range(parts)) and len(g) == parts <= max(splits, 1)
            assert {q[3] for q in g} == {parts}
            assert g[0][0] == 0 and g[-1][1] == tiles and all(a[1] == c[0] for a, c in zip(g, g[1:]))
