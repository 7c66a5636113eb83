"""How a decode step is cut into workgroups: ``step_plan`` and the kernel's own ``first_segment`` /
``next_segment`` / ``run_of``, built for the host (``step_cut_host``).  For any batch, every
16-token tile of every sequence falls to exactly one workgroup and one of its waves, a
sequence's parts are numbered 0 .. n-1 in order with one agreed n, and n never exceeds the rows
there are (``num_kv_splits``).
"""
import random

import pytest

import step_cut_host as host
import test_gpu_parts as parts


def up(a, b):
    return -(-a // b)


def check_cut(lens, splits, p):
    got = {}
    for x in range(p.nx):
        for b, t0, t1, part, parts in host.segments(lens, splits, p, x):
            assert 0 <= t0 < t1
            got.setdefault(b, []).append((t0, t1, part, parts))
            runs = [host.run_of(t1 - t0, p.sw, s) for s in range(p.sw)]
            assert runs[0][0] == 0 and runs[-1][1] == t1 - t0
            assert all(a[1] == c[0] for a, c in zip(runs, runs[1:]))
    for b, n in enumerate(lens):
        g, tiles = sorted(got.get(b, [])), (max(n, 0) + 15) >> 4
        assert bool(g) == bool(tiles)
        if not tiles:
            continue
        parts = g[0][3]
        assert [q[2] for q in g] == list(range(parts)) and len(g) == parts <= max(splits, 1)
        assert {q[3] for q in g} == {parts}
        assert g[0][0] == 0 and g[-1][1] == tiles and all(a[1] == c[0] for a, c in zip(g, g[1:]))


@pytest.mark.parametrize("seed", range(8))
def test_every_tile_has_one_wave(seed):
    r = random.Random(seed)
    for _ in range(60):
        batch = r.choice([1, 2, 3, 5, 8, 13, 24, 48, 64, 65, 100, 130, 200, 256, 300, 520])
        nvh, splits = r.choice([1, 2, 3, 4, 5, 6, 8, 12, 16]), r.choice([1, 2, 3, 8, 16, 32, 64, 300])
        longest = r.choice([1, 10, 100, 1000, 8192, 32768])
        if r.random() < 0.3:
            lens = [r.randint(0, longest)] * batch
        else:
            lens = [r.choice([0, 1, 16, 17, r.randint(0, longest), r.randint(0, longest), longest, -1])
                    for _ in range(batch)]
        bs = r.choice([16, 16, 64])
        blocks = max(1, up(max(lens), bs)) * r.choice([1, 1, 3, 40])
        p = host.plan(batch, nvh, blocks, splits, block_size=bs, whole_lines=r.random() < 0.5,
                      have_parts=r.random() < 0.9)
        assert nvh % p.vw == 0 and p.vw * p.sw <= host.waves()
        check_cut(lens, splits, p)


def test_the_host_build_sees_more_than_64_sequences_and_long_lists():
    """The carry past the first 64 sequences, and weights beyond 2^24 tiles."""
    for lens in ([16 * (1 + i % 7) for i in range(200)], [2 ** 24 * 3] * 5 + [1] * 70, [0] * 64 + [5000] * 70):
        check_cut(lens, 32, host.plan(len(lens), 8, up(max(lens), 16), 32))


@pytest.mark.parametrize("nvh", [1, 2, 3, 4, 5, 6, 8, 12, 16])
def test_small_workgroups_do_not_rotate_the_query(nvh):
    """One or two waves would stage the rotation matrix in eight or four rounds for every segment.  Four
    waves and more keep the rotation, and so does the one workgroup of a whole sequence."""
    for batch in (1, 2, 8, 16, 64, 128, 256, 400):
        for blocks, splits in ((20, 32), (256, 32), (2048, 16), (256, 2), (256, 1)):
            for lines in (True, False):
                p = host.plan(batch, nvh, blocks, splits, whole_lines=lines)
                assert p.rotates == (p.vw * p.sw >= 4 or (p.whole and p.vw == nvh))
    p = host.plan(64, nvh, 500, 32)  # 64 sequences of up to 8000 tokens: one wave per head part (two for one part)
    assert p.rotates == (nvh % 4 == 0)


@pytest.mark.parametrize("batch,nvh,lo,hi,table,splits,most", [
    (16, 1, 30, 500, 2048, 32, 1),    # short sequences under a backend's wide table: a workgroup each
    (64, 8, 250, 4000, 250, 2, 1),    # two rows per sequence leave no room for stretches
    (64, 8, 3900, 4096, 256, 32, 4),
    (16, 8, 30, 500, 2048, 32, 8),
])
def test_sequences_have_workgroups_of_their_own(batch, nvh, lo, hi, table, splits, most):
    """Where that is no slower no workgroup takes a second segment, and no sequence more than `most`."""
    lens = [lo + (hi - lo) * i // (batch - 1) for i in range(batch)]
    p = host.plan(batch, nvh, table, splits)
    assert not p.whole
    cut = [host.segments(lens, splits, p, x) for x in range(p.nx)]
    assert max(len(c) for c in cut) == 1
    assert max(s[4] for c in cut for s in c) == most
    check_cut(lens, splits, p)


@pytest.mark.parametrize("batch,lo,hi", [(64, 512, 8192), (140, 4000, 4000), (200, 100, 2000), (100, 200, 3000)])
def test_uneven_batches_are_cut_into_stretches(batch, lo, hi):
    lens = [lo + (hi - lo) * i // (batch - 1) for i in range(batch)]
    p = host.plan(batch, 8, up(hi, 16), 32)
    assert not p.whole
    assert max(len(host.segments(lens, 32, p, x)) for x in range(p.nx)) > 1


@pytest.mark.parametrize("batch,nvh,tokens,whole", [
    (200, 8, 500, True), (200, 8, 2000, False), (135, 8, 350, True), (135, 8, 700, False), (220, 8, 1000, True),
    (128, 8, 500, False), (400, 4, 700, True), (520, 8, 600, True), (520, 4, 600, True), (520, 4, 1500, False), (300, 8, 300, True),
    (400, 8, 1000, False),
    (256, 6, 700, True), (256, 6, 4000, False)])
def test_batches_past_half_a_round_stay_whole_for_small_tables(batch, nvh, tokens, whole):
    """One wave per head part: a second segment and the merge cost more than even stretches gain."""
    p = host.plan(batch, nvh, up(tokens, 16), 32)
    assert p.whole == whole
    assert not whole or p.sw == 1


def form(lens, splits, hk, group, block, whole_lines, blocks=0):
    nvh = hk * (1 if group <= 4 else up(group, 8))
    p = host.plan(len(lens), nvh, max(blocks, 1, up(max(lens), block)), splits, block_size=block,
                  whole_lines=whole_lines)
    cut = [host.segments(lens, splits, p, x) for x in range(p.nx)]
    return dict(whole=p.whole, vw=p.vw, sw=p.sw, rotates=p.rotates, segs=max(len(c) for c in cut),
                parts=max((s[4] for c in cut for s in c), default=0),
                wave_tiles=max((up(s[2] - s[1], p.sw) for c in cut for s in c), default=0))


@pytest.mark.parametrize("name", parts.CASES)
def test_gpu_cases_take_the_form_they_name(name):
    lens, splits, hk, group, block, layout, blocks, expected = parts.CASES[name]
    got = form(lens, splits, hk, group, block, layout == "soa", blocks)
    assert {k: got[k] for k in expected} == expected


@pytest.mark.parametrize("layout,hk,group,bs,lens,expected", parts.PRESET_CASES)
def test_gpu_preset_cases_take_the_form_they_name(layout, hk, group, bs, lens, expected):
    if expected is not None:
        got = form(lens, 16, hk, group, bs, False)
        assert {k: got[k] for k in expected} == expected


def test_gpu_sink_and_nan_cases_run_in_parts():
    got = form(parts.SINK_LENS, 32, 8, 4, 16, True)
    assert not got["whole"] and got["parts"] > 1
    for lens, splits, _ in parts.NAN_CASES:
        got = form(lens, splits, 8, 4, 16, True)
        assert not got["whole"] and got["parts"] == min(splits, 6)


@pytest.mark.parametrize("batch,hk,lo,hi", [(12, 2, 888, 14213), (3, 1, 93, 1500), (16, 1, 312, 5000), (24, 2, 94, 1500)])
def test_a_segment_costs_every_wave_of_a_head_part(batch, hk, lo, hi):
    """Workgroups of several waves per head part: a second segment takes as long as with one wave, in which
    they do as many times the tiles, so a stretch is worth cutting short of the next sequence."""
    lens = [lo + (hi - lo) * i // (batch - 1) for i in range(batch)]
    p = host.plan(batch, hk, up(hi, 16), 32)
    assert not p.whole and p.sw > 1
    assert max(len(host.segments(lens, 32, p, x)) for x in range(p.nx)) == 1
