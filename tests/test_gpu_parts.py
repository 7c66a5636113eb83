"""The full decode step as one kernel plus (where a sequence has several workgroups) the merge:
the list of all sequences' 16-token tiles cut into stretches, one row per workgroup and head.

Sizes are where the cut, the waves' runs, the part count and the block-table guess can go
wrong: lengths around tile edges, fewer tiles than waves, as many parts as rows (no count mark)
and more than the merge reads at once, stretches over several sequences and sequences over
several stretches, batches past 64 sequences and past the device, one to eight head parts per
workgroup, blocks of several tiles with full and partly used tables, tables much wider than the
lengths, waves with more tiles than address lanes (64) and than block-table entries in LDS (512).
Each case names the form that it is there for; ``test_step_cut`` checks on the CPU that the plan
and the cut give it.  Bar, against the float64 / C oracle: 1e-4 on outputs and LSE (fp32
outputs; the Stage1 requirement)."""
import numpy as np
import pytest
import torch

from conftest import to_dev
from oracle import native
from oracle import stage1 as ostage
from tq4_decode import aos_decode, codebook, ops, soa_decode, workloads
from tq4_decode.layout import slot_bytes_fp8, slot_bytes_preset

pytestmark = pytest.mark.gpu

EDGES = [1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 0, 1023]


def _mostly_short(n, **longer):
    lens = [5] * n
    for at, length in longer.items():
        lens[int(at[1:])] = length
    return lens


def _ragged(seed, lo, hi, n):
    return [int(v) for v in np.random.default_rng(seed).integers(lo, hi, n)]


# 512, 513, 1025 and 1063 tiles: the last position of a full table, one ring turn past it, a third table
PAST_TABLE = _mostly_short(256, s3=8192, s70=8200, s100=16400, s200=17003)
CASES = {
    # name: lengths, splits, kv-heads, group, block size, layout, table blocks (0: as the lengths need), form
    "tile edges": (EDGES, 32, 8, 4, 16, "soa", 0, dict(whole=True, sw=8)),
    "tile edges, aos": (EDGES, 32, 8, 4, 16, "aos", 0, dict(whole=True, sw=8)),
    "group of 8": (EDGES, 16, 4, 8, 16, "soa", 0, dict(whole=True, sw=8)),
    "two parts per kv-head": (EDGES[:6], 8, 2, 16, 16, "soa", 0, dict(whole=True, sw=8)),
    "tile edges, wide table": (EDGES, 32, 8, 4, 16, "soa", 2048, dict(whole=False, vw=4, sw=2, parts=8)),
    "tile edges, wide table, aos": (EDGES, 32, 8, 4, 16, "aos", 2048, dict(whole=False, vw=4, sw=2, parts=8)),
    "group of 8, wide table": (EDGES, 16, 4, 8, 16, "soa", 2048, dict(whole=False, vw=2, sw=4, parts=4)),
    "two parts per kv-head, wide table": (EDGES[:6], 8, 2, 16, 16, "soa", 600, dict(whole=False, parts=1)),
    "two rows": ([3000, 17, 16, 0, 1], 2, 8, 4, 16, "soa", 0, dict(whole=False, parts=2)),
    "as many parts as rows": ([3000, 2999, 17], 3, 8, 4, 16, "soa", 0, dict(whole=False, parts=3)),
    "more parts than one merge chunk": ([36000, 9000], 300, 1, 4, 16, "soa", 0, dict(whole=False, parts=71)),
    "runs of 20 tiles": ([5000, 4999, 4096, 1], 2, 8, 8, 16, "soa", 0, dict(whole=False, sw=8, wave_tiles=20)),
    "runs past the address lanes": (_mostly_short(256, s0=1024, s1=1040, s9=2100), 16, 8, 4, 16, "soa", 0,
                                    dict(whole=True, sw=1, wave_tiles=132)),
    "runs past the block-table entries": (PAST_TABLE, 16, 8, 4, 16, "soa", 0, dict(whole=True, sw=1, wave_tiles=1063)),
    "runs past the block-table entries, aos": (PAST_TABLE, 16, 8, 4, 16, "aos", 0,
                                               dict(whole=True, sw=1, wave_tiles=1063)),
    "runs past the block-table entries, blocks of 64": (PAST_TABLE, 16, 4, 16, 64, "soa", 0,
                                                        dict(whole=True, sw=1, wave_tiles=1063)),
    "parts past the block-table entries": ([140000, 100], 2, 1, 4, 16, "soa", 0,
                                           dict(whole=False, sw=8, parts=2, wave_tiles=547)),
    "equal, whole table, blocks of 64": ([2048] * 8, 32, 8, 4, 64, "soa", 0, dict(whole=False, parts=16, segs=1)),
    "equal, odd, blocks of 64": ([2041] * 64, 32, 8, 4, 64, "soa", 0, dict(whole=False, vw=8, sw=1, parts=4)),
    "equal, one tile": ([7] * 9, 32, 8, 4, 32, "soa", 0, dict(whole=True)),
    "all empty": ([0] * 5, 32, 8, 4, 16, "soa", 0, dict(whole=True)),
    "all empty, wide table": ([0] * 5, 32, 8, 4, 16, "soa", 500, dict(whole=False, parts=0)),
    "one long sequence": ([20011], 32, 8, 4, 16, "soa", 0, dict(whole=False, parts=32)),
    "one long sequence, one row": ([3001], 1, 8, 4, 16, "soa", 0, dict(whole=True)),
    "long and short": ([9000, 1, 40, 0, 700], 8, 4, 8, 16, "aos", 0, dict(whole=False, parts=8)),
    "three kv-heads": ([1500, 700, 1, 0, 90, 333], 32, 3, 4, 16, "soa", 0, dict(whole=False, vw=1, parts=3)),
    "five kv-heads, group of 6": ([1500, 700, 1, 0, 90, 333], 32, 5, 6, 16, "aos", 0, dict(whole=False, parts=3)),
    "five kv-heads, one wave": (_ragged(8, 1, 900, 100), 32, 5, 4, 16, "soa", 0,
                                dict(whole=False, vw=1, sw=1, rotates=False)),
    "one kv-head, two waves": (_ragged(9, 1, 4000, 64), 32, 1, 8, 16, "soa", 0,
                               dict(whole=False, vw=1, sw=2, rotates=False)),
    "eight waves of one head part": ([4000, 3000], 16, 1, 8, 32, "soa", 0, dict(whole=False, sw=8, parts=8)),
    "130 equal sequences": ([1000] * 130, 16, 8, 4, 16, "soa", 0, dict(whole=False, segs=2)),
    "130 ragged sequences": (_ragged(6, 0, 900, 130), 16, 8, 4, 16, "soa", 0, dict(whole=False, segs=2)),
    "300 ragged sequences": (_ragged(7, 0, 600, 300), 8, 8, 8, 16, "soa", 0, dict(whole=True)),
    "400 ragged sequences, wide table": (_ragged(10, 50, 1000, 400), 8, 8, 4, 16, "soa", 200, dict(whole=False, segs=4)),
    "one token each, 200 sequences, wide table": ([1] * 199 + [2000], 16, 8, 4, 16, "soa", 0, dict(whole=False, parts=11)),
    "ragged, 150 sequences": (_ragged(5, 0, 700, 150), 32, 2, 4, 16, "soa", 0, dict(whole=True, sw=4)),
    "ragged, 150 sequences, wide table": (_ragged(5, 0, 700, 150), 32, 2, 4, 16, "soa", 500, dict(whole=False, sw=1)),
}


def _widen(table, blocks):
    """The block table with at least ``blocks`` columns (zeros, as a backend's unused entries)."""
    if blocks <= table.shape[1]:
        return table
    out = np.zeros((table.shape[0], blocks), np.int32)
    out[:, :table.shape[1]] = table
    return out


@pytest.mark.parametrize("name", CASES)
def test_parts_match_the_oracle(dev, name):
    lens, splits, hk, group, block, layout, blocks, _ = CASES[name]
    seed = 900 + list(CASES).index(name)
    rng = np.random.default_rng(seed)
    batch, hq = len(lens), hk * group
    w = workloads.small(seed, batch, lens, splits, num_q_heads=hq, num_kv_heads=hk, block_size=block)
    cache = workloads.soa_to_aos(w.kv_cache, w.centroids, hk) if layout == "aos" else w.kv_cache
    query = torch.from_numpy(rng.standard_normal((batch, hq, 128)).astype(np.float32)).half()
    rot = workloads.random_orthogonal(rng, 128)
    t = lambda a: to_dev(a, dev)  # noqa: E731
    ws = ops.DecodeWorkspace(batch, hq, splits, dev, torch.float32)
    ws.mid_o.fill_(float("nan"))
    print(name, flush=True)
    out, lse = ops.full_decode(query.to(dev), t(rot), t(cache), t(_widen(w.block_table, blocks)), t(w.seq_lens),
                               t(w.centroids), splits, layout=layout, out_dtype=torch.float32, workspace=ws)
    torch.cuda.synchronize()
    q_rot = (query.double().numpy() @ rot.astype(np.float64)).astype(np.float32)
    mid = native.stage1(q_rot, cache, w.block_table, w.seq_lens, w.centroids, splits, num_kv_heads=hk,
                        block_size=block, is_aos=layout == "aos")
    ro, rl = native.stage2(mid, w.seq_lens)
    got, gl = out.cpu().numpy(), lse.cpu().numpy()
    live = w.seq_lens > 0
    assert np.isnan(got[~live]).all() and np.isneginf(gl[~live]).all()
    if live.any():
        assert np.abs(got[live] - ro[live]).max() <= 1e-4
        assert np.abs(gl[live] - rl[live]).max() <= 1e-4


SINK_LENS = [3000, 1, 16, 1333]  # parts: two sequences of several, two of one


def test_sinks_enter_the_first_part_only(dev):
    rng = np.random.default_rng(930)
    w = workloads.small(930, 4, SINK_LENS, 32)
    query = torch.from_numpy(rng.standard_normal((4, 32, 128)).astype(np.float32)).half()
    rot = workloads.random_orthogonal(rng, 128)
    sinks = rng.normal(0.0, 3.0, 32).astype(np.float32)
    t = lambda a: to_dev(a, dev)  # noqa: E731
    out, lse = ops.full_decode(query.to(dev), t(rot), t(w.kv_cache), t(w.block_table), t(w.seq_lens),
                               t(w.centroids), 32, out_dtype=torch.float32, sinks=t(sinks))
    torch.cuda.synchronize()
    q_rot = (query.double().numpy() @ rot.astype(np.float64)).astype(np.float32)
    ro, rl = ostage.stage2(ostage.stage1(q_rot, w.kv_cache, w.block_table, w.seq_lens, w.centroids, 1,
                                         num_kv_heads=8, sinks=sinks), w.seq_lens)
    assert np.abs(out.cpu().numpy() - ro).max() <= 1e-4
    assert np.abs(lse.cpu().numpy() - rl).max() <= 1e-4


# (lengths, splits, where a NaN norm goes): fewer parts than rows (the count mark is there), as many parts
# as rows (the last LSE has the slot that the mark would take), one part
NAN_CASES = [([3000, 2999, 17], 32, [(0, 0), (1, 2998)]), ([3000, 2999, 17], 3, [(0, 2999), (1, 5)]),
             ([3000, 2999, 17], 3, [(2, 16)])]


def _nan_case(dev, lens, splits, cache_bytes=None, sinks=None):
    """(out, lse) of the step on the cache as ``cache_bytes`` changes it, and the oracle's of the cache as it is."""
    rng = np.random.default_rng(935)
    w = workloads.small(935, len(lens), lens, splits)
    query = torch.from_numpy(rng.standard_normal((len(lens), 32, 128)).astype(np.float32)).half()
    rot = workloads.random_orthogonal(rng, 128)
    t = lambda a: to_dev(a, dev)  # noqa: E731
    q_rot = (query.double().numpy() @ rot.astype(np.float64)).astype(np.float32)
    finite = None if sinks is None else np.nan_to_num(sinks)
    ro, rl = ostage.stage2(ostage.stage1(q_rot, w.kv_cache, w.block_table, w.seq_lens, w.centroids, 1, num_kv_heads=8,
                                         sinks=finite), w.seq_lens)
    cache = w.kv_cache.copy().reshape(w.kv_cache.shape[0], -1)
    if cache_bytes:
        cache_bytes(cache, w.block_table)
    out, lse = ops.full_decode(query.to(dev), t(rot), t(cache.reshape(w.kv_cache.shape)), t(w.block_table),
                               t(w.seq_lens), t(w.centroids), splits, out_dtype=torch.float32,
                               sinks=None if sinks is None else t(sinks))
    torch.cuda.synchronize()
    return out.cpu().numpy(), lse.cpu().numpy(), ro, rl


@pytest.mark.parametrize("bits", [0x7E00, 0xFE00, 0xFFFF])
@pytest.mark.parametrize("lens,splits,at", NAN_CASES)
def test_a_nan_norm_stays_in_its_sequence_and_kv_head(dev, lens, splits, at, bits):
    """Its heads' outputs are NaN (their LSE is unspecified), all others as without it."""
    bs, hk, head = 16, 8, 3
    bad = np.zeros((len(lens), 32), bool)

    def put(cache, table):  # fp16 norms follow the block's records: [kv-head][norm, scale, zero][token]
        for b, token in at:
            word = bs * hk * 128 + head * 3 * bs * 2 + (token % bs) * 2
            cache[table[b, token // bs], word:word + 2] = np.array([bits], np.uint16).view(np.uint8)
            bad[b, 4 * head:4 * head + 4] = True

    got, gl, ro, rl = _nan_case(dev, lens, splits, put)
    assert bad.sum() == 4 * len(at) and np.isnan(got[bad]).all()
    assert np.abs(got[~bad] - ro[~bad]).max() <= 1e-4 and np.abs(gl[~bad] - rl[~bad]).max() <= 1e-4


@pytest.mark.parametrize("bits", [0x7FC00000, 0xFFC00000, 0xFFC00002, 0xFFFFFFFF])
@pytest.mark.parametrize("lens,splits", [c[:2] for c in NAN_CASES[:2]])
def test_a_nan_lse_is_not_taken_for_the_count_of_parts(dev, lens, splits, bits):
    """A NaN sink makes the first part's LSE NaN, and the count of parts is a NaN in a row's last LSE."""
    sinks = np.random.default_rng(936).normal(0.0, 3.0, 32).astype(np.float32)
    sinks[[5, 31]] = np.array([bits], np.uint32).view(np.float32)
    got, gl, ro, rl = _nan_case(dev, lens, splits, sinks=sinks)
    bad = np.isnan(sinks)
    assert np.isnan(got[:, bad]).all() and np.isnan(gl[:, bad]).all()
    assert np.abs(got[:, ~bad] - ro[:, ~bad]).max() <= 1e-4 and np.abs(gl[:, ~bad] - rl[:, ~bad]).max() <= 1e-4


def _preset_cache(dev, rng, bits, blocks, bs, hk, layout):
    """A cache written by the writer from random keys and values (every block full)."""
    kb, vb = bits
    slot = slot_bytes_fp8(128) if kb == 8 else slot_bytes_preset(128, kb, vb)
    cache = torch.zeros(blocks, bs, hk, slot, dtype=torch.uint8, device=dev)
    n = blocks * bs
    gen = torch.Generator(device=dev).manual_seed(int(rng.integers(1 << 31)))
    k, v = (torch.randn(n, hk, 128, generator=gen, device=dev).bfloat16() for _ in range(2))
    slots = torch.arange(n, dtype=torch.int32, device=dev)
    if kb == 8:
        return ops.store_fp8(k, v, cache, slots, layout=layout), None
    cents = to_dev(codebook.centroids(128, kb), dev)
    rot = to_dev(workloads.random_orthogonal(rng, 128), dev)
    ops.store_preset(k, v, cache, slots, rot, to_dev(codebook.midpoints(128, kb), dev), cents, key_bits=kb,
                     value_bits=vb, layout=layout, norm_correction=layout == "soa")
    return cache, cents


# (layout, kv-heads, group, block size, lengths, form: None on the VALU kernel, which block size 8 takes: rotation or
# conversion, Stage1 and Stage2 as before)
MANY = _ragged(12, 1, 2000, 70)
PRESET_CASES = [
    ("soa", 8, 4, 16, EDGES, dict(whole=True)), ("aos", 8, 4, 16, EDGES, dict(whole=True)),
    ("soa", 4, 8, 32, EDGES, dict(whole=True)), ("aos", 4, 6, 16, EDGES, dict(whole=True)),
    ("soa", 2, 16, 16, [700] * 5, dict(whole=True)), ("soa", 8, 4, 8, EDGES[:6], None),
    ("soa", 8, 4, 16, [40] * 300, dict(whole=True, sw=1)),
    ("soa", 8, 4, 16, MANY, dict(whole=False, vw=4, sw=1, segs=2)),
    ("aos", 8, 4, 16, MANY, dict(whole=False, vw=4, sw=1, segs=2)),
    ("soa", 2, 16, 32, MANY, dict(whole=False, vw=4, sw=1, parts=11)),
    ("aos", 1, 8, 16, MANY, dict(whole=False, vw=1, sw=2, rotates=False)),
    ("soa", 8, 4, 16, [3000, 17, 1333], dict(whole=False, vw=1, sw=8)),
    ("soa", 8, 4, 16, PAST_TABLE, dict(whole=True, vw=4, sw=1, wave_tiles=1063)),
]


@pytest.mark.parametrize("layout,hk,group,bs,lens", [
    pytest.param(*c[:5], id=f"{c[0]}-{c[1]}-{c[2]}-{c[3]}-{i}") for i, c in enumerate(PRESET_CASES)])
@pytest.mark.parametrize("bits", [(8, 4), (3, 4), (3, 3)])
@pytest.mark.parametrize("view", ["contiguous", "strided", "off by 2 bytes", "sinks"])
def test_preset_step_matches_the_separate_launches(dev, bits, layout, hk, group, bs, lens, view):
    """Outputs in fp16 against Stage1 over 16 splits + Stage2: both merge fp32 sums, so they differ
    by 1e-5 before the last rounding and by one fp16 unit (2^-10) after it."""
    if view == "off by 2 bytes" and bits != (8, 4):
        pytest.skip("the rotation takes 16-byte aligned queries")
    rng = np.random.default_rng(940 + bits[0] + hk)
    batch, hq = len(lens), hk * group
    need = [max(1, -(-n // bs)) for n in lens]
    cache, cents = _preset_cache(dev, rng, bits, sum(need), bs, hk, layout)
    table = np.zeros((batch, max(need)), np.int32)
    perm = rng.permutation(sum(need))
    for b, n in enumerate(need):
        table[b, :n] = perm[sum(need[:b]):sum(need[:b]) + n]
    bt, sl = to_dev(table, dev), to_dev(np.asarray(lens, np.int32), dev)
    x = to_dev(rng.standard_normal(batch * hq * 128 * 2 + 1).astype(np.float32), dev).half()
    if view == "strided":
        query = x[1:].view(batch, hq, 256)[:, :, ::2]
    else:
        query = x[1 if "off" in view else 0:][:batch * hq * 128].view(batch, hq, 128)
    pit = to_dev(workloads.random_orthogonal(rng, 128), dev)
    sinks = to_dev(rng.normal(0.0, 3.0, hq).astype(np.float32), dev) if view == "sinks" else None
    entry = (soa_decode if layout == "soa" else aos_decode).triton_turboquant_decode_attention
    print(bits, view, flush=True)
    got = entry(query, cache, bt, sl, pit.t().contiguous(), cents, 128 ** -0.5, bits[0],
                128 if bits[0] == 8 else 16 * bits[0] + 2, bits[1], key_fp8=bits[0] == 8, norm_correction=True,
                PiT=pit, max_num_kv_splits=16, sinks=sinks)
    if bits[0] == 8:
        mid = ops.stage1_fp8(query.float().contiguous(), cache, bt, sl, num_kv_splits=16, layout=layout,
                             sinks=sinks)
    else:
        mid = ops.stage1_preset(ops.rotate_query(query.contiguous(), pit), cache, bt, sl, cents, key_bits=bits[0],
                                value_bits=bits[1], num_kv_splits=16, layout=layout, sinks=sinks)
    ref, _ = ops.stage2(mid, sl)
    torch.cuda.synchronize()
    a, r = got.float().cpu().numpy(), ref.cpu().numpy()
    live = np.asarray(lens) > 0
    assert np.isnan(a[~live]).all()
    assert np.all(np.abs(a[live] - r[live]) <= 1e-5 + 2.0 ** -10 * np.abs(r[live]))
