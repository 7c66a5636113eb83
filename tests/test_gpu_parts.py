"""The full decode step as one kernel plus (where a sequence has several workgroups) the merge:
the list of all sequences' 16-token tiles cut into equal stretches, one row per workgroup and
head.

Sizes are where the cut, the waves' runs, the part count and the block-table guess can go
wrong: lengths around tile edges, fewer tiles than waves, as many parts as rows (no count mark)
and more than the merge reads at once, stretches over several sequences and sequences over
several stretches, batches past 64 sequences and past the device, one to eight head parts per
workgroup, blocks of several tiles with full and partly used tables.  Bar, against the float64 /
C oracle: 1e-4 on outputs and LSE (fp32 outputs; the Stage1 requirement)."""
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
CASES = {
    # name: lengths, splits, kv-heads, group, block size, layout
    "tile edges": (EDGES, 32, 8, 4, 16, "soa"),
    "tile edges, aos": (EDGES, 32, 8, 4, 16, "aos"),
    "group of 8": (EDGES, 16, 4, 8, 16, "soa"),
    "two parts per kv-head": (EDGES[:6], 8, 2, 16, 16, "soa"),
    "two rows": ([3000, 17, 16, 0, 1], 2, 8, 4, 16, "soa"),
    "as many parts as rows": ([512] * 4, 32, 8, 4, 16, "soa"),
    "more parts than one merge chunk": ([9001], 300, 1, 4, 16, "soa"),
    "chunks of 64 tiles": ([5000, 4999, 4096, 1], 2, 8, 8, 16, "soa"),
    "equal, whole table, blocks of 64": ([2048] * 8, 32, 8, 4, 64, "soa"),
    "equal, odd, blocks of 64": ([2041] * 64, 32, 8, 4, 64, "soa"),
    "equal, one tile": ([7] * 9, 32, 8, 4, 32, "soa"),
    "all empty": ([0] * 5, 32, 8, 4, 16, "soa"),
    "one long sequence": ([20011], 32, 8, 4, 16, "soa"),
    "one long sequence, one row": ([3001], 1, 8, 4, 16, "soa"),
    "long and short": ([9000, 1, 40, 0, 700], 8, 4, 8, 16, "aos"),
    "three kv-heads": ([1500, 700, 1, 0, 90, 333], 32, 3, 4, 16, "soa"),
    "five kv-heads, group of 6": ([1500, 700, 1, 0, 90, 333], 32, 5, 6, 16, "aos"),
    "eight waves of one head part": ([4000, 3000], 16, 1, 8, 32, "soa"),
    "130 equal sequences": ([1000] * 130, 16, 8, 4, 16, "soa"),
    "130 ragged sequences": (list(np.random.default_rng(6).integers(0, 900, 130)), 16, 8, 4, 16, "soa"),
    "300 ragged sequences": (list(np.random.default_rng(7).integers(0, 600, 300)), 8, 8, 8, 16, "soa"),
    "one token each, 200 sequences, wide table": ([1] * 199 + [2000], 16, 8, 4, 16, "soa"),
    "ragged, 150 sequences": (list(np.random.default_rng(5).integers(0, 700, 150)), 32, 2, 4, 16, "soa"),
}


@pytest.mark.parametrize("name", CASES)
def test_parts_match_the_oracle(dev, name):
    lens, splits, hk, group, block, layout = CASES[name]
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
    out, lse = ops.full_decode(query.to(dev), t(rot), t(cache), t(w.block_table), t(w.seq_lens), t(w.centroids),
                               splits, layout=layout, out_dtype=torch.float32, workspace=ws)
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


def test_sinks_enter_the_first_part_only(dev):
    rng = np.random.default_rng(930)
    lens = [700, 1, 16, 333]
    w = workloads.small(930, 4, lens, 32)
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


def _preset_cache(dev, rng, bits, blocks, bs, hk, layout):
    """A cache written by the writer from random keys and values (every block full)."""
    kb, vb = bits
    slot = slot_bytes_fp8(128) if kb == 8 else slot_bytes_preset(128, kb, vb)
    cache = torch.zeros(blocks, bs, hk, slot, dtype=torch.uint8, device=dev)
    n = blocks * bs
    k, v = (to_dev(rng.standard_normal((n, hk, 128)).astype(np.float32), dev).bfloat16() for _ in range(2))
    slots = torch.arange(n, dtype=torch.int32, device=dev)
    if kb == 8:
        return ops.store_fp8(k, v, cache, slots, layout=layout), None
    cents = to_dev(codebook.centroids(128, kb), dev)
    rot = to_dev(workloads.random_orthogonal(rng, 128), dev)
    ops.store_preset(k, v, cache, slots, rot, to_dev(codebook.midpoints(128, kb), dev), cents, key_bits=kb,
                     value_bits=vb, layout=layout, norm_correction=layout == "soa")
    return cache, cents


# (block size 8 runs on the VALU kernel: rotation or conversion, Stage1 and Stage2 as before)
@pytest.mark.parametrize("layout,hk,group,bs,lens", [
    ("soa", 8, 4, 16, EDGES), ("aos", 8, 4, 16, EDGES), ("soa", 4, 8, 32, EDGES), ("aos", 4, 6, 16, EDGES),
    ("soa", 2, 16, 16, [700] * 5), ("soa", 8, 4, 8, EDGES[:6]), ("soa", 8, 4, 16, [40] * 300)])
@pytest.mark.parametrize("bits", [(8, 4), (3, 4), (3, 3)])
@pytest.mark.parametrize("view", ["contiguous", "strided", "off by 2 bytes"])
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
    entry = (soa_decode if layout == "soa" else aos_decode).triton_turboquant_decode_attention
    got = entry(query, cache, bt, sl, pit.t().contiguous(), cents, 128 ** -0.5, bits[0],
                128 if bits[0] == 8 else 16 * bits[0] + 2, bits[1], key_fp8=bits[0] == 8, norm_correction=True,
                PiT=pit, max_num_kv_splits=16)
    if bits[0] == 8:
        mid = ops.stage1_fp8(query.float().contiguous(), cache, bt, sl, num_kv_splits=16, layout=layout)
    else:
        mid = ops.stage1_preset(ops.rotate_query(query.contiguous(), pit), cache, bt, sl, cents, key_bits=bits[0],
                                value_bits=bits[1], num_kv_splits=16, layout=layout)
    ref, _ = ops.stage2(mid, sl)
    torch.cuda.synchronize()
    a, r = got.float().cpu().numpy(), ref.cpu().numpy()
    live = np.asarray(lens) > 0
    assert np.isnan(a[~live]).all()
    assert np.all(np.abs(a[live] - r[live]) <= 1e-5 + 2.0 ** -10 * np.abs(r[live]))
