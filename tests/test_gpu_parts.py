"""The full decode step's part rows: a sequence's 16-token tiles divided among its Stage1 waves,
one row per wave, merged by ``merge_parts_kernel``.

Sizes are where the division, the part count and the block-table guess can go wrong: lengths
around tile edges, fewer tiles than waves, as many parts as split rows (no count mark), more
parts than the merge reads at once, batches past the ranked deal's 64 sequences, blocks of
several tiles with full and partly used tables.  Bar, against the float64 / C oracle: 1e-4 on
outputs and LSE (fp32 outputs; the Stage1 requirement)."""
import numpy as np
import pytest
import torch

from conftest import to_dev
from oracle import native
from oracle import stage1 as ostage
from tq4_decode import ops, workloads

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
