"""The work whose speed counts: decode attention over the quantised paged cache and the cache
writer, through the entry points a serving backend calls.

Kinds:

* ``decode``: one attention step of a layer, ``triton_turboquant_decode_attention`` of
  ``tq4_decode.soa_decode`` / ``aos_decode`` (rotation, Stage1, Stage2; output rows in the
  query type), with the workspaces on the layer's ``buf_holder``;
* ``stage1``: the split attention alone, ``launch_tq4_v2_stage1``;
* ``store``: the cache writer, ``triton_turboquant_store`` of ``soa_store`` / ``aos_store``.

Presets: ``4bit`` (4-bit K and V), ``k8v4`` (FP8 keys), ``k3v4`` and ``3bit``.  Layouts: ``soa``,
``aos``, and ``aos_heads`` (the ``transpose(1, 2)`` view of head-major AoS blocks that the
backend passes).  Caches hold what the writer leaves for Gaussian keys and values: Lloyd-Max
codes of N(0, 1/128) coordinates, min / max 4- or 3-bit value codes, fp16 scalars; block tables
are random permutations of the pool.
"""
import math
import os
import sys
import types

import torch

_PKG = os.path.join(os.getcwd(), "turboquant-cuda-decode_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from tq4_decode import aos_decode, aos_store, codebook, ops, soa_decode, soa_store  # noqa: E402

D = 128
BITS = {"4bit": (4, 4), "k8v4": (8, 4), "k3v4": (3, 4), "3bit": (3, 3)}
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
MOST_TOKEN_HEADS = 256 * 2048 * 8  # (token, kv-head) records of the largest decode case
MOST_STORE_ROWS = 65536 * 8        # (token, kv-head) rows of the largest writer case


def _decode(name, batch, ctx, hq, hk, splits, layout="soa", preset="4bit", dtype="bf16", lo=0, block=16,
            sinks=False, kind="decode"):
    """``lo`` > 0: ragged lengths, spread evenly over [lo, ctx]."""
    case = dict(kind=kind, batch=batch, ctx=ctx, lo=lo, hq=hq, hk=hk, splits=splits, layout=layout,
                preset=preset, dtype=dtype, block=block, sinks=sinks)
    return dict(name=name, **case) if name else case


def _store(name, tokens, hk, layout="soa", preset="4bit", dtype="bf16", block=16):
    case = dict(kind="store", tokens=tokens, hk=hk, layout=layout, preset=preset, dtype=dtype, block=block)
    return dict(name=name, **case) if name else case


def listed():
    return [
        # one user typing: a single short sequence, where launches and latency are everything
        _decode("decode_b1_ctx333", 1, 333, 32, 8, 32),
        # one user with a long document
        _decode("decode_b1_ctx32768", 1, 32768, 32, 8, 32),
        # the reference's headline shape as a full step
        _decode("decode_b64_ctx4096", 64, 4096, 32, 8, 32),
        # continuous batching: every sequence at another length
        _decode("decode_ragged_b64", 64, 8192, 32, 8, 32, lo=512),
        # a throughput server's large batch; fp16, fewer splits
        _decode("decode_b256_ctx2048", 256, 2048, 32, 8, 16, dtype="fp16"),
        # the same step over the array-of-slots cache that the backend keeps by default
        _decode("decode_aos_b64_ctx4096", 64, 4096, 32, 8, 32, layout="aos"),
        # FP8 keys, a moderate ragged batch with a GQA group of 8
        _decode("decode_k8v4_ragged_b24", 24, 6001, 64, 8, 32, preset="k8v4", lo=1001),
        # the 3-bit preset for caches that have to be small
        _decode("decode_3bit_b48_ctx4096", 48, 4096, 32, 8, 32, preset="3bit"),
        # long contexts, Stage1 alone with a GQA group of 8
        _decode("stage1_gqa8_b8_ctx32768", 8, 32768, 64, 8, 64, kind="stage1"),
        # the writer in a decode step: one token for each of 64 sequences
        _store("store_decode_64", 64, 8),
        # the writer behind a prefill chunk, an odd number of tokens
        _store("store_chunk_8191", 8191, 8),
        # the writer behind a large batched prefill
        _store("store_prefill_65536", 65536, 8),
    ]


def _log_uniform(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    preset = rng.choice(["4bit", "4bit", "4bit", "k8v4", "k3v4", "3bit"])
    layout = rng.choice(["soa", "soa", "aos", "aos_heads"])
    block = rng.choice([16, 16, 32, 64])
    if rng.random() < 0.3:
        hk = rng.choice([2, 4, 8])
        return _store(None, _log_uniform(rng, 1, MOST_STORE_ROWS // 8 // 2), hk, layout, preset,
                      rng.choice(["bf16", "bf16", "fp16", "fp32"]), block)
    hk = rng.choice([1, 2, 4, 8, 8])
    group = rng.choice([1, 2, 4, 4, 6, 8, 16]) if hk < 8 else rng.choice([2, 4, 4, 6, 8])
    splits = rng.choice([8, 16, 32, 32, 64])
    batch = _log_uniform(rng, 1, 256)
    while batch * hk * group * splits > 256 * 32 * 16:  # rows of split results
        splits //= 2
    room = MOST_TOKEN_HEADS // 2 // (batch * hk * max(1, group // 4))
    ctx = min(_log_uniform(rng, 17, 32768), room)
    lo = max(1, ctx // 16) if batch > 1 and rng.random() < 0.5 else 0
    return _decode(None, batch, ctx, hk * group, hk, splits, layout, preset, rng.choice(["bf16", "fp16"]), lo,
                   block, rng.random() < 0.15)


def _slot_bytes(preset):
    kb, vb = BITS[preset]
    return D * kb // 8 + (0 if preset == "k8v4" else 2) + D * vb // 8 + 4


def _lengths(case):
    """The batch's lengths in increasing order (a seed permutes them)."""
    n, lo, hi = case["batch"], case["lo"], case["ctx"]
    if lo <= 0 or n == 1:
        return [hi] * n
    return [lo + (hi - lo) * i // (n - 1) for i in range(n)]


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) % (1 << 62))


def _rotation(gen):
    q, r = torch.linalg.qr(torch.randn(D, D, generator=gen, device="cuda", dtype=torch.float64).cpu())
    return (q * torch.sign(torch.diagonal(r))).float().cuda().contiguous()


def _codebook(preset):
    bits = BITS[preset][0]
    if bits == 8:
        return None, None
    return (torch.from_numpy(codebook.centroids(D, bits).copy()).cuda(),
            torch.from_numpy(codebook.midpoints(D, bits).copy()).cuda())


def _pack(codes, bits):
    """Codes [..., 128] -> bytes, least significant bits first."""
    if bits == 4:
        return codes[..., 0::2] | (codes[..., 1::2] << 4)
    c = codes.reshape(codes.shape[:-1] + (D // 8, 8)).to(torch.int32)
    word = sum(c[..., i] << (3 * i) for i in range(8))
    out = torch.stack([word & 255, (word >> 8) & 255, word >> 16], dim=-1).to(torch.uint8)
    return out.reshape(codes.shape[:-1] + (D * 3 // 8,))


def _lay_out(k, v, fields, layout):
    """Blocks [n, bs * hk * slot] from K / V bytes [n, bs, hk, .] and fp16 scalars [n, bs, hk] (SoA: data
    records, then [hk][field][bs]; AoS: K, norm, V, scale, zero in each slot)."""
    n = k.shape[0]
    as_bytes = lambda t: t.contiguous().view(torch.uint8)  # noqa: E731
    if layout == "soa":
        meta = torch.stack([f.transpose(1, 2) for f in fields], dim=2)  # [n, hk, field, bs]
        return torch.cat([torch.cat([k, v], dim=-1).reshape(n, -1), as_bytes(meta).reshape(n, -1)], dim=1)
    cells = [as_bytes(f.unsqueeze(-1)) for f in fields]
    slots = torch.cat([k] + cells[:-2] + [v] + cells[-2:], dim=-1)
    return (slots.transpose(1, 2) if layout == "aos_heads" else slots).reshape(n, -1)


def _fill_cache(case, gen, blocks, keep):
    """The cache tensor of `blocks` blocks, and with `keep` also the unpacked codes and scalars."""
    bs, hk, preset, layout = case["block"], case["hk"], case["preset"], case["layout"]
    kb, vb = BITS[preset]
    cents, mids = _codebook(preset)
    cache = torch.empty(blocks, bs * hk * _slot_bytes(preset), dtype=torch.uint8, device="cuda")
    kept = []
    step = max(1, (1 << 25) // (bs * hk * D))
    for b0 in range(0, blocks, step):
        shape = (min(step, blocks - b0), bs, hk)
        x = torch.randn(shape + (D,), generator=gen, device="cuda")
        fields = []
        if preset == "k8v4":
            kc = x.to(torch.float8_e4m3fn).view(torch.uint8)
            kbytes = kc
        else:
            kc = torch.bucketize(x * (1.0 / math.sqrt(D)), mids, right=True, out_int32=True)
            norm = 8.0 + 6.0 * torch.rand(shape, generator=gen, device="cuda")
            if layout == "soa":  # the norm of the decoded direction folded in
                norm = norm / cents[kc].square().sum(-1).sqrt()
            fields.append(norm.half())
            kc = kc.to(torch.uint8)
            kbytes = _pack(kc, kb)
        x = torch.randn(shape + (D,), generator=gen, device="cuda")
        zero, top = x.amin(-1), (1 << vb) - 1
        scale = (x.amax(-1) - zero) / top
        vc = ((x - zero[..., None]) / scale[..., None] + 0.5).clamp(0, top).to(torch.uint8)
        fields += [scale.half(), zero.half()]
        cache[b0:b0 + shape[0]] = _lay_out(kbytes, _pack(vc, vb), fields, layout)
        if keep:
            kept.append((kc, vc, fields))
    raw = None
    if keep:
        raw = (torch.cat([k for k, _, _ in kept]), torch.cat([v for _, v, _ in kept]),
               [torch.cat([f[i] for _, _, f in kept]) for i in range(len(kept[0][2]))])
    if layout == "aos_heads":
        return cache.view(blocks, hk, bs, -1).transpose(1, 2), raw
    return cache.view(blocks, bs, hk, -1), raw


def _decode_inputs(case, seed, keep=False):
    gen = _generator(seed)
    bs, n = case["block"], case["batch"]
    order = torch.randperm(n, generator=gen, device="cuda").cpu()
    lens = torch.tensor(_lengths(case), dtype=torch.int32)[order]
    need = (lens + bs - 1) // bs
    pool = int(need.sum())
    pages = torch.randperm(pool, generator=gen, device="cuda").to(torch.int32)
    table = torch.zeros(n, int(need.max()), dtype=torch.int32, device="cuda")
    at = 0
    for b, k in enumerate(need.tolist()):
        table[b, :k] = pages[at:at + k]
        at += k
    cache, raw = _fill_cache(case, gen, pool, keep)
    dtype = DTYPES[case["dtype"]] if case["kind"] == "decode" else torch.float32
    query = torch.randn(n, case["hq"], D, generator=gen, device="cuda").to(dtype)
    pi_t = _rotation(gen)
    sinks = torch.randn(case["hq"], generator=gen, device="cuda") if case["sinks"] else None
    return dict(query=query, cache=cache, table=table, lens=lens.cuda(), pi_t=pi_t, sinks=sinks, raw=raw)


def _store_inputs(case, seed):
    gen = _generator(seed)
    n, hk, bs = case["tokens"], case["hk"], case["block"]
    blocks = (n + bs - 1) // bs + 7
    dtype = DTYPES[case["dtype"]]
    key = torch.randn(n, hk, D, generator=gen, device="cuda")
    key *= 0.5 + torch.rand(n, hk, 1, generator=gen, device="cuda")
    value = torch.randn(n, hk, D, generator=gen, device="cuda")
    if n >= 1024:  # prefill: whole pages in order, pages anywhere in the pool
        pages = torch.randperm(blocks, generator=gen, device="cuda")
        slots = (pages[:, None] * bs + torch.arange(bs, device="cuda")).reshape(-1)[:n]
    else:          # decode: one token in each of n sequences' own pages
        slots = torch.randperm(blocks * bs, generator=gen, device="cuda")[:n]
    shape = (blocks, hk, bs) if case["layout"] == "aos_heads" else (blocks, bs, hk)
    cache = torch.zeros(shape + (_slot_bytes(case["preset"]),), dtype=torch.uint8, device="cuda")
    if case["layout"] == "aos_heads":
        cache = cache.transpose(1, 2)
    return dict(key=key.to(dtype), value=value.to(dtype), cache=cache, slots=slots.to(torch.int32),
                pi_t=_rotation(gen))


def prepare(case, seed):
    kb, vb = BITS[case["preset"]]
    cents, mids = _codebook(case["preset"])
    key_packed = D if kb == 8 else D * kb // 8 + 2
    s = types.SimpleNamespace(case=case, cents=cents, mids=mids, kb=kb, vb=vb, key_packed=key_packed,
                              fp8=kb == 8)
    for name, value in (_store_inputs if case["kind"] == "store" else _decode_inputs)(case, seed).items():
        setattr(s, name, value)
    if case["kind"] == "decode":
        s.pi = s.pi_t.t().contiguous()
        s.layer = types.SimpleNamespace()  # keeps the call's workspaces, as a backend's layer does
    elif case["kind"] == "stage1":
        s.lut = ops.pair_lut_device(cents)
        s.mid_o = torch.zeros(case["batch"], case["hq"], case["splits"], D + 1, device="cuda")
    return s


def run(s):
    case = s.case
    soa = case["layout"] == "soa"
    if case["kind"] == "decode":
        entry = (soa_decode if soa else aos_decode).triton_turboquant_decode_attention
        return entry(s.query, s.cache, s.table, s.lens, s.pi, s.cents, 1.0 / math.sqrt(D), s.kb, s.key_packed,
                     s.vb, key_fp8=s.fp8, norm_correction=True, PiT=s.pi_t, buf_holder=s.layer,
                     max_num_kv_splits=case["splits"], sinks=s.sinks)
    if case["kind"] == "stage1":
        return ops.launch_tq4_v2_stage1(s.query, s.cache, s.table, s.lens, s.cents, s.lut, s.mid_o)
    if soa:
        soa_store.triton_turboquant_store(s.key, s.value, s.cache, s.slots, s.pi_t, s.mids, s.kb, s.key_packed,
                                          s.vb, key_fp8=s.fp8, centroids=s.cents, norm_correction=not s.fp8)
    else:
        aos_store.triton_turboquant_store(s.key, s.value, s.cache, s.slots, s.pi_t, s.mids, s.kb, s.key_packed,
                                          s.vb, key_fp8=s.fp8)
    return s.cache


def work(case):
    slot = _slot_bytes(case["preset"])
    if case["kind"] == "store":
        size = 4 if case["dtype"] == "fp32" else 2
        rows = case["tokens"] * case["hk"]
        rotated = case["preset"] != "k8v4"
        return {"bytes": rows * (2 * D * size + slot) + 4 * case["tokens"] + (4 * D * D if rotated else 0),
                "flops": rows * (2 * D * D if rotated else D)}
    tokens, rows = sum(_lengths(case)), case["batch"] * case["hq"]
    moved = tokens * case["hk"] * slot + 4 * sum(-(-n // case["block"]) for n in _lengths(case))
    flops = 4 * tokens * case["hq"] * D
    if case["kind"] == "stage1":
        return {"bytes": moved + rows * D * 4 + rows * case["splits"] * (D + 1) * 4, "flops": flops}
    return {"bytes": moved + rows * D * 2 * 2 + 4 * D * D, "flops": flops + 2 * rows * D * D}


def tolerance(case):
    if case["kind"] == "store":
        return "exact"  # bytes: codes and fp16 scalars
    if case["kind"] == "stage1":
        # fp32 sums over splits of hundreds of tokens: 5.9e-7 (largest 3.5e-6) against float64
        return {"rel": 2.4e-6, "max": 1.5e-5}
    # one rounding to the output type of fp32 sums in another order: a few elements move by one
    # unit in the last place.  Against the rounded float64 result: bf16 up to 1.7e-4 (largest
    # 7.6e-3), fp16 up to 8.9e-5 (largest 9.8e-4)
    return {"rel": 7e-4, "max": 3e-2} if case["dtype"] == "bf16" else {"rel": 3.6e-4, "max": 4e-3}


def _keys_values(case, raw, cents, pages, length):
    """K and V of one sequence in float64, [hk, length, D] each."""
    kc, vc, fields = raw
    take = lambda t: t[pages].flatten(0, 1)[:length]  # noqa: E731
    if case["preset"] == "k8v4":
        k = take(kc).view(torch.float8_e4m3fn).double()
    else:
        k = cents.double()[take(kc).long()]
        if case["layout"] != "soa":
            k = k / (k.square().sum(-1, keepdim=True) + 1e-16).sqrt()
        k = k * take(fields[0]).double()[..., None]
    v = take(vc).double() * take(fields[-2]).double()[..., None] + take(fields[-1]).double()[..., None]
    return k.transpose(0, 1).contiguous(), v.transpose(0, 1).contiguous()


def exact(case, seed):
    if case["kind"] == "store":
        return None  # bytes, compared as they are
    x = _decode_inputs(case, seed, keep=True)
    cents, _ = _codebook(case["preset"])
    n, hq, hk, splits = case["batch"], case["hq"], case["hk"], case["splits"]
    q = x["query"].double()
    if case["kind"] == "decode" and case["preset"] != "k8v4":
        q = q.reshape(-1, D) @ x["pi_t"].double()
    q = q.reshape(n, hk, hq // hk, D) * (1.0 / math.sqrt(D))
    stage1 = case["kind"] == "stage1"
    out = torch.zeros((n, hq, splits, D + 1) if stage1 else (n, hq, D), dtype=torch.float64, device="cuda")
    for b, length in enumerate(x["lens"].tolist()):
        pages = x["table"][b, :-(-length // case["block"])].long()
        k, v = _keys_values(case, x["raw"], cents, pages, length)
        scores = torch.matmul(q[b], k.transpose(1, 2).contiguous())  # [hk, group, length]
        if not stage1:
            if x["sinks"] is not None:
                sink = x["sinks"].double().reshape(hk, -1, 1)
                p = torch.softmax(torch.cat([sink, scores], dim=-1), dim=-1)[..., 1:].contiguous()
            else:
                p = torch.softmax(scores, dim=-1)
            out[b] = torch.matmul(p, v).reshape(hq, D)
            continue
        step = -(-length // splits)
        for s, t0 in enumerate(range(0, length, step)):
            part = scores[..., t0:t0 + step].contiguous()
            lse = torch.logsumexp(part, dim=-1, keepdim=True)
            o = torch.matmul(torch.exp(part - lse), v[:, t0:t0 + step].contiguous())
            out[b, :, s] = torch.cat([o, lse], dim=-1).reshape(hq, D + 1)
    return out
