"""The calls this library is used for, as timed cases over their real range of sizes.

A serving program keeps one paged K/V pool and, per layer and step, calls: the Q8_0 weight
projections, the fused decode step (RoPE, append, attention), prefill attention of a prompt
chunk, and bulk append and gather of K/V rows. Each case is one such call, or the few calls
of one layer, on sizes of the configurations of bench.py (TinyLlama, Llama-3-8B and
Llama-3-70B heads) or generic ones between them. Kinds of case:

  step     one decode step of one layer over n_seqs histories
  prefill  attention of n_seqs prompt chunks behind their histories
  proj     the projections of one layer (q/k/v, output, gate/up, down) for n_tokens rows
  layer    DecodeAttentionLayer.forward: q/k/v, decode step, output projection
  store    bulk append of a prompt chunk, then a gather of whole histories
"""
import math

import numpy as np
import torch

import ferrum_amd as fa

DEV = "cuda"
BLOCK = 16
THETA = 500000.0
F16, Q8_0 = "f16", "q8_0"
DTYPES = {F16: 1, Q8_0: 8}
CHUNK = 1 << 16  # tokens of one append while histories are filled


def listed():
    return [
        # A chat on a small model, alone on the GPU: one short history. Launches and latency.
        dict(name="step_tinyllama_1x575", kind="step", kv=F16, n_heads=32, n_kv_heads=4,
             head_dim=64, n_seqs=1, ctx_min=575, ctx_max=575, rope=True),
        # The ordinary decode step of a serving batch, histories of all lengths.
        dict(name="step_llama3_8b_64x4096", kind="step", kv=F16, n_heads=32, n_kv_heads=8,
             head_dim=128, n_seqs=64, ctx_min=128, ctx_max=4096, rope=True),
        # The same on the quantized cache that long histories are kept in.
        dict(name="step_llama3_8b_q8_24x8192", kind="step", kv=Q8_0, n_heads=32, n_kv_heads=8,
             head_dim=128, n_seqs=24, ctx_min=5001, ctx_max=8192, rope=True),
        # One very long document on a large model's heads.
        dict(name="step_llama3_70b_1x131072", kind="step", kv=F16, n_heads=64, n_kv_heads=8,
             head_dim=128, n_seqs=1, ctx_min=131072, ctx_max=131072, rope=False),
        # Prompt chunks of four requests behind their histories, as continuous batching runs them.
        dict(name="prefill_llama3_8b_4x512", kind="prefill", kv=F16, n_heads=32, n_kv_heads=8,
             head_dim=128, n_seqs=4, q_min=512, q_max=512, hist_min=1536, hist_max=4096),
        # One request's ragged chunk on the quantized cache.
        dict(name="prefill_llama3_8b_q8_1x389", kind="prefill", kv=Q8_0, n_heads=32, n_kv_heads=8,
             head_dim=128, n_seqs=1, q_min=389, q_max=389, hist_min=2011, hist_max=2011),
        # One sequence's projections: a layer's weights read once for one row.
        dict(name="proj_llama3_8b_1", kind="proj", embd=4096, q_rows=4096, kv_rows=1024,
             ffn=14336, n_tokens=1),
        # A few sequences on a small model, whose FFN width is no multiple of 1024.
        dict(name="proj_tinyllama_5", kind="proj", embd=2048, q_rows=2048, kv_rows=256,
             ffn=5632, n_tokens=5),
        # The projections of a decode batch.
        dict(name="proj_llama3_8b_64", kind="proj", embd=4096, q_rows=4096, kv_rows=1024,
             ffn=14336, n_tokens=64),
        # The projections of a prompt chunk.
        dict(name="proj_llama3_8b_512", kind="proj", embd=4096, q_rows=4096, kv_rows=1024,
             ffn=14336, n_tokens=512),
        # The attention half of a decode layer for a batch of two dozen sequences.
        dict(name="layer_llama3_8b_24x1500", kind="layer", kv=F16, n_heads=32, n_kv_heads=8,
             head_dim=128, embd=4096, n_seqs=24, ctx_min=100, ctx_max=1500),
        # Prompt chunks stored into the quantized cache and whole histories read back as
        # Q8_0 blocks (to keep a prefix, or to move a sequence).
        dict(name="store_llama3_8b_q8_16x512", kind="store", kv=Q8_0, n_kv_heads=8, head_dim=128,
             n_seqs=16, new=512, hist_min=0, hist_max=3000),
    ]


def _log(rng, lo, hi):
    """An integer of [lo, hi], even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["step", "step", "prefill", "proj", "proj", "proj", "layer", "store"])
    heads = rng.choice([(32, 4, 64), (32, 8, 128), (64, 8, 128)])
    c = dict(kind=kind)
    if kind != "proj":
        c.update(n_kv_heads=heads[1], head_dim=heads[2])
    if kind == "step":
        n = _log(rng, 1, 64)
        top = _log(rng, 64, min(65536, 200000 // n))
        c.update(kv=rng.choice([F16, F16, Q8_0]), n_heads=heads[0], n_seqs=n,
                 ctx_min=rng.randint(1, top), ctx_max=top, rope=rng.random() < 0.7)
    elif kind == "prefill":
        n = rng.randint(1, 4)
        q = _log(rng, 8, 512)
        h = rng.choice([0, _log(rng, 16, 4096 if heads[0] == 32 else 2048)])
        c.update(kv=rng.choice([F16, F16, Q8_0]), n_heads=heads[0], n_seqs=n,
                 q_min=rng.randint(max(1, q // 3), q), q_max=q, hist_min=rng.randint(0, h),
                 hist_max=h)
    elif kind == "proj":
        embd = 32 * rng.randint(24, 128)
        if rng.random() < 0.7:  # widths that models have: mostly multiples of 256
            embd = -(-embd // 256) * 256
        ffn = rng.choice([-(-int(embd * 2.7) // 256) * 256, embd * 7 // 2 // 32 * 32])
        c.update(embd=embd, q_rows=embd, kv_rows=rng.choice([embd // 4, embd // 8, embd]),
                 ffn=ffn, n_tokens=_log(rng, 1, 512))
    elif kind == "layer":
        hq, hkv, d = rng.choice([(32, 4, 64), (32, 8, 128)])
        c.update(kv=rng.choice([F16, F16, Q8_0]), n_heads=hq, n_kv_heads=hkv, head_dim=d,
                 embd=hq * d, n_seqs=_log(rng, 1, 48), ctx_min=rng.randint(1, 400),
                 ctx_max=rng.randint(400, 1500))
    else:
        h = _log(rng, 16, 3000)
        c.update(kv=rng.choice([F16, Q8_0]), n_seqs=_log(rng, 1, 16), new=_log(rng, 1, 512),
                 hist_min=rng.randint(0, h), hist_max=h)
    return c


# -- sizes and inputs -------------------------------------------------------------------


def _spread(lo, hi, n):
    """n lengths from lo to hi, evenly spaced, in an order that is not sorted."""
    if n == 1:
        return [hi]
    step = next(s for s in range(n // 2 + 1, 2 * n + 1) if math.gcd(s, n) == 1)
    return [lo + (hi - lo) * (i * step % n) // (n - 1) for i in range(n)]


def _lens(case):
    """(positions attended or gathered, new rows) of each sequence."""
    n = case["n_seqs"]
    if case["kind"] in ("step", "layer"):
        return _spread(case["ctx_min"], case["ctx_max"], n), [1] * n
    if case["kind"] == "prefill":
        new = _spread(case["q_min"], case["q_max"], n)
    else:
        new = [case["new"]] * n
    hist = _spread(case["hist_min"], case["hist_max"], n)
    return [h + q for h, q in zip(hist, new)], new


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _rows(gen, n, heads, dim, outliers):
    """n rows of K or V: N(0, 1), for the quantized cache with 1% of outliers at 20 sigma."""
    x = torch.randn((n, heads, dim), device=DEV, generator=gen)
    if outliers:
        hit = torch.rand((n, heads, dim), device=DEV, generator=gen) < 0.01
        x = torch.where(hit, torch.copysign(torch.full_like(x, 20.0), x), x)
    return x


def _kv(case, seed):
    """Every sequence's K and V rows, one after the other."""
    gen, total = _gen(seed), sum(_lens(case)[0])
    shape = (total, case["n_kv_heads"], case["head_dim"], case["kv"] == Q8_0)
    return _rows(gen, *shape), _rows(gen, *shape)


def _q(case, seed):
    rows = sum(_lens(case)[1])
    return torch.randn((rows, case["n_heads"], case["head_dim"]), device=DEV,
                       generator=_gen(seed + 1000003))


def _weight(gen, rows, cols):
    """Q8_0 rows as trained weights have them: normal quants, positive binary16 scales."""
    nb = cols // 32
    w = torch.empty((rows, nb, 34), dtype=torch.int8, device=DEV)
    q = torch.randn((rows, nb, 32), device=DEV, generator=gen).mul_(45.0)
    w[:, :, 2:] = q.round_().clamp_(-127, 127).to(torch.int8)
    d = torch.rand((rows, nb), device=DEV, generator=gen).mul_(3e-4).add_(2e-4).half()
    w[:, :, :2] = d.view(torch.int8).view(rows, nb, 2)
    return w.view(torch.uint8).view(-1)


def _proj_shapes(case):
    """The calls of one layer: (columns, row counts of the matrices that share them)."""
    e, kv, f = case["embd"], case["kv_rows"], case["ffn"]
    return [(e, [case["q_rows"], kv, kv]), (case["q_rows"], [e]), (e, [f, f]), (f, [e])]


def _proj_inputs(case, seed):
    gen, calls = _gen(seed), []
    for cols, rows in _proj_shapes(case):
        ws = [_weight(gen, r, cols) for r in rows]
        calls.append((cols, rows, ws, torch.randn((case["n_tokens"], cols), device=DEV,
                                                  generator=gen)))
    return calls


def _layer_inputs(case, seed):
    gen = _gen(seed + 2000003)
    e, q, kv = case["embd"], case["n_heads"] * case["head_dim"], case["n_kv_heads"] * case["head_dim"]
    ws = [_weight(gen, r, c) for r, c in ((q, e), (kv, e), (kv, e), (e, q))]
    return ws, torch.randn((case["n_seqs"], e), device=DEV, generator=gen)


# -- what a program keeps, and one pass ---------------------------------------------------


class _Storage:
    """The pool's device storage, for torch.as_tensor."""

    def __init__(self, pool):
        self.pool = pool  # lives as long as the view
        self.__cuda_array_interface__ = dict(shape=(pool.pool_bytes,), typestr="|u1", version=3,
                                             data=(pool.info().device_base, False))


def _pool(case, seed):
    """A pool that holds the histories under scattered block tables."""
    total, new = _lens(case)
    need = [-(-c // BLOCK) for c in total]
    n_blocks = sum(need) + 8
    pool = fa.PagedKvPool(fa.PagedConfig(
        n_layers=1, n_kv_heads=case["n_kv_heads"], head_dim=case["head_dim"],
        num_blocks=n_blocks, block_size=BLOCK, kv_dtype=DTYPES[case["kv"]]))
    pool.fill(0)
    order = np.random.default_rng(seed).permutation(n_blocks).astype(np.int32)
    tables = np.zeros((len(total), max(need)), dtype=np.int32)
    at = 0
    for s, b in enumerate(need):
        tables[s, :b] = order[at:at + b]
        at += b
    slots = [tables[s, np.arange(c) // BLOCK].astype(np.int64) * BLOCK + np.arange(c) % BLOCK
             for s, c in enumerate(total)]
    k, v = _kv(case, seed)
    # the newest rows of a step and of a store come with the call
    late = new if case["kind"] != "prefill" else [0] * len(new)
    first = np.concatenate([[0], np.cumsum(total)])
    old = np.concatenate([np.arange(first[s], first[s + 1] - late[s]) for s in range(len(total))])
    flat = torch.from_numpy(np.concatenate(slots)).to(DEV)
    for i in range(0, old.size, CHUNK):
        at = torch.from_numpy(old[i:i + CHUNK]).to(DEV)
        pool.append(0, k[at], v[at], flat[at])
    fresh = np.concatenate([np.arange(first[s + 1] - late[s], first[s + 1])
                            for s in range(len(total))])
    at = torch.from_numpy(fresh).to(DEV)
    return dict(pool=pool, tables=torch.from_numpy(tables).to(DEV),
                ctx=torch.tensor(total, dtype=torch.int32, device=DEV), max_ctx=max(total),
                k=k[at].contiguous(), v=v[at].contiguous(), slots=flat[at].contiguous(),
                first=torch.from_numpy(first[:-1].astype(np.int64)).to(DEV))


def _scratch(nbytes):
    return torch.empty(max(nbytes, 16), dtype=torch.uint8, device=DEV)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "proj":
        calls, n = _proj_inputs(case, seed), case["n_tokens"]
        ws = _scratch(max(fa.gemm_q8_0_batched_workspace_bytes(c, n) for c, _, _, _ in calls))
        ys = [[torch.empty((n, r), device=DEV) for r in rows] for _, rows, _, _ in calls]
        return dict(case=case, calls=calls, ys=ys, ws=ws)
    st = _pool(case, seed)
    st["case"] = case
    pool, n = st["pool"], case["n_seqs"]
    if kind == "step":
        st["q"] = _q(case, seed)
        st["out"] = torch.empty_like(st["q"])
        if case["rope"]:
            st["ws"] = _scratch(pool.rope_attention_workspace_bytes(case["n_heads"], n, st["max_ctx"]))
        else:
            st["ws"] = _scratch(pool.attention_workspace_bytes(case["n_heads"], n, st["max_ctx"]))
    elif kind == "prefill":
        new = _lens(case)[1]
        st["q"] = _q(case, seed)
        st["out"] = torch.empty_like(st["q"])
        st["q_lens"] = torch.tensor(new, dtype=torch.int32, device=DEV)
        st["q_first"] = torch.tensor(np.cumsum([0] + new[:-1]), dtype=torch.int64, device=DEV)
        st["max_q"] = max(new)
        st["ws"] = _scratch(pool.prefill_workspace_bytes(case["n_heads"], n, st["max_q"], st["max_ctx"]))
    elif kind == "layer":
        ws, st["x"] = _layer_inputs(case, seed)
        st["layer"] = fa.DecodeAttentionLayer(
            pool, 0, *ws, n_heads=case["n_heads"], n_embd=case["embd"], rope_dim=case["head_dim"],
            theta=THETA, max_seqs=n, max_ctx_len=st["max_ctx"])
        st["y"] = torch.empty_like(st["x"])
    else:
        total, row = sum(_lens(case)[0]), case["n_kv_heads"] * case["head_dim"]
        per_row = row * 2 if case["kv"] == F16 else row // 32 * 34
        st["out"] = [torch.empty((total, per_row), dtype=torch.uint8, device=DEV) for _ in "kv"]
    # A small cache is an output too, beside the rows computed from it.
    if kind == "layer" or (kind == "step" and pool.pool_bytes <= 64 << 20):
        st["image"] = torch.as_tensor(_Storage(pool), device=DEV)
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "proj":
        for (cols, rows, ws, x), ys in zip(st["calls"], st["ys"]):
            fa.gemm_q8_0_batched(ws, rows, cols, x, case["n_tokens"], ys, workspace=st["ws"])
        return [y for ys in st["ys"] for y in ys]
    pool = st["pool"]
    if kind == "step":
        args = (0, st["k"], st["v"], st["q"], st["out"], st["tables"], st["ctx"], st["max_ctx"])
        if case["rope"]:
            pool.rope_append_decode_attention(*args, case["head_dim"], THETA, workspace=st["ws"])
        else:
            pool.append_decode_attention(*args, workspace=st["ws"])
        return [st["out"]] + ([st["image"]] if "image" in st else [])
    if kind == "prefill":
        pool.prefill_attention(0, st["q"], st["out"], st["tables"], st["ctx"], st["q_lens"],
                               st["q_first"], st["max_q"], st["max_ctx"], workspace=st["ws"])
        return [st["out"]]
    if kind == "layer":
        st["layer"].forward(st["x"], st["tables"], st["ctx"], st["max_ctx"], st["y"])
        return [st["y"], st["image"]]
    pool.append(0, st["k"], st["v"], st["slots"])
    pool.gather_tables(0, st["tables"], st["ctx"], st["first"], st["max_ctx"], *st["out"],
                       fmt=fa.GATHER_RAW)
    return st["out"]


# -- what a pass cannot do without, and how exact it is -----------------------------------


def _attention_work(case):
    total, new = _lens(case)
    hq, hkv, d = case["n_heads"], case["n_kv_heads"], case["head_dim"]
    e = 2.0 if case["kv"] == F16 else 34 / 32
    nbytes = sum(c * hkv * d * 2 * e + q * hq * d * 8 + -(-c // BLOCK) * 4 + 4
                 for c, q in zip(total, new))
    if case["kind"] != "prefill":  # the new rows, read and stored
        nbytes += len(total) * 2 * hkv * d * (4 + e)
    keys = sum(q * (c - q) + q * (q + 1) // 2 for c, q in zip(total, new))
    return nbytes, 4.0 * d * hq * keys


def work(case):
    kind, nbytes, flops = case["kind"], 0.0, 0.0
    if kind == "proj":
        n, shapes = case["n_tokens"], _proj_shapes(case)
    elif kind == "layer":
        n, q, kv = (case["n_seqs"], case["n_heads"] * case["head_dim"],
                    case["n_kv_heads"] * case["head_dim"])
        shapes = [(case["embd"], [q, kv, kv]), (q, [case["embd"]])]
    elif kind == "store":
        total, new = _lens(case)
        row = 2 * case["n_kv_heads"] * case["head_dim"]
        e = 2.0 if case["kv"] == F16 else 34 / 32
        nbytes = sum(new) * (row * (4 + e) + 8) + sum(total) * row * 2 * e
        return dict(bytes=nbytes, flops=0.0)
    if kind in ("step", "prefill", "layer"):
        nbytes, flops = _attention_work(case)
    if kind in ("proj", "layer"):
        for cols, rows in shapes:
            nbytes += sum(rows) * (cols // 32 * 34) + n * cols * 4 + n * sum(rows) * 4
            flops += 2.0 * n * cols * sum(rows)
    return dict(bytes=nbytes, flops=flops)


def tolerance(case):
    if case["kind"] in ("proj", "store"):
        # Q8_0 products are defined to the bit (integer dots, scales and sums in order)
        return "exact"
    if case["kind"] == "layer":
        # attention rows a little apart round some activations to the other 8-bit value:
        # 1.5e-3 to 1.7e-3 from 64-bit attention between the same products
        return dict(rel=7e-3)
    # softmax weights in binary16: 1.2e-4 to 2.6e-4 from 64 bits
    return dict(rel=1e-3)


def _stored(x, kv):
    """Rows of K or V as the cache keeps them, in 64 bits."""
    if kv == F16:
        return x.half().double()
    q, d = _quantize(x)
    return (q.double() * d.double()[..., None]).reshape(x.shape)


def _quantize(x):
    """(quants [..., 32], binary16 scale) of each run of 32 values, as Q8_0 defines them."""
    b = x.reshape(*x.shape[:-1], -1, 32)
    d = b.abs().amax(-1) / 127.0
    q = b * torch.where(d != 0, 1.0 / d, torch.zeros_like(d))[..., None]
    q = torch.copysign((q.double().abs() + 0.5).floor(), q.double())
    return q.clamp(-128, 127), d.half()


def _product(w, rows, cols, x):
    """x of [n, cols], quantized, by the Q8_0 matrix w, in 64 bits."""
    q, d = _quantize(x)
    xq = (q * d.double()[..., None]).reshape(x.shape)
    blk = w.view(torch.int8).view(rows, cols // 32, 34)
    ws = blk[:, :, :2].contiguous().view(torch.float16).double()
    return xq @ (blk[:, :, 2:].double() * ws).reshape(rows, cols).t().contiguous()


def _rotate(x, pos):
    """RoPE of x [n, heads, dim] at pos [n]: pairs (2i, 2i + 1), angles kept in 32 bits."""
    d = x.shape[-1]
    e = np.float32(2.0) * np.arange(d // 2, dtype=np.float32) / np.float32(d)
    den = torch.from_numpy(np.float32(THETA) ** e).to(DEV)
    f = (pos.float()[:, None] / den).double()[:, None, :]
    a, b = x[..., 0::2].double(), x[..., 1::2].double()
    return torch.stack([a * f.cos() - b * f.sin(), a * f.sin() + b * f.cos()], -1).reshape(x.shape)


def _attend(q, k, v, n_kv):
    """Causal attention of q [n, heads, dim] at the end of k, v [c, kv heads, dim], in 64 bits."""
    n, hq, d = q.shape
    c, g = k.shape[0], hq // n_kv
    out = torch.empty((n, hq, d), dtype=torch.float64, device=DEV)
    hide = torch.arange(c, device=DEV)[None, :] > torch.arange(c - n, c, device=DEV)[:, None]
    for h in range(hq):
        s = q[:, h].double() @ k[:, h // g].t().contiguous() * fa.default_scale(d)
        p = torch.softmax(s.masked_fill_(hide, -math.inf), -1)
        out[:, h] = p @ v[:, h // g]
    return out


def _attention_exact(case, seed, q, k_new=None, v_new=None):
    """Attention of q over the case's histories; k_new and v_new are each one's last row."""
    total, new = _lens(case)
    k, v = _kv(case, seed)
    outs, at, qat = [], 0, 0
    for s, (c, n) in enumerate(zip(total, new)):
        ks, vs = k[at:at + c], v[at:at + c]
        if k_new is not None:
            ks, vs = ks.clone(), vs.clone()
            ks[-1], vs[-1] = k_new[s].to(ks.dtype), v_new[s].to(vs.dtype)
        outs.append(_attend(q[qat:qat + n], _stored(ks, case["kv"]), _stored(vs, case["kv"]),
                            case["n_kv_heads"]))
        at, qat = at + c, qat + n
    return torch.cat(outs)


def exact(case, seed):
    kind = case["kind"]
    if kind == "store":
        return None  # bytes
    if kind == "proj":
        return [_product(w, r, cols, x) for cols, rows, ws, x in _proj_inputs(case, seed)
                for w, r in zip(ws, rows)]
    total = _lens(case)[0]
    pos = torch.tensor(total, device=DEV) - 1
    if kind == "layer":
        (wq, wk, wv, wo), x = _layer_inputs(case, seed)
        hq, hkv, d, e = case["n_heads"], case["n_kv_heads"], case["head_dim"], case["embd"]
        q = _rotate(_product(wq, hq * d, e, x).view(-1, hq, d), pos)
        k = _rotate(_product(wk, hkv * d, e, x).view(-1, hkv, d), pos)
        v = _product(wv, hkv * d, e, x).view(-1, hkv, d)
        o = _attention_exact(case, seed, q, k, v)
        return [_product(wo, e, hq * d, o.float().view(-1, hq * d)), None]
    q = _q(case, seed)
    if kind == "prefill":
        return [_attention_exact(case, seed, q)]
    if case["rope"]:
        k, v = _kv(case, seed)
        last = torch.tensor(np.cumsum(total) - 1, device=DEV)
        out = _attention_exact(case, seed, _rotate(q, pos), _rotate(k[last], pos), v[last])
    else:
        out = _attention_exact(case, seed, q)
    return [out] + ([None] if _image_kept(case) else [])


def _image_kept(case):
    """Whether a step's outputs hold the cache (see prepare)."""
    row = case["n_kv_heads"] * case["head_dim"] * 2
    per_block = BLOCK * (row * 2 if case["kv"] == F16 else row // 32 * 34)
    return (sum(-(-c // BLOCK) for c in _lens(case)[0]) + 8) * per_block <= 64 << 20
