"""The work this framework is measured on: paged decode and prefill attention,
beam selection, the KV-cache writes of a decode step, and one whole model call,
each through the public entry points a decoding program calls.

A case is a dict of plain values; ``listed()`` are the standing ones, ``draw``
gives more of the same ranges, ``prepare`` / ``run`` execute one, ``work`` is
what it cannot do without, ``exact`` its result in 64 bits by plain torch.
"""

import math
import random

import numpy as np
import torch

from beam_engine_amd import (BatchDecodeWithPagedKVCacheWrapper, BatchPrefillWithPagedKVCacheWrapper,
                             MultiLevelCascadeAttentionWrapper, PageTable, beam_topk, decode_k)
from beam_engine_amd.llama import LlamaConfig, LlamaDecoder

DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
SIZE = {"float32": 4, "float16": 2, "bfloat16": 2}
WORKSPACE = 256 << 20       # the engine's attention workspace


def _decode(name, requests, beams, prefix, suffix, ragged, strategy, hq, hkv, d, page, dtype, layers):
    return dict(name=name, kind="decode", requests=requests, beams=beams, prefix=prefix, suffix=suffix, ragged=ragged,
                strategy=strategy, hq=hq, hkv=hkv, d=d, page=page, dtype=dtype, layers=layers)


def listed():
    return [
        # one request, four beams, full-precision cache: the smallest decode call, bound by launches and latency
        _decode("decode-fp32-small", 1, 4, 512, 32, False, "cascade", 8, 8, 64, 16, "float32", 1),
        # one request on PageTable's default page size and storage type: an interactive prompt of a few hundred
        # tokens, eight beams, some twenty tokens into the answer; a decode step's attention over eight layers
        _decode("decode-fp16-page8", 1, 8, 350, 24, True, "cascade", 32, 8, 128, 8, "float16", 8),
        # the serving step: 8 requests x 16 beams, short private tails (eight of the model's layers)
        _decode("decode-step", 8, 16, 1136, 24, True, "cascade", 32, 8, 128, 16, "bfloat16", 8),
        # the same batch on a 4k prompt with longer answers: the HBM-bound headline shape
        _decode("decode-prefix4k", 8, 16, 4096, 128, False, "cascade", 32, 8, 128, 16, "bfloat16", 4),
        # a small model's heads (head_dim 64)
        _decode("decode-d64", 4, 8, 2048, 128, True, "cascade", 32, 8, 64, 16, "bfloat16", 8),
        # long context, wide beams, a large model's layer: the largest decode call
        _decode("decode-long", 2, 64, 32768, 512, True, "cascade", 64, 8, 128, 16, "bfloat16", 1),
        # the batch's prompts, fresh, one layer after another
        dict(name="prefill-prompts", kind="prefill", requests=8, longest=1024, cached=0, ragged=False, hq=32, hkv=8,
             d=128, page=16, dtype="bfloat16", layers=2),
        # prompts of different lengths that continue a cached conversation, default page size and storage type
        dict(name="prefill-page8", kind="prefill", requests=3, longest=1500, cached=400, ragged=True, hq=32, hkv=8,
             d=128, page=8, dtype="float16", layers=2),
        # selection of the serving step: 8 requests x 16 beams over a 128k vocabulary
        dict(name="topk-step", kind="topk", requests=8, beam=16, vocab=128256, dtype="bfloat16", temperature=1.0),
        # selection of one small request on full-precision logits
        dict(name="topk-small", kind="topk", requests=1, beam=4, vocab=32000, dtype="float32", temperature=1.0),
        # the cache writes of a serving step: forked pages copied on every layer, then RoPE and append per layer
        dict(name="kv-step", kind="kv", requests=8, beams=16, forks=40, hq=32, hkv=8, d=128, page=16,
             dtype="bfloat16", layers=16),
        # a whole prefill call of a decoder (two layers of the serving model), prompt ids to logits
        dict(name="model-prefill", kind="model", requests=2, prompt=512, layers=2, page=16, dtype="bfloat16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["decode", "prefill", "topk", "kv"], [9, 5, 3, 2])[0]
    dtype = rng.choice(["bfloat16", "bfloat16", "bfloat16", "float16", "float16", "float32"])
    hq, hkv = rng.choice([(32, 8), (32, 8), (64, 8), (8, 8), (16, 4)])
    d = rng.choice([128, 128, 128, 64])
    page = rng.choice([16, 16, 16, 8, 8, 4, 32])
    if dtype == "float32":          # full precision is for small models and for checking
        hq, hkv, d = 8, rng.choice([8, 2]), rng.choice([64, 128])
    if kind == "decode":
        requests, beams, suffix = _log(rng, 1, 12), _log(rng, 2, 40), _log(rng, 1, 400)
        most = 20000 if dtype == "float32" else 100000
        prefix = max(30, min(20000, _log(rng, 2000, most) // requests))
        seen = requests * beams * (prefix + suffix)
        flat = seen < 100000 and rng.random() < 0.3
        tokens = seen if flat else requests * (prefix + beams * suffix)
        return dict(kind=kind, requests=requests, beams=beams, prefix=prefix, suffix=suffix, ragged=rng.random() < 0.8,
                    strategy="flat" if flat else "cascade", hq=hq, hkv=hkv, d=d, page=page, dtype=dtype,
                    layers=max(1, min(rng.choice([1, 2, 4, 8]), 120000 // tokens)))
    if kind == "prefill":
        requests, longest = _log(rng, 1, 10), _log(rng, 24, 3000)
        cached = rng.choice([0, 0, _log(rng, 10, 1500)])
        most = 4e9 if dtype == "float32" else 1.2e11
        while longest > 24 and 4.0 * d * hq * requests * longest * (longest / 2 + cached) > most:
            longest = longest * 4 // 5 + rng.randrange(3)
        return dict(kind=kind, requests=requests, longest=longest, cached=cached, ragged=rng.random() < 0.7, hq=hq, hkv=hkv,
                    d=d, page=page, dtype=dtype, layers=1)
    if kind == "topk":
        requests = _log(rng, 1, 8)
        return dict(kind=kind, requests=requests, beam=_log(rng, 1, 32 if requests < 4 else 16), vocab=_log(rng, 8000, 130000),
                    dtype=dtype, temperature=rng.choice([1.0, 1.0, 0.7, 1.3]))
    requests, beams = _log(rng, 1, 12), _log(rng, 2, 32)
    return dict(kind=kind, requests=requests, beams=beams, forks=rng.randint(1, requests * beams), hq=hq, hkv=hkv, d=d,
                page=page, dtype="bfloat16" if dtype == "float32" else dtype, layers=rng.choice([4, 8, 16]))


# ------------------------------------------------------------------ shapes of a case
def _fixed(case, salt):
    """Lengths belong to the case, not to the seed of its values."""
    return random.Random(salt + "/".join(f"{k}={case[k]}" for k in sorted(case) if k != "name"))


def _suffixes(case):
    r, n = _fixed(case, "suffix"), case["requests"] * case["beams"]
    return [r.randint(1, case["suffix"]) if case["ragged"] else case["suffix"] for _ in range(n)]


def _prompts(case):
    """(new tokens, cached tokens) of each request."""
    r, out = _fixed(case, "prompt"), []
    for _ in range(case["requests"]):
        n = r.randint(max(1, case["longest"] // 4), case["longest"]) if case["ragged"] else case["longest"]
        c = r.randint(0, case["cached"]) if case["ragged"] else case["cached"]
        out.append((n, c))
    return out


class _Pages:
    """Pages in the shuffled order a pool in use hands them out."""

    def __init__(self, case, total):
        self.order = list(range(total))
        _fixed(case, "pages").shuffle(self.order)

    def take(self, tokens, page):
        n = -(-tokens // page)
        got, self.order = self.order[:n], self.order[n:]
        return got, tokens - (n - 1) * page


def _decode_layout(case):
    """Per request (prefix pages, last), per beam (suffix pages, last); pages in the pool.  Beams share the
    prompt's whole pages, as the engine's trie does (a partial page is copied to each beam at the fork)."""
    page, suf = case["page"], _suffixes(case)
    whole = max(1, case["prefix"] // page) * page
    total = case["requests"] * (whole // page) + sum(-(-s // page) for s in suf)
    pool = _Pages(case, total)
    pre, tails = [], []
    for r in range(case["requests"]):
        pre.append(pool.take(whole, page))
        tails.append([pool.take(s, page) for s in suf[r * case["beams"]:(r + 1) * case["beams"]]])
    return pre, tails, total


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _attention_inputs(case, seed, queries, pages):
    """q and the paged cache of every layer: normalised heads, scores of unit variance."""
    g, dt = _generator(seed), DTYPES[case["dtype"]]
    q, kv = [], []
    for _ in range(case["layers"]):
        q.append(torch.randn((queries, case["hq"], case["d"]), generator=g, device="cuda", dtype=torch.float32).to(dt))
        kv.append(torch.randn((pages, 2, case["page"], case["hkv"], case["d"]), generator=g, device="cuda",
                              dtype=dt if dt != torch.float16 else torch.float32).to(dt))
    return q, kv


# ------------------------------------------------------------------ prepare / run
def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return state[0](*state[1:])


def _run_layers(wrapper, q, kv):
    return [wrapper.run(a, b) for a, b in zip(q, kv)]


def _prepare_decode(case, seed):
    pre, tails, total = _decode_layout(case)
    beams, n = case["beams"], case["requests"] * case["beams"]
    q, kv = _attention_inputs(case, seed, n, total)
    ws = torch.empty(WORKSPACE, dtype=torch.uint8, device="cuda")
    dt, heads = DTYPES[case["dtype"]], (case["hq"], case["hkv"], case["d"], case["page"])
    tail = [t for ts in tails for t in ts]
    if case["strategy"] == "flat":
        w = BatchDecodeWithPagedKVCacheWrapper(ws)
        ind, ptr = [], [0]
        for r, ts in enumerate(tails):
            for p, _ in ts:
                ind += pre[r][0] + p
                ptr.append(len(ind))
        w.plan(ptr, ind, [last for _, last in tail], *heads, q_data_type=dt)
    else:
        w = MultiLevelCascadeAttentionWrapper(2, ws)
        levels = [[], [], [], []]
        for groups, per in ((pre, beams), (tail, 1)):
            ptr, ind = [0], []
            for p, _ in groups:
                ind += p
                ptr.append(len(ind))
            for lv, x in zip(levels, ([i * per for i in range(len(groups) + 1)], ptr, ind, [last for _, last in groups])):
                lv.append(x)
        w.plan(*levels, *heads, causal=True, q_data_type=dt)
    return _run_layers, w, q, kv


def _prepare_prefill(case, seed):
    lens, page = _prompts(case), case["page"]
    pool = _Pages(case, sum(-(-(n + c) // page) for n, c in lens))
    total = len(pool.order)
    qo, ptr, ind, last = [0], [0], [], []
    for n, c in lens:
        p, l = pool.take(n + c, page)
        ind += p
        ptr.append(len(ind))
        last.append(l)
        qo.append(qo[-1] + n)
    q, kv = _attention_inputs(case, seed, qo[-1], total)
    w = BatchPrefillWithPagedKVCacheWrapper(torch.empty(WORKSPACE, dtype=torch.uint8, device="cuda"))
    w.plan(qo, ptr, ind, last, case["hq"], case["hkv"], case["d"], page, causal=True, q_data_type=DTYPES[case["dtype"]])
    return _run_layers, w, q, kv


def _logits(case, seed):
    """Logits as a language-model head gives them (a few units wide, some tokens well ahead of the rest), and
    the beams' accumulated log-probabilities."""
    g, rows = _generator(seed), case["requests"] * case["beam"]
    x = torch.randn((rows, case["vocab"]), generator=g, device="cuda") * 2.0
    x += torch.randn((rows, case["vocab"]), generator=g, device="cuda").clamp_(min=2.5).sub_(2.5).mul_(4.0)
    parents = -6.0 * torch.rand(rows, generator=g, device="cuda", dtype=torch.float64)
    return x.to(DTYPES[case["dtype"]]), parents


def _run_topk(logits, k, parents, beam, temperature, rows):
    return beam_topk(logits, k, parents, beam, temperature, request_rows=rows)


def _prepare_topk(case, seed):
    x, parents = _logits(case, seed)
    return (_run_topk, x, decode_k(case["beam"], case["vocab"]), parents, case["beam"], case["temperature"],
            [case["beam"]] * case["requests"])


def _run_kv(table, copies, qkv, hq, positions, cos, sin, pages, slots):
    table.copy_pages(copies)
    q = [table.write_rope_qkv(l, x, hq, positions, cos, sin, pages, slots) for l, x in enumerate(qkv)]
    return q + [table.kv_pool]


def _kv_inputs(case, seed):
    """A pool, the fork copies of a step (source page, new page, tokens), the projections and where they go.
    Every beam has a page of its own; new pages and written slots are distinct, as the trie hands them out."""
    g, r, dt = _generator(seed), _fixed(case, "kv"), DTYPES[case["dtype"]]
    n = case["requests"] * case["beams"]
    total = 2 * n + case["forks"]
    order = list(range(total))
    r.shuffle(order)
    own, new = order[:n], order[2 * n:]
    copies = np.array([[own[r.randrange(n)], p, r.randint(1, case["page"])] for p in new], dtype=np.int32)
    slots = torch.tensor([r.randrange(case["page"]) for _ in range(n)], dtype=torch.int32, device="cuda")
    pages = torch.tensor(order[n:2 * n], dtype=torch.int32, device="cuda")
    positions = torch.tensor([r.randrange(2048) for _ in range(n)], dtype=torch.int64, device="cuda")
    width = (case["hq"] + 2 * case["hkv"]) * case["d"]
    pool = torch.randn((case["layers"], total, 2, case["page"], case["hkv"], case["d"]), generator=g, device="cuda",
                       dtype=torch.float32).to(dt)
    qkv = [torch.randn((n, width), generator=g, device="cuda", dtype=torch.float32).to(dt) for _ in range(case["layers"])]
    d = case["d"]
    freq = torch.outer(torch.arange(2048, dtype=torch.float64, device="cuda"),
                       500000.0 ** (-torch.arange(0, d, 2, dtype=torch.float64, device="cuda") / d))
    emb = torch.cat([freq, freq], dim=-1)
    return pool, copies, qkv, positions, emb.cos().to(dt), emb.sin().to(dt), pages, slots


def _prepare_kv(case, seed):
    pool, copies, qkv, positions, cos, sin, pages, slots = _kv_inputs(case, seed)
    table = PageTable(case["layers"], page_size=case["page"], max_num_pages=pool.shape[1], head_num=case["hkv"],
                      head_dim=case["d"], store_dtype=pool.dtype)
    table.kv_pool.copy_(pool)
    return _run_kv, table, copies, qkv, case["hq"], positions, cos, sin, pages, slots


def _model(case, seed):
    cfg = LlamaConfig.llama3_8b()
    cfg.num_hidden_layers = case["layers"]
    cfg.max_position_embeddings = 2048
    ids = torch.randint(0, cfg.vocab_size, (case["requests"], case["prompt"]), generator=_generator(seed), device="cuda")
    return LlamaDecoder(cfg, dtype=DTYPES[case["dtype"]], seed=seed), ids


def _run_model(model, ids, table, pages):
    return model.prefill(ids, table, pages)


def _prepare_model(case, seed):
    model, ids = _model(case, seed)
    per = -(-case["prompt"] // case["page"])
    table = PageTable(case["layers"], page_size=case["page"], max_num_pages=per * case["requests"] + 8,
                      head_num=model.cfg.num_key_value_heads, head_dim=model.cfg.head_dim, store_dtype=model.dtype)
    return _run_model, model, ids, table, [[table.allocate_block() for _ in range(per)] for _ in range(case["requests"])]


_PREPARE = {"decode": _prepare_decode, "prefill": _prepare_prefill, "topk": _prepare_topk, "kv": _prepare_kv,
            "model": _prepare_model}


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    kind, es = case["kind"], SIZE[case["dtype"]]
    if kind == "decode":
        suf, n = _suffixes(case), case["requests"] * case["beams"]
        pre = max(1, case["prefix"] // case["page"]) * case["page"]
        tokens = case["requests"] * pre + sum(suf)
        seen = n * pre + sum(suf)
        kv, qo = tokens * case["hkv"] * case["d"] * 2 * es, 2 * n * case["hq"] * case["d"] * es
        return {"bytes": case["layers"] * (kv + qo), "flops": case["layers"] * 4.0 * case["d"] * case["hq"] * seen}
    if kind == "prefill":
        lens = _prompts(case)
        seen = sum(n * c + n * (n + 1) // 2 for n, c in lens)
        kv = sum(n + c for n, c in lens) * case["hkv"] * case["d"] * 2 * es
        qo = 2 * sum(n for n, _ in lens) * case["hq"] * case["d"] * es
        return {"bytes": case["layers"] * (kv + qo), "flops": case["layers"] * 4.0 * case["d"] * case["hq"] * seen}
    if kind == "topk":
        rows = case["requests"] * case["beam"]
        return {"bytes": rows * (case["vocab"] * es + 8 + 8 * decode_k(case["beam"], case["vocab"]) + 16), "flops": 0}
    if kind == "kv":
        n, slot = case["requests"] * case["beams"], 2 * case["hkv"] * case["d"] * es
        copied = sum(int(c[2]) for c in _kv_copies(case))
        rows = 2 * n * (case["hq"] + 2 * case["hkv"]) * case["d"] * es
        return {"bytes": case["layers"] * (2 * copied * slot + rows), "flops": 0}
    cfg, t = LlamaConfig.llama3_8b(), case["requests"] * case["prompt"]
    per = cfg.hidden_size * (cfg.hidden_size * 2 + 2 * cfg.num_key_value_heads * cfg.head_dim + 3 * cfg.intermediate_size)
    head = cfg.vocab_size * cfg.hidden_size
    att = 4.0 * cfg.hidden_size * case["requests"] * case["prompt"] * (case["prompt"] + 1) / 2
    kv = 2 * t * cfg.num_key_value_heads * cfg.head_dim * es
    return {"bytes": case["layers"] * (per * es + kv) + head * es + t * cfg.hidden_size * es,
            "flops": case["layers"] * (2.0 * per * t + att) + 2.0 * head * case["requests"]}


def _kv_copies(case):
    """The copies _kv_inputs makes, without its tensors."""
    r, n = _fixed(case, "kv"), case["requests"] * case["beams"]
    order = list(range(2 * n + case["forks"]))
    r.shuffle(order)
    return [[order[r.randrange(n)], p, r.randint(1, case["page"])] for p in order[2 * n:]]


def tolerance(case):
    """Measured on the start against ``exact``; about four times that.  16-bit attention rounds its
    probabilities and its result to the storage type; selection and copies have one right answer (RoPE's two
    products and their sum are rounded to the storage type in a fixed order)."""
    if case["kind"] in ("topk", "kv"):
        return "exact"
    if case["kind"] == "model":
        return {"rel": 0.03, "max": 0.3}
    return {"float32": {"rel": 4e-6, "max": 1e-4}, "float16": {"rel": 2e-3, "max": 2e-2},
            "bfloat16": {"rel": 1.2e-2, "max": 0.12}}[case["dtype"]]


# ------------------------------------------------------------------ 64-bit results
def _attend(q, k, v, first_seen=None):
    """softmax(q k^T / sqrt(d)) v in float64; q [n, hq, d], k / v [t, hkv, d]; query i sees first_seen + i keys."""
    n, hq, d = q.shape
    hkv, t = k.shape[1], k.shape[0]
    out = torch.empty((n, hq, d), dtype=torch.float64, device=q.device)
    mask = None
    if first_seen is not None:
        mask = torch.arange(t, device=q.device)[None, :] >= first_seen + torch.arange(n, device=q.device)[:, None]
    for h in range(hq):
        kh = h // (hq // hkv)
        s = (q[:, h].double() @ k[:, kh].double().t().contiguous()) * d ** -0.5
        if mask is not None:
            s = s.masked_fill(mask, -math.inf)
        out[:, h] = torch.softmax(s, dim=-1) @ v[:, kh].double().contiguous()
    return out


def _paged(kv, pages, tokens):
    p = kv[torch.tensor(pages, device=kv.device)]
    return p[:, 0].reshape(-1, *kv.shape[3:])[:tokens], p[:, 1].reshape(-1, *kv.shape[3:])[:tokens]


def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)


def _merged_prefix(q, k, v):
    """Unnormalised attention of all beams of a request over its shared prefix: (sum e^(s - m) v, sum, m)."""
    n, hq, d = q.shape
    hkv = k.shape[1]
    g = hq // hkv
    o = torch.empty((n, hq, d), dtype=torch.float64, device=q.device)
    z = torch.empty((n, hq), dtype=torch.float64, device=q.device)
    m = torch.empty((n, hq), dtype=torch.float64, device=q.device)
    for kh in range(hkv):
        qq = q[:, kh * g:(kh + 1) * g].double().reshape(n * g, d)
        s = (qq @ k[:, kh].double().t().contiguous()) * d ** -0.5
        mm = s.max(dim=-1).values
        e = torch.exp(s - mm[:, None])
        o[:, kh * g:(kh + 1) * g] = (e @ v[:, kh].double().contiguous()).reshape(n, g, d)
        z[:, kh * g:(kh + 1) * g] = e.sum(-1).reshape(n, g)
        m[:, kh * g:(kh + 1) * g] = mm.reshape(n, g)
    return o, z, m


def _exact_decode(case, seed):
    pre, tails, total = _decode_layout(case)
    beams, page = case["beams"], case["page"]
    q, kv = _attention_inputs(case, seed, case["requests"] * beams, total)
    out = []
    for a, b in zip(q, kv):
        o = torch.empty(a.shape, dtype=torch.float64, device=a.device)
        for r, (pp, plast) in enumerate(pre):
            rows = a[r * beams:(r + 1) * beams]
            k, v = _paged(b, pp, (len(pp) - 1) * page + plast)
            po, pz, pm = _merged_prefix(rows, k, v)
            for i, (tp, tlast) in enumerate(tails[r]):
                k, v = _paged(b, tp, (len(tp) - 1) * page + tlast)
                to, tz, tm = _merged_prefix(rows[i:i + 1], k, v)
                m = torch.maximum(pm[i], tm[0])
                x, y = torch.exp(pm[i] - m), torch.exp(tm[0] - m)
                o[r * beams + i] = (po[i] * x[:, None] + to[0] * y[:, None]) / (pz[i] * x + tz[0] * y)[:, None]
        out.append(o)
    return out


def _exact_prefill(case, seed):
    lens, page = _prompts(case), case["page"]
    pool = _Pages(case, sum(-(-(n + c) // page) for n, c in lens))
    q, kv = _attention_inputs(case, seed, sum(n for n, _ in lens), len(pool.order))
    pages = [pool.take(n + c, page)[0] for n, c in lens]
    out = []
    for a, b in zip(q, kv):
        parts, at = [], 0
        for (n, c), p in zip(lens, pages):
            k, v = _paged(b, p, n + c)
            parts.append(_attend(a[at:at + n], k, v, c + 1))
            at += n
        out.append(torch.cat(parts))
    return out


def _exact_topk(case, seed):
    x, _ = _logits(case, seed)
    logp = torch.log_softmax(x.double() / case["temperature"], dim=-1)
    return logp.topk(decode_k(case["beam"], case["vocab"]), dim=-1).values, None, (None, None, None)


def _exact_kv(case, seed):
    pool, copies, qkv, positions, cos, sin, pages, slots = _kv_inputs(case, seed)
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    pool = pool.double()
    for s, t, l in copies.tolist():
        pool[:, t, :, :l] = pool[:, s, :, :l]
    c, sn, out = cos[positions].double()[:, None], sin[positions].double()[:, None], []
    for l, x in enumerate(qkv):
        x = x.double().reshape(x.shape[0], hq + 2 * hkv, d)
        rot = torch.cat([-x[..., d // 2:], x[..., :d // 2]], dim=-1)
        y = x * c + rot * sn
        out.append(y[:, :hq])
        pool[l, pages.long(), 0, slots.long()] = y[:, hq:hq + hkv]
        pool[l, pages.long(), 1, slots.long()] = x[:, hq + hkv:]
    return out + [pool]


def _exact_model(case, seed):
    model, ids = _model(case, seed)
    cfg = model.cfg
    hq, hkv, d = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim
    r, s = ids.shape

    def norm(x, w):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + cfg.rms_norm_eps) * w.double()

    def rope(x):
        rot = torch.cat([-x[..., d // 2:], x[..., :d // 2]], dim=-1)
        return x * model.cos[:s].double()[None, :, None] + rot * model.sin[:s].double()[None, :, None]

    x = model.embed[ids].double()
    for w in model.layers:
        y = norm(x, w["ln1"]) @ w["wqkv"].double().t()
        q, k, v = (t.unflatten(-1, (-1, d)) for t in y.split([hq * d, hkv * d, hkv * d], dim=-1))
        q, k = rope(q), rope(k)
        o = torch.stack([_attend(q[i], k[i], v[i], 1) for i in range(r)])
        x = x + o.reshape(r, s, hq * d) @ w["wo"].double().t()
        gate, up = (norm(x, w["ln2"]) @ w["wgu"].double().t()).chunk(2, dim=-1)
        x = x + (torch.nn.functional.silu(gate) * up) @ w["wd"].double().t()
    return norm(x[:, -1], model.norm) @ model.lm_head.double().t()


_EXACT = {"decode": _exact_decode, "prefill": _exact_prefill, "topk": _exact_topk, "kv": _exact_kv,
          "model": _exact_model}
