"""The calls of the paged int4-KIVI cache whose speed is followed.

A program that serves a model calls this package once per layer and token: it
appends the new tokens to the cache, quantising what leaves the fp16 residual
window, and attends over it.  The cases are those calls, through the public
entry points (``PagedKiviCache`` and the torch ops of the reference's binding),
from the smallest model's single sequence to a batch whose cache is 6 GB.

A case names the call (``op``), the geometry and the lengths:

  decode   PagedKiviCache.decode: one query per sequence
  step     PagedKiviCache.write_decode: append one token, then decode, one launch
  append   PagedKiviCache.append: ``new`` tokens to every sequence
  token    ops kivi_cache_write_dsl + kivi_decode_dsl: the reference's per-token pair
  chunk    ops kivi_cache_write_batched_dsl + kivi_decode_batched_dsl: one sub-chunk
           of the reference's batched prefill
  sparse   PagedKiviCache.decode_sparse_retained: one sequence whose old pages were
           partly evicted

Lengths spread evenly over [lo, hi] (the lengths before the call), whatever the
seed, which only says which sequence has which; the values are N(0,1) with a few
outlier K channels per kv head, as the workloads of jacq_amd.workloads have them.
"""
from __future__ import annotations

import math

import torch

from jacq_amd import kivi, torch_ops

GROUP = 32
POOL = ("k_code", "k_scale", "k_zero", "v_code", "v_scale", "v_zero", "k_scr", "v_scr")
MAX_NEW_V1 = 159  # the most tokens of one v1 sub-chunk that ages no group out
V1 = {"hd": 128, "page": 32, "residual": 128, "batch": 1}
DRAWN_MOST = 2_700_000_000  # tokens x kv heads x HD of a drawn decode: half of the largest listed


def case(op, nh, nkv, hd, batch, lo, hi, name=None, page=16, residual=128, **more):
    c = {"op": op, "nh": nh, "nkv": nkv, "hd": hd, "page": page, "residual": residual,
         "batch": batch, "lo": lo, "hi": hi, **more}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one user of a 1B model (TinyLlama heads, short window): latency and launches alone
        case("step", 32, 4, 64, 1, 512, 512, "step_tinyllama", residual=32),
        # a small model served to a few users (Qwen2.5-0.5B heads): the cache fits the caches
        case("decode", 14, 2, 64, 16, 2048, 2048, "decode_qwen05b"),
        # an ordinary server batch in step (Mistral-7B heads)
        case("step", 32, 8, 128, 32, 4096, 4096, "step_mistral7b"),
        # the benchmark: Qwen2.5-14B heads, ragged contexts, one token each
        case("step", 40, 8, 128, 64, 1024, 16384, "step_qwen14b"),
        # the largest: long ragged contexts of a 70B model's heads, 6 GB of cache
        case("decode", 64, 8, 128, 256, 4096, 32768, "decode_long"),
        # 16 query heads per kv head and 32-token pages, more than 64 sequences, odd lengths
        case("decode", 32, 2, 128, 80, 101, 6007, "decode_gqa16", page=32),
        # the write of a program that keeps write and decode apart: one token per sequence,
        # of which about 2 in 64 age a group out
        case("append", 40, 8, 128, 64, 1024, 16384, "append_token", new=1),
        # a prompt of odd length in one call
        case("append", 40, 8, 128, 1, 0, 0, "append_prompt", new=8191),
        # chunked prefill of a batch whose sequences are at different places
        case("append", 40, 8, 128, 64, 1024, 16384, "append_chunk", new=512),
        # the reference's own per-token pair at its fixed geometry
        case("token", 40, 8, name="v1_token", lo=2900, hi=2900, **V1),
        # the reference's batched prefill: a sub-chunk short of an age-out, its causal queries
        case("chunk", 40, 8, name="v1_chunk", lo=2048, hi=2048, new=31, **V1),
        # one long sequence after half of its old pages were evicted
        case("sparse", 40, 8, 128, 1, 16001, 16001, "sparse_16k", keep=0.5),
    ]


# (query heads, kv heads, head dim) of the workloads and the tests
HEADS = ((32, 4, 64), (14, 2, 64), (18, 2, 64), (24, 2, 64), (32, 8, 128), (40, 8, 128),
         (20, 4, 128), (64, 8, 128), (32, 2, 128), (36, 4, 128), (8, 8, 128))


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(("decode", "decode", "step", "step", "append", "append", "token", "chunk",
                     "sparse"))
    if op in ("token", "chunk"):
        nh, nkv = rng.choice(((40, 8), (20, 4)))
        if op == "token":
            n = _log(rng, 8, 4095)
            return case("token", nh, nkv, lo=n, hi=n, **V1)
        # where a sub-chunk may start: an empty cache, or one whose window has just been shifted
        n = rng.choice((0, 128 + GROUP * _log(rng, 1, 120)))
        new = rng.randint(2, MAX_NEW_V1 if n == 0 else GROUP - 1)
        return case("chunk", nh, nkv, lo=n, hi=n, new=new, **V1)
    nh, nkv, hd = rng.choice(HEADS)
    page, residual = rng.choice((16, 16, 32)), rng.choice((32, 64, 128, 128))
    if op == "sparse":
        n = _log(rng, 300, 32768)
        return case(op, nh, nkv, hd, 1, n, n, page=page, residual=residual,
                    keep=round(rng.uniform(0.1, 0.9), 2))
    if op == "append" and rng.random() < 0.7:  # a prompt or a chunk; else one token each
        new = _log(rng, 2, 16384)
        batch = _log(rng, 1, min(256, max(1, 65536 // new)))
        lo = 0 if rng.random() < 0.5 else _log(rng, 16, 4096)
        return case(op, nh, nkv, hd, batch, lo, lo * rng.randint(1, 3), page=page,
                    residual=residual, new=new)
    batch, hi = _log(rng, 1, 256), _log(rng, 48, 32768)
    while batch * (hi + residual) * nkv * hd > DRAWN_MOST:
        batch, hi = max(1, batch * 3 // 4), hi * 3 // 4
    lo = rng.choice((hi, max(1, hi // 2), max(1, hi // 16)))
    more = {"new": 1} if op == "append" else {}
    return case(op, nh, nkv, hd, batch, lo, hi, page=page, residual=residual, **more)


def old_tokens(n, residual):
    return max(0, n - residual) // GROUP * GROUP


def lengths(c):
    """Lengths before the call, one per sequence, spread over [lo, hi] by the golden
    ratio: evenly, but at all places of a 32-token group."""
    lo, hi = c["lo"], c["hi"]
    return [lo + int((hi - lo + 1) * ((i + 1) * 0.6180339887498949 % 1)) for i in range(c["batch"])]


def new_tokens(c):
    return {"decode": 0, "sparse": 0, "step": 1, "token": 1}.get(c["op"], c.get("new", 0))


def retained_groups(c):
    return int(old_tokens(c["lo"], c["residual"]) // GROUP * c["keep"])


def group_bytes(c):  # a quantised group of one kv head: codes, K and V scales and zeros
    hd = c["hd"]
    return GROUP * hd + 4 * hd + 4 * GROUP * (hd // GROUP)


def work(c):
    nh, nkv, hd, res = c["nh"], c["nkv"], c["hd"], c["residual"]
    row = 4 * nkv * hd  # K and V of one token in fp16
    total = flops = 0
    for n in lengths(c):
        new = new_tokens(c)
        end = n + new
        old0, old1 = old_tokens(n, res), old_tokens(end, res)
        if new:
            total += new * row  # the new tokens
            total += (old1 - old0) // GROUP * nkv * group_bytes(c)  # the groups that age out
            # the window's rows: those appended, or all where they move up
            total += (new if old1 == old0 else end - old1) * row
            if old1 > old0:
                total += (n - old0) * row  # the rows before the call: they age out or move
        if c["op"] == "append":
            continue
        old = GROUP * retained_groups(c) if c["op"] == "sparse" else old1
        queries = new if c["op"] == "chunk" else 1
        total += old // GROUP * nkv * group_bytes(c) + (end - old1) * row
        total += queries * nh * hd * 6 + 4 * (old // c["page"]) + 4 * queries  # Q, O, table
        # a chunk's queries end one token after another
        seen = sum(old + end - old1 - q for q in range(queries))
        flops += 4 * nh * hd * seen
    return {"bytes": total, "flops": flops}


def tolerance(c):
    # appended bytes are the reference's, bit for bit
    if c["op"] == "append":
        return "exact"
    # P and the dequantised V enter the matrix cores in fp16, sums are fp32: measured against
    # exact(), 1.6e-4 to 5.1e-4 of the output's norm and at most 8.8e-3 of its root mean square
    return {"rel": 2e-3, "max": 3.5e-2, "differ": 0.0}


# ---- state ----

def quantise(k, v):
    """Groups [N, heads, 32, HD] -> codes [N, heads, 32, HD / 2], scales and zeros of K
    [N, heads, HD] and V [N, heads, 32, HD / 32], in the dtype of the arguments."""
    def code(x, lo, scale):
        x = ((x - lo) / scale).round_().clamp_(0, 15).to(torch.uint8)
        return x[..., 0::2] | (x[..., 1::2] << 4)

    def span(lo, hi):
        s = (hi - lo) / 15
        return torch.where(s > 0, s, torch.ones_like(s))

    n, h, _, hd = k.shape
    kz = k.amin(2)
    ks = span(kz, k.amax(2))
    kc = code(k, kz[:, :, None], ks[:, :, None])
    v5 = v.reshape(n, h, GROUP, hd // GROUP, GROUP)
    vz = v5.amin(4)
    vs = span(vz, v5.amax(4))
    vc = code(v5, vz[..., None], vs[..., None]).reshape(n, h, GROUP, hd // 2)
    return kc, ks, kz, vc, vs, vz


def to_pages(c, x, per_group):
    """A group's array [N, heads, 32 or -, ...] as its pages' [N * pages, heads, ...]."""
    ppg = GROUP // c["page"]
    if per_group:  # K scales and zeros: one copy in every page of the group
        return x.repeat_interleave(ppg, 0)
    n, h, _, w = x.shape
    return x.reshape(n, h, ppg, c["page"], w).transpose(1, 2).reshape(n * ppg, h, c["page"], w)


class Values:
    """Seeded K and V tokens on the device: N(0,1), outlier K channels per kv head."""

    def __init__(self, c, seed):
        self.c, self.gen = c, torch.Generator(device="cuda").manual_seed(seed)
        nkv, hd = c["nkv"], c["hd"]
        out = torch.rand((nkv, hd), generator=self.gen, device="cuda").argsort(1)[:, :hd // 16]
        self.k_scale = torch.ones((nkv, hd), device="cuda", dtype=torch.float16)
        self.k_scale.scatter_(1, out, 10.0)

    def randn(self, *shape):
        return torch.randn(shape, generator=self.gen, device="cuda", dtype=torch.float16)

    def k(self, *lead):  # [..., tokens, heads, HD]
        return self.randn(*lead, self.c["nkv"], self.c["hd"]) * self.k_scale

    def k_rows(self, *lead):  # [..., heads, tokens, HD]
        return self.randn(*lead[:-1], self.c["nkv"], lead[-1], self.c["hd"]) * self.k_scale[:, None]

    def v_rows(self, *lead):
        return self.randn(*lead[:-1], self.c["nkv"], lead[-1], self.c["hd"])


def prepare(c, seed):
    nkv, hd, page, res, batch = c["nkv"], c["hd"], c["page"], c["residual"], c["batch"]
    val = Values(c, seed)
    order = torch.randperm(batch, generator=val.gen, device="cuda").tolist()
    even = lengths(c)
    lens = [even[i] for i in order]
    new = new_tokens(c)
    ppg = GROUP // page
    # a table as wide as the longest sequence will need, the pool as large as all do
    need = [max(ppg, old_tokens(n + new + GROUP - 1, res) // page) for n in lens]
    if c["op"] in ("token", "chunk"):
        width, pages = 124, 124
    else:
        width, pages = max(need), sum(need)
    perm = torch.randperm(pages, generator=val.gen, device="cuda").to(torch.int32)
    tables = torch.zeros((batch, width), dtype=torch.int32, device="cuda")
    at = 0
    for b, k in enumerate(need):
        tables[b, :k] = perm[at:at + k]
        at += k
    geo = kivi.KiviGeometry(c["nh"], nkv, hd, page, GROUP, res, width, pages)
    cache = kivi.PagedKiviCache(geo, batch)
    if c["op"] != "append":  # an append writes pages and reads none
        used = torch.cat([tables[b, :old_tokens(n, res) // page]
                          for b, n in enumerate(lens)]).long()
        step = 4096 * ppg
        for p0 in range(0, used.numel(), step):
            to = used[p0:p0 + step]
            n = to.numel() // ppg
            got = quantise(val.k_rows(n, GROUP).float(), val.v_rows(n, GROUP).float())
            for name, x in zip(POOL, got):
                dst = getattr(cache, name)
                dst[to] = to_pages(c, x, name in ("k_scale", "k_zero")).to(dst.dtype)
    cache.k_scr.copy_(val.k_rows(batch, res + GROUP))
    cache.v_scr.copy_(val.v_rows(batch, res + GROUP))

    s = {"op": c["op"], "case": c, "cache": cache, "tables": tables, "lens": lens,
         "start": torch.tensor(lens, dtype=torch.int32, device="cuda")}
    s["after"] = s["start"] + new
    if c["op"] in ("token", "chunk"):
        s["ops"] = torch_ops.load()
        s["pool"] = [getattr(cache, n) for n in POOL[:6]] + [cache.k_scr[0], cache.v_scr[0]]
        s["slots"] = torch.zeros(new, dtype=torch.int64, device="cuda")
        s["seq_len"] = lens[0] + new
    if c["op"] in ("step", "token"):
        s["nk"], s["nv"] = val.k(batch), val.randn(batch, nkv, hd)
    elif new:
        s["nk"], s["nv"] = val.k(batch, new), val.randn(batch, new, nkv, hd)
    queries = new if c["op"] == "chunk" else batch
    if c["op"] != "append":
        s["q"] = val.randn(queries, c["nh"], hd)
        s["out"] = torch.empty((queries, c["nh"], hd), dtype=torch.float32, device="cuda")
    if c["op"] == "chunk":
        s["query_lens"] = torch.arange(lens[0] + 1, lens[0] + new + 1, dtype=torch.int32,
                                       device="cuda")
    if c["op"] == "sparse":
        groups, keep = old_tokens(lens[0], res) // GROUP, retained_groups(c)
        kept = torch.randperm(groups, generator=val.gen, device="cuda")[:keep].sort().values
        s["retained"] = tables[0, :groups * ppg].view(groups, ppg)[kept].reshape(-1).contiguous()
        s["num_retained"] = keep * ppg
    return s


def run(s):
    cache, op = s["cache"], s["op"]
    if op == "decode":
        return cache.decode(s["q"], s["after"], s["tables"], out=s["out"])
    if op == "sparse":
        return cache.decode_sparse_retained(s["q"][0], s["lens"][0], s["retained"],
                                            s["num_retained"], out=s["out"][0])
    if op == "step":
        o = cache.write_decode(s["q"], s["nk"], s["nv"], s["after"], s["tables"], out=s["out"])
        return {"o": o, **{n: getattr(cache, n) for n in POOL}}
    if op == "append":
        cache.append(s["nk"], s["nv"], s["tables"], s["start"])
        return {n: getattr(cache, n) for n in POOL}
    ops, pool, table = s["ops"], s["pool"], s["tables"][0]
    if op == "token":
        ops.kivi_cache_write_dsl(*pool, s["nk"][0], s["nv"][0], s["slots"], table, s["seq_len"])
        ops.kivi_decode_dsl(s["q"][0], table, *pool, s["seq_len"], s["out"][0])
    else:
        new = s["slots"].numel()
        ops.kivi_cache_write_batched_dsl(*pool, s["nk"][0], s["nv"][0], s["slots"], table,
                                         s["lens"][0], new)
        ops.kivi_decode_batched_dsl(s["q"], s["query_lens"], table, *pool, new, s["out"])
    return {"o": s["out"], **dict(zip(POOL, pool))}


# ---- the same in 64 bits, in plain torch ----

def nibbles(x):
    return torch.stack((x & 15, x >> 4), -1).flatten(-2).double()


def old_rows(c, cache, pages):
    """K and V [heads, tokens, HD] of the groups in `pages`, dequantised."""
    ppg, hd, nkv = GROUP // c["page"], c["hd"], c["nkv"]
    scale, zero = cache.k_scale[pages].double(), cache.k_zero[pages].double()
    # a group's K scales: those of its first page
    scale = scale[::ppg].repeat_interleave(ppg, 0)[:, :, None]
    zero = zero[::ppg].repeat_interleave(ppg, 0)[:, :, None]
    k = nibbles(cache.k_code[pages]) * scale + zero
    v = nibbles(cache.v_code[pages]).unflatten(3, (hd // GROUP, GROUP))
    v = (v * cache.v_scale[pages].double()[..., None]
         + cache.v_zero[pages].double()[..., None]).flatten(3)
    return [x.transpose(0, 1).reshape(nkv, -1, hd) for x in (k, v)]


def attend(c, q, k, v):
    """q [NH, HD] over k, v [heads, tokens, HD]."""
    nh, nkv, hd = c["nh"], c["nkv"], c["hd"]
    qt = q.double().view(nkv, nh // nkv, hd).transpose(1, 2).contiguous()
    p = torch.softmax(torch.matmul(k, qt) / math.sqrt(hd), 1).transpose(1, 2).contiguous()
    return torch.matmul(p, v.contiguous()).reshape(nh, hd)


def exact(c, seed):
    s = prepare(c, seed)
    cache, res, op = s["cache"], c["residual"], c["op"]
    new = new_tokens(c)
    ppg = GROUP // c["page"]
    state = {n: getattr(cache, n).double() for n in POOL if "code" not in n} if new else {}
    outs = []
    for b, n in enumerate(s["lens"]):
        old0, end = old_tokens(n, res), n + new
        old1, r0 = old_tokens(end, res), n - old_tokens(n, res)
        k, v = cache.k_scr[b, :, :r0].double(), cache.v_scr[b, :, :r0].double()
        aged = []
        if new:
            nk, nv = (s[x][b].double().reshape(new, c["nkv"], c["hd"]).transpose(0, 1)
                      for x in ("nk", "nv"))
            k, v = torch.cat((k, nk), 1), torch.cat((v, nv), 1)
            if r0 + new <= res + GROUP:  # the new rows, before any shift
                state["k_scr"][b, :, r0:r0 + new], state["v_scr"][b, :, r0:r0 + new] = nk, nv
            d = old1 - old0
            if d:
                x = [t[:, :d].unflatten(1, (d // GROUP, GROUP)).transpose(0, 1) for t in (k, v)]
                aged = quantise(*x)
                to = s["tables"][b, old0 // c["page"]:old1 // c["page"]].long()
                for name, t in zip(POOL, aged):
                    if name in state:
                        state[name][to] = to_pages(c, t, name in ("k_scale", "k_zero"))
                k, v = k[:, d:], v[:, d:]
                state["k_scr"][b, :, :end - old1] = k
                state["v_scr"][b, :, :end - old1] = v
        if op == "append":
            continue
        if op == "sparse":
            ok, ov = old_rows(c, cache, s["retained"].long())
        else:
            if aged:  # the groups as they are stored
                to = s["tables"][b, old0 // c["page"]:old1 // c["page"]].long()
                for name, t in zip(POOL, aged):
                    dst = getattr(cache, name)
                    dst[to] = to_pages(c, t, name in ("k_scale", "k_zero")).to(dst.dtype)
            ok, ov = old_rows(c, cache, s["tables"][b, :old1 // c["page"]].long())
        k, v = torch.cat((ok, k), 1), torch.cat((ov, v), 1)
        if op == "chunk":
            for i in range(new):
                m = k.shape[1] - new + 1 + i
                outs.append(attend(c, s["q"][i], k[:, :m], v[:, :m]))
        else:
            outs.append(attend(c, s["q"][b], k, v))
    o = torch.stack(outs) if outs else None
    if op == "decode":
        return o
    if op == "sparse":
        return o[0]
    both = {n: state.get(n) for n in POOL}
    if op == "append":
        return both
    if op in ("token", "chunk"):
        both["k_scr"], both["v_scr"] = both["k_scr"][0], both["v_scr"][0]
    return {"o": o, **both}
