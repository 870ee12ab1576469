"""The workloads this framework is timed on, through its public entry points.

A case is a dict of plain values; its "kind" says which path it takes:

  prefill   block_route_budget + sparse_attention: one routed causal prefill attention layer
  layer     gemma_ssa.ssa_attention_forward on a transformers-layout prefill of any length
  generate  the same entry point as a generation uses it: a prefill, then one token at a time
  decode    RoutedDecoder.step: routed decode on a long KV cache
  train     ssa_swap.ssa_masked forward and backward (continued training through the swap)
  ivf       ivf_route + sparse_attention: prefill with the sub-linear IVF router
  cascade   ccc_prefill: prefill with the streaming certified cascade

Whole numbers (block lists, certificates) have to be equal; the tolerances of computed outputs are
about four times the difference from the 64-bit restatement in exact().
"""
from __future__ import annotations

import math
from types import SimpleNamespace

import torch

from ssa_amd import cascade_router, gemma_ssa, ivf_decode, ivf_kernel, ssa_kernel, ssa_swap

DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
NEG = float("-inf")


def listed():
    return [
        # one fp32 head of 4096 tokens: the smallest prefill, where launches and latency count
        dict(name="prefill_fp32_4k", kind="prefill", dtype="fp32", B=1, hq=1, hkv=1, n=4096, d=64,
             block=64, top_c=8, local=1, keys="normal"),
        # a grouped-query layer at an ordinary 32K prompt with fine blocks
        dict(name="prefill_bf16_32k", kind="prefill", dtype="bf16", B=1, hq=14, hkv=2, n=32768,
             d=64, block=64, top_c=32, local=2, keys="mixture"),
        # the headline: the same layer over a 128K prompt
        dict(name="prefill_bf16_128k", kind="prefill", dtype="bf16", B=1, hq=14, hkv=2, n=131072,
             d=64, block=128, top_c=64, local=2, keys="mixture"),
        # the longest context: one head over 12M tokens
        dict(name="prefill_fp16_12m", kind="prefill", dtype="fp16", B=1, hq=1, hkv=1, n=12582912,
             d=64, block=256, top_c=64, local=1, keys="normal"),
        # a wide-head layer of a hybrid model at a prompt length that fills no block, budget routing
        dict(name="layer_bf16_d512", kind="layer", dtype="bf16", B=1, hq=16, hkv=8, n=8100, d=512,
             block=256, frac=0.25, local=1),
        # a short prompt and the first tokens after it, through the transformers interface
        dict(name="generate_bf16_1500", kind="generate", dtype="bf16", B=1, hq=14, hkv=2, n=1500,
             d=64, block=128, frac=0.25, local=1, tokens=8),
        # decode at a 1M-token cache; the steps cross a block's completion
        dict(name="decode_bf16_1m", kind="decode", dtype="bf16", B=1, hq=14, hkv=2, n=1048572,
             d=64, block=128, top_c=64, local=1, tokens=8),
        # batched serving decode: eight sequences of about 32K tokens, wider heads
        dict(name="decode_fp16_batch8", kind="decode", dtype="fp16", B=8, hq=32, hkv=8, n=32701,
             d=128, block=128, top_c=16, local=1, tokens=8),
        # continued training through the swap at the GPT-2 attention shape
        dict(name="train_bf16", kind="train", dtype="bf16", B=4, hq=12, hkv=12, n=1024, d=64,
             block=64, top_c=4, local=2),
        # the same in fp32 with sequences that fill no block
        dict(name="train_fp32_ragged", kind="train", dtype="fp32", B=4, hq=12, hkv=12, n=1000,
             d=64, block=64, top_c=4, local=2),
        # the sub-linear router at 1M tokens (index build, search and attention)
        dict(name="ivf_fp16_1m", kind="ivf", dtype="fp16", B=1, hq=1, hkv=1, n=1048576, d=64,
             block=128, top_c=8, local=1),
        # the streaming selector over 1M tokens, certified
        dict(name="cascade_fp16_1m", kind="cascade", dtype="fp16", n=1048576, d=64, block=128,
             chunk_blocks=1024),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _heads(rng):
    hkv = rng.choice([1, 2, 4, 8])
    return hkv * rng.choice([1, 2, 4, 7]), hkv


def draw(rng):
    while True:
        c = _draw(rng)
        if work(c)["flops"] <= 5e12:  # no drawn case costs as much as the 12M-token prefill
            return c


def _draw(rng):
    kind = rng.choice(["prefill", "prefill", "layer", "generate", "decode", "decode", "train",
                       "train", "ivf", "cascade"])
    if kind == "prefill":
        dtype = rng.choice(["bf16", "fp16", "bf16", "fp32"])
        hq, hkv = _heads(rng) if dtype != "fp32" else (rng.choice([1, 2, 3]), 1)
        block = rng.choice([64, 128, 256])
        d = 64 if dtype == "fp32" else rng.choice([64, 64, 128])
        nb = _log_int(rng, 8, 100 if dtype == "fp32" else 1500)
        return dict(kind=kind, dtype=dtype, B=1, hq=hq, hkv=hkv, n=nb * block, d=d, block=block,
                    top_c=_log_int(rng, 4, 64), local=rng.choice([1, 2]),
                    keys=rng.choice(["normal", "mixture"]))
    if kind in ("layer", "generate"):
        hq, hkv = _heads(rng)
        c = dict(kind=kind, dtype=rng.choice(["bf16", "fp16"]), B=1, hq=hq, hkv=hkv,
                 n=_log_int(rng, 300, 16000), d=rng.choice([64, 128, 256, 512]),
                 block=rng.choice([128, 256]), frac=rng.choice([0.06, 0.12, 0.25]), local=1)
        if kind == "generate":
            c["tokens"] = rng.randint(2, 16)
        return c
    if kind == "decode":
        hq, hkv = _heads(rng)
        B = rng.choice([1, 2, 8])
        return dict(kind=kind, dtype=rng.choice(["bf16", "fp16"]), B=B, hq=hq, hkv=hkv,
                    n=_log_int(rng, 2000, 2000000 // (B * hkv)), d=rng.choice([64, 128]),
                    block=rng.choice([64, 128, 256]), top_c=_log_int(rng, 4, 64), local=1,
                    tokens=rng.randint(4, 12))
    if kind == "train":
        h = rng.randint(2, 16)
        return dict(kind=kind, dtype=rng.choice(["bf16", "fp16", "fp32"]), B=rng.randint(1, 4),
                    hq=h, hkv=h, n=_log_int(rng, 130, 2048), d=64, block=rng.choice([32, 64, 128]),
                    top_c=rng.randint(2, 8), local=rng.randint(0, 2))
    if kind == "ivf":
        hkv = rng.choice([1, 2])
        return dict(kind=kind, dtype=rng.choice(["bf16", "fp16"]), B=1, hq=hkv * rng.choice([1, 4]),
                    hkv=hkv, n=128 * _log_int(rng, 300, 16000), d=64, block=128,
                    top_c=rng.choice([4, 8, 16]), local=1)
    return dict(kind=kind, dtype=rng.choice(["bf16", "fp16"]), n=128 * _log_int(rng, 300, 12000),
                d=64, block=128, chunk_blocks=1024)


# ---------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------

def _randn(g, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=g, device="cuda").to(dtype)


def _keys(g, c, n, dtype):
    """Keys drawn token by token, or (mixture) around one of 256 component means that stays the
    same over runs of 32 tokens, as the keys of neighbouring tokens do."""
    shape = (c["B"], c["hkv"], n, c["d"])
    if c.get("keys", "mixture") == "normal":
        return _randn(g, *shape, dtype=dtype)
    means = _randn(g, c["hkv"], 256, c["d"])
    comp = torch.randint(0, 256, (c["B"], c["hkv"], -(-n // 32)), generator=g, device="cuda")
    k = torch.empty(shape, device="cuda", dtype=dtype)
    for b in range(c["B"]):
        for h in range(c["hkv"]):
            centre = means[h][comp[b, h]].repeat_interleave(32, 0)[:n]
            k[b, h] = (centre + 0.3 * _randn(g, n, c["d"])).to(dtype)
    return k


def _plant(g, q, k, v, block):
    """Sparse strong matches: keys along a later query, their values one-hot (normal keys only)."""
    n, d = q.shape[2], q.shape[3]
    m = max(8, n // 12288)
    t = torch.randint(3 * n // 4, n, (m,), generator=g, device="cuda")
    p = torch.randint(0, 3 * n // 4 - 2 * block, (m,), generator=g, device="cuda")
    p, keep = torch.unique(p, return_inverse=True)
    t = torch.zeros_like(p).scatter_(0, keep, t)
    qt = q[0, 0, t].float()
    k[0, 0, p] = (3.0 * qt / qt.norm(dim=-1, keepdim=True)).to(k.dtype)
    v[0, 0, p] = torch.eye(d, device="cuda", dtype=v.dtype)[torch.arange(len(p), device="cuda") % d]


def _inputs(c, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt = DTYPES[c["dtype"]]
    kind, n, d = c["kind"], c["n"], c["d"]
    if kind == "cascade":  # clustered keys, one cluster per 32 tokens, and queries near clusters
        nc = max(8, int((n // 32) ** 0.5))
        ctr = _randn(g, nc, d)
        a = torch.randint(0, nc, (n // 32,), generator=g, device="cuda")
        b = torch.randint(0, nc, (n // c["block"],), generator=g, device="cuda")
        k = (ctr[a].repeat_interleave(32, 0) + 0.1 * _randn(g, n, d)).to(dt)
        q = (ctr[b].repeat_interleave(c["block"], 0) + 0.2 * _randn(g, n, d)).to(dt)
        return dict(q=q.view(1, 1, n, d), k=k.view(1, 1, n, d),
                    v=_randn(g, 1, 1, n, d, dtype=dt))
    B, hq, hkv = c["B"], c["hq"], c["hkv"]
    if kind in ("prefill", "ivf"):
        q = _randn(g, B, hq, n, d, dtype=dt)
        k = _keys(g, c, n, dt)
        v = _randn(g, B, hkv, n, d, dtype=dt)
        if c.get("keys") == "normal":
            _plant(g, q, k, v, c["block"])
        return dict(q=q, k=k, v=v)
    if kind in ("layer", "generate"):  # (B, n, heads, d) projections seen as (B, heads, n, d)
        total = n + c.get("tokens", 0)
        q = _randn(g, B, total, hq, d, dtype=dt).transpose(1, 2)
        k = _keys(g, c, total, dt).transpose(1, 2).contiguous().transpose(1, 2)
        v = _randn(g, B, total, hkv, d, dtype=dt).transpose(1, 2)
        return dict(q=q, k=k, v=v)
    if kind == "decode":
        k = _keys(g, c, n + c["tokens"], dt)
        v = _randn(g, B, hkv, n + c["tokens"], d, dtype=dt)
        return dict(q=_randn(g, c["tokens"], B, hq, d, dtype=dt), k=k, v=v)
    return dict(q=_randn(g, B, hq, n, d, dtype=dt), k=_randn(g, B, hkv, n, d, dtype=dt),
                v=_randn(g, B, hkv, n, d, dtype=dt), g=_randn(g, B, hq, n, d, dtype=dt))


def prepare(case, seed):
    s = _inputs(case, seed)
    s["c"] = c = case
    if c["kind"] == "decode":
        dec = ivf_decode.RoutedDecoder(c["B"], c["hq"], c["hkv"], c["d"], c["n"] + c["tokens"],
                                       block=c["block"], top_c=c["top_c"], local=c["local"],
                                       dtype=DTYPES[c["dtype"]])
        dec.prefill(s["k"][:, :, :c["n"]], s["v"][:, :, :c["n"]])
        s["dec"] = dec
        s["new"] = [(s["k"][:, :, c["n"] + t].contiguous(), s["v"][:, :, c["n"] + t].contiguous())
                    for t in range(c["tokens"])]
        del s["k"], s["v"]
    elif c["kind"] == "train":
        for x in "qkv":
            s[x].requires_grad_(True)
    elif c["kind"] in ("layer", "generate"):
        s["cfg"] = gemma_ssa.SSAConfig(block=c["block"], budget_frac=c["frac"],
                                       local_w=c["local"], impl="hip")
        s["module"] = SimpleNamespace(layer_idx=0, is_sliding=False, scaling=c["d"] ** -0.5)
    return s


def run(state):
    c, kind = state["c"], state["c"]["kind"]
    if kind == "decode":
        dec, outs = state["dec"], []
        dec.pos = c["n"]  # a rewind: the same tokens are appended again
        for t, (k_new, v_new) in enumerate(state["new"]):
            outs.append(dec.step(state["q"][t], k_new, v_new))
        return outs, dec.kv_num, dec.kv_idx, dec.mu, dec.var, dec.kcache, dec.vcache
    q, k, v = state["q"], state["k"], state["v"]
    if kind == "prefill":
        kv_num, kv_idx, _ = ssa_kernel.block_route_budget(q, k, c["block"], top_c=c["top_c"],
                                                          local=c["local"], compact=True)
        return ssa_kernel.sparse_attention(q, k, v, kv_num, kv_idx, c["block"]), kv_num, kv_idx
    if kind == "ivf":
        kv_num, kv_idx = ivf_kernel.ivf_route(q, k, c["block"], c["top_c"], c["local"])
        return ssa_kernel.sparse_attention(q, k, v, kv_num, kv_idx, c["block"]), kv_num, kv_idx
    if kind == "cascade":
        return cascade_router.ccc_prefill(q, k, v, c["block"], certify=True,
                                          chunk_blocks=c["chunk_blocks"])
    if kind == "train":
        out = ssa_swap.ssa_masked(q, k, v, c["block"], c["top_c"], c["local"])
        return (out, *torch.autograd.grad(out, (q, k, v), state["g"]))
    gemma_ssa.CFG = state["cfg"]
    m, n = state["module"], c["n"]
    with torch.no_grad():
        outs = [gemma_ssa.ssa_attention_forward(m, q[:, :, :n], k[:, :, :n], v[:, :, :n])[0]]
        for t in range(n, n + c.get("tokens", 0)):
            outs.append(gemma_ssa.ssa_attention_forward(m, q[:, :, t:t + 1], k[:, :, :t + 1],
                                                        v[:, :, :t + 1])[0])
    return outs


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------

def _pairs(n, block, keep, local):
    """Query-key pairs of a causal routed pass: whole blocks but for the query's own."""
    nb = -(-n // block)
    total = 0
    for i in range(nb):
        rows = min(n, (i + 1) * block) - i * block
        past = min(i, max(keep(i), min(i, local)) + (local if keep(i) < i else 0))
        total += rows * past * block + rows * (rows + 1) // 2
    return total


def work(case):
    c, kind, n, d = case, case["kind"], case["n"], case["d"]
    es = 4 if c["dtype"] == "fp32" else 2
    if kind == "cascade":
        return dict(bytes=4 * n * d * es, flops=4 * d * _pairs(n, c["block"], lambda i: 8, 1))
    B, hq, hkv = c["B"], c["hq"], c["hkv"]
    if kind == "decode":  # summaries of the cache, then the K / V of the selected blocks
        nb = c["n"] // c["block"]
        keys = min(nb, c["top_c"] + c["local"] + 1) * c["block"]
        rows = B * c["tokens"]
        # (the query heads of a group select different blocks)
        return dict(bytes=rows * (hkv * nb * d * 8 + hkv * min(keys * hq // hkv, n) * d * 2 * es),
                    flops=rows * hq * (4 * nb * d + 4 * keys * d))
    if kind == "train":
        nb = -(-n // c["block"])
        keys = min(nb, c["top_c"] + c["local"] + 1) * c["block"]
        pairs = sum(min(t + 1, keys) for t in range(n))
        return dict(bytes=B * (hq * 4 + hkv * 4) * n * d * es,
                    flops=B * hq * (14 * d * pairs + 4 * d * n * nb))
    if kind in ("layer", "generate"):
        frac = c["frac"]
        pairs = _pairs(n, c["block"], lambda i: max(1, math.ceil(frac * i)), c["local"])
        nb, extra = n // c["block"], c.get("tokens", 0)
        keys = min(nb, max(1, math.ceil(frac * nb)) + c["local"] + 1) * c["block"]
        return dict(bytes=B * d * es * (2 * (hq + hkv) * n + extra * 2 * hkv * keys),
                    flops=B * hq * d * 4 * (pairs + extra * (keys + nb)))
    pairs = _pairs(n, c["block"], lambda i: c["top_c"], c["local"])
    nb = n // c["block"]
    route = 4 * d * nb * nb // 2 if kind == "prefill" else 2 * d * nb * int(nb ** 0.5)
    return dict(bytes=B * 2 * (hq + hkv) * n * d * es,
                flops=B * hq * (4 * d * pairs + route))


def tolerance(case):
    # seen against exact(): 2.6e-3 and 0.14 in bf16, 3.5e-4 in fp16, 5.2e-7 and 1.3e-5 in fp32
    return {"bf16": {"rel": 1e-2, "max": 0.5}, "fp16": {"rel": 1.5e-3, "max": 0.1},
            "fp32": {"rel": 2.5e-6, "max": 6e-5}}[case["dtype"]]


# ---------------------------------------------------------------------------------------------
# the same results in 64 bits (statistics and scores rounded to fp32 where the contract rounds
# them, so that the selections are the same)
# ---------------------------------------------------------------------------------------------

def _f32(x):
    return x.float().double()


def _means(x, block):
    """Block means of x (..., n, d), a last short block padded with zero rows."""
    n = x.shape[-2]
    x = torch.nn.functional.pad(x.double(), (0, 0, 0, -n % block))
    return _f32(x.unflatten(-2, (-1, block)).mean(-2))


def _stats(x, block, unbiased=False):
    """Block mean and variance over the rows that exist (unbiased: zero rows count as rows)."""
    n, nb = x.shape[-2], -(-x.shape[-2] // block)
    x = torch.nn.functional.pad(x.double(), (0, 0, 0, nb * block - n)).unflatten(-2, (nb, block))
    real = (torch.arange(nb * block, device=x.device) < (nb * block if unbiased else n))
    real = real.view(nb, block, 1).double()
    cnt = real.sum(1)
    mu = x.sum(-2) / cnt
    var = (((x - mu.unsqueeze(-2)) ** 2) * real).sum(-2) / (cnt - 1 if unbiased else cnt)
    return _f32(mu), _f32(var)


def _scores(rows, mu, var, coef2):
    """fl32(<q, mu>) + fl32(coef2 fl32(<q*q, var>)), summed in fp32; one head."""
    r = (rows @ mu.mT.contiguous()).float()
    return r + coef2 * (_f32(rows * rows) @ var.mT.contiguous()).float()


def _lists(r, ncand, keep, own, local):
    """Scores r (R, nb) -> sorted ids (R, W) with repeats and padding marked nb: the `keep` best of
    the first `ncand` blocks (ties to the lower), the own block and its predecessors."""
    R, nb = r.shape
    col = torch.arange(nb, device=r.device)
    r = r.masked_fill(col >= ncand[:, None], NEG)
    kmax = min(nb, int(keep.max()))
    top = torch.sort(r, dim=1, descending=True, stable=True).indices[:, :kmax]
    kept = torch.minimum(keep, ncand)[:, None]
    top = torch.where(torch.arange(kmax, device=r.device) < kept, top, nb)
    loc = own[:, None] - torch.arange(local + 1, device=r.device)
    return _unique(torch.cat([top, torch.where(loc >= 0, loc, nb)], 1), nb)


def _unique(ids, nb):
    ids = ids.sort(1).values
    ids[:, 1:] = torch.where(ids[:, 1:] == ids[:, :-1], nb, ids[:, 1:])
    return ids


def _attend(q, pos, k, v, ids, block, scale):
    """q (R, m, d) fp64 at positions pos (R, m) over the blocks ids (R, W) of k, v (n, d)."""
    n, d = k.shape
    nb = -(-n // block)
    j = (ids[:, :, None] * block + torch.arange(block, device=k.device)).flatten(1)
    ok = (ids < nb).repeat_interleave(block, 1) & (j < n)
    j = j.clamp(max=n - 1)
    s = torch.bmm(q, k[j].double().mT.contiguous()) * scale
    s.masked_fill_(~(ok[:, None, :] & (j[:, None, :] <= pos[:, :, None])), NEG)
    return torch.bmm(torch.softmax(s, -1), v[j].double())


def _prefill64(q, k, v, block, lists_of, scale):
    """Attention of q, k, v (B, H, n, d); lists_of(b, h, i0, i1) gives the block lists."""
    B, hq, n, d = q.shape
    G = hq // k.shape[1]
    nb = -(-n // block)
    out = torch.zeros(B, hq, n, d, device=q.device, dtype=torch.float64)
    step = None
    for b in range(B):
        for h in range(hq):
            kk, vv = k[b, h // G], v[b, h // G]
            qq = torch.nn.functional.pad(q[b, h].double(), (0, 0, 0, nb * block - n))
            qq = qq.view(nb, block, d)
            i0 = 0
            while i0 < nb:
                i1 = min(nb, i0 + (step or 1))
                ids = lists_of(b, h, i0, i1)
                step = max(1, (1 << 25) // (block * block * ids.shape[1]))
                i = torch.arange(i0, i1, device=q.device)
                pos = i[:, None] * block + torch.arange(block, device=q.device)
                o = _attend(qq[i0:i1], pos, kk, vv, ids, block, scale).flatten(0, 1)
                out[b, h, i0 * block:min(n, i1 * block)] = o[:n - i0 * block]
                i0 = i1
    return out


def _budget_lists(q, k, block, top_c, frac, local):
    """The query-block budget router's lists, by (b, h, i0, i1)."""
    qm = _means(q, block)
    mu, var = _stats(k, block)
    G = q.shape[1] // k.shape[1]

    def keep_of(i):
        if top_c is not None:
            return torch.full_like(i, top_c)
        return torch.ceil((torch.tensor(frac, device=i.device) * i.float())).long().clamp(min=1)

    def lists_of(b, h, i0, i1):
        i = torch.arange(i0, i1, device=q.device)
        r = _scores(qm[b, h, i0:i1], mu[b, h // G], var[b, h // G], 1.0)
        return _lists(r, i, keep_of(i), i, local)
    return lists_of


def _rows64(q, pos, k, v, mu, var, block, top_c, frac, local, scale):
    """One query per head, q (B, Hq, d) at `pos`, routed over the blocks complete there."""
    B, hq, d = q.shape
    hkv = k.shape[1]
    nc = (pos + 1) // block
    keep = top_c if top_c is not None else max(1, math.ceil(float(torch.tensor(frac)) * nc))
    out = torch.empty(B, hq, d, device=q.device, dtype=torch.float64)
    dev = q.device
    one = torch.ones(hq // hkv, device=dev, dtype=torch.long)
    for b in range(B):
        for g in range(hkv):
            hs = slice(g * len(one), (g + 1) * len(one))
            rows = q[b, hs].double()
            r = _scores(rows, mu[b, g, :nc], var[b, g, :nc], 1.0)
            r = torch.nn.functional.pad(r, (0, pos // block + 1 - nc), value=NEG)
            ids = _lists(r, one * nc, one * keep, one * (pos // block), local)
            p = torch.full((len(one), 1), pos, device=dev)
            out[b, hs] = _attend(rows[:, None], p, k[b, g, :pos + 1], v[b, g, :pos + 1], ids,
                                 block, scale)[:, 0]
    return out


def _train64(s, c):
    q, k, v = (s[x].double().requires_grad_(True) for x in "qkv")
    B, H, n, d = q.shape
    block = c["block"]
    mu, var = _stats(k.detach(), block, unbiased=True)
    t = torch.arange(n, device=q.device)
    outs = []
    for b in range(B):
        for h in range(H):
            r = _scores(q[b, h].detach(), mu[b, h], var[b, h], 0.5)
            ids = _lists(r, t // block + 1, torch.full_like(t, c["top_c"]), t // block, c["local"])
            sel = torch.zeros(n, mu.shape[2] + 1, device=q.device, dtype=torch.bool)
            sel.scatter_(1, ids, True)
            ok = sel[:, t // block] & (t[None, :] <= t[:, None])
            a = (q[b, h] @ k[b, h].T) * d ** -0.5
            outs.append(torch.softmax(a.masked_fill(~ok, NEG), -1) @ v[b, h])
    out = torch.stack(outs).view(B, H, n, d)
    return (out.detach(), *torch.autograd.grad(out, (q, k, v), s["g"].double()))


def _dot(a, b):
    return (a @ b.mT.contiguous()).float()


def _unit(x):
    nrm = x.norm(dim=-1, keepdim=True)
    return torch.where(nrm > 0, _f32(x / nrm), _f32(x))


def _ivf_lists(q, k, c):
    """The IVF router's lists per (b, h): spherical k-means over the block means, the four lists
    of best centroids, the 2 top_c best members, the first top_c of them that are not later."""
    block, top_c, local = c["block"], c["top_c"], c["local"]
    qb, mu = _means(q, block), _means(k, block)
    nb = mu.shape[2]
    nlist = min(nb, max(4, int(nb ** 0.5)))
    G = q.shape[1] // k.shape[1]
    found = {}
    for b in range(k.shape[0]):
        for g in range(k.shape[1]):
            m = mu[b, g]
            cent = _unit(m[torch.arange(nlist, device=m.device) * nb // nlist])
            for it in range(11):
                a = _best(_dot(m, cent))
                if it == 10:
                    break
                tot = torch.zeros_like(cent).index_add_(0, a, m)
                cent = torch.where(tot.norm(dim=1, keepdim=True) > 0, _unit(tot), cent)
            found[b, g] = cent, a

    def lists_of(b, h, i0, i1):
        cent, a = found[b, h // G]
        rows = qb[b, h, i0:i1]
        i = torch.arange(i0, i1, device=rows.device)
        order = torch.sort(_dot(rows, cent), dim=1, descending=True, stable=True).indices
        probed = torch.zeros(len(i), nlist, device=rows.device, dtype=torch.bool)
        probed.scatter_(1, order[:, :4], True)
        fine = _dot(rows, mu[b, h // G]).masked_fill(~probed[:, a], NEG)
        best = torch.sort(fine, dim=1, descending=True, stable=True)
        sk = min(2 * top_c, nb)
        ids, sc = best.indices[:, :sk], best.values[:, :sk]
        ok = (sc > NEG) & (ids <= i[:, None])
        ok &= ok.cumsum(1) <= top_c
        loc = i[:, None] - torch.arange(local + 1, device=rows.device)
        return _unique(torch.cat([torch.where(ok, ids, nb), torch.where(loc >= 0, loc, nb)], 1), nb)
    return lists_of


def _best(s):
    """Column of each row's largest score, the lowest where several are equal."""
    col = torch.arange(s.shape[1], device=s.device)
    return torch.where(s == s.max(1, keepdim=True).values, col, s.shape[1]).min(1).values


def _top(s, m):
    """Mask of each row's m largest scores above -inf, ties to the lower column."""
    order = torch.sort(s, dim=1, descending=True, stable=True)
    keep = torch.zeros_like(s, dtype=torch.bool)
    return keep.scatter_(1, order.indices[:, :m], order.values[:, :m] > NEG), order.values


class _Cells:
    """The cascade's index over its committed sub-block means: centroids, cells and radii."""

    def __init__(self, x, nlist, cent=None):
        n = x.shape[0]
        if cent is None:
            cent = x[torch.arange(nlist, device=x.device) * n // nlist]
        for _ in range(6):
            a = _best(_dot(x, cent))
            cnt = torch.bincount(a, minlength=nlist)[:, None]
            tot = torch.zeros_like(cent).index_add_(0, a, x)
            cent = torch.where(cnt > 0, _f32(tot / cnt.clamp(min=1)), cent)
        self.cent, self.of = cent, torch.empty(0, device=x.device, dtype=torch.long)
        self.radius = torch.zeros(nlist, device=x.device)
        self.built = n
        self.add(x)

    def add(self, x):
        a = _best(_dot(x, self.cent))
        r = (x - self.cent[a]).square().sum(1).sqrt().float()
        self.radius.scatter_reduce_(0, a, r, "amax")
        self.of = torch.cat([self.of, a])


def _cascade64(q, k, c, top_c=8, local=1, sub=32, search_k=32, cap=4):
    """The cascade's lists (nb, W) and certificates, chunk by chunk as the stream runs."""
    n, d, block = c["n"], c["d"], c["block"]
    dev, spb, nb = q.device, block // sub, n // block
    nlist = max(4, int((n / sub) ** 0.5))
    means, outl = torch.empty(0, d, device=dev, dtype=torch.float64), []
    cells, com, ids, certs = None, 0, [], []
    for t0 in range(0, n, c["chunk_blocks"] * block):
        t1 = min(n, t0 + c["chunk_blocks"] * block)
        if means.shape[0] > com:  # the chunk staged before this one is committed
            old, com = com, means.shape[0]
            if cells is not None:
                cells.add(means[old:])
                if com >= 2 * cells.built:
                    cells = _Cells(means, nlist, cells.cent)
            elif com >= max(4 * nlist, 16384):
                cells = _Cells(means, nlist)
        x = k[0, 0, t0:t1].double()
        mu = _means(x, sub)
        far = (x - mu.repeat_interleave(sub, 0)).square().sum(1).float()
        far = torch.sort(far, descending=True, stable=True).indices[:max(1, int(1e-3 * (t1 - t0)))]
        outl.append((x[far], (t0 + far) // block))
        means = torch.cat([means, mu])
        okey, opar = (torch.cat(z) for z in zip(*outl))

        blk = torch.arange(t0 // block, t1 // block, device=dev)
        qr = _means(q[0, 0, t0:t1], block)
        qn = qr.square().sum(1).sqrt().float()[:, None]
        sc, osc = _dot(qr, means), _dot(qr, okey)
        parent = torch.arange(means.shape[0], device=dev) // spb
        staged = (parent >= com // spb) & (parent < blk[:, None])
        staged = _top(sc.masked_fill(~staged, NEG), search_k)[0]
        todo = torch.arange(len(blk), device=dev)
        out = torch.empty(len(blk), top_c + cap + local + 1, device=dev, dtype=torch.long)
        cert = torch.zeros(len(blk), device=dev, dtype=torch.bool)
        nprobe, sk = min(4, nlist), search_k
        for rnd in range(3):
            s, b = sc[todo], blk[todo]
            open_ = (torch.arange(means.shape[0], device=dev) < com).expand_as(s).clone()
            last = torch.full((len(todo),), NEG, device=dev)
            if cells is not None:
                cs = _dot(qr[todo], cells.cent)
                probed = _top(cs, nprobe)[0]
                open_[:, :com] = probed[:, cells.of]
            kc = min(sk, com)
            if kc:
                open_, vals = _top(s.masked_fill(~open_, NEG), kc)
                last = vals[:, kc - 1]
            per = s.masked_fill(~(open_ | staged[todo]), NEG).unflatten(1, (-1, spb)).amax(2)
            kept, vals = _top(per, top_c)
            nkept = kept.sum(1)
            tau = vals.gather(1, (nkept - 1).clamp(min=0)[:, None])[:, 0]
            tau = torch.where(nkept > 0, tau, NEG)
            hit = (opar < b[:, None]) & (osc[todo] > tau[:, None])
            hit = _top(osc[todo].masked_fill(~hit, NEG), cap)[0]
            sel = torch.zeros(len(todo), nb + 1, device=dev, dtype=torch.bool)
            sel[:, :per.shape[1]] = kept
            sel.scatter_(1, torch.where(hit, opar, nb), True)
            loc = b[:, None] - torch.arange(local + 1, device=dev)
            sel.scatter_(1, torch.where(loc >= 0, loc, nb), True)
            sel[:, nb] = False
            order = torch.sort(sel.int(), dim=1, descending=True, stable=True)
            w = min(out.shape[1], nb)
            out[todo] = nb
            out[todo, :w] = torch.where(order.values[:, :w] > 0, order.indices[:, :w], nb)
            sure = (nkept >= b.clamp(max=top_c)) & ((tau > NEG) | (b == 0))
            if cells is not None:
                rest = (cs + qn[todo] * cells.radius).masked_fill(probed, NEG).amax(1)
                sure &= (tau > NEG) & (rest < tau) & (last < tau)
            cert[todo] = sure
            todo = todo[~sure]
            if cells is None or not len(todo):
                break
            nprobe, sk = min(4 * nprobe, nlist), min(2 * sk, com)
        ids.append(out)
        certs.append(cert)
    return torch.cat(ids), torch.cat(certs)


def exact(case, seed):
    c, kind = case, case["kind"]
    if work(c)["flops"] > 2e13:
        return None  # too long in 64 bits
    s = _inputs(c, seed)
    if kind == "train":
        return _train64(s, c)
    q, k, v, scale = s["q"], s["k"], s["v"], c["d"] ** -0.5
    if kind == "prefill":
        lists = _budget_lists(q, k, c["block"], c["top_c"], None, c["local"])
        return _prefill64(q, k, v, c["block"], lists, scale), None, None
    if kind == "ivf":
        return _prefill64(q, k, v, c["block"], _ivf_lists(q, k, c), scale), None, None
    if kind == "cascade":
        ids, _ = _cascade64(q, k, c)
        out = _prefill64(q, k, v, c["block"], lambda b, h, i0, i1: ids[i0:i1], scale)
        return out, None, None, None
    n, block, tokens = c["n"], c["block"], c.get("tokens", 0)
    mu, var = _stats(k[:, :, :(n + tokens) // block * block], block)
    if kind == "decode":
        outs = [_rows64(q[t], n + t, k, v, mu, var, block, c["top_c"], None, c["local"], scale)
                for t in range(tokens)]
        return outs, None, None, None, None, None, None
    lists = _budget_lists(q[:, :, :n], k[:, :, :n], block, None, c["frac"], c["local"])
    outs = [_prefill64(q[:, :, :n], k[:, :, :n], v[:, :, :n], block, lists, scale).transpose(1, 2)]
    for t in range(n, n + tokens):
        outs.append(_rows64(q[:, :, t], t, k, v, mu, var, block, None, c["frac"], c["local"],
                            scale)[:, None])
    return outs
