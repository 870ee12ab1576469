"""GPU parity tests: the HIP kernels (through the C ABI, via the ssa_amd drop-in API) against the
CPU oracle and the reference's golden outputs, on the seeded configurations and edge cases.

Bars: selections bit-exact against the oracle and equal to the reference's float32 selections
except on certified float32 near-ties; summaries within 1 ulp of the oracle; attention outputs
within 2e-2 (bf16/fp16) or 1e-5 (fp32) max-abs of the oracle's float64 masked softmax."""
import functools
import math

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from oracle import ssa_oracle as O
from ssa_amd import gemma_ssa as G
from ssa_amd import ivf_decode as D
from ssa_amd import ssa_kernel as K
from ssa_amd import workloads as WL
from tests import golden_util as GU
from tests.test_oracle import (ROUTE_CASES, certificate_d, certificate_inputs, oracle_route,
                               resolve_kw)

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 1e-5, torch.float16: 2e-2, torch.bfloat16: 2e-2}


def dev(x, dtype, cuda):
    return WL.to_device(x, dtype, cuda)


def np_of(t):
    return t.detach().float().cpu().numpy()


def ulp_diff(a, b):
    a = np.ascontiguousarray(a, dtype=np.float32).view(np.int32).astype(np.int64)
    b = np.ascontiguousarray(b, dtype=np.float32).view(np.int32).astype(np.int64)
    return np.abs(a - b)


# ---- a1 / a2 summaries -------------------------------------------------------------------------

@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_block_summary_matches_oracle(cuda, dtype):
    rng = np.random.default_rng(7)
    x = WL.round_to(rng.standard_normal((2, 3, 1000, 64)).astype(np.float32) * 3 + 1, dtype)
    xt = dev(x, dtype, cuda)
    mu, var, m3 = K.block_summary(xt, 128, "pop", n_real=990, with_m3=True)
    omu, ovar, om3 = O.block_stats(x, 128, "pop", n_real=990)
    assert ulp_diff(np_of(mu), omu).max() <= 1
    assert ulp_diff(np_of(var), ovar).max() <= 1
    assert np.abs(np_of(m3) - om3).max() <= 1e-6 * np.abs(om3).max()
    mu_u, var_u, _ = K.block_summary(xt[:, :, :896], 128, "unbiased")
    _, ovar_u, _ = O.block_stats(x[:, :, :896], 128, "unbiased")
    assert ulp_diff(np_of(var_u), ovar_u).max() <= 1
    qb = K.block_summary(xt, 128, "qmean")
    assert ulp_diff(np_of(qb), O.qmean(x, 128)).max() <= 1


@pytest.mark.parametrize("d", [24, 96, 128, 200, 512])
def test_block_summary_other_head_dims(cuda, d):
    """Head dims other than 64: 128 takes the one-wave-per-block kernel with 4 row groups per
    wave; the others the workgroup-per-block kernel, whose 8-column groups do not all divide the
    256 threads (the last threads idle)."""
    rng = np.random.default_rng(8)
    x = WL.round_to(rng.standard_normal((1, 2, 700, d)).astype(np.float32) * 2 - 1, torch.bfloat16)
    xt = dev(x, torch.bfloat16, cuda)
    mu, var, m3 = K.block_summary(xt, 64, "pop", n_real=690, with_m3=True)
    omu, ovar, om3 = O.block_stats(x, 64, "pop", n_real=690)
    assert ulp_diff(np_of(mu), omu).max() <= 1
    assert ulp_diff(np_of(var), ovar).max() <= 1
    assert np.abs(np_of(m3) - om3).max() <= 1e-6 * np.abs(om3).max()
    assert ulp_diff(np_of(K.block_summary(xt, 64, "qmean")), O.qmean(x, 64)).max() <= 1


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_block_summary_counts_zero_rows_past_n(cuda, dtype):
    """n_real > n: rows [n, n_real) count as zero rows (the zero padding ssa_swap applies before
    its block statistics) -- equal to the statistics of the explicitly zero-padded tensor."""
    rng = np.random.default_rng(9)
    x = WL.round_to(rng.standard_normal((1, 2, 300, 64)).astype(np.float32) + 0.5, dtype)
    xp = np.zeros((1, 2, 320, 64), dtype=np.float32)
    xp[:, :, :300] = x
    for mode in ("pop", "unbiased"):
        mu, var, m3 = K.block_summary(dev(x, dtype, cuda), 64, mode, n_real=320, with_m3=True)
        omu, ovar, om3 = O.block_stats(xp, 64, mode)
        assert ulp_diff(np_of(mu), omu).max() <= 1 and ulp_diff(np_of(var), ovar).max() <= 1
        assert np.abs(np_of(m3) - om3).max() <= 1e-6 * np.abs(om3).max()
        # n_real beyond the last block is capped there
        mu2, var2, _ = K.block_summary(dev(x, dtype, cuda), 64, mode, n_real=10**6)
        assert torch.equal(mu2, mu) and torch.equal(var2, var)


def test_block_summary_strided_input(cuda):
    """A (b, n, h, d) buffer viewed as (b, h, n, d) needs no copy and gives the same stats."""
    rng = np.random.default_rng(8)
    x = rng.standard_normal((1, 512, 4, 64)).astype(np.float32)
    xt = dev(x, torch.float32, cuda).transpose(1, 2)
    mu, var, _ = K.block_summary(xt, 64, "pop")
    omu, ovar, _ = O.block_stats(x.transpose(0, 2, 1, 3), 64, "pop")
    assert ulp_diff(np_of(mu), omu).max() <= 1 and ulp_diff(np_of(var), ovar).max() <= 1


# ---- a3-a5 router ------------------------------------------------------------------------------

def gpu_route(p, mode, kw, cuda):
    cfg = p["cfg"]
    kw = resolve_kw(cfg, kw, pair_as="object")
    q = dev(p["q"], cfg.dtype, cuda)
    k = dev(p["k"], cfg.dtype, cuda)
    if mode == "flat":
        kv_num, kv_idx, _ = K.block_route(q, k, cfg.block, compact=True, **kw)
    else:
        kv_num, kv_idx, _ = K.block_route_budget(q, k, cfg.block, compact=True, **kw)
    return kv_num.cpu().numpy(), kv_idx.cpu().numpy()


@pytest.mark.parametrize("case", list(ROUTE_CASES))
def test_route_bit_exact_vs_oracle_and_reference(cuda, case):
    cfg_name, variant, mode, kw = ROUTE_CASES[case]
    p = WL.make(cfg_name, variant)
    kv_num, kv_idx = gpu_route(p, mode, dict(kw), cuda)
    onum, oidx = oracle_route(p, mode, dict(kw))
    n, n_eq, _, bad = GU.compare_selections(kv_num, kv_idx, onum, oidx)
    assert n_eq == n, f"{n - n_eq} rows differ from the oracle: {bad[:3]}"
    assert (kv_num == onum).all()
    g = GU.load(case)
    r64, mag = certificate_inputs(p, mode, kw)
    n, n_eq, n_cert, bad = GU.compare_selections(kv_num, kv_idx, g["kv_num"], g["kv_idx"], r64, mag,
                                                 d=certificate_d(p["cfg"], kw))
    print(f"{case}: {n} rows, {n_eq} identical to the reference, {n_cert} certified near-ties")
    assert not bad, bad[:3]


def test_route_budget_frac_and_edge_rows(cuda):
    """budget_frac keep in float32, top_c >= #blocks (dense), top_c = 0 (local window only),
    a single block, and beta = 0 == centroid routing (test_share_route.py:27-37)."""
    rng = np.random.default_rng(9)
    q = rng.standard_normal((1, 2, 40 * 32, 64)).astype(np.float32)
    k = rng.standard_normal((1, 2, 40 * 32, 64)).astype(np.float32)
    qt, kt = dev(q, torch.float32, cuda), dev(k, torch.float32, cuda)
    for kw in (dict(budget_frac=0.1, local=1), dict(budget_frac=0.3, local=0),
               dict(budget_frac=1.0, local=1), dict(top_c=999, local=1), dict(top_c=0, local=2),
               dict(top_c=3, local=1, beta=0.0)):
        a, b, _ = K.block_route_budget(qt, kt, 32, compact=True, **kw)
        on, oi = O.route_budget(q, k, 32, **{"top_c": None, **kw})
        n, n_eq, _, bad = GU.compare_selections(a.cpu().numpy(), b.cpu().numpy(), on, oi)
        assert n_eq == n, (kw, bad[:3])
    one, onei, _ = K.block_route_budget(qt[:, :, :32], kt[:, :, :32], 32, compact=True, top_c=4)
    assert one.cpu().tolist() == [[[1], [1]]] and onei.cpu().tolist() == [[[[0]], [[0]]]]
    a0 = K.block_route_budget(qt, kt, 32, top_c=3, local=1, beta=0.0, compact=True)
    ac = K.route(K.block_summary(qt, 32, "qmean"), K.block_summary(kt, 32, "pop")[0], None, None,
                 "budget", 3, 0.0, 1, 0.0)
    assert torch.equal(a0[0], ac[0]) and torch.equal(a0[1], ac[1])


def test_route_ties_take_lowest_index(cuda):
    """Identical key blocks tie exactly: the lowest block indices win."""
    x = np.ones((1, 1, 16 * 32, 8), dtype=np.float32)
    xt = dev(x, torch.float32, cuda)
    kv_num, kv_idx, _ = K.block_route_budget(xt, xt, 32, top_c=3, local=0, compact=True)
    rows = GU.row_sets(kv_num.cpu().numpy(), kv_idx.cpu().numpy())
    for i, s in enumerate(rows):
        assert s == frozenset(list(range(min(3, i))) + [i]), (i, s)


@pytest.mark.parametrize("nbk", [600, 6000])
@pytest.mark.parametrize("case", ["near_ties", "exact_ties", "distinct_tiles", "boundary_tie"])
def test_certified_router_band_cases(cuda, nbk, case):
    """The certified MFMA router (more than 16 rows per key head: 2 query heads x 40 rows) on
    inputs that stress its certificate, against the exact oracle selection row by row.
    near_ties: every candidate mean lies within 1e-6 relative of one vector, so every score
    falls inside the error band -- the whole row is ranked exactly (a wave-uniform rescoring
    loop for 600 blocks, the wide-band fallback for 6000). exact_ties: 100 identical best blocks
    straddle the keep-th place (lowest indices win). distinct_tiles: 64 planted winners, one per
    64-block tile at 6000 blocks, so the tile-maximum filter keeps exactly keep candidates and
    the band reaches below its threshold (at 600 blocks, 9 tiles, the winners lie anywhere).
    boundary_tie: as distinct_tiles plus an exact copy of the weakest winner outside the winners'
    tiles (a band of two, ranked by index)."""
    rng = np.random.default_rng(31)
    d, block, keep, rows_per_head = 64, 64, 64, 40
    q = rng.standard_normal((1, 2, rows_per_head, d)).astype(np.float32)
    mu = rng.standard_normal((1, 1, nbk, d)).astype(np.float32) * 0.1
    var = rng.uniform(0.5, 1.5, (1, 1, nbk, d)).astype(np.float32)
    if case == "near_ties":
        base = rng.standard_normal(d).astype(np.float32)
        mu[0, 0] = base * (1.0 + 1e-6 * rng.standard_normal((nbk, 1))).astype(np.float32)
        var[:] = 1.0
    elif case == "exact_ties":
        best = rng.choice(nbk, 100, replace=False)
        var[0, 0, best] = 4.0
        mu[0, 0, best] = 0.0
    else:
        if nbk // 64 >= keep:
            tiles = rng.choice(nbk // 64, keep, replace=False)
            won = tiles * 64 + rng.integers(0, 64, keep)
        else:  # fewer tiles than winners (the one-wave select): winners anywhere
            won = rng.choice(nbk, keep, replace=False)
            tiles = np.unique(won // 64)
        var[0, 0, won] = (6.0 + 0.01 * np.arange(keep))[:, None]
        mu[0, 0, won] = 0.0
        if case == "boundary_tie":
            weakest = won[0]
            free = np.setdiff1d(np.arange(nbk), won)
            free_tiles = np.setdiff1d(np.arange(nbk // 64), tiles)
            twin = free_tiles[0] * 64 + 5 if len(free_tiles) else free[0]
            var[0, 0, twin] = var[0, 0, weakest]
            mu[0, 0, twin] = mu[0, 0, weakest]
    pos0 = nbk * block - rows_per_head
    kv_num, kv_idx = K.route(dev(q, torch.float32, cuda), dev(mu, torch.float32, cuda),
                             dev(var, torch.float32, cuda), None, "query", keep, 0.0, 1, 1.0,
                             query_pos=pos0, block=block)
    gn, gi = kv_num.cpu().numpy(), kv_idx.cpu().numpy()
    keys = O.score_keys(O.scores(q, mu, var, 1.0))
    for h in range(2):
        for r in range(rows_per_head):
            sel = O.select_row(keys[0, h, r], r, "query", keep, 0.0, 1, pos0, block)
            assert gi[0, h, r, :gn[0, h, r]].tolist() == sel, (case, nbk, h, r)


@pytest.mark.parametrize("d, terms, pool, limit", [
    (64, "mu", 1, None), (64, "mu_var", 1, None), (64, "mu_var_m3", 1, None),
    (128, "mu_var", 1, None), (32, "mu_var", 1, 6 << 20), (64, "mu_var", 2, None)])
def test_route_strip_scoring_matches_oracle(cuda, d, terms, pool, limit):
    """Rows of more than 1024 candidates score with the row operands held in registers, a strip
    of 128 rows per workgroup (contractions of 64, 128, 192 and 256 values: d x terms). Budget
    mode over 1300 blocks with 2 query heads per key head: 2600 rows in 21 strips (the last one
    partial, one straddling the heads), rows of 0 to 1299 candidates (21 tiles, two segments);
    one case routes in row chunks (a 6 MiB workspace), one max-pools 2 sub-blocks per block (no
    tile maxima). Every row against the oracle's selection."""
    rng = np.random.default_rng(47)
    nb, hq, keep = 1300, 2, 64
    rows = rng.standard_normal((1, hq, nb, d)).astype(np.float32)
    mu = (rng.standard_normal((1, 1, nb * pool, d)) * 0.3).astype(np.float32)
    var = rng.uniform(0.5, 1.5, (1, 1, nb * pool, d)).astype(np.float32) if "var" in terms else None
    m3 = (rng.standard_normal((1, 1, nb * pool, d)) * 0.2).astype(np.float32) \
        if "m3" in terms else None
    coef2, coef3 = (1.0 if var is not None else 0.0), (0.25 if m3 is not None else 0.0)
    t = lambda x: None if x is None else dev(x, torch.float32, cuda)
    kw = {} if limit is None else {"workspace_limit": limit}
    kv_num, kv_idx = K.route(t(rows), t(mu), t(var), t(m3), "budget", keep, 0.0, 1, coef2,
                             coef3, pool=pool, **kw)
    gn, gi = kv_num.cpu().numpy(), kv_idx.cpu().numpy()
    keys = O.score_keys(O.pool_max(O.scores(rows, mu, var, coef2, m3, coef3), pool))
    for h in range(hq):
        for i in range(nb):
            sel = O.select_row(keys[0, h, i], i, "budget", keep, 0.0, 1)
            assert gi[0, h, i, :gn[0, h, i]].tolist() == sel, (d, terms, pool, h, i)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", [(4, 1, 3, 40, "started"), (2, 1, 1, 500, "query"),
                                   (4, 2, 24, 300, "query"), (1, 1, 200, 200, "budget")])
def test_route_16bit_rows_equal_fp32_rows(cuda, dtype, shape):
    """The router reads fp16 / bf16 query rows directly (their fp32 values are exact): the same
    lists as for the fp32 copy, on each score kernel (fused <= 64 blocks, few rows, tiles)."""
    hq, hkv, nbq, nbk, mode = shape
    rng = np.random.default_rng(31)
    rows = WL.round_to(rng.standard_normal((1, hq, nbq, 64)).astype(np.float32), dtype)
    mu = rng.standard_normal((1, hkv, nbk, 64)).astype(np.float32)
    var = rng.uniform(0.5, 1.5, (1, hkv, nbk, 64)).astype(np.float32)
    r16, r32 = dev(rows, dtype, cuda), dev(rows, torch.float32, cuda)
    assert r16.dtype == dtype
    kw = dict(query_pos=nbk * 64 - nbq - 5, block=64) if mode != "budget" else {}
    a = K.route(r16, dev(mu, torch.float32, cuda), dev(var, torch.float32, cuda), None, mode, 8,
                0.0, 1, 1.0, **kw)
    b = K.route(r32, dev(mu, torch.float32, cuda), dev(var, torch.float32, cuda), None, mode, 8,
                0.0, 1, 1.0, **kw)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


@pytest.mark.parametrize("nbk", [200, 300, 3000, 12000, 20000])
@pytest.mark.parametrize("case", ["random", "top_ties", "all_equal"])
def test_route_long_rows_match_oracle(cuda, case, nbk):
    """Query rows over 200 to 20000 key blocks, keep 64, through every select: one wave per row
    (200, 300), the two-stage chunked select (3000, 12000) and the filtered radix select (20000,
    more than fit in LDS). Random scores, ties at the top (100 identical best blocks: the lowest
    indices win) and all scores equal (ties spread over every lane and slot; for 20000 the
    filter keeps too much and the select falls back to the whole row)."""
    rng = np.random.default_rng(21)
    d, block = 64, 64
    mu = rng.standard_normal((1, 1, nbk, d)).astype(np.float32)
    var = rng.uniform(0.5, 1.5, (1, 1, nbk, d)).astype(np.float32)
    rows = rng.standard_normal((1, 2, 3, d)).astype(np.float32)
    if case == "top_ties":
        best = rng.choice(nbk, 100, replace=False)
        mu[0, 0, best] = 3.0 * rows[0, 0, 0] / np.linalg.norm(rows[0, 0, 0])
        var[0, 0, best] = 1.0
    elif case == "all_equal":
        mu[:] = mu[0, 0, 0]
        var[:] = var[0, 0, 0]
    pos0 = nbk * block - 3
    kv_num, kv_idx = K.route(dev(rows, torch.float32, cuda), dev(mu, torch.float32, cuda),
                             dev(var, torch.float32, cuda), None, "query", 64, 0.0, 1, 1.0,
                             query_pos=pos0, block=block)
    gn, gi = kv_num.cpu().numpy(), kv_idx.cpu().numpy()
    keys = O.score_keys(O.scores(rows, mu, var, 1.0))
    for h in range(2):
        for r in range(3):
            sel = O.select_row(keys[0, h, r], r, "query", 64, 0.0, 1, pos0, block)
            assert gi[0, h, r, :gn[0, h, r]].tolist() == sel, (case, h, r)


def test_block_route_budget_sub_identity_and_recall(cuda):
    """sub=None is identical to the default; with centroid scores sub=32 finds a planted
    coherent 32-key sub-block whose block mean is diluted (test_cascade_router.py:147-167)."""
    rng = np.random.default_rng(23)
    n, block = 8 * 128, 128
    q = WL.round_to(rng.standard_normal((1, 1, n, 64)).astype(np.float32), torch.float16)
    k = WL.round_to(rng.standard_normal((1, 1, n, 64)).astype(np.float32), torch.float16)
    qt, kt = dev(q, torch.float16, cuda), dev(k, torch.float16, cuda)
    a = K.block_route_budget(qt, kt, block, top_c=2, local=1)
    b = K.block_route_budget(qt, kt, block, top_c=2, local=1, sub=None)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1]) and torch.equal(a[2], b[2])
    u = rng.standard_normal(64)
    u = (u / np.linalg.norm(u)).astype(np.float32)
    q2, k2 = q.copy(), k.copy()
    q2[0, 0, n - block:] = WL.round_to(u[None], torch.float16)   # last query block points at u
    k2[0, 0, block:block + 32] = WL.round_to(u[None], torch.float16)  # block 1, sub-block 0
    q2t, k2t = dev(q2, torch.float16, cuda), dev(k2, torch.float16, cuda)
    qblk = (n - 1) // block
    _, _, sub_sel = K.block_route_budget(q2t, k2t, block, top_c=1, local=0, sub=32, beta=0.0)
    assert bool(sub_sel[0, 0, qblk, 1]), "sub-block routing should select the coherent block"
    for beta in (0.0, 2.0):
        on, oi = O.route_budget(q2, k2, block, top_c=1, local=0, sub=32, beta=beta)
        gn, gi, _ = K.block_route_budget(q2t, k2t, block, top_c=1, local=0, sub=32, beta=beta,
                                         compact=True)
        assert (gn.cpu().numpy() == on).all() and (gi.cpu().numpy() == oi).all()


def test_block_route_budget_proj_identity(cuda):
    """proj = identity reproduces centroid-only (beta = 0) routing exactly
    (test_share_route.py:27-37)."""
    torch.manual_seed(0)
    q = torch.randn(1, 1, 8 * 128, 64, device=cuda)
    k = torch.randn_like(q)
    a = K.block_route_budget(q, k, 128, top_c=3, local=1, proj=torch.eye(64))
    b = K.block_route_budget(q, k, 128, top_c=3, local=1, beta=0.0)
    assert torch.equal(a[0], b[0]) and torch.equal(a[2], b[2])


def test_route_reference_dense_outputs(cuda):
    """Default (non-compact) returns the reference's (kv_num, argsort-order kv_idx, sel)."""
    rng = np.random.default_rng(10)
    q = rng.standard_normal((1, 2, 8 * 64, 64)).astype(np.float32)
    k = rng.standard_normal((1, 2, 8 * 64, 64)).astype(np.float32)
    kv_num, kv_full, sel = K.block_route_budget(dev(q, torch.float32, cuda),
                                                dev(k, torch.float32, cuda), 64, top_c=2, local=1)
    assert sel.dtype == torch.bool and sel.shape == (1, 2, 8, 8)
    ref = torch.argsort(sel.cpu().int(), dim=-1, descending=True, stable=True).int()
    assert torch.equal(kv_full.cpu(), ref)
    assert torch.equal(kv_num.cpu(), sel.cpu().sum(-1).int())
    qi = torch.arange(8)
    assert not (sel.cpu() & (qi[:, None] < qi[None, :])).any()


# ---- a6-a8 attention ---------------------------------------------------------------------------

def test_ssa_flex_c1_fp32_matches_reference_flexattention(cuda):
    g = GU.load("c1_flex_out")
    p = WL.make("C1")
    q, k, v = (dev(p[x], torch.float32, cuda) for x in ("q", "k", "v"))
    out = K.ssa_flex(q, k, v, block=64, top_c=8, local=1)
    err = np.abs(np_of(out) - g["out"]).max()
    assert err < 1e-5, err


@functools.lru_cache(maxsize=1)
def c3_inputs():
    """The C3 bench input (host arrays), generated once per test session."""
    return WL.make("C3")


@pytest.mark.parametrize("cfg_name,n,qblocks", [("C2", 8192, [0, 1, 5, 63, 127]),
                                                ("C2", 32768, [0, 2, 100, 311, 511]),
                                                ("C3", 131072, [0, 3, 64, 511, 1023])])
def test_sparse_attention_matches_oracle(cuda, cfg_name, n, qblocks):
    p = c3_inputs() if cfg_name == "C3" else WL.make(cfg_name, n=n)
    cfg = p["cfg"]
    q, k, v = (dev(p[x], cfg.dtype, cuda) for x in ("q", "k", "v"))
    kv_num, kv_idx, _ = K.block_route_budget(q, k, cfg.block, top_c=cfg.top_c, local=cfg.local,
                                             beta=cfg.beta, compact=True)
    out = K.sparse_attention(q, k, v, kv_num, kv_idx, cfg.block)
    heads = [0, 6, 13]
    ref = O.sparse_attention(p["q"], p["k"], p["v"], kv_num.cpu().numpy(), kv_idx.cpu().numpy(),
                             cfg.block, qblocks=qblocks, heads=heads)
    o = np_of(out)
    for h in heads:
        for i in qblocks:
            sl = slice(i * cfg.block, (i + 1) * cfg.block)
            err = np.abs(o[0, h, sl] - ref[0, h, sl]).max()
            assert err < TOL[cfg.dtype], (h, i, err)
    assert torch.isfinite(out).all()


def test_c3_attention_whole_heads_match_oracle(cuda):
    """Every query block (all 1,024) of query heads 0 and 13 -- one per key head -- of the C3
    bench input against the float64 oracle (every C3 workgroup takes the bounded-row path)."""
    p = c3_inputs()
    cfg = p["cfg"]
    q, k, v = (dev(p[x], cfg.dtype, cuda) for x in ("q", "k", "v"))
    kv_num, kv_idx, _ = K.block_route_budget(q, k, cfg.block, top_c=cfg.top_c, local=cfg.local,
                                             beta=cfg.beta, compact=True)
    out = np_of(K.sparse_attention(q, k, v, kv_num, kv_idx, cfg.block))
    heads = [0, 13]
    ref = O.sparse_attention(p["q"], p["k"], p["v"], kv_num.cpu().numpy(), kv_idx.cpu().numpy(),
                             cfg.block, heads=heads)
    err = max(float(np.abs(out[0, h] - ref[0, h]).max()) for h in heads)
    print(f"C3 heads {heads}, all {cfg.n // cfg.block} query blocks: max |err| {err:.3g}")
    assert err < TOL[cfg.dtype], err


@pytest.mark.parametrize("seed", [0, 1, 2])
def test_c3_shape_rows_near_the_bound(cuda, seed):
    """C3-shaped inputs (14q/2kv, d 64, block 128, top_c 64 + local 2, beta 2, keys from the
    segmented Gaussian mixture, n = 32,768) with every query row rescaled so that
    scale*log2e*|q|*max|k| (max over the key head) lies in [0.9, 0.995] of the bf16 admission
    bound: every workgroup takes the bounded-row path with rows at its edge. 48 query blocks of
    4 heads against the float64 oracle."""
    cfg = WL.C3
    n, c = 32768, math.log2(math.e) / 8.0
    rng = np.random.default_rng(1000 + seed)
    q = rng.standard_normal((1, cfg.Hq, n, cfg.d), dtype=np.float32)
    k = WL.round_to(WL._gmm_keys(rng, cfg.Hkv, n, cfg.d), cfg.dtype)
    v = WL.round_to(rng.standard_normal((1, cfg.Hkv, n, cfg.d), dtype=np.float32), cfg.dtype)
    kmax = np.sqrt((k.astype(np.float64) ** 2).sum(-1)).max(-1)  # (1, Hkv)
    G = cfg.Hq // cfg.Hkv
    u = rng.uniform(0.9, 0.995, size=(1, cfg.Hq, n, 1))
    target = u * FAST_BOUND[cfg.dtype] / (c * np.repeat(kmax, G, axis=1)[:, :, None, None])
    q = q / np.linalg.norm(q, axis=-1, keepdims=True) * target
    q = WL.round_to(q.astype(np.float32), cfg.dtype)
    qmax = np.linalg.norm(q.astype(np.float64), axis=-1).max(-1)  # (1, Hq)
    bound = float((c * qmax * np.repeat(kmax, G, axis=1)).max())
    assert 0.95 * FAST_BOUND[cfg.dtype] < bound < FAST_BOUND[cfg.dtype], bound
    qt, kt, vt = (dev(x, cfg.dtype, cuda) for x in (q, k, v))
    kv_num, kv_idx, _ = K.block_route_budget(qt, kt, cfg.block, top_c=cfg.top_c, local=cfg.local,
                                             beta=cfg.beta, compact=True)
    out = np_of(K.sparse_attention(qt, kt, vt, kv_num, kv_idx, cfg.block))
    qblocks = sorted(set(rng.choice(n // cfg.block, 47, replace=False).tolist()) | {n // cfg.block - 1})
    heads = [0, 6, 7, 13]
    ref = O.sparse_attention(q, k, v, kv_num.cpu().numpy(), kv_idx.cpu().numpy(), cfg.block,
                             qblocks=qblocks, heads=heads)
    err = max(float(np.abs(out[0, h, i * cfg.block:(i + 1) * cfg.block] -
                        ref[0, h, i * cfg.block:(i + 1) * cfg.block]).max())
              for h in heads for i in qblocks)
    print(f"seed {seed}: max bound {bound:.2f}, max |err| {err:.3g}")
    assert err < TOL[cfg.dtype], err


@pytest.mark.parametrize("dtype,block", [(torch.bfloat16, 128), (torch.float16, 256)])
def test_rotated_walk_and_exact_flag(cuda, dtype, block):
    """rotate=True: each bounded-row workgroup starts its walk over its key blocks at a position
    taken from the GPU clock (lists of <= 128 entries), so the summation order, and the output's
    last bits, vary between calls; the default walks in list order and repeats bit for bit, as
    does rotate=True under torch.use_deterministic_algorithms(True). Every output -- and that of
    exact=True, which sends every workgroup to the exact path -- within 2e-2 of the oracle on
    sampled blocks, rotated within 4e-3 of the list-order output."""
    rng = np.random.default_rng(77)
    n, hq, hkv = 16384, 4, 2
    q, k, v = (WL.round_to(rng.standard_normal((1, h_, n, 64)).astype(np.float32), dtype)
               for h_ in (hq, hkv, hkv))
    qt, kt, vt = (dev(x, dtype, cuda) for x in (q, k, v))
    kv_num, kv_idx, _ = K.block_route_budget(qt, kt, block, top_c=32, local=1, beta=2.0,
                                             compact=True)
    det = [K.sparse_attention(qt, kt, vt, kv_num, kv_idx, block) for _ in range(2)]
    rot = [K.sparse_attention(qt, kt, vt, kv_num, kv_idx, block, rotate=True) for _ in range(3)]
    prev = torch.are_deterministic_algorithms_enabled()
    torch.use_deterministic_algorithms(True, warn_only=True)
    try:
        det.append(K.sparse_attention(qt, kt, vt, kv_num, kv_idx, block, rotate=True))
    finally:
        torch.use_deterministic_algorithms(prev)
    assert torch.equal(det[0], det[1]) and torch.equal(det[0], det[2])
    spread = max(float((r.float() - det[0].float()).abs().max()) for r in rot)
    print(f"{dtype} block {block}: rotated vs list-order walk max |diff| {spread:.3g}")
    assert spread < 4e-3, spread
    # exact=True: every workgroup on the exact (running-max, fp32-scaled) path
    ex = K.sparse_attention(qt, kt, vt, kv_num, kv_idx, block, exact=True)
    rot.append(ex)
    qblocks = [0, 1, n // block // 2, n // block - 1]
    ref = O.sparse_attention(q, k, v, kv_num.cpu().numpy(), kv_idx.cpu().numpy(), block,
                             qblocks=qblocks, heads=[0, 3])
    for o in det[:1] + rot:
        oo = np_of(o)
        for h in (0, 3):
            for i in qblocks:
                sl = slice(i * block, (i + 1) * block)
                assert np.abs(oo[0, h, sl] - ref[0, h, sl]).max() < TOL[dtype]


def two_key_case(dtype, target, rounding, seed=0, n=2048, block=128, amp=1.0, scale=0.125):
    """A case built against the bounded-row path's one approximation, the rounding of
    q*scale*log2e before the QK product. Query block i (i >= 1) repeats one query row q_i with
    scale*log2e*|q_i|*8 = target; key block i-1 starts with two keys k+- = a*qh +- b*w (|k+-| =
    8, a = 4, qh = q_i/|q_i|) whose exact scores are equal, w being the part orthogonal to qh of
    the rounding error of q_i*scale*log2e in `rounding` (float16: what the kernel rounds to;
    bfloat16: what it rounded to before) -- so that rounding moves the two scores in opposite
    directions by the largest amount its error allows. Their values are +-amp*e_(i mod 64): the
    exact output there is 0 and a score difference of x log2 units shows as amp*tanh(x ln2/2).
    The other keys: random directions of norm 2.4, values ~0.1 N(0,1). Lists: [i-1, i]."""
    rng = np.random.default_rng(seed)
    d, c, kn = 64, scale * math.log2(math.e), 8.0
    nb = n // block
    q = np.zeros((1, 1, n, d), np.float32)
    for i in range(nb):
        x = rng.standard_normal(d)
        q[0, 0, i * block:(i + 1) * block] = x / np.linalg.norm(x) * (target / (c * kn))
    q = WL.round_to(q, dtype)
    r = rng.standard_normal((1, 1, n, d))
    k = (r / np.linalg.norm(r, axis=-1, keepdims=True) * 0.3 * kn).astype(np.float32)
    v = (0.1 * rng.standard_normal((1, 1, n, d))).astype(np.float32)
    a = 0.5 * kn
    b = math.sqrt(kn * kn - a * a) * 0.999
    for i in range(1, nb):
        x = q[0, 0, i * block].astype(np.float64)
        qc = x * c
        delta = WL.round_to(qc.astype(np.float32), rounding).astype(np.float64) - qc
        qh = x / np.linalg.norm(x)
        w = delta - (delta @ qh) * qh
        w /= np.linalg.norm(w)
        p0 = (i - 1) * block
        k[0, 0, p0], k[0, 0, p0 + 1] = a * qh + b * w, a * qh - b * w
        v[0, 0, p0:p0 + 2] = 0.0
        v[0, 0, p0, i % d], v[0, 0, p0 + 1, i % d] = amp, -amp
    k, v = WL.round_to(k, dtype), WL.round_to(v, dtype)
    kv_num = np.full((1, 1, nb), 2, np.int32)
    kv_num[0, 0, 0] = 1
    kv_idx = np.array([[[[max(i - 1, 0), i] for i in range(nb)]]], np.int32)
    return q, k, v, kv_num, kv_idx, block, scale


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("target", [16.0, 31.0, 40.0])
@pytest.mark.parametrize("rounding", [torch.float16, torch.bfloat16])
def test_bounded_rows_constructive_rounding(cuda, dtype, target, rounding):
    """two_key_case: rounding errors of q*scale*log2e added constructively along k. Just under
    the admission bound (31) the bounded path rounds q*scale*log2e to fp16 and stays well within
    2e-2 (the earlier bf16 rounding gave 0.040 here); above it (40) the exact path, whose scores
    are scaled in fp32, shows only the rounding of P."""
    q, k, v, num, idx, block, scale = two_key_case(dtype, target, rounding)
    ref = O.sparse_attention(q, k, v, num, idx, block, scale=scale)
    qt, kt, vt = (dev(x, dtype, cuda) for x in (q, k, v))
    out = np_of(K.sparse_attention(qt, kt, vt, torch.from_numpy(num).to(cuda),
                                   torch.from_numpy(idx).to(cuda), block, scale=scale))
    err = float(np.abs(out - ref).max())
    print(f"{dtype} target {target} rounding {rounding}: max |err| {err:.3g}")
    assert np.isfinite(out).all()
    assert err < 1e-2, err


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("block", [64, 128, 256])
def test_unbounded_rows_take_the_exact_path(cuda, dtype, block):
    """Query blocks whose |q| max|k| bound exceeds the fp32-safe range (every other block scaled
    by 40: scaled logits up to ~500) run the exact running-max softmax, the others the bounded
    path: every row matches the float64 oracle, and the scaled rows stay finite."""
    rng = np.random.default_rng(12)
    n, G = 1024, 2
    q = rng.standard_normal((1, 2 * G, n, 64)).astype(np.float32)
    for i in range(0, n // block, 2):
        q[:, :, i * block:(i + 1) * block] *= 40.0
    q = WL.round_to(q, dtype)
    k = WL.round_to(rng.standard_normal((1, 2, n, 64)).astype(np.float32), dtype)
    v = WL.round_to(rng.standard_normal((1, 2, n, 64)).astype(np.float32), dtype)
    qt, kt, vt = (dev(x, dtype, cuda) for x in (q, k, v))
    kv_num, kv_idx, _ = K.block_route_budget(qt, kt, block, top_c=4, local=1, beta=2.0,
                                             compact=True)
    out = K.sparse_attention(qt, kt, vt, kv_num, kv_idx, block)
    ref = O.sparse_attention(q, k, v, kv_num.cpu().numpy(), kv_idx.cpu().numpy(), block)
    assert torch.isfinite(out).all()
    assert np.abs(np_of(out) - ref).max() < TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("jump", [40.0, 90.0, 220.0])
@pytest.mark.parametrize("exact", [False, True])
def test_exact_path_score_jump_after_the_first_sub_tile(cuda, dtype, jump, exact):
    """The exact path (bf16) takes the running max on a wave's first sub-tile only and offsets the
    later sub-tiles' P = 2^(s - m) by it; a row whose sum then reaches 2^100 sends its workgroup
    through its list again with the running max of every sub-tile (fp16 inputs always take the
    running max of every sub-tile). Query block i (i >= 2) repeats one direction q_i with |q_i| =
    40 and walks [0, i - 1, i]: block 0 holds short random keys (its scores, the first sub-tile's
    max, a few log2 units), block i - 1 starts with a needle along q_i whose score lies `jump`
    log2 units above them, value e_(i mod 64). jump 40 / 90: the offset pass keeps every sum
    finite; 220: it overflows and the second walk runs. Both the exact launch of unbounded rows
    (exact=False: |q| max|k| is far over the bounded path's limit) and exact=True. Every row within
    2e-2 of the float64 oracle."""
    rng = np.random.default_rng(31)
    n, block, d, scale = 1024, 128, 64, 0.125
    c = scale * math.log2(math.e)
    nb = n // block
    qn = 40.0
    q = np.zeros((1, 1, n, d), np.float32)
    k = (0.05 * rng.standard_normal((1, 1, n, d))).astype(np.float32)
    v = (0.1 * rng.standard_normal((1, 1, n, d))).astype(np.float32)
    kv_num = np.full((1, 1, nb), 3, np.int32)
    kv_idx = np.zeros((1, 1, nb, 3), np.int32)
    kv_num[0, 0, 0], kv_num[0, 0, 1] = 1, 2
    kv_idx[0, 0, 0, 0] = 0
    kv_idx[0, 0, 1, :2] = [0, 1]
    for i in range(nb):
        x = rng.standard_normal(d)
        qh = x / np.linalg.norm(x)
        q[0, 0, i * block:(i + 1) * block] = qh * qn
        if i >= 2:
            p0 = (i - 1) * block
            k[0, 0, p0] = qh * (jump / (c * qn))  # score c * |q| * |k| = jump log2 units
            v[0, 0, p0] = 0.0
            v[0, 0, p0, i % d] = 1.0
            kv_idx[0, 0, i] = [0, i - 1, i]
    q, k, v = (WL.round_to(x, dtype) for x in (q, k, v))
    # block 0's scores: the first sub-tile's row maxima lie far below the needle
    s0 = c * (q[0, 0, 2 * block:].astype(np.float64) @ k[0, 0, :block].astype(np.float64).T)
    assert s0.max() < 10.0, s0.max()
    ref = O.sparse_attention(q, k, v, kv_num, kv_idx, block, scale=scale)
    qt, kt, vt = (dev(x, dtype, cuda) for x in (q, k, v))
    out = K.sparse_attention(qt, kt, vt, torch.from_numpy(kv_num).to(cuda),
                             torch.from_numpy(kv_idx).to(cuda), block, scale=scale, exact=exact)
    o = np_of(out)
    err = float(np.abs(o - ref).max())
    print(f"{dtype} jump {jump} exact={exact}: max |err| {err:.3g}")
    assert np.isfinite(o).all()
    assert err < TOL[dtype], err
    # the needle dominates its rows
    i = nb - 1
    assert abs(o[0, 0, i * block + 5, i % d] - ref[0, 0, i * block + 5, i % d]) < TOL[dtype]


# admission bounds of the bounded-row path (log2 units of scale * q.k): attn.hip fast_bound<DT>
FAST_BOUND = {torch.float16: 32.0, torch.bfloat16: 32.0}


@pytest.mark.parametrize("dtype,target,aligned", [
    (torch.float16, 14.0, True), (torch.float16, 22.0, True), (torch.float16, 31.0, True),
    (torch.float16, 33.0, True), (torch.float16, 250.0, True), (torch.float16, 31.0, False),
    (torch.float16, 250.0, False), (torch.bfloat16, 14.0, True), (torch.bfloat16, 31.0, True),
    (torch.bfloat16, 33.0, True), (torch.bfloat16, 60.0, True)])
def test_rows_near_the_fast_path_bound(cuda, dtype, target, aligned):
    """Every row's |q| is set so that the key-norm bound scale*log2e*|q|*max|k| equals `target`:
    just under the admission bound (32) the rows take the bounded path (q*scale*log2e rounded to
    fp16 must stay within tolerance; fp16: P = 2^(S - m0), m0 the largest score of the row's
    first sub-tile, overflows when a later score exceeds m0 + 16, and the query block is then
    redone exactly), just over it the exact path. aligned: keys lean on the queries' direction so
    that scores reach the bound (largest scores near `target`, a peaked softmax); not aligned:
    random keys, scores far below the bound, so at fp16 31 the scores of later sub-tiles can
    exceed m0 + 16 (overflow and redo). The output must be finite and within 2e-2 of the float64
    oracle either way."""
    rng = np.random.default_rng(21)
    n, block, scale = 1024, 128, 0.125
    q = rng.standard_normal((1, 2, n, 64)).astype(np.float32)
    k = rng.standard_normal((1, 1, n, 64)).astype(np.float32)
    v = rng.standard_normal((1, 1, n, 64)).astype(np.float32)
    # a shared direction u: keys lean on it so that some scores approach the Cauchy-Schwarz bound
    u = rng.standard_normal(64).astype(np.float32)
    u /= np.linalg.norm(u)
    if aligned:
        q += 2.0 * u
        k += 1.5 * rng.standard_normal((1, 1, n, 1)).astype(np.float32) * u
    k = WL.round_to(k, dtype)
    kmax = float(np.sqrt((k.astype(np.float64) ** 2).sum(-1)).max())
    qn = np.sqrt((q.astype(np.float64) ** 2).sum(-1, keepdims=True))
    q = q / qn * (target / (scale * math.log2(math.e) * kmax))
    q, v = WL.round_to(q, dtype), WL.round_to(v, dtype)
    bound = scale * math.log2(math.e) * float(np.sqrt((q.astype(np.float64) ** 2).sum(-1)).max()) * kmax
    assert (bound < FAST_BOUND[dtype]) == (target < FAST_BOUND[dtype]), bound
    qt, kt, vt = (dev(x, dtype, cuda) for x in (q, k, v))
    kv_num, kv_idx, _ = K.block_route_budget(qt, kt, block, top_c=3, local=1, beta=2.0,
                                             compact=True)
    out = K.sparse_attention(qt, kt, vt, kv_num, kv_idx, block, scale=scale)
    ref = O.sparse_attention(q, k, v, kv_num.cpu().numpy(), kv_idx.cpu().numpy(), block,
                             scale=scale)
    assert torch.isfinite(out).all()
    assert np.abs(np_of(out) - ref).max() < TOL[dtype]


@pytest.mark.parametrize("block", [64, 128, 256])
def test_fp16_bounded_rows_overflow_redone_exactly(cuda, block):
    """fp16 bounded rows take P = 2^(S - m0) with m0 the largest score of the row's first
    sub-tile. Here every query leans on one direction u and a needle key along u sits in key
    block 5, while the other keys are random: the rows' first sub-tiles (earlier blocks) score
    far below the needle (about |q| |k|/8 against |q| |k|), so the needle's P overflows fp16 and
    the query blocks that attend block 5 must be redone by the exact launch. Every row within
    2e-2 of the float64 oracle, the output finite."""
    rng = np.random.default_rng(41)
    n, scale = max(1024, 8 * block), 0.125
    u = rng.standard_normal(64).astype(np.float32)
    u /= np.linalg.norm(u)
    q = (0.1 * rng.standard_normal((1, 2, n, 64)) + u).astype(np.float32)
    k = rng.standard_normal((1, 1, n, 64)).astype(np.float32)
    v = rng.standard_normal((1, 1, n, 64)).astype(np.float32)
    k[0, 0, 5 * block + 3] = 20.0 * u  # the needle
    c2 = scale * math.log2(math.e)
    # |q| max|k| scale log2e ~ 31: inside the admission bound (32)
    q *= 31.0 / (c2 * np.linalg.norm(q, axis=-1, keepdims=True) * 20.0)
    q, k, v = (WL.round_to(x, torch.float16) for x in (q, k, v))
    qt, kt, vt = (dev(x, torch.float16, cuda) for x in (q, k, v))
    kv_num, kv_idx, _ = K.block_route_budget(qt, kt, block, top_c=3, local=1, beta=2.0,
                                             compact=True)
    idx, num = kv_idx.cpu().numpy(), kv_num.cpu().numpy()
    # rows whose needle score exceeds their first sub-tile's largest score by more than 16
    q64, k64 = q.astype(np.float64), k.astype(np.float64)
    over = 0
    for h in range(2):
        for i in range(6, n // block):
            sel = idx[0, h, i, :num[0, h, i]]
            if 5 not in sel:
                continue
            k0 = sel[0] * block
            rows = np.arange(i * block, (i + 1) * block)
            m0 = (c2 * q64[0, h, rows] @ k64[0, 0, k0:k0 + 64].T).max(-1)
            over += int((c2 * q64[0, h, rows] @ k64[0, 0, 5 * block + 3] - m0 > 16.5).sum())
    assert over > 0  # the overflow path is exercised
    out = K.sparse_attention(qt, kt, vt, kv_num, kv_idx, block, scale=scale)
    ref = O.sparse_attention(q, k, v, kv_num.cpu().numpy(), idx, block, scale=scale)
    assert torch.isfinite(out).all()
    assert np.abs(np_of(out) - ref).max() < TOL[torch.float16]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("block", [64, 128, 256])
def test_full_budget_matches_dense_sdpa(cuda, dtype, block):
    """Every causal block selected -> dense causal attention (test_ssa_kernel.py:8-18)."""
    torch.manual_seed(0)
    n = 4 * 256
    q = torch.randn(1, 2, n, 64, device=cuda, dtype=dtype)
    k, v = torch.randn_like(q), torch.randn_like(q)
    out = K.ssa_flex(q, k, v, block=block, top_c=n // block, local=n // block)
    ref = F.scaled_dot_product_attention(q.float(), k.float(), v.float(), is_causal=True)
    assert (out.float() - ref).abs().max().item() < TOL[dtype]


@pytest.mark.parametrize("dtype,block,n", [(torch.float16, 256, 1000), (torch.bfloat16, 128, 300),
                                           (torch.bfloat16, 64, 333), (torch.float32, 64, 200)])
def test_ragged_length_gqa_matches_oracle(cuda, dtype, block, n):
    """n not a block multiple (pad keys masked, pad queries not written), GQA 3:1, lse."""
    rng = np.random.default_rng(12)
    q = WL.round_to(rng.standard_normal((1, 6, n, 64)).astype(np.float32), dtype)
    k = WL.round_to(rng.standard_normal((1, 2, n, 64)).astype(np.float32), dtype)
    v = WL.round_to(rng.standard_normal((1, 2, n, 64)).astype(np.float32), dtype)
    qt, kt, vt = (dev(x, dtype, cuda) for x in (q, k, v))
    kv_num, kv_idx = K.route(K.block_summary(qt, block, "qmean"),
                             *K.block_summary(kt, block, "pop", n_real=n)[:2], None, "budget", 2,
                             0.0, 1, 1.0)
    out, lse = K.sparse_attention(qt, kt, vt, kv_num, kv_idx, block, scale=0.2, return_lse=True)
    ref = O.sparse_attention(q, k, v, kv_num.cpu().numpy(), kv_idx.cpu().numpy(), block, scale=0.2)
    assert np.abs(np_of(out) - ref).max() < TOL[dtype]
    assert torch.isfinite(lse).all()


def test_hf_layout_output_without_copies(cuda):
    """(b, n, h, d) buffers viewed as (b, h, n, d): strided q/k/v and output."""
    torch.manual_seed(1)
    b, n, hq, hkv = 1, 512, 4, 2
    qb = torch.randn(b, n, hq, 64, device=cuda, dtype=torch.bfloat16)
    kb = torch.randn(b, n, hkv, 64, device=cuda, dtype=torch.bfloat16)
    vb = torch.randn(b, n, hkv, 64, device=cuda, dtype=torch.bfloat16)
    q, k, v = qb.transpose(1, 2), kb.transpose(1, 2), vb.transpose(1, 2)
    kv_num, kv_idx, _ = K.block_route_budget(q, k, 128, top_c=2, local=0, compact=True)
    outb = torch.empty(b, n, hq, 64, device=cuda, dtype=torch.bfloat16)
    K.sparse_attention(q, k, v, kv_num, kv_idx, 128, out=outb.transpose(1, 2))
    ref = K.sparse_attention(q.contiguous(), k.contiguous(), v.contiguous(), kv_num, kv_idx, 128)
    assert torch.equal(outb.transpose(1, 2), ref)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_no_future_leak(cuda, dtype):
    """Perturbing keys/values after position `cut` leaves outputs <= cut unchanged: bit for bit
    in the query blocks that end before `cut`'s block (no key they read changed, and their
    softmax path is chosen from the keys they read), and within the reference's own bar
    (test_flex_swap.py:78-91, atol 2e-2) in `cut`'s block, whose rows share one workgroup with
    later rows and may take the other softmax path when the perturbed keys raise its bound. The
    perturbation (+5, |k| ~ 40) pushes the bound past both dtypes' fast-path limits."""
    torch.manual_seed(0)
    n, cut, block = 1024, 300, 128
    q = torch.randn(1, 2, n, 64, device=cuda, dtype=dtype)
    k, v = torch.randn_like(q), torch.randn_like(q)
    o1 = K.ssa_flex(q, k, v, block=block, top_c=2, local=1)
    k2, v2 = k.clone(), v.clone()
    k2[:, :, cut + 1:] += 5
    v2[:, :, cut + 1:] += 5
    o2 = K.ssa_flex(q, k2, v2, block=block, top_c=2, local=1)
    whole = cut // block * block
    assert torch.equal(o1[:, :, :whole], o2[:, :, :whole])
    assert (o1[:, :, :cut + 1].float() - o2[:, :, :cut + 1].float()).abs().max().item() < 2e-2


def test_c5_full_length_properties_and_sampled_rows(cuda):
    """C5 at its full 12.6M-token length (49152 blocks of 256, fp16): list structure for every
    row, summaries of sampled blocks, the selections of sampled rows recomputed by the oracle from
    the device summaries, and the attention of sampled query blocks against the oracle on the
    gathered blocks (only the diagonal block is masked, so the gathered blocks keep the
    geometry)."""
    d5 = WL.make_c5_device(cuda)
    c5 = d5["cfg"]
    q, k, v = d5["q"], d5["k"], d5["v"]
    blk, nb, T = c5.block, c5.nb, c5.top_c
    qbar = K.block_summary(q, blk, "qmean")
    mu, var, _ = K.block_summary(k, blk, "pop")
    kv_num, kv_idx = K.route(qbar, mu, var, None, "budget", T, 0.0, c5.local, 0.5 * c5.beta)
    out = K.sparse_attention(q, k, v, kv_num, kv_idx, blk)
    torch.cuda.synchronize()
    assert torch.isfinite(out).all()

    num = kv_num[0, 0].long()
    idx = kv_idx[0, 0].long()
    i = torch.arange(nb, device=cuda)
    # rows i <= top_c keep every earlier block; later rows keep top_c of them plus i-1 and i
    assert torch.equal(num[:T + 1], i[:T + 1] + 1)
    assert bool(((num[T + 1:] >= T + 1) & (num[T + 1:] <= T + 2)).all())
    j = torch.arange(idx.shape[1], device=cuda)
    valid = j[None, :] < num[:, None]
    assert bool((idx.gather(1, (num - 1)[:, None])[:, 0] == i).all())
    assert bool((idx.gather(1, (num - 2).clamp(min=0)[:, None])[1:, 0] == i[1:] - 1).all())
    inc = (idx[:, 1:] > idx[:, :-1]) | ~valid[:, 1:]
    assert bool(inc.all())
    assert bool(((idx >= 0) & ((idx <= i[:, None]) | ~valid)).all())

    rows = sorted({0, 1, 63, 64, 65, 66, 1000, 9999, 30000, nb - 2, nb - 1}
                  | set(np.random.default_rng(5).integers(0, nb, 16).tolist()))
    # summaries of the sampled blocks against the oracle (within 1 ulp)
    for c in rows[:6] + rows[-3:]:
        sl = slice(c * blk, (c + 1) * blk)
        kb, qb = np_of(k[:, :, sl]), np_of(q[:, :, sl])
        m_o, v_o, _ = O.block_stats(kb, blk, "pop")
        assert ulp_diff(np_of(mu[:, :, c:c + 1]), m_o).max() <= 1
        assert ulp_diff(np_of(var[:, :, c:c + 1]), v_o).max() <= 1
        assert ulp_diff(np_of(qbar[:, :, c:c + 1]), O.qmean(qb, blk)).max() <= 1

    mu_h, var_h, qbar_h = np_of(mu), np_of(var), np_of(qbar)
    num_h, idx_h = kv_num.cpu().numpy(), kv_idx.cpu().numpy()
    for r in rows:
        sc = O.scores(qbar_h[:, :, r:r + 1], mu_h, var_h, 0.5 * c5.beta)
        sel = O.select_row(O.score_keys(sc)[0, 0, 0], r, "budget", T, 0.0, c5.local)
        assert idx_h[0, 0, r, :num_h[0, 0, r]].tolist() == sel, r

    for r in (0, 65, nb // 2, nb - 1):
        ids = idx_h[0, 0, r, :num_h[0, 0, r]].tolist()
        gk = np.concatenate([np_of(k[:, :, c * blk:(c + 1) * blk]) for c in ids], axis=2)
        gv = np.concatenate([np_of(v[:, :, c * blk:(c + 1) * blk]) for c in ids], axis=2)
        gq = np.zeros_like(gk)
        gq[:, :, -blk:] = np_of(q[:, :, r * blk:(r + 1) * blk])
        m = len(ids)
        gnum = np.array([[[m] * m]], dtype=np.int32)
        gidx = np.broadcast_to(np.arange(m, dtype=np.int32), (1, 1, m, m)).copy()
        ref = O.sparse_attention(gq, gk, gv, gnum, gidx, blk, qblocks=[m - 1])
        err = np.abs(np_of(out[:, :, r * blk:(r + 1) * blk]) - ref[:, :, -blk:]).max()
        assert err < TOL[c5.dtype], (r, err)


# ---- a10-a12 decode ----------------------------------------------------------------------------

def test_decode_attend_matches_oracle_and_prefill_row(cuda):
    rng = np.random.default_rng(13)
    n, block = 12 * 128, 128
    q = WL.round_to(rng.standard_normal((1, 1, n, 64)).astype(np.float32), torch.bfloat16)
    k = WL.round_to(rng.standard_normal((1, 1, n, 64)).astype(np.float32), torch.bfloat16)
    v = WL.round_to(rng.standard_normal((1, 1, n, 64)).astype(np.float32), torch.bfloat16)
    qt, kt, vt = (dev(x, torch.bfloat16, cuda) for x in (q, k, v))
    kv_num, kv_idx, _ = K.block_route_budget(qt, kt, block, top_c=4, local=1, compact=True)
    pre = K.sparse_attention(qt, kt, vt, kv_num, kv_idx, block)
    blocks = kv_idx[0, 0, 11, :int(kv_num[0, 0, 11])].tolist() + [3, 3]   # duplicates attend once
    row = D.decode_attend(qt[0, 0, n - 1], kt[0, 0], vt[0, 0], blocks, n - 1, block)
    ref = O.decode_attend(q[0, 0, n - 1], k[0, 0], v[0, 0], blocks, n - 1, block)
    assert np.abs(np_of(row) - ref).max() < 2e-2
    assert (row.float() - pre[0, 0, n - 1].float()).abs().max().item() < 2e-2
    # a block past pos contributes nothing; pos inside a block clips it
    row2 = D.decode_attend(qt[0, 0, 700], kt[0, 0], vt[0, 0], [0, 5, 9], 700, block)
    ref2 = O.decode_attend(q[0, 0, 700], k[0, 0], v[0, 0], [0, 5, 9], 700, block)
    assert np.abs(np_of(row2) - ref2).max() < 2e-2


def test_dense_decode_baselines_agree_with_full_selection(cuda):
    """The dense decode baselines (ssa/ivf_decode.py:65-85; the reference pins dense_decode
    against dense_decode_naive) equal each other, the oracle's softmax row and decode_attend over
    every block of the prefix."""
    rng = np.random.default_rng(17)
    n, block, pos = 9 * 128, 128, 9 * 128 - 40
    q, k, v = (WL.round_to(rng.standard_normal(s).astype(np.float32), torch.bfloat16)
               for s in ((64,), (n, 64), (n, 64)))
    qt, kt, vt = (dev(x, torch.bfloat16, cuda) for x in (q, k, v))
    a = D.dense_decode(qt, kt, vt, pos)
    b = D.dense_decode_naive(qt, kt, vt, pos)
    c = D.decode_attend(qt, kt, vt, list(range(9)), pos, block)
    ref = O.decode_attend(q, k, v, list(range(9)), pos, block)
    for got in (a, b, c):
        assert got.dtype == torch.bfloat16 and np.abs(np_of(got) - ref).max() < 2e-2


def test_decoder_folded_append_equals_separate_append(cuda):
    """RoutedDecoder.step with contiguous query rows folds the cache append into the attend
    launch (no prep launch; the router reads the bf16 q); with strided rows it appends and
    converts in a launch of its own. Over steps that complete a block and steps that do not,
    both give identical selections, outputs and caches."""
    rng = np.random.default_rng(29)
    hq, hkv, d, block, n0, steps = 4, 2, 64, 64, 64 * 5 + 60, 10
    k, v = (WL.round_to(rng.standard_normal((1, hkv, n0 + steps, d)).astype(np.float32),
                        torch.bfloat16) for _ in range(2))
    q = WL.round_to(rng.standard_normal((steps, 1, hq, d)).astype(np.float32), torch.bfloat16)
    kt, vt = dev(k, torch.bfloat16, cuda), dev(v, torch.bfloat16, cuda)
    qc = dev(q, torch.bfloat16, cuda)                        # step t: qc[t] contiguous
    qs = qc.permute(1, 2, 0, 3).contiguous().permute(2, 0, 1, 3)  # same values, strided rows
    assert qc[0].is_contiguous() and not qs[0].is_contiguous()
    decs = [D.RoutedDecoder(1, hq, hkv, d, n0 + steps, block=block, top_c=3, local=1,
                            dtype=torch.bfloat16, device=cuda) for _ in range(2)]
    for dec in decs:
        dec.prefill(kt[:, :, :n0], vt[:, :, :n0])
    for t in range(steps):  # positions 380..389: the step at 383 completes block 5
        outs = [dec.step(qq[t], kt[:, :, n0 + t], vt[:, :, n0 + t])
                for dec, qq in zip(decs, (qc, qs))]
        assert torch.equal(outs[0], outs[1]), t
        assert torch.equal(decs[0].kv_num, decs[1].kv_num) and torch.equal(decs[0].kv_idx, decs[1].kv_idx)
    for a, b in ((decs[0].kcache, decs[1].kcache), (decs[0].vcache, decs[1].vcache)):
        assert torch.equal(a[:, :, :n0 + steps], b[:, :, :n0 + steps])
    assert torch.equal(decs[0].kcache[:, :, :n0 + steps], kt)


def test_routed_decoder_step_under_torch_compile(cuda):
    """RoutedDecoder.step compiled (dynamo + aot_eager: the ssa_amd::decode_step op's in-place
    writes to the caches, summaries and selection are functionalised and written back): 8 steps
    crossing a block completion give outputs, selections, caches and summaries bit-identical to
    an eager decoder's, and the advancing position (self.pos, read inside the compiled step)
    costs at most one recompilation: after the first change dynamo makes it a symbolic int."""
    import torch._dynamo.testing as DT
    torch._dynamo.reset()
    Hq, Hkv, d, block, prefix, steps = 14, 2, 64, 128, 1020, 8
    rng = np.random.default_rng(17)
    total = prefix + steps
    k = WL.round_to(rng.standard_normal((1, Hkv, total, d)).astype(np.float32), torch.bfloat16)
    v = WL.round_to(rng.standard_normal((1, Hkv, total, d)).astype(np.float32), torch.bfloat16)
    q = WL.round_to(rng.standard_normal((steps, 1, Hq, d)).astype(np.float32), torch.bfloat16)
    kd, vd, qd = (dev(x, torch.bfloat16, cuda) for x in (k, v, q))
    eager, comp = (D.RoutedDecoder(1, Hq, Hkv, d, total, block=block, top_c=8, local=1,
                                   dtype=torch.bfloat16, device=cuda) for _ in range(2))
    for dec in (eager, comp):
        dec.prefill(kd[:, :, :prefix], vd[:, :, :prefix])
    cnt = DT.CompileCounterWithBackend("aot_eager")
    step_c = torch.compile(lambda q_, k_, v_: comp.step(q_, k_, v_), backend=cnt)
    for t in range(steps):
        pos = prefix + t
        k_new, v_new = kd[:, :, pos].contiguous(), vd[:, :, pos].contiguous()
        out_e = eager.step(qd[t], k_new, v_new)
        out_c = step_c(qd[t], k_new, v_new)
        assert torch.equal(out_e, out_c), t
        assert torch.equal(eager.kv_num, comp.kv_num) and torch.equal(eager.kv_idx, comp.kv_idx), t
    print(f"compiled decode steps: {cnt.frame_count} compilation(s) over {steps} steps", flush=True)
    assert comp.pos == eager.pos == total
    assert torch.equal(eager.kcache, comp.kcache) and torch.equal(eager.vcache, comp.vcache)
    assert torch.equal(eager.mu, comp.mu) and torch.equal(eager.var, comp.var)
    assert 1 <= cnt.frame_count <= 2, cnt.frame_count


def test_routed_decoder_matches_reference_router_and_oracle(cuda):
    """RoutedDecoder on a C4-shaped cache: the selection at each fixture position equals the
    reference _selection_mask (float32) and the oracle; the output matches the oracle row."""
    g = GU.load("c4_query")
    p = WL.make("C4", n=65536 + 128)
    cfg = p["cfg"]
    positions = g["positions"].tolist()
    dec = D.RoutedDecoder(1, cfg.Hq, cfg.Hkv, cfg.d, 65536 + 128, block=cfg.block,
                          top_c=cfg.top_c, local=cfg.local, beta=cfg.beta, dtype=cfg.dtype,
                          device=cuda)
    start = positions[0]
    dec.prefill(dev(p["k"][:, :, :start], cfg.dtype, cuda), dev(p["v"][:, :, :start], cfg.dtype, cuda))
    G_ = cfg.Hq // cfg.Hkv
    for pos in range(start, positions[-1] + 1):
        q = dev(p["q"][:, :, pos], cfg.dtype, cuda)
        out = dec.step(q, dev(p["k"][:, :, pos], cfg.dtype, cuda), dev(p["v"][:, :, pos], cfg.dtype, cuda))
        if pos not in positions:
            continue
        a = positions.index(pos)
        kn, ki = dec.kv_num.cpu().numpy(), dec.kv_idx.cpu().numpy()
        onum, oidx = O.route_query(p["q"][:, :, pos:pos + 1], p["k"], cfg.block, pos,
                                   top_c=cfg.top_c, local=cfg.local, beta=cfg.beta, kv_len=pos + 1)
        n_, n_eq, _, bad = GU.compare_selections(kn, ki, onum[:, :, 0], oidx[:, :, 0])
        assert n_eq == n_, (pos, bad)
        mu, var, _ = O.block_stats(p["k"][:, :, :pos + 1], cfg.block, "pop")
        r64, mag = O.exact_scores64(p["q"][:, :, pos:pos + 1], mu, var, 0.5 * cfg.beta)
        n_, n_eq, n_cert, bad = GU.compare_selections(kn, ki, g["kv_num"][a][None],
                                                      g["kv_idx"][a][None], r64[:, :, 0], mag[:, :, 0])
        assert not bad, (pos, bad)
        for h in (0, 7, 13):
            ids = ki[0, h, :kn[0, h]]
            ref = O.decode_attend(p["q"][0, h, pos], p["k"][0, h // G_], p["v"][0, h // G_], ids,
                                  pos, cfg.block)
            assert np.abs(np_of(out[0, h]) - ref).max() < 2e-2


def test_routed_decoder_full_1m_cache_matches_reference(cuda):
    """RoutedDecoder over the bench's C4 decode workload at its full size: a 1,048,576-token
    cache, then decode steps t = 0..127 appending one token each (8193 complete blocks by the
    last). At the fixture steps (t = 127 completes a block) the selection equals the reference's
    float32 _selection_mask (or differs on a certified near-tie) and the oracle's bit for bit,
    and every head's output is within 2e-2 of the oracle's decode_attend."""
    g = GU.load("c4_query_1m")
    p = WL.make_decode(steps=GU.C4_1M_STEPS)
    cfg, n = p["cfg"], p["n_cache"]
    assert GU.sha(p["q"], p["k"]) == str(g["inputs_sha256"])
    steps = g["steps"].tolist()
    print(f"c4 1M decode: cache {n}, steps up to {steps[-1]}", flush=True)
    dec = D.RoutedDecoder(1, cfg.Hq, cfg.Hkv, cfg.d, n + GU.C4_1M_STEPS, block=cfg.block,
                          top_c=cfg.top_c, local=cfg.local, beta=cfg.beta, dtype=cfg.dtype,
                          device=cuda)
    kd, vd = dev(p["k"], cfg.dtype, cuda), dev(p["v"], cfg.dtype, cuda)
    qd = dev(p["q"], cfg.dtype, cuda)
    dec.prefill(kd[:, :, :n], vd[:, :, :n])
    G_ = cfg.Hq // cfg.Hkv
    # summaries of every block complete at the checked steps (all lie in the first n + 128)
    assert steps[-1] < 128
    mu, var, _ = O.block_stats(p["k"][:, :, :n + 128], cfg.block, "pop")
    for t in range(steps[-1] + 1):
        out = dec.step(qd[:, :, t].contiguous(), kd[:, :, n + t].contiguous(),
                       vd[:, :, n + t].contiguous())
        if t not in steps:
            continue
        a, pos = steps.index(t), n + t
        kn, ki = dec.kv_num.cpu().numpy(), dec.kv_idx.cpu().numpy()
        qrow = p["q"][:, :, t:t + 1]
        onum, oidx = O.route_query_summaries(qrow, mu, var, cfg.block, pos, top_c=cfg.top_c,
                                             local=cfg.local, beta=cfg.beta)
        n_, n_eq, _, bad = GU.compare_selections(kn, ki, onum[:, :, 0], oidx[:, :, 0])
        assert n_eq == n_, (t, bad)
        r64, mag = O.exact_scores64(qrow, mu, var, 0.5 * cfg.beta)
        n_, n_eq, n_cert, bad = GU.compare_selections(kn, ki, g["kv_num"][a][None],
                                                      g["kv_idx"][a][None], r64[:, :, 0],
                                                      mag[:, :, 0])
        print(f"step {t}: {n_eq}/{n_} heads identical to the reference, {n_cert} certified",
              flush=True)
        assert not bad, (t, bad)
        o = np_of(out)
        for h in range(cfg.Hq):
            ref = O.decode_attend(p["q"][0, h, t], p["k"][0, h // G_], p["v"][0, h // G_],
                                  ki[0, h, :kn[0, h]], pos, cfg.block)
            assert np.abs(o[0, h] - ref).max() < 2e-2, (t, h)


def test_c5_geometry_prefix_router_matches_reference(cuda):
    """The router at C5's geometry (fp16, block 256, top_c 64 + local 1, beta 2) over a
    2,097,152-token prefix (8192 query blocks x 8192 candidate blocks): bit-exact against the
    oracle and equal to the reference's float32 block_route_budget except on certified near-ties;
    sampled query blocks' attention within 2e-2 of the oracle."""
    g = GU.load("c5_prefix")
    p = WL.make_c5_prefix()
    cfg = p["cfg"]
    assert GU.sha(p["q"], p["k"]) == str(g["inputs_sha256"])
    q, k, v = (dev(p[x], cfg.dtype, cuda) for x in ("q", "k", "v"))
    kv_num, kv_idx, _ = K.block_route_budget(q, k, cfg.block, top_c=cfg.top_c, local=cfg.local,
                                             beta=cfg.beta, compact=True)
    kn, ki = kv_num.cpu().numpy(), kv_idx.cpu().numpy()
    onum, oidx = O.route_budget(p["q"], p["k"], cfg.block, top_c=cfg.top_c, local=cfg.local,
                                beta=cfg.beta)
    n, n_eq, _, bad = GU.compare_selections(kn, ki, onum, oidx)
    assert n_eq == n, bad[:3]
    qb = O.qmean(p["q"], cfg.block)
    mu, var, _ = O.block_stats(p["k"], cfg.block, "pop")
    r64, mag = O.exact_scores64(qb, mu, var, 0.5 * cfg.beta)
    n, n_eq, n_cert, bad = GU.compare_selections(kn, ki, g["kv_num"], g["kv_idx"], r64, mag)
    print(f"c5 prefix: {n} rows, {n_eq} identical to the reference, {n_cert} certified")
    assert not bad, bad[:3]
    out = K.sparse_attention(q, k, v, kv_num, kv_idx, cfg.block)
    blocks = [0, 1, 64, 4095, 8191]
    ref = O.sparse_attention(p["q"], p["k"], p["v"], kn, ki, cfg.block, qblocks=blocks)
    o = np_of(out)
    for i in blocks:
        sl = slice(i * cfg.block, (i + 1) * cfg.block)
        assert np.abs(o[0, 0, sl] - ref[0, 0, sl]).max() < 2e-2, i


# ---- a9 real-model boundary --------------------------------------------------------------------

def _mod(groups=1, scaling=0.125, layer_idx=0):
    from types import SimpleNamespace
    return SimpleNamespace(num_key_value_groups=groups, is_sliding=False, scaling=scaling,
                           layer_idx=layer_idx)


@pytest.mark.parametrize("impl", ["flex", "analytic"])
def test_gemma_full_budget_matches_sdpa(cuda, impl):
    """test_flex_swap.py:82-93 / test_gemma_ssa.py:45-52 restated, GQA 2:1, n=300 ragged."""
    torch.manual_seed(0)
    for n in (512, 300):
        q = torch.randn(1, 4, n, 64, device=cuda, dtype=torch.float16)
        k = torch.randn(1, 2, n, 64, device=cuda, dtype=torch.float16)
        v = torch.randn_like(k)
        G.CFG = G.SSAConfig(block=128, budget_frac=1.0, impl=impl)
        out, _ = G.ssa_attention_forward(_mod(groups=2), q, k, v, scaling=1 / 8)
        ref = F.scaled_dot_product_attention(q.float(), G.repeat_kv(k, 2).float(),
                                             G.repeat_kv(v, 2).float(), is_causal=True,
                                             scale=1 / 8).transpose(1, 2)
        assert out.shape == (1, n, 4, 64)
        assert (out.float() - ref).abs().max().item() < 2e-2


def test_gemma_analytic_matches_reference_fixture(cuda):
    g = GU.load("analytic_gqa")
    rng = np.random.default_rng(11)
    q = rng.standard_normal((1, 4, 300, 64))
    k = rng.standard_normal((1, 2, 300, 64))
    v = rng.standard_normal((1, 2, 300, 64))
    G.CFG = G.SSAConfig(block=64, budget_frac=0.5, local_w=1, beta=2.0, impl="analytic")
    qt, kt, vt = (torch.from_numpy(x).float().to(cuda) for x in (q, k, v))
    out, _ = G.ssa_attention_forward(_mod(groups=2), qt, kt, vt, scaling=0.125)
    assert np.abs(np_of(out) - g["out"]).max() < 1e-5
    inc, _ = G.ssa_attention_forward(_mod(groups=2), qt[:, :, -1:], kt, vt, scaling=0.125)
    assert np.abs(np_of(inc) - g["out_last"]).max() < 1e-5


def test_gemma_analytic_edgeworth_matches_reference_fixture(cuda):
    """ssa_attention_forward(impl='analytic', edgeworth=True): the per-query router adds
    beta^2/6 <q^3, m3> (ssa/gemma_ssa.py:101-102 via :237) on skewed keys, where the term changes
    the selection of 418 of the 1200 (head, query) rows; prefill rows and a q_len = 1 row match
    the reference's float64 output within 1e-5."""
    g = GU.load("analytic_gqa_edgeworth")
    q, k, v = GU.analytic_inputs(12, skew=0.7)
    assert GU.sha(q, k, v) == str(g["inputs_sha256"])
    G.CFG = G.SSAConfig(block=64, budget_frac=0.5, local_w=1, beta=2.0, impl="analytic",
                        edgeworth=True)
    qt, kt, vt = (torch.from_numpy(x).float().to(cuda) for x in (q, k, v))
    out, _ = G.ssa_attention_forward(_mod(groups=2), qt, kt, vt, scaling=0.125)
    assert np.abs(np_of(out) - g["out"]).max() < 1e-5
    inc, _ = G.ssa_attention_forward(_mod(groups=2), qt[:, :, -1:], kt, vt, scaling=0.125)
    assert np.abs(np_of(inc) - g["out_last"]).max() < 1e-5
    # without the term the output differs from the fixture (the fixture pins the term)
    G.CFG = G.SSAConfig(block=64, budget_frac=0.5, local_w=1, beta=2.0, impl="analytic")
    plain, _ = G.ssa_attention_forward(_mod(groups=2), qt, kt, vt, scaling=0.125)
    assert np.abs(np_of(plain) - g["out"]).max() > 1e-2


@pytest.mark.parametrize("d,dtype", [(128, torch.bfloat16), (256, torch.float16),
                                     (96, torch.bfloat16), (128, torch.float32)])
def test_prefill_other_head_dims_match_oracle(cuda, d, dtype):
    """impl='flex' prefill at head dims other than 64 (the reference's flex branch serves any
    head size, ssa/gemma_ssa.py:169-180): ragged n, GQA 2:1, against the oracle."""
    rng = np.random.default_rng(33)
    n, block = 700, 128
    q = WL.round_to(rng.standard_normal((1, 4, n, d)).astype(np.float32), dtype)
    k = WL.round_to(rng.standard_normal((1, 2, n, d)).astype(np.float32), dtype)
    v = WL.round_to(rng.standard_normal((1, 2, n, d)).astype(np.float32), dtype)
    G.CFG = G.SSAConfig(block=block, budget_frac=0.5, local_w=1, beta=2.0, impl="flex")
    qt, kt, vt = (dev(x, dtype, cuda) for x in (q, k, v))
    out, _ = G.ssa_attention_forward(_mod(groups=2), qt, kt, vt, scaling=d ** -0.5)
    kv_num, kv_idx = O.route_budget(q, k, block, budget_frac=0.5, local=1, beta=2.0, n_real=n)
    ref = O.sparse_attention(q, k, v, kv_num, kv_idx, block, scale=d ** -0.5)
    assert np.abs(np_of(out).transpose(0, 2, 1, 3) - ref).max() < TOL[dtype]


def _lse64(q, k, kv_num, kv_idx, block, scale):
    """Natural-log sum-exp of every query row over its selected keys j <= t, j < n (float64)."""
    B, Hq, n, d = q.shape
    G_ = Hq // k.shape[1]
    out = np.empty((B, Hq, n))
    for b, h, i in np.ndindex(B, Hq, kv_num.shape[2]):
        t0, t1 = i * block, min(n, (i + 1) * block)
        keys = np.concatenate([np.arange(c * block, min(n, (c + 1) * block))
                               for c in kv_idx[b, h, i, :kv_num[b, h, i]]])
        s = scale * (q[b, h, t0:t1].astype(np.float64) @ k[b, h // G_, keys].astype(np.float64).T)
        s = np.where(keys[None, :] <= np.arange(t0, t1)[:, None], s, -np.inf)
        m = s.max(axis=1, keepdims=True)
        out[b, h, t0:t1] = (m + np.log(np.exp(s - m).sum(axis=1, keepdims=True)))[:, 0]
    return out


@pytest.mark.parametrize("d,dtype,block", [(128, torch.bfloat16, 128), (128, torch.float16, 64),
                                           (128, torch.bfloat16, 256), (256, torch.bfloat16, 256),
                                           (256, torch.float16, 128), (256, torch.bfloat16, 64),
                                           (512, torch.bfloat16, 256), (512, torch.float16, 128),
                                           (512, torch.bfloat16, 64)])
def test_tiled_prefill_wide_head_dims_match_oracle(cuda, d, dtype, block):
    """The tiled MFMA prefill kernels at head dims 128 and 256 (4 waves x 32 query rows per
    128-row query tile, 2 waves for block 64; 64-key sub-tiles, 32-key at head dim 256; exact
    running-max softmax) and 512 (sparse_attn_wide_kernel, which serves calls this small: 4 waves
    split the head dim over one 32-row query group, 32-key sub-tiles): ragged n, GQA 3:1, the oracle router's lists (budget
    0.4 + local 1), every query row against the oracle within 2e-2, lse within 2^-8 of the
    float64 log-sum-exp (the row sum adds each P after rounding it to the 16-bit input type, a
    relative error of at most 2^-9 per term, so |d lse| <= 2^-9 plus fp32 accumulation), and a
    caller-supplied V^T (transpose_v) giving the identical output."""
    rng = np.random.default_rng(35 + d + block)
    n, hq, hkv = 1500, 6, 2
    q, k, v = (WL.round_to(rng.standard_normal((1, h_, n, d)).astype(np.float32), dtype)
               for h_ in (hq, hkv, hkv))
    kv_num, kv_idx = O.route_budget(q, k, block, budget_frac=0.4, local=1, beta=2.0, n_real=n)
    qt, kt, vt_ = (dev(x, dtype, cuda) for x in (q, k, v))
    num_t = torch.from_numpy(kv_num).to(cuda)
    idx_t = torch.from_numpy(kv_idx).to(cuda)
    scale = d ** -0.5
    out, lse = K.sparse_attention(qt, kt, vt_, num_t, idx_t, block, return_lse=True)
    ref = O.sparse_attention(q, k, v, kv_num, kv_idx, block, scale=scale)
    assert np.abs(np_of(out) - ref).max() < TOL[dtype]
    assert np.abs(np_of(lse) - _lse64(q, k, kv_num, kv_idx, block, scale)).max() < 2.0 ** -8
    vtr = K.transpose_v(vt_, block)
    out2 = K.sparse_attention(qt, kt, vt_, num_t, idx_t, block, vt=vtr)
    assert torch.equal(out, out2)


@pytest.mark.parametrize("dtype,d,block,exact", [(torch.bfloat16, 64, 128, False),
                                                (torch.float16, 64, 256, False),
                                                (torch.bfloat16, 64, 128, True),
                                                (torch.bfloat16, 128, 128, False),
                                                (torch.float16, 512, 64, False)])
def test_prepared_attention_matches_unprepared(cuda, dtype, d, block, exact):
    """prepare_attention on a second stream (V^T and the key-norm pass, overlapping nothing here
    but ordered by an event) + sparse_attention(prepared=...) gives the same output, bit for bit,
    as the call that prepares for itself; a PreparedKV serves one call and must match k, v and
    the block."""
    rng = np.random.default_rng(d + block)
    n, hq, hkv = 1100, 4, 2
    q, k, v = (WL.round_to(rng.standard_normal((1, h_, n, d)).astype(np.float32), dtype)
               for h_ in (hq, hkv, hkv))
    kv_num, kv_idx = O.route_budget(q, k, block, budget_frac=0.4, local=1, beta=2.0, n_real=n)
    qt, kt, vt_ = (dev(x, dtype, cuda) for x in (q, k, v))
    num_t, idx_t = torch.from_numpy(kv_num).to(cuda), torch.from_numpy(kv_idx).to(cuda)
    ref = K.sparse_attention(qt, kt, vt_, num_t, idx_t, block, exact=exact)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        prep = K.prepare_attention(kt, vt_, block)
        done = torch.cuda.Event()
        done.record(side)
    torch.cuda.current_stream().wait_event(done)
    out = K.sparse_attention(qt, kt, vt_, num_t, idx_t, block, exact=exact, prepared=prep)
    assert torch.equal(out, ref)
    with pytest.raises(ValueError):
        K.sparse_attention(qt, kt, vt_, num_t, idx_t, block, prepared=prep)
    if d == 64 and block == 128:
        with pytest.raises(ValueError):
            K.sparse_attention(qt, kt, vt_, num_t, idx_t, 256, prepared=K.prepare_attention(
                kt, vt_, block))


def test_d512_tiled_prefill_gemma_shape_beats_per_row_path(cuda):
    """The reference's Gemma attention shape (16 query heads, 8 key heads, head dim 512, block
    256, budget 0.25 + local 1, bf16) at n = 8192: the tiled d = 512 kernel agrees with the
    per-row kernel (ssa_decode_attend over every query row) within 2e-2 and is at least 10x
    faster than it (median of 5 timed calls each, after a warm-up call)."""
    torch.manual_seed(512)
    n, hq, hkv, d, block = 8192, 16, 8, 512, 256
    print(f"d512 gemma shape n={n}", flush=True)
    q = torch.randn(1, hq, n, d, device=cuda, dtype=torch.bfloat16)
    k = torch.randn(1, hkv, n, d, device=cuda, dtype=torch.bfloat16)
    v = torch.randn(1, hkv, n, d, device=cuda, dtype=torch.bfloat16)
    kv_num, kv_idx, _ = K.block_route_budget(q, k, block, budget_frac=0.25, local=1,
                                             compact=True)
    scale = d ** -0.5

    def timed(fn):
        fn()
        ts = []
        for _ in range(5):
            a, b_ = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            fn()
            b_.record()
            torch.cuda.synchronize()
            ts.append(a.elapsed_time(b_))
        return float(np.median(ts))

    out_t = torch.empty_like(q)
    out_r = torch.empty_like(q)
    t_tiled = timed(lambda: K.sparse_attention(q, k, v, kv_num, kv_idx, block, out=out_t))
    t_rows = timed(lambda: K._sparse_attention_rows(q, k, v, kv_num, kv_idx, block, scale,
                                                    out_r))
    print(f"tiled {t_tiled:.3f} ms, per-row {t_rows:.3f} ms, x{t_rows / t_tiled:.1f}", flush=True)
    assert (out_t.float() - out_r.float()).abs().max().item() < 2e-2
    assert t_rows >= 10.0 * t_tiled, (t_tiled, t_rows)


@pytest.mark.parametrize("case,top_c,nblk", [("all_equal", 64, 3000), ("top_ties", 64, 3000),
                                             ("random", 64, 3000), ("random", 4, 12000)])
def test_fused_decode_step_ties_match_oracle(cuda, case, top_c, nblk):
    """The fused two-launch decode step on exact score ties (identical key blocks have identical
    summaries, so identical scores for any query): the lowest block indices win, as in the
    oracle. all_equal: every complete block holds one pattern -- every chunk keeps K equal keys,
    the 16-entry prefix pass hands over to the whole lists, and the row's survivors exceed what
    one wave holds (the workgroup-wide search runs); top_ties: 100 identical copies of a block
    aligned with the key head's queries among random blocks (ties straddle the K-th key);
    random: no ties. 3000 candidate blocks of 16 keys (47 route chunks of 64), top_c 64 + local
    1; and 12000 blocks at top_c 4 (94 chunks of 128: the merge must load every chunk list
    although K is small). Selections bit-exact against the oracle; outputs within 2e-2 of the
    oracle's decode_attend."""
    rng = np.random.default_rng(43)
    hq, hkv, d, block = 4, 2, 64, 16
    G_ = hq // hkv
    n0 = nblk * block + 5  # the step's position: nblk complete blocks before it
    k = rng.standard_normal((1, hkv, n0 + 1, d)).astype(np.float32)
    v = rng.standard_normal((1, hkv, n0 + 1, d)).astype(np.float32)
    q = rng.standard_normal((1, hq, d)).astype(np.float32)
    if case == "all_equal":
        pat = rng.standard_normal((hkv, block, d)).astype(np.float32)
        k[0, :, :nblk * block] = np.tile(pat, (1, nblk, 1))
    elif case == "top_ties":
        for kvh in range(hkv):
            qd_ = q[0, kvh * G_:(kvh + 1) * G_].sum(0)
            pat = 2.5 * qd_ / np.linalg.norm(qd_) + 0.3 * rng.standard_normal((block, d))
            for c in rng.choice(nblk, 100, replace=False):
                k[0, kvh, c * block:(c + 1) * block] = pat
    k, v, q = (WL.round_to(x, torch.bfloat16) for x in (k, v, q))
    dec = D.RoutedDecoder(1, hq, hkv, d, n0 + 1, block=block, top_c=top_c, local=1,
                          dtype=torch.bfloat16, device=cuda)
    dec.prefill(dev(k[:, :, :n0], torch.bfloat16, cuda), dev(v[:, :, :n0], torch.bfloat16, cuda))
    out = dec.step(dev(q, torch.bfloat16, cuda), dev(k[:, :, n0], torch.bfloat16, cuda),
                   dev(v[:, :, n0], torch.bfloat16, cuda))
    kn, ki = dec.kv_num.cpu().numpy(), dec.kv_idx.cpu().numpy()
    onum, oidx = O.route_query(q[:, :, None], k, block, n0, top_c=top_c, local=1, kv_len=n0 + 1)
    for h in range(hq):
        sel = ki[0, h, :kn[0, h]].tolist()
        assert sel == oidx[0, h, 0, :onum[0, h, 0]].tolist(), (case, h)
        ref = O.decode_attend(q[0, h], k[0, h // G_], v[0, h // G_], sel, n0, block)
        assert np.abs(np_of(out[0, h]) - ref).max() < 2e-2, (case, h)


def test_attention_and_decoder_reject_mismatched_arguments(cuda):
    """A V^T of another length or dtype, and decode inputs of the wrong dtype or shape, raise
    instead of being read as the cache's layout."""
    q = torch.randn(1, 2, 512, 64, device=cuda, dtype=torch.bfloat16)
    k, v = torch.randn_like(q), torch.randn_like(q)
    kv_num, kv_idx, _ = K.block_route_budget(q, k, 128, top_c=2, local=1, compact=True)
    with pytest.raises(ValueError):
        K.sparse_attention(q, k, v, kv_num, kv_idx, 128, vt=K.transpose_v(v[:, :, :384], 128))
    with pytest.raises(ValueError):
        K.sparse_attention(q, k, v, kv_num, kv_idx, 128, vt=K.transpose_v(v.half(), 128))
    out = K.sparse_attention(q, k, v, kv_num, kv_idx, 128, vt=K.transpose_v(v, 128))
    assert torch.equal(out, K.sparse_attention(q, k, v, kv_num, kv_idx, 128))
    dec = D.RoutedDecoder(1, 2, 1, 64, 512, block=128, top_c=2, dtype=torch.bfloat16, device=cuda)
    qd = torch.randn(1, 2, 64, device=cuda, dtype=torch.bfloat16)
    kn = torch.randn(1, 1, 64, device=cuda, dtype=torch.bfloat16)
    with pytest.raises(TypeError):
        dec.step(qd.float(), kn, kn)
    with pytest.raises(ValueError):
        dec.step(qd[:, :1], kn, kn)
    with pytest.raises(ValueError):
        dec.step(torch.randn(1, 2, 128, device=cuda, dtype=torch.bfloat16)[..., ::2], kn, kn)
    assert dec.pos == 0
    dec.step(qd, kn, kn)
    assert dec.pos == 1


def test_gemma_decode_equals_prefill_last_row(cuda):
    """test_gemma_ssa.py:86-98 restated on the HIP per-query path."""
    torch.manual_seed(2)
    q = torch.randn(1, 4, 640, 64, device=cuda, dtype=torch.float32)
    k = torch.randn(1, 2, 640, 64, device=cuda, dtype=torch.float32)
    v = torch.randn_like(k)
    for frac in (0.5, 0.25):
        G.CFG = G.SSAConfig(block=64, budget_frac=frac, impl="analytic")
        full, _ = G.ssa_attention_forward(_mod(groups=2), q, k, v, scaling=1.0)
        inc, _ = G.ssa_attention_forward(_mod(groups=2), q[:, :, -1:], k, v, scaling=1.0)
        assert (inc[:, 0] - full[:, -1]).abs().max().item() < 1e-5


@pytest.mark.parametrize("edgeworth", [False, True])
def test_gemma_decode_resident_summaries(cuda, monkeypatch, edgeworth):
    """Decode steps through ssa_attention_forward keep the key-block summaries resident and
    summarise only the block a step completes (ssa/ivf_decode.py:133-135 grows its index the same
    way): over 150 steps crossing two block boundaries every output equals, bit for bit, the same
    call with the summaries recomputed from the whole cache; a prefill, a shorter cache and a
    non-consecutive position each start over."""
    torch.manual_seed(5)
    n0, steps, block = 1000, 150, 128
    q = torch.randn(1, 4, n0 + steps, 64, device=cuda, dtype=torch.bfloat16)
    k = torch.randn(1, 2, n0 + steps, 64, device=cuda, dtype=torch.bfloat16)
    v = torch.randn_like(k)
    G.CFG = G.SSAConfig(block=block, budget_frac=0.3, impl="hip", edgeworth=edgeworth)
    G.reset_decode_state()
    lens = []
    real = G.block_summary

    def recording(x, *a, **kw):
        lens.append(x.shape[2])
        return real(x, *a, **kw)
    mod = _mod(groups=2, layer_idx=3)
    for t in range(n0, n0 + steps):
        args = (q[:, :, t:t + 1], k[:, :, :t + 1], v[:, :, :t + 1])
        monkeypatch.setattr(G, "block_summary", recording)
        inc, _ = G.ssa_attention_forward(mod, *args, scaling=0.125,
                                         cache_position=torch.tensor([t], device=cuda))
        monkeypatch.setattr(G, "block_summary", real)
        saved = dict(G._DECODE)
        G.reset_decode_state()
        ref, _ = G.ssa_attention_forward(mod, *args, scaling=0.125)
        G._DECODE.clear()
        G._DECODE.update(saved)
        assert torch.equal(inc, ref), t
    # the first step summarised the prefix's complete blocks, later ones only completed blocks
    assert lens[0] == (n0 + 1) // block * block and all(x == block for x in lens[1:]), lens
    assert len(lens) == 1 + (n0 + steps) // block - (n0 + 1) // block
    st = G._DECODE[("layer", 3)]
    assert st["kv_len"] == n0 + steps and st["nc"] == (n0 + steps) // block
    # a shorter cache (a new sequence) and a position gap each start over
    G.ssa_attention_forward(mod, q[:, :, 499:500], k[:, :, :500], v[:, :, :500], scaling=0.125)
    assert G._DECODE[("layer", 3)]["kv_len"] == 500
    G.ssa_attention_forward(mod, q[:, :, 600:601], k[:, :, :601], v[:, :, :601], scaling=0.125)
    assert G._DECODE[("layer", 3)]["kv_len"] == 601 and G._DECODE[("layer", 3)]["nc"] == 4
    # a prefill drops the layer's decode summaries
    G.CFG = G.SSAConfig(block=block, budget_frac=0.3, impl="hip")
    G.ssa_attention_forward(mod, q[:, :, :512], k[:, :, :512], v[:, :, :512], scaling=0.125)
    assert ("layer", 3) not in G._DECODE
    G.reset_decode_state()


def test_gemma_flex_no_future_leak_and_sharing(cuda):
    """ssa/tests/test_flex_swap.py:78-90 restated (outputs up to `cut` within 2e-2 when later
    keys/values change), plus bit-equality for the query blocks wholly before cut's block: the
    rows of cut's own block may take the other softmax path when the later keys of that block
    change its key-norm bound (outputs equal to rounding). Then cross-layer sharing: the donor's
    selection object is reused by the consumer layer."""
    torch.manual_seed(0)
    n, cut = 512, 256
    q = torch.randn(1, 2, n, 64, device=cuda, dtype=torch.float16)
    k = torch.randn(1, 2, n, 64, device=cuda, dtype=torch.float16)
    v = torch.randn_like(k)
    G.CFG = G.SSAConfig(block=128, budget_frac=0.5, impl="flex")
    o1, _ = G.ssa_attention_forward(_mod(), q, k.clone(), v.clone(), scaling=1 / 8)
    k2, v2 = k.clone(), v.clone()
    k2[:, :, cut + 1:] += 5.0 * torch.randn_like(k2[:, :, cut + 1:])
    v2[:, :, cut + 1:] += 5.0 * torch.randn_like(v2[:, :, cut + 1:])
    o2, _ = G.ssa_attention_forward(_mod(), q, k2, v2, scaling=1 / 8)
    whole = cut // 128 * 128
    assert torch.equal(o1[:, :whole], o2[:, :whole])
    assert (o1[:, :cut + 1].float() - o2[:, :cut + 1].float()).abs().max().item() < 2e-2
    # donor layer 0 stashes its selection; consumer layer 1 reuses the same object
    G.CFG = G.SSAConfig(block=128, budget_frac=0.25, impl="flex", share_route_from=0)
    G._SHARE["sig"] = None
    G._SHARE["bm"] = None
    G.ssa_attention_forward(_mod(layer_idx=0), q, k, v, scaling=1 / 8)
    bm0 = G._SHARE["bm"]
    assert bm0 is not None
    G.ssa_attention_forward(_mod(layer_idx=1), q, k, v, scaling=1 / 8)
    assert G._SHARE["bm"] is bm0


def test_gemma_full_budget_shared_equals_dense(cuda):
    """test_share_route.py:61-74 restated: full budget with cross-layer sharing still reproduces
    dense causal attention on the consumer layer; a forward of another shape is not served the
    stashed selection (the signature check), and layers below the donor route on their own."""
    torch.manual_seed(0)
    n, d = 384, 64
    q = torch.randn(1, 1, n, d, device=cuda, dtype=torch.float16)
    k = torch.randn(1, 1, n, d, device=cuda, dtype=torch.float16)
    v = torch.randn_like(k)
    G.CFG = G.SSAConfig(block=128, budget_frac=1.0, impl="flex", share_route_from=0)
    G._SHARE["sig"] = None
    G._SHARE["bm"] = None
    G.ssa_attention_forward(_mod(groups=1, layer_idx=0), q, k, v, scaling=1.0 / d ** 0.5)
    out, _ = G.ssa_attention_forward(_mod(groups=1, layer_idx=1), q, k, v, scaling=1.0 / d ** 0.5)
    ref = F.scaled_dot_product_attention(q, k, v, is_causal=True).transpose(1, 2)
    assert (out.float() - ref.float()).abs().max().item() < 2e-2
    # budget 0.25: a consumer of another length routes itself (matches an unshared forward)
    G.CFG = G.SSAConfig(block=128, budget_frac=0.25, impl="flex", share_route_from=0)
    G.ssa_attention_forward(_mod(groups=1, layer_idx=0), q, k, v, scaling=1.0 / d ** 0.5)
    q2, k2, v2 = q[:, :, :256], k[:, :, :256], v[:, :, :256]
    shared, _ = G.ssa_attention_forward(_mod(groups=1, layer_idx=1), q2, k2, v2,
                                        scaling=1.0 / d ** 0.5)
    G.CFG = G.SSAConfig(block=128, budget_frac=0.25, impl="flex")
    own, _ = G.ssa_attention_forward(_mod(groups=1, layer_idx=1), q2, k2, v2,
                                     scaling=1.0 / d ** 0.5)
    assert torch.equal(shared, own)


def test_gemma_decode_ignores_sharing(cuda):
    """test_share_route.py:77-84 restated: with sharing configured, a q_len = 1 step takes the
    per-query path and equals the per-query prefill's last row (sharing is prefill-only)."""
    torch.manual_seed(4)
    q = torch.randn(1, 4, 160 * 4, 64, device=cuda, dtype=torch.float32)
    k = torch.randn(1, 2, 160 * 4, 64, device=cuda, dtype=torch.float32)
    v = torch.randn_like(k)
    G.CFG = G.SSAConfig(block=32, budget_frac=0.5, impl="analytic", share_route_from=0)
    G._SHARE["sig"] = None
    G._SHARE["bm"] = None
    full, _ = G.ssa_attention_forward(_mod(groups=2, layer_idx=2), q, k, v, scaling=1.0)
    inc, _ = G.ssa_attention_forward(_mod(groups=2, layer_idx=2), q[:, :, -1:], k, v, scaling=1.0)
    assert (inc[:, 0] - full[:, -1]).abs().max().item() < 1e-5
    assert G._SHARE["bm"] is None  # nothing stashed outside the prefill kernel path


def _dense_ref(q, k, v, scaling):
    G_ = q.shape[1] // k.shape[1]
    kr = k.repeat_interleave(G_, dim=1).double()
    vr = v.repeat_interleave(G_, dim=1).double()
    s = (q.double() @ kr.transpose(-1, -2)) * scaling
    n = q.shape[2]
    s = s.masked_fill(torch.ones(n, n, dtype=torch.bool, device=q.device).triu(1), float("-inf"))
    return (torch.softmax(s, -1) @ vr).transpose(1, 2)


def test_gemma_needle_known_answer_d512(cuda):
    """test_gemma_ssa.py:100-121 restated on the HIP per-query path at the Gemma head size
    (d = 512): with top_c = 1 and no local window, the probe query at the last position routes to
    the block holding a key 12x aligned with it, and its output is that key's value."""
    torch.manual_seed(0)
    n, d = 128, 512
    q = torch.randn(1, 1, n, d, device=cuda, dtype=torch.float32)
    k = torch.randn(1, 1, n, d, device=cuda, dtype=torch.float32)
    v = torch.randn(1, 1, n, d, device=cuda, dtype=torch.float32)
    u = F.normalize(torch.randn(d, device=cuda), dim=0)
    q[0, 0, n - 1] = u
    k[0, 0, 40] = 12.0 * u
    v[0, 0, 40] = torch.arange(d, device=cuda, dtype=torch.float32) / d
    G.CFG = G.SSAConfig(block=32, top_c=1, local_w=0, beta=2.0)
    out, _ = G.ssa_attention_forward(_mod(groups=1), q, k, v, scaling=1.0)
    ref = _dense_ref(q, k, v, 1.0)
    assert (out[0, n - 1].double() - ref[0, n - 1]).abs().max().item() < 3e-3
    assert (out[0, n - 1] - v[0, 0, 40]).abs().max().item() < 3e-3


def test_gemma_d512_gqa_full_budget_and_budget_monotone(cuda):
    """test_gemma_ssa.py:45-84,156-168 restated at d = 512, GQA 2:1 on the per-query path: full
    budget (and top_c >= blocks) equals dense causal attention; the attended key count shrinks
    strictly with the budget."""
    torch.manual_seed(1)
    n, d = 160, 512
    q = torch.randn(1, 4, n, d, device=cuda, dtype=torch.float32)
    k = torch.randn(1, 2, n, d, device=cuda, dtype=torch.float32)
    v = torch.randn(1, 2, n, d, device=cuda, dtype=torch.float32)
    ref = _dense_ref(q, k, v, 1.0 / math.sqrt(d))
    for cfg in (G.SSAConfig(block=32, budget_frac=1.0), G.SSAConfig(block=32, top_c=99)):
        G.CFG = cfg
        out, _ = G.ssa_attention_forward(_mod(groups=2), q, k, v, scaling=1.0 / math.sqrt(d))
        assert (out.double() - ref).abs().max().item() < 1e-5
    counts = []
    mu, var, _ = K.block_summary(k, 32, "pop", n_real=n)
    for frac in (1.0, 0.5, 0.25, 0.1):
        kn, ki = K.route(q.float(), mu, var, None, "query", None, frac, 0, 1.0, query_pos=0,
                         block=32)
        sets = GU.row_sets(kn.cpu().numpy(), ki.cpu().numpy())
        # attended keys: keys <= row of the selected blocks
        tot = 0
        for r, blocks in enumerate(sets):
            i = r % n
            tot += sum(min(32, i + 1 - 32 * c) for c in blocks if 32 * c <= i)
        counts.append(tot)
    assert counts[0] > counts[1] > counts[2] > counts[3], counts


def test_gemma_selection_mask_matches_attention_and_budget(cuda):
    """G._selection_mask (ssa/gemma_ssa.py:85-137) on the HIP router: masked dense softmax with it
    equals the per-query attention path, its kept blocks equal the oracle's route, and the
    attended key count shrinks strictly with the budget (test_gemma_ssa.py:156-168)."""
    torch.manual_seed(5)
    n, d = 256, 64
    q = torch.randn(1, 2, n, d, device=cuda, dtype=torch.float32)
    k = torch.randn(1, 2, n, d, device=cuda, dtype=torch.float32)
    v = torch.randn(1, 2, n, d, device=cuda, dtype=torch.float32)
    G.CFG = G.SSAConfig(block=32, budget_frac=0.25, local_w=1)
    m = G._selection_mask(q, k, G.CFG)
    s = (q @ k.transpose(-1, -2)) * 0.125 + m
    ref = (torch.softmax(s, -1) @ v).transpose(1, 2)
    out, _ = G.ssa_attention_forward(_mod(groups=1), q, k, v, scaling=0.125)
    assert (out - ref).abs().max().item() < 1e-5
    onum, oidx = O.route_query(np_of(q), np_of(k), 32, 0, top_c=None, budget_frac=0.25, local=1,
                               beta=2.0)
    first = np_of(m)[..., ::32] == 0.0  # first key of each block kept <=> block selected
    for r in (40, 100, 255):
        want = set(oidx[0, 0, r, :onum[0, 0, r]].tolist())
        got = {c for c in range(n // 32) if first[0, 0, r, c] and 32 * c <= r}
        assert got == want, (r, got, want)
    counts = []
    for frac in (1.0, 0.5, 0.25, 0.1):
        G.CFG = G.SSAConfig(block=32, budget_frac=frac, local_w=0)
        counts.append(int((G._selection_mask(q[:, :1], k[:, :1], G.CFG) == 0.0).sum().item()))
    assert counts[0] > counts[1] > counts[2] > counts[3], counts
    mu, var, m3, nb = G._block_stats(k, 48)
    omu, ovar, om3 = O.block_stats(np_of(k), 48, "pop")
    assert nb == 6 and ulp_diff(np_of(mu), omu).max() <= 1 and ulp_diff(np_of(var), ovar).max() <= 1


def test_gemma_sliding_layer_falls_back(cuda):
    """test_gemma_ssa.py:146-153: a sliding layer defers to the installed fallback untouched."""
    G.CFG = G.SSAConfig(block=32, budget_frac=0.1, route_full_only=True)
    sentinel = object()
    saved = G._FALLBACK
    try:
        G._FALLBACK = lambda module, q, k, v, mask=None, scaling=None, dropout=0.0, **kw: (sentinel, None)
        from types import SimpleNamespace
        mod = SimpleNamespace(num_key_value_groups=1, is_sliding=True, scaling=1.0, layer_idx=0)
        q = torch.randn(1, 1, 64, 64, device=cuda)
        out, _ = G.ssa_attention_forward(mod, q, q, q, scaling=1.0)
        assert out is sentinel
    finally:
        G._FALLBACK = saved


def test_gemma_proj_path_identity_equals_centroid_routing(cuda, tmp_path):
    """A routing projection saved in the reference's RoutingProjection format is loaded at
    install time (weights_only) and used by the prefill router; identity projections give the
    centroid (beta = 0) selection exactly."""
    torch.manual_seed(3)
    q = torch.randn(1, 2, 1024, 64, device=cuda, dtype=torch.bfloat16)
    k = torch.randn(1, 2, 1024, 64, device=cuda, dtype=torch.bfloat16)
    v = torch.randn_like(k)
    path = tmp_path / "proj.pt"
    torch.save({"W_q": torch.eye(64), "W_k": torch.eye(64), "meta": {"d": 64}}, path)

    class _Model:  # install_ssa needs only .config
        config = type("C", (), {"_attn_implementation": "sdpa"})()

    G.install_ssa(_Model(), block=128, budget_frac=0.25, impl="flex", proj_path=str(path))
    assert G._PROJ is not None and G._PROJ.meta == {"d": 64}
    o_proj, _ = G.ssa_attention_forward(_mod(), q, k, v, scaling=1 / 8)
    G.install_ssa(_Model(), block=128, budget_frac=0.25, impl="flex", beta=0.0)
    assert G._PROJ is None
    o_cent, _ = G.ssa_attention_forward(_mod(), q, k, v, scaling=1 / 8)
    assert torch.equal(o_proj, o_cent)


def test_transformers_qwen2_full_budget_matches_sdpa(cuda):
    """install_ssa on a transformers Qwen2 model with the Qwen2.5-0.5B attention shape (896
    hidden, 14 query / 2 key heads, d 64; 2 layers, random weights: no checkpoint can be
    fetched here): at full budget the logits and loss reproduce the same weights on SDPA (the
    reference's smoke gate, loss within 5e-2); at budget 0.25 the routed model runs end to end."""
    from transformers import Qwen2Config, Qwen2ForCausalLM
    cfg = Qwen2Config(vocab_size=512, hidden_size=896, intermediate_size=1024,
                      num_hidden_layers=2, num_attention_heads=14, num_key_value_heads=2,
                      max_position_embeddings=4096, attn_implementation="sdpa")
    torch.manual_seed(0)
    model = Qwen2ForCausalLM(cfg).to(device=cuda, dtype=torch.bfloat16).eval()
    ids = torch.randint(0, 512, (1, 1024), device=cuda)
    with torch.no_grad():
        ref = model(ids, labels=ids)
        G.install_ssa(model, block=128, budget_frac=1.0, impl="hip")
        full = model(ids, labels=ids)
        G.install_ssa(model, block=128, budget_frac=0.25, impl="hip")
        sparse = model(ids, labels=ids)
    assert model.config._attn_implementation == "ssa"
    assert abs(full.loss.item() - ref.loss.item()) < 5e-2
    assert (full.logits.float() - ref.logits.float()).abs().max().item() < 0.25
    assert torch.isfinite(sparse.logits).all() and math.isfinite(sparse.loss.item())
    assert not torch.equal(sparse.logits, full.logits)  # the routed layers attended fewer keys


def _qwen2_tiny(cuda):
    from transformers import Qwen2Config, Qwen2ForCausalLM
    cfg = Qwen2Config(vocab_size=512, hidden_size=896, intermediate_size=1024,
                      num_hidden_layers=2, num_attention_heads=14, num_key_value_heads=2,
                      max_position_embeddings=4096, attn_implementation="sdpa")
    torch.manual_seed(0)
    return Qwen2ForCausalLM(cfg).to(device=cuda, dtype=torch.bfloat16).eval()


def test_torch_compile_qwen2_uses_the_custom_ops(cuda):
    """torch.compile of a transformers Qwen2 model (0.5B attention shape, 2 layers) with
    install_ssa(impl='hip'): the traced graph calls the ssa_amd:: ops (summaries, router,
    block-sparse attention) and its logits equal the uncompiled model's bit for bit (a backend
    that runs the captured graph eagerly: same kernels, same order)."""
    torch._dynamo.reset()
    model = _qwen2_tiny(cuda)
    G.install_ssa(model, block=128, budget_frac=0.25, impl="hip")
    ids = torch.randint(0, 512, (1, 1024), device=cuda)
    targets = []

    def recording_backend(gm, example_inputs):
        targets.extend(str(n.target) for n in gm.graph.nodes if n.op == "call_function")
        return gm.forward

    with torch.no_grad():
        ref = model(ids).logits
        out = torch.compile(model, backend=recording_backend)(ids).logits
    ops = {t for t in targets if "ssa_amd" in t}
    assert {"ssa_amd.block_qmean.default", "ssa_amd.block_stats.default",
            "ssa_amd.route.default", "ssa_amd.sparse_attention.default"} <= ops, ops
    assert torch.equal(out, ref)


def test_torch_compile_inductor_qwen2_matches_eager(cuda):
    """The default inductor backend around the opaque ssa_amd:: ops. Inductor fuses the rest of
    the model with its own bf16 rounding, which perturbs the query-block means enough to flip
    routing near-ties on some rows: the loss agrees closely and the logits on average (a routing
    flip moves a few rows by up to ~0.5)."""
    torch._dynamo.reset()
    model = _qwen2_tiny(cuda)
    G.install_ssa(model, block=128, budget_frac=0.25, impl="hip")
    ids = torch.randint(0, 512, (1, 1024), device=cuda)
    with torch.no_grad():
        ref = model(ids, labels=ids)
        out = torch.compile(model)(ids, labels=ids)
    assert abs(out.loss.item() - ref.loss.item()) < 2e-2
    assert (out.logits.float() - ref.logits.float()).abs().mean().item() < 0.05
