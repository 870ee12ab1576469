"""GPU kernels at the sizes where their tilings change or leave remainders, against the CPU oracle
(float64)."""
import re
from pathlib import Path

import numpy as np
import pytest
import torch

from oracle import ssa_oracle as O
from ssa_amd import ssa_kernel as K
from ssa_amd import workloads as WL

pytestmark = pytest.mark.gpu


def np_of(t):
    return t.detach().float().cpu().numpy()


def random_lists(rng, rows, nb, W):
    """Ascending block lists of 1 to min(W, i + 2) blocks (a later block may be among them)."""
    kv_num = np.zeros((1, rows, nb), np.int32)
    kv_idx = np.zeros((1, rows, nb, W), np.int32)
    for h in range(rows):
        for i in range(nb):
            m = int(rng.integers(1, min(W, i + 2, nb) + 1))
            ids = np.sort(rng.permutation(min(i + 2, nb))[:m])
            kv_num[0, h, i], kv_idx[0, h, i, :m] = m, ids
    return kv_num, kv_idx


# 16-row groups (fewer than 1024) and 32-row groups; a single row; a part of a unit; lists longer
# than the 64-entry register window
@pytest.mark.parametrize("hq,hkv,n,block,W", [(1, 1, 1, 64, 2), (2, 1, 79, 64, 3),
                                              (3, 1, 700, 128, 4), (1, 1, 4608, 64, 72),
                                              (8, 2, 2075, 64, 6), (6, 6, 3000, 384, 5)])
def test_fp32_attention_tiles_match_oracle(cuda, hq, hkv, n, block, W):
    """1e-5: the bar of every fp32 attention test (64-term fp32 dots of N(0,1) at scale 1/8)."""
    rng = np.random.default_rng(n)
    q, k, v = (rng.standard_normal((1, h, n, 64)).astype(np.float32) for h in (hq, hkv, hkv))
    nb = -(-n // block)
    kv_num, kv_idx = random_lists(rng, hq, nb, min(W, nb))
    out, lse = K.sparse_attention(*(torch.from_numpy(x).to(cuda) for x in (q, k, v)),
                                  torch.from_numpy(kv_num).to(cuda),
                                  torch.from_numpy(kv_idx).to(cuda), block, return_lse=True)
    ref = O.sparse_attention(q, k, v, kv_num, kv_idx, block)
    assert np.abs(np_of(out) - ref).max() < 1e-5
    h, i = hq - 1, nb - 1  # lse of the last row
    js = [j for c in kv_idx[0, h, i, :kv_num[0, h, i]] for j in range(c * block,
                                                                       min(n, (c + 1) * block))]
    s = k[0, h // (hq // hkv), js].astype(np.float64) @ q[0, h, n - 1].astype(np.float64) / 8
    assert abs(float(lse[0, h, n - 1]) - np.log(np.exp(s).sum())) < 1e-5


# head dim 512: fewer than 96 groups of 128 rows (32-row workgroups, also at block 64), 4-wave
# groups, 8-wave groups; lengths that end inside a wave's rows and inside a 32-key sub-tile
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,n,block,W", [(2, 1, 300, 64, 3), (16, 4, 797, 128, 4),
                                              (32, 32, 261, 64, 5), (24, 8, 1043, 256, 3),
                                              (48, 8, 400, 384, 2)])
def test_d512_attention_tiles_match_oracle(cuda, dtype, hq, hkv, n, block, W):
    """2e-2: the bar of every 16-bit attention test. The layout is the transformers one (heads
    inside rows), so no stride is the contiguous one."""
    rng = np.random.default_rng(n)
    x = [WL.round_to(rng.standard_normal((1, n, h, 512)).astype(np.float32), dtype)
         for h in (hq, hkv, hkv)]
    q, k, v = (a.transpose(0, 2, 1, 3) for a in x)
    nb = -(-n // block)
    kv_num, kv_idx = random_lists(rng, hq, nb, min(W, nb))
    qt, kt, vt = (WL.to_device(a, dtype, cuda).transpose(1, 2) for a in x)
    out, lse = K.sparse_attention(qt, kt, vt, torch.from_numpy(kv_num).to(cuda),
                                  torch.from_numpy(kv_idx).to(cuda), block, return_lse=True)
    heads = [0, hq // 2, hq - 1]
    ref = O.sparse_attention(q, k, v, kv_num, kv_idx, block, heads=heads)
    assert np.abs(np_of(out)[:, heads] - ref[:, heads]).max() < 2e-2
    none = ~np.isfinite(ref[0, 0]).all(-1) | (ref[0, 0] == 0).all(-1)
    assert (torch.isneginf(lse[0, 0]).cpu().numpy() == none).all()


# head dim 512 from 96 groups of 128 rows on, which reads V itself: block 64 (4-wave groups), 4- and
# 8-wave groups, also with a V^T or a prepared workspace, whose V^T such a call does not read
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,n,block,W", [(48, 8, 261, 64, 3), (16, 4, 850, 128, 3),
                                              (24, 8, 1043, 256, 3)])
def test_d512_attention_given_workspaces(cuda, dtype, hq, hkv, n, block, W):
    """2e-2: the bar of every 16-bit attention test; the given workspaces change no bit."""
    src = (Path(__file__).resolve().parents[1] / "ssa_amd/csrc/attn.hip").read_text()
    nb = -(-n // block)
    least = int(re.search(r"kWide16Min = (\d+)", src).group(1))
    assert nb * block // 64 * hq // 2 >= least, "the case no longer reaches the 128-row kernel"
    rng = np.random.default_rng(n)
    q, k, v = (WL.round_to(rng.standard_normal((1, h, n, 512)).astype(np.float32), dtype)
               for h in (hq, hkv, hkv))
    kv_num, kv_idx = random_lists(rng, hq, nb, min(W, nb))
    qt, kt, vt = (WL.to_device(a, dtype, cuda) for a in (q, k, v))
    num, idx = torch.from_numpy(kv_num).to(cuda), torch.from_numpy(kv_idx).to(cuda)
    out = K.sparse_attention(qt, kt, vt, num, idx, block)
    heads = [0, hq - 1]
    ref = O.sparse_attention(q, k, v, kv_num, kv_idx, block, heads=heads)
    assert np.abs(np_of(out)[:, heads] - ref[:, heads]).max() < 2e-2
    given = K.sparse_attention(qt, kt, vt, num, idx, block, vt=K.transpose_v(vt, block))
    assert torch.equal(given, out)
    given = K.sparse_attention(qt, kt, vt, num, idx, block,
                               prepared=K.prepare_attention(kt, vt, block))
    assert torch.equal(given, out)


# cascade route: query blocks and rows that fill no 64 x 128 score tile, and candidates in rising
# score order (every run of the streaming search passes the threshold it set, so the run is cut);
# scored ahead and row by row (no room for the scores)
@pytest.mark.parametrize("limit", [None, 0])
@pytest.mark.parametrize("rising", [False, True])
@pytest.mark.parametrize("d,blocks,nbq", [(64, 2700, 70), (96, 700, 1), (32, 130, 129)])
def test_cascade_route_scores_match_oracle(cuda, monkeypatch, d, blocks, nbq, rising, limit):
    from ssa_amd import cascade_router as C
    if limit is not None:
        monkeypatch.setattr(C, "SCORE_WORKSPACE_LIMIT", limit)
    rng = np.random.default_rng(d)
    n, past = blocks * 128, (blocks - nbq) * 128
    if rising:
        k = np.ones((n, d)) * np.repeat(np.arange(n // 32) + 1.0, 32)[:, None] / 1024
        q = np.ones((nbq * 128, d))
    else:
        k, q = rng.standard_normal((n, d)), rng.standard_normal((nbq * 128, d))
    k, q = (x.astype(np.float16) for x in (k, q))
    got, ref = C.CausalCascade(d, search_k=48), O.CascadeOracle(d, search_k=48)
    got.build_threshold = ref.build_threshold = 1 << 30  # every committed mean is scanned
    for a, b in ((0, past // 2), (past // 2, past), (past, n)):
        got.append(torch.from_numpy(k[a:b]).to(cuda))
        ref.append(k[a:b].astype(np.float32))
    kn, ki, cert, _ = got.route(torch.from_numpy(q).to(cuda), past, certify=True)
    rn, rl, rc, _ = ref.route(q.astype(np.float32), past, certify=True)
    assert (kn.cpu().numpy() == rn).all() and (cert.cpu().numpy() == rc).all()
    for i in range(nbq):
        assert ki[i, :rn[i]].tolist() == rl[i], i


# the same for query blocks at and before the staged means' first block (none, one or two are past)
@pytest.mark.parametrize("limit", [None, 0])
def test_cascade_route_before_the_staged_means(cuda, monkeypatch, limit):
    from ssa_amd import cascade_router as C
    if limit is not None:
        monkeypatch.setattr(C, "SCORE_WORKSPACE_LIMIT", limit)
    rng = np.random.default_rng(5)
    k = rng.standard_normal((24 * 128, 64)).astype(np.float16)
    q = rng.standard_normal((8 * 128, 64)).astype(np.float16)
    got, ref = C.CausalCascade(64, search_k=48), O.CascadeOracle(64, search_k=48)
    for a, b in ((0, 16), (16, 24)):
        got.append(torch.from_numpy(k[a * 128:b * 128]).to(cuda))
        ref.append(k[a * 128:b * 128].astype(np.float32))
    for first in (14, 16):  # (staged: blocks 16 .. 23)
        kn, ki, _, _ = got.route(torch.from_numpy(q).to(cuda), first * 128)
        rn, rl, _, _ = ref.route(q.astype(np.float32), first * 128)
        assert (kn.cpu().numpy() == rn).all()
        for i in range(8):
            assert ki[i, :rn[i]].tolist() == rl[i], (first, i)


# list building: one wave, one tile and several, with remainders; one list, a list per mean, the most
@pytest.mark.parametrize("nb,nlist", [(33, 1), (64, 64), (256, 17), (257, 257), (1000, 300),
                                      (2300, 2048)])
def test_ivf_lists_match_oracle(cuda, nb, nlist):
    from ssa_amd import ivf_kernel as I
    rng = np.random.default_rng(nb)
    mu = rng.standard_normal((2, nb, 32)).astype(np.float32)
    ix = I.build_ivf(torch.from_numpy(mu).to(cuda), nlist=nlist, niter=1)
    off, ids = ix.list_offsets.cpu().numpy(), ix.list_ids.cpu().numpy()
    for h in range(2):
        cent, lists = O.ivf_build(mu[h], nlist, 1)
        assert (ix.centroids[h].cpu().numpy() == cent).all()
        for c in range(nlist):
            assert ids[h, off[h, c]:off[h, c + 1]].tolist() == lists[c].tolist(), (h, c)


# list scoring (16-centroid tiles, 32 means a wave) and updates (runs of 64 members): every head dim
# the kernels are built for, remainders of each tile, lists of one member, of a run and of several
@pytest.mark.parametrize("nb,nlist,d", [(1100, 2, 64), (500, 33, 96), (97, 16, 128), (130, 5, 160),
                                        (1, 1, 192), (129, 128, 224), (700, 3, 256)])
def test_ivf_scores_and_updates_match_oracle(cuda, nb, nlist, d):
    from ssa_amd import ivf_kernel as I
    rng = np.random.default_rng(d)
    mu = rng.standard_normal((2, nb, d)).astype(np.float32)
    ix = I.build_ivf(torch.from_numpy(mu).to(cuda), nlist=nlist, niter=3)
    off, ids = ix.list_offsets.cpu().numpy(), ix.list_ids.cpu().numpy()
    for h in range(2):
        cent, lists = O.ivf_build(mu[h], nlist, 3)
        assert (ix.centroids[h].cpu().numpy() == cent).all()
        for c in range(nlist):
            assert ids[h, off[h, c]:off[h, c + 1]].tolist() == lists[c].tolist(), (h, c)


# masked attention: one block per key tile and several, a block of two tiles, a length that
# ends inside a wave's rows, more than the 64 tiles of a mask round (4100 tokens), grouped heads
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,n,block,top_c", [(2, 1, 200, 64, 2), (3, 3, 129, 128, 1),
                                                  (2, 2, 150, 24, 3), (4, 2, 65, 16, 2),
                                                  (1, 1, 4100, 64, 3)])
def test_masked_attention_tiles_match_oracle(cuda, dtype, hq, hkv, n, block, top_c):
    """The bars of the masked attention's tests: 2e-2 of the largest gradient, 1e-5 in fp32."""
    from ssa_amd import ssa_swap as S
    rng = np.random.default_rng(n)
    q, k, v, g = (WL.round_to(rng.standard_normal((1, h, n, 64)).astype(np.float32), dtype)
                  for h in (hq, hkv, hkv, hq))
    t = [WL.to_device(x, dtype, cuda).requires_grad_(True) for x in (q, k, v)]
    kn, ki = S.route_masked(t[0].detach(), t[1].detach(), block, top_c, 1)
    kn, ki = kn.cpu().numpy(), ki.cpu().numpy()
    lists = np.empty((1, hq, n), dtype=object)
    for at in np.ndindex(*lists.shape):
        lists[at] = ki[at][:kn[at]].tolist()
    out = S.ssa_masked(*t, block, top_c, 1)
    grads = torch.autograd.grad(out, t, WL.to_device(g, dtype, cuda))
    ref, _ = O.masked_forward(q, k, v, lists, block)
    tol = 1e-5 if dtype == torch.float32 else 2e-2
    assert np.abs(np_of(out) - ref).max() < tol
    for got, want in zip(grads, O.masked_grads(q, k, v, lists, g, block)):
        assert np.abs(np_of(got) - want).max() < tol * max(1.0, np.abs(want).max())


# routed decode step: head dim 128 over parts of a block of less, exactly and more than 32 keys, the
# new token first and last in its block; contexts of one chunk list, of one and of two a wave and
# of the most (more than 64 chunks: 4200 blocks), at head dim 64 too (test_gpu_decode_shapes.py:
# the lengths between)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("d,block,n,top_c", [(128, 16, 33, 2), (128, 64, 640, 4),
                                             (128, 512, 1800, 2), (128, 128, 131072, 8),
                                             (64, 128, 66000, 64), (128, 16, 67196, 64),
                                             (64, 16, 67196, 64)])
def test_decode_step_tiles_match_oracle(cuda, dtype, d, block, n, top_c):
    """Selections exact; outputs within the bars of the decode tests (2e-2, fp32 1e-5)."""
    from ssa_amd.ivf_decode import RoutedDecoder
    rng = np.random.default_rng(n + d)
    hq, hkv, steps = 4, 2, 3
    k, v = (WL.round_to(rng.standard_normal((1, hkv, n + steps, d)).astype(np.float32), dtype)
            for _ in range(2))
    q = WL.round_to(rng.standard_normal((steps, 1, hq, d)).astype(np.float32), dtype)
    kt, vt, qt = (WL.to_device(a, dtype, cuda) for a in (k, v, q))
    dec = RoutedDecoder(1, hq, hkv, d, n + steps, block=block, top_c=top_c, local=1, dtype=dtype,
                        device=cuda)
    dec.prefill(kt[:, :, :n], vt[:, :, :n])
    tol = 1e-5 if dtype == torch.float32 else 2e-2
    for t in range(steps):
        out = np_of(dec.step(qt[t], kt[:, :, n + t], vt[:, :, n + t]))
        on, oi = O.route_query(q[t][:, :, None], k, block, n + t, top_c=top_c, local=1,
                               kv_len=n + t + 1)
        kn, ki = dec.kv_num.cpu().numpy(), dec.kv_idx.cpu().numpy()
        for h in range(hq):
            sel = oi[0, h, 0, :on[0, h, 0]].tolist()
            assert ki[0, h, :kn[0, h]].tolist() == sel, (t, h)
            ref = O.decode_attend(q[t][0, h], k[0, h // 2], v[0, h // 2], sel, n + t, block)
            assert np.abs(out[0, h] - ref).max() < tol, (t, h)
