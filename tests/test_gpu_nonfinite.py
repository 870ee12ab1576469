"""GPU kernels on inputs with infinities: a value that takes no part in a row (a weight of zero, a
key or a row past the end) leaves no trace in it. Against the CPU oracle (float64)."""
import numpy as np
import pytest
import torch

from oracle import ssa_oracle as O
from ssa_amd import workloads as WL

pytestmark = pytest.mark.gpu
INF = float("inf")


def np_of(t):
    return t.detach().float().cpu().numpy()


def same(got, ref, tol):
    """Equal infinities, no NaN where the reference has none, finite values within tol."""
    f = np.isfinite(ref)
    assert (np.isfinite(got) == f).all()
    assert (got[~f] == ref[~f]).all()
    assert np.abs(got[f] - ref[f]).max() < tol


def decode_all_blocks(cuda, dtype, d, block, n, poison, steps=2):
    """Steps of a decoder that selects every block of an n-token cache, and the oracle's rows.
    poison(k, v): sets values of the n + steps tokens before they are used (CPU arrays)."""
    from ssa_amd.ivf_decode import RoutedDecoder
    rng = np.random.default_rng(n + d + block)
    hq, hkv = 4, 2
    k, v = (WL.round_to(rng.standard_normal((1, hkv, n + steps, d)).astype(np.float32), dtype)
            for _ in range(2))
    q = WL.round_to(rng.standard_normal((steps, 1, hq, d)).astype(np.float32), dtype)
    q[..., 0] = np.abs(q[..., 0]) + 0.5
    nb = -(-(n + steps) // block)
    dec = RoutedDecoder(1, hq, hkv, d, n + steps, block=block, top_c=nb, local=1, dtype=dtype,
                        device=cuda)
    kt, vt, qt = (WL.to_device(a, dtype, cuda) for a in (k, v, q))
    dec.prefill(kt[:, :, :n], vt[:, :, :n])  # (the routing summaries stay finite)
    poison(k, v)
    kt, vt = (WL.to_device(a, dtype, cuda) for a in (k, v))
    dec.kcache[:, :, :n], dec.vcache[:, :, :n] = kt[:, :, :n], vt[:, :, :n]
    for t in range(steps):
        out = np_of(dec.step(qt[t], kt[:, :, n + t], vt[:, :, n + t]))
        sel = list(range((n + t) // block + 1))
        for h in range(hq):
            assert dec.kv_idx[0, h, :int(dec.kv_num[0, h])].tolist() == sel
            ref = O.decode_attend(q[t][0, h], k[0, h // 2], v[0, h // 2], sel, n + t, block)
            yield out[0, h], ref


# the first 32 keys of a half block score -inf (block 128), a whole half does (block 64)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("block", [64, 128])
def test_decode_step_keys_of_minus_infinity(cuda, dtype, block):
    n = 3 * block + 5 * block // 8

    def poison(k, v):
        for half in (block, 3 * block):  # a half of a complete block, and of the own one
            k[:, :, half:half + 32, 0] = -INF
    for got, ref in decode_all_blocks(cuda, dtype, 128, block, n, poison):
        same(got, ref, 2e-2)


# the last key of a part whose length fills no 32-key load: whole halves of 8, 16 and 32 keys, and
# the whole block
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d,block", [(128, 16), (128, 32), (128, 64), (64, 32)])
def test_decode_step_value_of_infinity_last_in_its_part(cuda, dtype, d, block):
    n = 10 * block + block // 4

    def poison(k, v):
        v[:, :, block + block // 2 - 1, 7] = INF
        v[:, :, 2 * block - 1, 9] = -INF
    for got, ref in decode_all_blocks(cuda, dtype, d, block, n, poison):
        same(got, ref, 2e-2)


# an infinite value in the last row of a length that fills no tile: rows that attend it are infinite
@pytest.mark.parametrize("dtype,d,hq,hkv,n,block", [(torch.float32, 64, 2, 1, 700, 64),
                                                    (torch.float32, 64, 8, 2, 2075, 128),
                                                    (torch.bfloat16, 128, 2, 1, 300, 64),
                                                    (torch.float16, 512, 16, 4, 797, 128),
                                                    (torch.bfloat16, 512, 24, 8, 1043, 256),
                                                    (torch.bfloat16, 512, 48, 8, 261, 64)])
def test_prefill_value_of_infinity_in_the_last_row(cuda, dtype, d, hq, hkv, n, block):
    from ssa_amd import ssa_kernel as K
    rng = np.random.default_rng(n)
    q, k, v = (WL.round_to(rng.standard_normal((1, h, n, d)).astype(np.float32), dtype)
               for h in (hq, hkv, hkv))
    v[:, :, n - 1, 3], v[:, :, n - 1, 5] = INF, -INF
    nb = -(-n // block)
    num = np.minimum(np.arange(nb) + 1, 3)
    idx = np.clip(np.arange(nb)[:, None] - num[:, None] + 1 + np.arange(3), 0, nb - 1)
    num, idx = (np.broadcast_to(a.astype(np.int32), (1, hq, *a.shape)).copy() for a in (num, idx))
    out = np_of(K.sparse_attention(*(WL.to_device(a, dtype, cuda) for a in (q, k, v)),
                                   torch.from_numpy(num).to(cuda), torch.from_numpy(idx).to(cuda),
                                   block))
    finite = v.copy()
    finite[:, :, n - 1, 3] = finite[:, :, n - 1, 5] = 0.0
    ref = O.sparse_attention(q, k, finite, num, idx, block)
    ref[:, :, n - 1, 3], ref[:, :, n - 1, 5] = INF, -INF
    # (head dims without the infinity everywhere, all head dims in the last row; rows before it
    # share a tile with the infinity at weight 0)
    rest = [e for e in range(d) if e not in (3, 5)]
    tol = 1e-5 if dtype == torch.float32 else 2e-2
    same(out[..., rest], ref[..., rest], tol)
    same(out[:, :, n - 1], ref[:, :, n - 1], tol)


# the same through the masked attention, forward and backward: an infinite value (a gradient) in the
# last row makes the output (dV) infinite for the rows (keys) that meet it there
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,n,block", [(2, 1, 200, 64), (2, 2, 1000, 64), (4, 2, 150, 24)])
def test_masked_attention_infinity_in_the_last_row(cuda, dtype, hq, hkv, n, block):
    from ssa_amd import ssa_swap as S
    rng = np.random.default_rng(n)
    q, k, v, g = (WL.round_to(rng.standard_normal((1, h, n, 64)).astype(np.float32), dtype)
                  for h in (hq, hkv, hkv, hq))
    kn, ki = S.route_masked(*(WL.to_device(x, dtype, cuda) for x in (q, k)), block, 2, 1)
    kn, ki = kn.cpu().numpy(), ki.cpu().numpy()
    lists = np.empty((1, hq, n), dtype=object)
    for at in np.ndindex(*lists.shape):
        lists[at] = ki[at][:kn[at]].tolist()
    tol = 1e-5 if dtype == torch.float32 else 2e-2
    rest = [e for e in range(64) if e != 3]

    def run(v, g):
        t = [WL.to_device(x, dtype, cuda).requires_grad_(True) for x in (q, k, v)]
        out = S.ssa_masked(*t, block, 2, 1)
        return np_of(out), np_of(torch.autograd.grad(out, t, WL.to_device(g, dtype, cuda))[2])

    out, dv = run(v, g)
    bad = v.copy()
    bad[:, :, n - 1, 3] = INF
    got, _ = run(bad, g)
    assert (got[:, :, n - 1, 3] == INF).all()
    same(got[..., rest], out[..., rest], tol)
    bad = g.copy()
    bad[:, hq - 1, n - 1, 3] = INF
    _, got = run(v, bad)
    h = hkv - 1
    seen = np.zeros(n, bool)  # the keys that the last row attends
    for c in lists[0, hq - 1, n - 1]:
        seen[c * block:(c + 1) * block] = True
    assert (got[0, h, seen, 3] == INF).all()
    same(got[0, :, :, rest], dv[0, :, :, rest], tol * max(1.0, np.abs(dv).max()))
