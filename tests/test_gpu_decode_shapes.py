"""Routed decode steps at the sizes where the attend launch changes its LDS, against the CPU oracle
(float64)."""
import numpy as np
import pytest
import torch

from oracle import ssa_oracle as O
from ssa_amd import workloads as WL

pytestmark = pytest.mark.gpu


def check_steps(cuda, dtype, B, hq, hkv, d, block, n, top_c, steps=2, rows=((0, 0), (-1, -1))):
    """Steps of a RoutedDecoder on an n-token cache: selections exact, outputs within the bars of the
    decode tests (2e-2, fp32 1e-5), at the (batch, head) rows given."""
    from ssa_amd.ivf_decode import RoutedDecoder
    rng = np.random.default_rng(n + d)
    k, v = (WL.round_to(rng.standard_normal((B, hkv, n + steps, d)).astype(np.float32), dtype)
            for _ in range(2))
    q = WL.round_to(rng.standard_normal((steps, B, hq, d)).astype(np.float32), dtype)
    kt, vt, qt = (WL.to_device(a, dtype, cuda) for a in (k, v, q))
    dec = RoutedDecoder(B, hq, hkv, d, n + steps, block=block, top_c=top_c, local=1, dtype=dtype,
                        device=cuda)
    dec.prefill(kt[:, :, :n], vt[:, :, :n])
    tol = 1e-5 if dtype == torch.float32 else 2e-2
    for t in range(steps):
        out = dec.step(qt[t], kt[:, :, n + t], vt[:, :, n + t]).detach().float().cpu().numpy()
        kn, ki = dec.kv_num.cpu().numpy(), dec.kv_idx.cpu().numpy()
        for b, h in rows:
            b, h = b % B, h % hq
            g = h // (hq // hkv)
            on, oi = O.route_query(q[t][b:b + 1, h:h + 1, None], k[b:b + 1, g:g + 1], block, n + t,
                                   top_c=top_c, local=1, kv_len=n + t + 1)
            sel = oi[0, 0, 0, :on[0, 0, 0]].tolist()
            assert ki[b, h, :kn[b, h]].tolist() == sel, (t, b, h)
            ref = O.decode_attend(q[t][b, h], k[b, g], v[b, g], sel, n + t, block)
            assert np.abs(out[b, h] - ref).max() < tol, (t, b, h)


# 480, 512, 560 and 640 attend workgroups, blocks of 256 and 512: two a CU or one
@pytest.mark.parametrize("B,hq,hkv,top_c", [(8, 30, 2, 6), (8, 32, 8, 4), (8, 14, 2, 16),
                                            (8, 20, 4, 12)])
@pytest.mark.parametrize("block", [256, 512])
def test_decode_step_two_workgroups_a_cu(cuda, B, hq, hkv, top_c, block):
    check_steps(cuda, torch.bfloat16, B, hq, hkv, 64, block, 6 * block + block // 3, top_c)


# the merge's segments: chunk lists that fill one, two, four and eight of a wave's 64-entry lists (up
# to 64 chunks) and the fixed array (more), with grids of more than 256 workgroups; head dim 64 also
# with a grid of one workgroup a CU, which takes the fixed array
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("d,hq,nblocks,top_c", [
    (128, 32, 60, 40), (128, 32, 700, 64), (128, 32, 1500, 64), (128, 32, 3500, 64),
    (128, 32, 4200, 64), (64, 32, 60, 40), (64, 32, 700, 64), (64, 32, 1500, 64),
    (64, 32, 3500, 64), (64, 4, 3500, 64)])
def test_decode_step_merge_segments(cuda, dtype, d, hq, nblocks, top_c):
    check_steps(cuda, dtype, 1, hq, 2, d, 16, 16 * nblocks + 5, top_c)
