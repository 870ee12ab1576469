"""The cascade route's workspace: bounded, routed in slices where the scores need more, and no
scores where the memory is not there. Selections equal the row-by-row search's in every case."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def cascade(cuda, seed, blocks, d, **kw):
    from ssa_amd import cascade_router as C
    g = torch.Generator(device=cuda).manual_seed(seed)
    cc = C.CausalCascade(d, search_k=48, **kw)
    for n in blocks:
        cc.append(torch.randn(n * 128, d, device=cuda, generator=g).half())
    return cc, g


def routed(cc, q, first, certify):
    """(block lists, certificates, rounds) of one route call, on the host."""
    kn, ki, cert, st = cc.route(q, first * 128, certify=certify)
    kn, ki = kn.cpu().numpy(), ki.cpu().numpy()
    return ([ki[i, :kn[i]].tolist() for i in range(len(kn))],
            None if cert is None else cert.cpu().numpy().tolist(),
            st["rounds"].cpu().numpy().tolist())


def test_workspace_stays_bounded(cuda, monkeypatch):
    """2048 query blocks against 65,664 rows: 0.5 GB of scores in one piece."""
    from ssa_amd import cascade_router as C
    cc, g = cascade(cuda, 1, (64, 16352), 32, outlier_rate=5e-4)
    q = torch.randn(2048 * 128, 32, device=cuda, generator=g).half()
    torch.cuda.synchronize()
    base = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    got = routed(cc, q, 16416 - 2048, False)
    assert torch.cuda.max_memory_allocated() - base < 300 << 20
    monkeypatch.setattr(C, "SCORE_WORKSPACE_LIMIT", 0)
    assert routed(cc, q, 16416 - 2048, False) == got


# slices of one score tile and of two, a remainder of one query block; with an index the slices
# share the escalation carry
@pytest.mark.parametrize("indexed", [False, True])
@pytest.mark.parametrize("nbq,tiles", [(129, 1), (200, 2), (64, 1), (63, 0)])
def test_slices_select_the_same(cuda, monkeypatch, indexed, nbq, tiles):
    from ssa_amd import cascade_router as C
    kw = dict(nlist=40, nprobe=2) if indexed else {}
    from_blocks = (700, 300)
    cc, g = cascade(cuda, nbq, (), 64, **kw)
    cc.build_threshold = 1000 if indexed else 1 << 30
    for n in from_blocks:
        cc.append(torch.randn(n * 128, 64, device=cuda, generator=g).half())
    assert (cc.index is not None) == indexed
    q = torch.randn(nbq * 128, 64, device=cuda, generator=g).half()
    ref = routed(cc, q, 1000 - nbq, True)
    rows = (cc.n_sub - cc.committed + 3) // 4 * 4 + (cc.n_out + 3) // 4 * 4
    rows += 0 if indexed else (cc.committed + 3) // 4 * 4
    monkeypatch.setattr(C, "SCORE_WORKSPACE_LIMIT", (64 * tiles + 1) * 4 * rows)
    assert cc._route_workspace(nbq, 0, cuda)[1] == (min(nbq, 64 * tiles) if tiles else nbq)
    assert routed(cc, q, 1000 - nbq, True) == ref


def test_no_memory_for_the_scores(cuda, monkeypatch):
    """The allocation of the scores fails: the call routes with the carry alone."""
    cc, g = cascade(cuda, 3, (), 64, nlist=40, nprobe=2)
    cc.build_threshold = 1000
    for n in (700, 300):
        cc.append(torch.randn(n * 128, 64, device=cuda, generator=g).half())
    q = torch.randn(100 * 128, 64, device=cuda, generator=g).half()
    ref = routed(cc, q, 900, True)
    empty, tried = torch.empty, []

    def short(*a, **k):
        if k.get("dtype") == torch.uint8 and a[0] > 400_000:
            tried.append(a[0])
            raise torch.OutOfMemoryError("no memory")
        return empty(*a, **k)
    monkeypatch.setattr(torch, "empty", short)
    got = routed(cc, q, 900, True)
    assert tried and got == ref


# short contexts, few query blocks: the scores ahead cost more launches than they save
@pytest.mark.parametrize("d,blocks,nbq,indexed,ahead", [
    (64, (30, 30), 8, False, False), (64, (150, 150), 1, False, False),
    (128, (300, 300), 64, True, False), (64, (1300, 1300), 1, False, True),
    (96, (700, 700), 1, False, True), (32, (550, 550), 129, False, True),
    (256, (300, 700), 300, True, True), (32, (700, 1100), 130, True, True),
    (64, (300, 300), 800, False, True)])
def test_scores_ahead_only_where_they_pay(cuda, monkeypatch, d, blocks, nbq, indexed, ahead):
    """The workspace shows whether the scores were written; the selection is the same."""
    from ssa_amd import cascade_router as C
    cc, g = cascade(cuda, d, (), d, **(dict(nlist=40, nprobe=2) if indexed else {}))
    cc.build_threshold = 1000 if indexed else 1 << 30
    for n in blocks:
        cc.append(torch.randn(n * 128, d, device=cuda, generator=g).half())
    assert (cc.index is not None) == indexed
    q = torch.randn(nbq * 128, d, device=cuda, generator=g).half()
    first = max(sum(blocks) - nbq, 200)
    empty, made = torch.empty, []

    def marked(*a, **k):
        t = empty(*a, **k)
        if k.get("dtype") == torch.uint8:
            made.append(t.fill_(0xA5))
        return t
    monkeypatch.setattr(torch, "empty", marked)
    got = routed(cc, q, first, False)
    assert len(made) == 1 and bool((made[0] != 0xA5).any()) == ahead
    monkeypatch.setattr(C, "SCORE_WORKSPACE_LIMIT", 0)
    assert routed(cc, q, first, False) == got


def test_centroids_at_any_float(cuda):
    """Assignment and k-means read a caller's centroids at 4-byte alignment."""
    from ssa_amd import _lib
    g = torch.Generator(device=cuda).manual_seed(5)
    n, nlist, d = 300, 37, 96
    x = torch.randn(n, d, device=cuda, generator=g)
    c = torch.randn(nlist, d, device=cuda, generator=g)
    ws = torch.empty(int(_lib.query("ssa_ccc_index_size", n, nlist, d)), dtype=torch.uint8,
                     device=cuda)
    res = []
    for shift in (0, 1, 2, 3):
        buf = torch.empty(nlist * d + 4, device=cuda)
        cent = buf[shift:shift + nlist * d]
        cent.copy_(c.view(-1))
        assign = torch.empty(n, dtype=torch.int32, device=cuda)
        _lib.call("ssa_ccc_assign", x.data_ptr(), n, d, cent.data_ptr(), nlist, assign.data_ptr(),
                  ws.data_ptr(), ws.numel(), _lib.stream_of(x))
        _lib.call("ssa_ccc_kmeans", x.data_ptr(), n, d, nlist, 2, 1, cent.data_ptr(),
                  ws.data_ptr(), ws.numel(), _lib.stream_of(x))
        res.append((assign.tolist(), cent.tolist()))
    assert all(r == res[0] for r in res[1:])
