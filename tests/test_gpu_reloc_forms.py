"""The relocalisation kernels where their bounds and splits can go wrong, against the oracle.

The matcher prices all pairs and evaluates only the chunks that can hold a query's two nearest:
its indices and distances are the exact scan's, bit for bit, also for ties, for magnitudes whose
products overflow or vanish, and for descriptors that are not finite.
"""
import numpy as np
import pytest
import torch

from fusion_amd import api as A
from oracle import binding as O

pytestmark = pytest.mark.gpu


def _descriptors(kind, nq, nt, seed=0):
    rng = np.random.default_rng(seed)
    t = rng.normal(size=(nt, 64)).astype(np.float32)
    t /= np.linalg.norm(t, axis=1, keepdims=True)
    q = t[rng.integers(0, nt, nq)] + rng.normal(0, 0.03, (nq, 64)).astype(np.float32)
    if kind == "ties":  # few values, many equal distances, every one several times
        t = rng.integers(0, 2, (nt, 64)).astype(np.float32) * np.float32(0.25)
        t[nt // 2 :] = t[: nt - nt // 2]
        q = t[rng.integers(0, nt, nq)].copy()
    elif kind == "mixed":  # magnitudes from vanishing to overflowing, zeros
        e = rng.choice([1e-30, 1e-22, 1e-10, 1.0, 1e10, 1e18, 3e19], nt).astype(np.float32)
        t *= e[:, None]
        t[rng.random(nt) < 0.1] = 0
        q = (t[rng.integers(0, nt, nq)] * np.float32(1.01)).astype(np.float32)
    elif kind == "huge":  # all products overflow, the differences do not
        t = (t * 0.01 + 2e19).astype(np.float32)
        q = t[rng.integers(0, nt, nq)].copy()
    elif kind == "holes":
        t[rng.random(nt) < 0.01, 5] = np.nan
        t[rng.random(nt) < 0.01, 60] = np.inf
        q[rng.random(nq) < 0.1, 7] = np.nan
        q[rng.random(nq) < 0.1, 9] = -np.inf
    return np.ascontiguousarray(q, dtype=np.float32), t


@pytest.mark.parametrize("kind", ["unit", "ties", "mixed", "huge", "holes"])
@pytest.mark.parametrize("nq,nt", [(1, 2), (33, 512), (31, 513), (129, 640), (64, 641), (200, 4133)])
def test_match_forms_exact(gpu, kind, nq, nt):
    print("match", kind, nq, nt, flush=True)
    q, t = _descriptors(kind, nq, nt)
    idx, dist = A.match_knn2(torch.from_numpy(q).cuda(), torch.from_numpy(t).cuda())
    io, do = O.match_knn2(q, t)
    assert np.array_equal(idx.cpu().numpy(), io)
    assert np.array_equal(dist.cpu().numpy().view(np.uint32), do.view(np.uint32))


@pytest.mark.parametrize("kind", ["unit", "few", "holes"])
@pytest.mark.parametrize("nq,nt", [(8193, 600), (16385, 3), (16384, 128), (8193, 4096), (300, 4200), (40, 33100)])
def test_match_dispatch_exact(gpu, kind, nq, nt):
    """both sides of the dispatch's lines, and queries left to the list of those that have too many
    chunks to scan: some of them, and more than a wave keeps the bounds of"""
    print("match dispatch", kind, nq, nt, flush=True)
    q, t = _descriptors("unit" if kind == "few" else kind, nq, nt)
    if kind == "few":  # zeros in every chunk, and queries that are zero among others
        t[::3] = 0
        q[::7] = 0
    idx, dist = A.match_knn2(torch.from_numpy(q).cuda(), torch.from_numpy(t).cuda())
    some = np.unique(np.concatenate([np.arange(min(nq, 300)), np.arange(max(0, nq - 100), nq)]))
    io, do = O.match_knn2(np.ascontiguousarray(q[some]), t)
    assert np.array_equal(idx.cpu().numpy()[some], io)
    assert np.array_equal(dist.cpu().numpy()[some].view(np.uint32), do.view(np.uint32))
    assert int(idx.min()) >= -1 and int(idx.max()) < nt


def _key_map(nk, max_keys, n_buckets, seed):
    rng = np.random.default_rng(seed)
    keys = np.zeros(nk, A.SURF_DTYPE)
    keys["valid"] = 1
    keys["pos"] = rng.uniform([-2, -2, 0.5], [2, 2, 4.0], (nk, 3)).astype(np.float32)
    keys["normal"] = rng.normal(size=(nk, 4)).astype(np.float32)
    keys["descriptor"] = rng.normal(size=(nk, 64)).astype(np.float32)
    km = A.KeyMap(max_keys=max_keys, n_buckets=n_buckets)
    km.InsertKeyPoints(A.surf_to_device(keys), torch.full((nk,), -1, dtype=torch.int32, device="cuda"))
    return km


@pytest.mark.parametrize("nk,max_keys,n_buckets", [(1, 1, 1), (64, 13, 5), (300, 1021, 2), (4000, 1021, 5), (2500, 70001, 3)])
def test_collect_forms(gpu, nk, max_keys, n_buckets):
    # sparse and full words of slots, several groups, counts that start in the middle of a group
    print("collect", nk, max_keys, n_buckets, flush=True)
    km = _key_map(nk, max_keys, n_buckets, nk)
    slots = km.read()
    want = slots[slots["valid"] != 0]
    for cap in (len(want) + 3, max(1, len(want) // 2)):
        out, n = km.CollectKeyPoints(cap)
        assert n == len(want)
        got = A.surf_from_device(out)
        m = min(cap, n)
        assert got[1:m].tobytes() == want[1:m].tobytes()
        assert not any(got[:1].tobytes()) and not any(got[m:].tobytes())
    km.close()


@pytest.mark.parametrize("share,iterations", [(0.6, 100), (0.04, 0), (0.04, 1), (0.04, 256), (0.04, 257), (0.02, 4500)])
def test_relocalise_equals_the_host_walk(gpu, share, iterations):
    # the inliers of the draws are counted on the device, at more draws in further launches (few
    # inliers: the confidence does not end the walk): the pose is that of the host's own counts
    nk = 1500
    km = _key_map(nk, 20011, 5, 3)
    out, n = km.CollectKeyPoints(nk + 8)
    rec = A.surf_from_device(out)[:n]
    rec[0] = np.zeros(1, A.SURF_DTYPE)
    rng = np.random.default_rng(5)
    seen = rng.choice(n, 500, replace=False)
    cam = rec["pos"][seen].astype(np.float64) + 0.25 + rng.normal(0, 0.002, (500, 3))
    lost = rng.random(500) >= share
    cam[lost] = rng.uniform(-3, 3, (int(lost.sum()), 3))
    desc = torch.from_numpy((rec["descriptor"][seen] + rng.normal(0, 0.05, (500, 64))).astype(np.float32)).cuda()
    idx, dist = A.match_knn2(desc, torch.from_numpy(np.ascontiguousarray(rec["descriptor"])).cuda())
    idx, dist = idx.cpu().numpy(), dist.cpu().numpy().astype(np.float64)
    take = np.nonzero((idx[:, 0] >= 0) & (dist[:, 0] < 0.90 * dist[:, 1]))[0]
    for seed in (1, 2):
        print("walk", share, iterations, seed, flush=True)
        got, npairs = km.relocalise(desc, cam, iterations=iterations, seed=seed)
        T, _ = A.pose_estimate(cam[take], rec["pos"][idx[take, 0]].astype(np.float64), iterations, seed)
        assert npairs == len(take) > 400
        assert (got is None) == (T is None)
        if T is not None:
            want = np.eye(4)
            for i in range(3):
                want[i, :3] = T[:3, i]
                want[i, 3] = -(T[0, i] * T[0, 3] + T[1, i] * T[1, 3] + T[2, i] * T[2, 3])
            assert np.array_equal(got, want)
    km.close()


@pytest.mark.parametrize("n,max_sel", [(2, 2), (3, 3), (5, 4), (6, 5), (40, 64), (300, 257), (1100, 1024)])
def test_selection_forms(gpu, n, max_sel):
    # counts about the refinement's groups of four pairs and its 256-pair passes, and a head whose
    # list fills; most pairs agree with the head, one in four excludes another
    rng = np.random.default_rng(n)
    C = (0.2 + 0.8 * rng.random((n, n))).astype(np.float32)
    C[rng.random((n, n)) < 2.0 / n] = 0.0
    print("select", n, max_sel, flush=True)
    g = A.select_subgraphs(torch.from_numpy(C).cuda(), 10, max_sel, 0.1)
    o = O.graph_select(C, 10, max_sel, 0.1)
    assert np.array_equal(g[2].view(np.uint32), o[2].view(np.uint32)) and np.array_equal(g[3], o[3])
    assert np.array_equal(g[0], o[0])
    for a, b in zip(g[1], o[1]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("n,max_sel,lists", [(1, 4, 3), (5, 1024, 4200), (70, 64, 300), (1100, 1024, 40), (300, 130, 125)])
def test_selection_of_many_lists(gpu, n, max_sel, lists):
    # more lists than a wave per pair is launched for: waves that take several pairs, lists that ranks end
    rng = np.random.default_rng(n + lists)
    C = (0.2 + 0.8 * rng.random((n, n))).astype(np.float32)
    C[rng.random((n, n)) < 2.0 / n] = 0.0
    print("select", n, max_sel, lists, flush=True)
    g = A.select_subgraphs(torch.from_numpy(C).cuda(), lists, max_sel, 0.1)
    o = O.graph_select(C, lists, max_sel, 0.1)
    assert np.array_equal(g[0], o[0])
    assert len(g[1]) == len(o[1]) == lists
    for a, b in zip(g[1], o[1]):
        assert np.array_equal(a, b)
