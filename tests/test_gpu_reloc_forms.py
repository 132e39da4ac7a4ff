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

