"""Calls that read a key map side by side, each on a stream and thread of its own: every collection
is the slots in order and every relocalisation the one of a call alone, from the first call after the
map has changed."""
import threading

import numpy as np
import pytest
import torch

from fusion_amd import api as A

pytestmark = pytest.mark.gpu


def _keys(rng, n):
    k = np.zeros(n, A.SURF_DTYPE)
    k["valid"] = 1
    k["pos"] = rng.uniform([-2, -2, 0.5], [2, 2, 4.0], (n, 3)).astype(np.float32)
    k["normal"] = rng.normal(size=(n, 4)).astype(np.float32)
    k["descriptor"] = rng.normal(size=(n, 64)).astype(np.float32)
    return k


@pytest.mark.parametrize("max_keys,n_buckets", [(20011, 3), (70001, 5)])
def test_reads_side_by_side(gpu, max_keys, n_buckets):
    rng = np.random.default_rng(max_keys)
    km = A.KeyMap(max_keys=max_keys, n_buckets=n_buckets)
    streams = [torch.cuda.Stream() for _ in range(4)]
    for rep, n in enumerate((600, 900, 0, 700)):  # 0: a reset
        print("side by side", max_keys, rep, flush=True)
        if n == 0:
            km.ResetKeyPoints()
            n = 500
        keys = _keys(rng, n)
        km.InsertKeyPoints(A.surf_to_device(keys), torch.full((n,), -1, dtype=torch.int32, device="cuda"))
        slots = km.read()
        want = slots[slots["valid"] != 0]
        pick = rng.choice(len(want) - 1, 200, replace=False) + 1
        desc = torch.from_numpy(want["descriptor"][pick] + np.float32(0.01)).cuda()
        cam = want["pos"][pick].astype(np.float64) + 0.25
        torch.cuda.synchronize()
        got = [None] * len(streams)
        barrier = threading.Barrier(len(streams))

        def work(i):
            out = []
            with torch.cuda.stream(streams[i]):
                barrier.wait(60)
                for k in range(6):
                    if (i + k) % 2:
                        out.append(km.relocalise(desc, cam, iterations=40, seed=3))
                    else:
                        o, m = km.CollectKeyPoints(len(want) + 2)
                        out.append((A.surf_from_device(o), m))
            got[i] = out

        threads = [threading.Thread(target=work, args=(i,)) for i in range(len(streams))]
        for t in threads:
            t.start()
        for t in threads:
            t.join(100)
        pose, pairs = km.relocalise(desc, cam, iterations=40, seed=3)
        assert pose is not None and pairs == len(pick)
        for i, out in enumerate(got):
            assert out is not None, i
            for k, (a, b) in enumerate(out):
                if (i + k) % 2:
                    assert b == pairs and np.array_equal(a, pose)
                else:
                    assert b == len(want) and a[1 : len(want)].tobytes() == want[1:].tobytes()
    km.close()


def test_number_of_keys_after_a_failed_insert(gpu):
    """an insert that fails part way (here refused by its stream, which is being captured) leaves the
    number of keys to be read from the device"""
    import ctypes as C

    from fusion_amd import native as N
    from tests.test_gpu_results import _hip

    rng = np.random.default_rng(4)
    km = A.KeyMap(max_keys=997, n_buckets=5)
    keys = _keys(rng, 300)
    km.InsertKeyPoints(A.surf_to_device(keys), torch.full((300,), -1, dtype=torch.int32, device="cuda"))
    slots = km.read()
    want = slots[slots["valid"] != 0]
    desc = torch.from_numpy(want["descriptor"][1:] + np.float32(0.01)).cuda()
    cam = want["pos"][1:].astype(np.float64) + 0.25
    pose, pairs = km.relocalise(desc, cam, iterations=40, seed=3)
    more, index = A.surf_to_device(_keys(rng, 50)), torch.full((50,), -1, dtype=torch.int32, device="cuda")
    hip, s, graph = _hip(), torch.cuda.Stream(), C.c_void_p()
    torch.cuda.synchronize()
    stream = C.c_void_p(s.cuda_stream)
    assert hip.hipStreamBeginCapture(stream, 2) == 0
    st = N.lib().fu_insert_key_points(km.handle, C.c_void_p(more.data_ptr()), C.c_void_p(index.data_ptr()), 50, stream)
    end = hip.hipStreamEndCapture(stream, C.byref(graph))
    hip.hipGetLastError()
    assert st != 0 and (end != 0 or not graph.value)
    again, n = km.relocalise(desc, cam, iterations=40, seed=3)
    assert pose is not None and np.array_equal(again, pose) and n == pairs == len(want) - 1
    km.InsertKeyPoints(more, index)
    assert km.CollectKeyPoints(4)[1] == int((km.read()["valid"] != 0).sum()) == len(want) + int((index >= 0).sum())
    km.close()
