"""Results on the host.  A pinned slot goes back to the pool only when its stream has been waited for,
also where an error that an earlier call left on the thread makes a launch look failed; a batch's
results are those of its call, whatever has become of its trackers since."""
import ctypes as C
import time

import numpy as np
import pytest
import torch

from fusion_amd import api as A
from fusion_amd import native as N
from fusion_amd.native import FusionError
from tests.test_gpu_icp import _pair, _plane_maps

pytestmark = pytest.mark.gpu


def _hip():
    """the HIP runtime that this process has loaded"""
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64" in line)
    return C.CDLL(path)


def _leave_error(hip):
    """a refused call (a device number that does not exist): its error stays on the thread"""
    assert hip.hipSetDevice(1 << 20) != 0
    return hip.hipPeekAtLastError() != 0


def test_slot_waits_for_its_stream(gpu):
    hip = _hip()
    K = (64.0, 64.0, 39.5, 29.5)
    v, nm = _plane_maps(80, 60, K)
    v, nm = (torch.from_numpy(a).cuda() for a in (v, nm))
    step = lambda: A.ICPStep(v, v, nm, nm, np.eye(4), np.eye(4), K)
    want = step()
    m = A.Mapping(num_buckets=64, num_excess=64, num_blocks=64, voxel_size=0.01, trunc_dist=0.03, max_new_blocks=64)
    stats = m.stats()
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    for call, fails in ((step, True), (m.stats, False)):
        with torch.cuda.stream(s):
            torch.cuda._sleep(20_000_000)  # the call's launch is behind this
            if not _leave_error(hip):
                pytest.skip("this runtime keeps no error between calls")
            t = time.perf_counter()
            if fails:
                with pytest.raises(FusionError):
                    call()
            else:
                assert call() == stats
            assert s.query(), "returned after %.6f s with its launch under way" % (time.perf_counter() - t)
    hip.hipGetLastError()
    for a, b in zip(step(), want):
        assert np.array_equal(a, b)
    m.close()


def test_batch_results_are_those_of_the_call(gpu):
    """results asked for on another stream than the call's, after its trackers have been used for
    another pair and after they are gone"""
    cols, rows, n = 160, 120, 3
    K, last, following, _ = _pair(0, 2, cols, rows)
    (lv, ln), (nv, nn) = ([[torch.from_numpy(m).cuda() for m in maps] for maps in pair] for pair in (last, following))
    first = [A.Tracker(cols, rows) for _ in range(n)]
    b = A.IcpBatch(n)
    want = b.ComputeSE3(first, [nv] * n, [nn] * n, [lv] * n, [ln] * n, [K] * n)
    assert all(r["iterations"] == 19 for r in want)
    trackers = [A.Tracker(cols, rows) for _ in range(n)]
    handles = (C.c_void_p * n)(*[t.handle.value for t in trackers])
    arr = lambda maps: (C.c_void_p * (3 * n))(*[m.data_ptr() for _ in range(n) for m in maps])
    Kf = (C.c_float * (4 * n))(*(list(K) * n))
    s = torch.cuda.Stream()
    out = (N.TrackResult * n)()
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        st = N.lib().fu_compute_se3_batch(b.handle, n, handles, arr(nv), arr(nn), arr(lv), arr(ln), Kf,
                                          (C.c_int32 * 3)(10, 5, 4), (C.c_int32 * 3)(2000, 1000, 100), 1e-4,
                                          s.cuda_stream)
        assert st == 0
        for t in trackers:
            assert not np.array_equal(t.ComputeSE3(lv, ln, lv, ln, K)["x"], want[0]["x"])
    del t
    trackers.clear()
    assert N.lib().fu_icp_batch_results(b.handle, n, out, None) == 0
    for r, w in zip(out, want):
        got = A._track_result(r)
        assert all(np.array_equal(got[k], w[k]) for k in w), (got, w)
    assert N.lib().fu_icp_batch_results(b.handle, n + 1, out, None) != 0
