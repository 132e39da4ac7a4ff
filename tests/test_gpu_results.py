"""Results through pinned slots: a slot goes back to the pool only when its stream has been waited
for, also where an error that an earlier call left on the thread makes a launch look failed."""
import ctypes as C
import time

import numpy as np
import pytest
import torch

from fusion_amd import api as A
from fusion_amd.native import FusionError
from tests.test_gpu_icp import _plane_maps

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
