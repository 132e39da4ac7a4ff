"""GPU ICP (Tracking/Reduction.cu, Tracking/Tracking.cc:296-409) against the FP64 oracle.

Bar: each ICP step's pose update within 1e-5 rad and 1e-5 m of the FP64
oracle on the same inputs; the reduced normal equations within FP32 summation error.
"""
import numpy as np
import pytest
import torch

from fusion_amd import api as A
from oracle import binding as O
from tests.helpers import scene_frames
from tests.test_gpu_pyramid import _pyr_oracle

pytestmark = pytest.mark.gpu


def _rot_err(Ra, Rb):
    c = (np.trace(Ra.T @ Rb) - 1) / 2
    return float(np.arccos(np.clip(c, -1, 1)))


def _pair(f0=0, f1=2, cols=640, rows=480):
    sc, K, fr = scene_frames(frames=(f0, f1), cols=cols, rows=rows)
    _, _, v0, n0 = _pyr_oracle(fr[0][0], K)
    _, _, v1, n1 = _pyr_oracle(fr[1][0], K)
    gt = np.linalg.inv(sc.pose(f0)) @ sc.pose(f1)
    return K, (v0, n0), (v1, n1), gt


def test_icp_step_sums(gpu):
    K, (v0, n0), (v1, n1), gt = _pair()
    cu = lambda a: torch.from_numpy(a).cuda()
    A_g, b_g, r_g = A.ICPStep(cu(v1[0]), cu(v0[0]), cu(n1[0]), cu(n0[0]), np.eye(4), np.eye(4), K)
    s32, s64 = O.icp_sums(v1[0], v0[0], n1[0], n0[0], np.eye(4), np.eye(4), K)
    A_o, b_o = O.unpack_sums(s64)
    assert r_g[1] == s64[28]  # the correspondence count is exact
    scale = np.abs(A_o).max()
    assert np.abs(A_g - A_o).max() <= 1e-6 * scale
    assert np.abs(b_g - b_o).max() <= 1e-6 * max(np.abs(b_o).max(), 1e-12) + 1e-6 * scale * 1e-3
    x_g = np.linalg.solve(A_g, b_g)
    x_o = O.solve6(A_o, b_o)
    assert np.abs(x_g - x_o).max() < 1e-6


def test_icp_step_at_a_moving_pose(gpu):
    """the true motion from frame 0 to frame 2 as the current pose: the association's
    projection (float invz and products, + 0.5 in double, Reduction.cu:237-239) decides pixels
    on these maps, so the correspondence count must equal the oracle's and an independent numpy
    restatement's exactly; A and b within FP32 summation error of the FP64 sums"""
    from tests.icp_numpy import associate
    K, (v0, n0), (v1, n1), gt = _pair()
    cu = lambda a: torch.from_numpy(a).cuda()
    A_g, b_g, r_g = A.ICPStep(cu(v1[0]), cu(v0[0]), cu(n1[0]), cu(n0[0]), gt, np.eye(4), K)
    _, s64 = O.icp_sums(v1[0], v0[0], n1[0], n0[0], gt, np.eye(4), K)
    ok, _, _ = associate(v1[0], n1[0], v0[0], n0[0], gt, np.eye(4), K)
    assert r_g[1] == s64[28] == ok.sum() > 200000
    A_o, b_o = O.unpack_sums(s64)
    scale = np.abs(A_o).max()
    assert np.abs(A_g - A_o).max() <= 1e-6 * scale
    assert np.abs(b_g - b_o).max() <= 1e-6 * max(np.abs(b_o).max(), 1e-12) + 1e-9 * scale


def _plane_maps(cols, rows, K, n=(0.1, -0.2, -1.0), c=-2.0, seed=0):
    """vertex and normal maps of the plane n.p = c seen from the origin, with a mild ripple"""
    fx, fy, cx, cy = K
    n = np.asarray(n, np.float64)
    n /= np.linalg.norm(n)
    x = (np.arange(cols) - cx) / fx
    y = (np.arange(rows) - cy) / fy
    d = np.stack(np.broadcast_arrays(x[None, :], y[:, None], np.ones((1, 1))), -1)
    t = c / (d @ n)
    t *= 1.0 + 0.002 * np.sin(np.arange(cols) / 37.0)[None, :] * np.cos(np.arange(rows) / 23.0)[:, None]
    v = np.concatenate([d * t[..., None], np.ones((rows, cols, 1))], -1)
    nm = np.concatenate([np.broadcast_to(n, (rows, cols, 3)), np.ones((rows, cols, 1))], -1)
    return np.ascontiguousarray(v, np.float32), np.ascontiguousarray(nm, np.float32)


def test_icp_step_sums_chunk_loop(gpu):
    """a frame of more pixels than 4096 work-groups of two pixels per lane cover (8.6M) takes
    the per-lane chunk loop with compensated sums (k_icp_step<kLoop>); its sums match FP64 and the
    correspondence count is exact"""
    cols, rows = 4096, 2112
    K = (2000.0, 2000.0, cols / 2 - 0.5, rows / 2 - 0.5)
    v, nm = _plane_maps(cols, rows, K)
    pc = np.eye(4)
    pc[:3, 3] = (0.002, -0.001, 0.003)
    cu = lambda a: torch.from_numpy(a).cuda()
    print("icp chunk loop %dx%d" % (cols, rows), flush=True)
    A_g, b_g, r_g = A.ICPStep(cu(v), cu(v), cu(nm), cu(nm), pc, np.eye(4), K)
    s32, s64 = O.icp_sums(v, v, nm, nm, pc, np.eye(4), K)
    A_o, b_o = O.unpack_sums(s64)
    assert r_g[1] == s64[28] and s64[28] > 0.9 * cols * rows
    scale = np.abs(A_o).max()
    assert np.abs(A_g - A_o).max() <= 1e-6 * scale
    assert np.abs(b_g - b_o).max() <= 1e-6 * max(np.abs(b_o).max(), 1e-12) + 1e-9 * scale


@pytest.mark.parametrize("cols,rows,f1", [(640, 480, 2), (320, 240, 3), (1280, 720, 1)])
def test_compute_se3_vs_fp64(gpu, cols, rows, f1):
    print("icp %dx%d" % (cols, rows), flush=True)
    K, (v0, n0), (v1, n1), gt = _pair(0, f1, cols, rows)
    t = A.Tracker(cols, rows)
    cu = lambda xs: [torch.from_numpy(x).cuda() for x in xs]
    t.set_last_pose(np.eye(4))
    r = t.ComputeSE3(cu(v1), cu(n1), cu(v0), cu(n0), K)
    st, pose_o, err_o, cnt_o = O.compute_se3(v1, n1, v0, n0, K, np.eye(4))
    assert r["status"] == st == 1
    assert _rot_err(r["pose"][:3, :3], pose_o[:3, :3]) <= 1e-5
    assert np.linalg.norm(r["pose"][:3, 3] - pose_o[:3, 3]) <= 1e-5
    # and the motion itself is recovered (at 1280x720 the depth noise of 0.0015 z^2 m spans
    # several pixel spacings, so the reference algorithm's estimate itself is off by ~1 cm
    # on this view; the requirement there is agreement with the FP64 oracle above)
    if cols <= 640:
        assert np.linalg.norm(r["pose"][:3, 3] - gt[:3, 3]) < 3e-3


def test_icp_too_few_points_rolls_back(gpu):
    K, (v0, n0), (v1, n1), gt = _pair()
    empty = [np.full_like(v, np.nan) for v in v1]
    t = A.Tracker(640, 480)
    P = np.eye(4)
    P[:3, 3] = [0.1, 0.2, 0.3]
    t.set_last_pose(P)
    cu = lambda xs: [torch.from_numpy(x).cuda() for x in xs]
    r = t.ComputeSE3(cu(empty), cu(empty), cu(v0), cu(n0), K)
    assert r["status"] == 2
    assert np.array_equal(r["pose"], P)
    st, pose_o, _, _ = O.compute_se3(empty, empty, v0, n0, K, P)
    assert st == 2 and np.array_equal(pose_o, P)


def test_icp_large_motion_rejected(gpu):
    """a 0.2 m jump between model and frame is not accepted (Tracking.cc:398-408)"""
    sc, K, fr = scene_frames(frames=(0,))
    _, _, v0, n0 = _pyr_oracle(fr[0][0], K)
    pose = sc.pose(0).copy()
    pose[:3, 3] += pose[:3, :3] @ np.array([0.0, 0.0, 0.2])
    d1, _ = sc.render_pose(pose)
    _, _, v1, n1 = _pyr_oracle(d1, K)
    t = A.Tracker(640, 480)
    cu = lambda xs: [torch.from_numpy(x).cuda() for x in xs]
    r = t.ComputeSE3(cu(v1), cu(n1), cu(v0), cu(n0), K)
    st, _, _, _ = O.compute_se3(v1, n1, v0, n0, K, np.eye(4))
    assert r["status"] == st
    assert r["status"] in (2, 3)
    assert np.array_equal(r["pose"], np.eye(4))


def test_compute_se3_batch_uneven_sizes(gpu):
    """Batched ComputeSE3 over frame pairs of uneven size (320x240, 640x480, 1280x720; more
    pairs than one launch takes, so they run in groups): every pair's result is identical to
    the tracker run alone, and within 1e-5 rad / 1e-5 m of the FP64 oracle"""
    sizes = [(320, 240)] * 50 + [(640, 480)] * 12 + [(1280, 720)] * 4
    rng = np.random.default_rng(3)
    rng.shuffle(sizes)
    cu = lambda xs: [torch.from_numpy(x).cuda() for x in xs]
    pairs, trackers, alone = [], [], []
    print("pairs", len(sizes), flush=True)
    for i, (cols, rows) in enumerate(sizes):
        f0 = int(rng.integers(0, 40))
        sc, K, fr = scene_frames(frames=(f0, f0 + 2), cols=cols, rows=rows)
        _, _, v0, n0 = _pyr_oracle(fr[0][0], K)
        _, _, v1, n1 = _pyr_oracle(fr[1][0], K)
        pairs.append((K, cu(v1), cu(n1), cu(v0), cu(n0), (v0, n0, v1, n1)))
        t = A.Tracker(cols, rows)
        alone.append(t.ComputeSE3(*[pairs[-1][k] for k in (1, 2, 3, 4)], K))
        t2 = A.Tracker(cols, rows)
        t2.set_last_pose(np.eye(4))
        trackers.append(t2)
    b = A.IcpBatch(128)
    res = b.ComputeSE3(trackers, [p[1] for p in pairs], [p[2] for p in pairs], [p[3] for p in pairs],
                       [p[4] for p in pairs], [p[0] for p in pairs])
    for i, (ra, rb) in enumerate(zip(alone, res)):
        assert ra["status"] == rb["status"], i
        assert np.array_equal(ra["pose"], rb["pose"]), i
    # the FP64 oracle's final pose after the whole coarse-to-fine loop (19 steps; the per-step
    # bar of 1e-5 rad / 1e-5 m is checked per step by test_icp_step_sums): within 3e-5
    checked = 0
    for i, (cols, rows) in enumerate(sizes):
        if checked >= 6 or (cols == 320 and checked >= 2):
            continue
        K, _, _, _, _, (v0, n0, v1, n1) = pairs[i]
        st, pose_o, _, _ = O.compute_se3(v1, n1, v0, n0, K, np.eye(4))
        assert res[i]["status"] == st, i
        if st == 1:
            er = _rot_err(res[i]["pose"][:3, :3], pose_o[:3, :3])
            et = np.linalg.norm(res[i]["pose"][:3, 3] - pose_o[:3, 3])
            print("pair %d %dx%d: rot %.2e rad, trans %.2e m vs FP64" % (i, cols, rows, er, et), flush=True)
            assert er <= 3e-5 and et <= 3e-5, i
        checked += 1
    assert sum(r["status"] == 1 for r in res) >= 0.9 * len(res)
