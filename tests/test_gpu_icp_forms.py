"""The work-group forms of an ICP iteration: a quarter of a 2048-pixel chunk, a chunk, and the
chunk loop per work-group.  The sums at the sizes where the form changes (1, 128 and 129 chunks,
a chunk that is not full; above 4096 chunks) against the FP64 oracle, ICP and photometric; the
forms of a batch against a tracker alone; the two ways in which a session's frame has its vertices."""
import numpy as np
import pytest
import torch

from fusion_amd import api as A
from oracle import binding as O
from tests.test_gpu_icp import _plane_maps

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cols,rows", [(33, 31), (64, 32), (65, 32), (512, 512), (513, 512)])
def test_sums_of_each_form(gpu, cols, rows):
    print("icp forms %dx%d" % (cols, rows), flush=True)
    K = (0.8 * cols, 0.8 * cols, cols / 2 - 0.5, rows / 2 - 0.5)
    v, nm = _plane_maps(cols, rows, K)
    pc = np.eye(4)
    pc[:3, 3] = (0.002, -0.001, 0.003)
    cu = lambda a: torch.from_numpy(a).cuda()
    s32, s64 = O.icp_sums(v, v, nm, nm, pc, np.eye(4), K)
    A_o, b_o = O.unpack_sums(s64)
    scale = np.abs(A_o).max()
    for rep in range(3):  # the arrival count is back at zero after each call
        A_g, b_g, r_g = A.ICPStep(cu(v), cu(v), cu(nm), cu(nm), pc, np.eye(4), K)
        assert r_g[1] == s64[28] and s64[28] > 0.9 * cols * rows
        # FP32 products (2^-24 each) added pairwise: far below 1e-6 of the largest sum
        assert np.abs(A_g - A_o).max() <= 1e-6 * scale
        assert np.abs(b_g - b_o).max() <= 1e-6 * max(np.abs(b_o).max(), 1e-12) + 1e-9 * scale
    # the photometric sums on the same maps
    rng = np.random.default_rng(cols)
    i0 = rng.integers(1, 250, (rows, cols)).astype(np.uint8)
    i1 = np.clip(i0.astype(int) + rng.integers(-5, 6, i0.shape), 1, 255).astype(np.uint8)
    dx, dy = (rng.integers(-300, 300, i0.shape).astype(np.int16) for _ in range(2))
    (cnt, sq), sigma, _, s64 = O.rgb_sums(i1, i0, v, v, dx, dy, pc, np.eye(4), K)
    A_o, b_o = O.unpack_sums(s64)
    scale = np.abs(A_o).max()
    for rep in range(3):
        A_g, b_g, r_g, (gc, gq) = A.RGBStep(cu(i1), cu(i0), cu(v), cu(v), cu(dx), cu(dy), pc, np.eye(4), K)
        assert (gc, gq) == (cnt, sq) and r_g[1] == s64[28] == cnt > 0
        # the bounds of test_rgb_step_matches_oracle; b's sums cancel, so against its rows' scale
        assert np.abs(A_g - A_o).max() <= 2e-6 * scale
        assert np.abs(b_g - b_o).max() <= 2e-6 * max(np.abs(b_o).max(), np.sqrt(scale * s64[27]))
        assert abs(r_g[0] - s64[27]) <= 2e-6 * s64[27]


@pytest.mark.parametrize("rgb", [False, True])
def test_batch_summed_by_a_second_launch(gpu, rgb):
    """steps of more than 4096 chunks (ten 1280x720 sessions and more) sum their rows in a second
    launch: the poses equal those of a session run alone"""
    K = (1050.0, 1050.0, 639.5, 359.5)
    sc = A.Scene(0, (4.0, 4.0, 3.0), 5)
    mp = dict(num_buckets=1 << 15, num_excess=1 << 15, num_blocks=1 << 15, voxel_size=0.01,
              trunc_dist=float(np.float32(0.01) * np.float32(8.0)), max_new_blocks=1 << 15)
    params = lambda: A.system_params(cols=1280, rows=720, K=K, use_rgb=int(rgb), map=mp)
    alone = A.System(params())
    n = 10
    bt, many = A.Batch(n), [A.System(params()) for _ in range(n)]
    for x in many:
        bt.attach(x)
    for f in range(3):
        print("batch rgb %d frame %d" % (rgb, f), flush=True)
        d, c = A.to_device(*sc.render(f, 1280, 720, K))
        alone.GrabImage(d, c)
        r = alone.result()
        assert r["track_status"] in (1, 4)
        bt.grab(many, [d] * n, [c] * n)
        for x in many:
            assert np.array_equal(x.result()["pose"], r["pose"]), f
    bt.close()


def _bumpy_maps(cols, rows, K, seed):
    """device vertex and normal maps of a surface that constrains every direction"""
    y, x = np.mgrid[0:rows, 0:cols].astype(np.float32)
    z = 2 + 0.3 * np.sin(x / cols * 9) * np.cos(y / rows * 7)
    z += 0.00005 * np.random.default_rng(seed).standard_normal(z.shape, dtype=np.float32)
    v = A.ComputeVMap(torch.from_numpy(z.astype(np.float32)).cuda(), *K, 3.0)
    return v, A.ComputeNMap(v)


def test_chunk_loop_of_a_tracked_pose(gpu):
    """frames of more than 4096 chunks: a tracker's iterations, and a batch's with the sums in the
    iterations' launch and, beside a small frame, in a second one"""
    cols, rows = 4096, 2112
    K = (2000.0, 2000.0, cols / 2 - 0.5, rows / 2 - 0.5)
    small = (160, 120, (140.0, 140.0, 79.5, 59.5))
    levels = lambda m: ([m[0]] * 3, [m[1]] * 3)  # no iterations at the others
    last, following = _bumpy_maps(cols, rows, K, 1), _bumpy_maps(cols, rows, K, 2)
    args = (*levels(following), *levels(last))
    poses = [np.eye(4)]
    lv, ln, nv, nn = (m.cpu().numpy() for m in (*last, *following))
    for k in (1, 2):
        print("chunk loop, %d iterations" % k, flush=True)
        kw = dict(iters=(k, 0, 0), min_count=(1000, 0, 0))
        r = A.Tracker(cols, rows).ComputeSE3(*args, K, **kw)
        assert r["iterations"] == k
        _, s64 = O.icp_sums(nv, lv, nn, ln, poses[-1], np.eye(4), K)
        A_o, b_o = O.unpack_sums(s64)
        # the bounds of test_icp_step_sums_chunk_loop; the pose of the second is the first's, in floats
        assert r["count"] == s64[28] > 0.5 * cols * rows
        scale = np.abs(A_o).max()
        assert np.abs(r["A"] - A_o).max() <= 1e-6 * scale
        assert np.abs(r["b"] - b_o).max() <= 1e-6 * max(np.abs(b_o).max(), np.sqrt(scale * s64[27]))
        poses.append(r["pose"])
        one = A.IcpBatch(1).ComputeSE3([A.Tracker(cols, rows)], *[[m] for m in args], [K], **kw)[0]
        sargs = (*levels(_bumpy_maps(*small, 4)), *levels(_bumpy_maps(*small, 3)))
        two = A.IcpBatch(2).ComputeSE3([A.Tracker(*small[:2]), A.Tracker(cols, rows)], *[[a, b] for a, b in zip(sargs, args)],
                                       [small[2], K], **kw)
        alone = A.Tracker(*small[:2]).ComputeSE3(*sargs, small[2], **kw)
        for got, want in ((one, r), (two[1], r), (two[0], alone)):
            assert all(np.array_equal(got[f], want[f]) for f in want), got


@pytest.mark.parametrize("rows", [1020, 1028])
def test_vertices_from_depth_and_from_the_map(gpu, rows):
    """a frame's iterations make its vertices from the depth where a pixel's row can be had by one
    multiplication (cols * cols * rows below 2^32), else read them: the pose is a tracker's on its maps"""
    cols = 2048
    K = (1600.0, 1600.0, cols / 2 - 0.5, rows / 2 - 0.5)
    sc = A.Scene(0, (4.0, 4.0, 3.0), 5)
    mp = dict(num_buckets=1 << 15, num_excess=1 << 15, num_blocks=1 << 15, voxel_size=0.02,
              trunc_dist=float(np.float32(0.02) * np.float32(4.0)), max_new_blocks=1 << 15)
    s = A.System(A.system_params(cols=cols, rows=rows, K=K, map=mp))
    print("vertices of a frame", cols, rows, flush=True)
    s.GrabImage(*A.to_device(*sc.render(0, cols, rows, K)))
    s.GrabImage(*A.to_device(*sc.render(1, cols, rows, K)))
    pose = s.result()["pose"]
    model = [(s.view("model_vmap").clone(), s.view("model_nmap").clone())]
    for _ in range(2):
        model.append(A.ResizeMap(*model[-1]))
    s.GrabImage(*A.to_device(*sc.render(2, cols, rows, K)))
    r = s.result()
    assert r["track_status"] in (1, 4) and not np.array_equal(r["pose"], pose)
    t = A.Tracker(cols, rows)
    t.set_last_pose(pose)
    p = s.params
    got = t.ComputeSE3([s.view("vmap", l) for l in range(3)], [s.view("nmap", l) for l in range(3)],
                       [m[0] for m in model], [m[1] for m in model], K, iters=tuple(p.iters), min_count=tuple(p.min_count),
                       thresh=p.icp_thresh)
    assert np.array_equal(got["pose"], r["pose"])
    s.close()
