"""The work-group forms of an ICP iteration: a quarter of a 2048-pixel chunk, a chunk, and the
chunk loop per work-group.  The sums at the sizes where the form changes (1, 128 and 129 chunks,
a chunk that is not full) against the FP64 oracle, ICP and photometric."""
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
