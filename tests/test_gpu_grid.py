"""The block grid in front of the hash table: maps whose blocks share grid cells (the same view
fused again a whole grid away, so that every cell of the second is taken) and maps outside the
grid's range take the hash table, with the oracle's raycast and mesh bit for bit; so does a map
loaded from a snapshot, whose grid is rebuilt."""
import numpy as np
import pytest

from fusion_amd import api as A
from tests.helpers import same_bits, scene_frames
from tests.test_gpu_map import _compare_maps, _fuse_both
from tests.test_gpu_render import _mesh_dict

pytestmark = pytest.mark.gpu
VOX = 0.02
CELLS = 32  # per axis, for maps of up to 2048 blocks


@pytest.mark.parametrize("axis,shift", [(0, CELLS * 8 * VOX), (1, -CELLS * 8 * VOX), (2, 2 * CELLS * 8 * VOX),
                                        (0, 600 * CELLS * 8 * VOX), (1, -600 * CELLS * 8 * VOX)])
def test_shared_cells_and_outside_the_grid(gpu, tmp_path, axis, shift):
    cols, rows = 160, 120
    sc, K, fr = scene_frames(frames=(0,), cols=cols, rows=rows)
    there = sc.pose(0).copy()
    there[axis, 3] += shift
    p = dict(num_buckets=1 << 10, num_excess=1 << 12, num_blocks=1 << 11, voxel_size=VOX,
             trunc_dist=float(np.float32(VOX) * np.float32(3.0)), max_new_blocks=1 << 12)
    g, o = _fuse_both(p, [fr[0], fr[0]], [sc.pose(0), there], K)
    n = _compare_maps(g, o)
    print("grid: axis %d shift %g, %d blocks" % (axis, shift, n), flush=True)
    assert 200 < n < 2048
    path = str(tmp_path / "m")
    g.save(path)
    h = A.Mapping(**p)
    h.load(path)
    for m in (g, h):
        for pose in (sc.pose(0), there):
            nv = m.CheckBlockVisibility(pose, cols, rows, K, 3.0, 0.1)
            assert nv == o.check_visibility(pose, cols, rows, K, 3.0, 0.1) > 50
            zg = m.CreateRenderingBlocks(20, 15, pose, nv, K)
            zo = o.create_rendering_blocks(20, 15, pose, nv, K)
            vg, ng = m.Raycast(cols, rows, zg[0], zg[1], pose, K)
            vo, no = o.raycast(cols, rows, zo[0], zo[1], pose, K)
            assert same_bits(vg.cpu().numpy(), vo) and same_bits(ng.cpu().numpy(), no)
            if abs(shift) < 100:
                assert np.isfinite(vo[..., 0]).mean() > 0.3
        v, nm, c, meta = (x.cpu().numpy() for x in m.MeshScene(max_triangles=1_000_000, with_meta=True))
        vo, no, co, mo, total = o.mesh()
        assert meta.shape[0] == total > 500
        dg, do = _mesh_dict(v, nm, c, meta), _mesh_dict(vo, no, co, mo)
        assert set(dg) == set(do)
        assert all(same_bits(dg[k][0], do[k][0]) and same_bits(dg[k][1], do[k][1]) for k in do)


def test_many_periods(gpu, tmp_path):
    """the same view at places whole periods apart: all but the first place's blocks go to the grid's
    second part, where some meet and are left to the hash table"""
    cols, rows = 128, 96
    sc, K, fr = scene_frames(frames=(0,), cols=cols, rows=rows)
    period = 2 * CELLS * 8 * VOX  # of maps of up to 2^14 blocks
    poses = []
    for x, y, z in ((0, 0, 0), (1, 0, 0), (0, 1, 0), (-1, 2, 0), (0, 0, 3), (5, -4, 1), (-2, -2, -2)):
        poses.append(sc.pose(0).copy())
        poses[-1][:3, 3] += np.array([x, y, z]) * period
    p = dict(num_buckets=1 << 13, num_excess=1 << 12, num_blocks=1 << 14, voxel_size=VOX,
             trunc_dist=float(np.float32(VOX) * np.float32(3.0)), max_new_blocks=1 << 14)
    g, o = _fuse_both(p, [fr[0]] * len(poses), poses, K)
    n = _compare_maps(g, o)
    print("grid: %d blocks of %d places" % (n, len(poses)), flush=True)
    assert 3000 < n < 1 << 14
    path = str(tmp_path / "m")
    g.save(path)
    h = A.Mapping(**p)
    h.load(path)
    for m in (g, h):
        for pose in poses:
            nv = m.CheckBlockVisibility(pose, cols, rows, K, 3.0, 0.1)
            assert nv == o.check_visibility(pose, cols, rows, K, 3.0, 0.1) > 50
            zg = m.CreateRenderingBlocks(16, 12, pose, nv, K)
            zo = o.create_rendering_blocks(16, 12, pose, nv, K)
            vg, ng = m.Raycast(cols, rows, zg[0], zg[1], pose, K)
            vo, no = o.raycast(cols, rows, zo[0], zo[1], pose, K)
            assert same_bits(vg.cpu().numpy(), vo) and same_bits(ng.cpu().numpy(), no)
            assert np.isfinite(vo[..., 0]).mean() > 0.3
        v, nm, c, meta = (x.cpu().numpy() for x in m.MeshScene(max_triangles=1_000_000, with_meta=True))
        vo, no, co, mo, total = o.mesh()
        assert meta.shape[0] == total > 500
        dg, do = _mesh_dict(v, nm, c, meta), _mesh_dict(vo, no, co, mo)
        assert set(dg) == set(do)
        assert all(same_bits(dg[k][0], do[k][0]) and same_bits(dg[k][1], do[k][1]) for k in do)
