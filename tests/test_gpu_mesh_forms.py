"""Marching cubes' case selection for every voxel format, over maps whose blocks span several
chunks of the triangle scan, against a dense numpy restatement of buildVertexList's tests
(MeshScene.cu:152-183) on the voxels read back; an empty map."""
import numpy as np
import pytest

from fusion_amd import api as A
from tests.helpers import scene_frames
from tests.test_gpu_map import _fuse_both

pytestmark = pytest.mark.gpu


def _cases(blocks, sdf):
    """{(x, y, z): cube} of the voxels that make triangles"""
    lo = blocks.min(0) * 8 - 2
    n = blocks.max(0) * 8 + 8 + 3 - lo
    vol = np.full(tuple(n[::-1]), np.nan, np.float32)  # z, y, x
    for b, s in zip(blocks, sdf):
        x, y, z = b * 8 - lo
        vol[z:z + 8, y:y + 8, x:x + 8] = s.reshape(8, 8, 8)
    nan = np.isnan(vol)
    bad, neg = nan | (vol == 1.0), vol < 0
    at = lambda a, dx, dy, dz: a[1 + dz:a.shape[0] - 2 + dz, 1 + dy:a.shape[1] - 2 + dy, 1 + dx:a.shape[2] - 2 + dx]
    corners = [(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)]
    ok, cube = True, 0
    for c, (dx, dy, dz) in enumerate(corners):
        ok = ok & ~at(bad, dx, dy, dz)
        for ex, ey, ez in ((1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1)):
            ok = ok & ~at(nan, dx + ex, dy + ey, dz + ez)
        cube = cube | at(neg, dx, dy, dz).astype(int) << c
    z, y, x = np.nonzero(ok & (cube > 0) & (cube < 255))
    return {tuple(k): int(v) for k, v in zip((np.stack([x, y, z], 1) + 1 + lo).tolist(), cube[z, y, x])}


@pytest.mark.parametrize("fmt,voxel,frames", [(0, 0.01, (0, 40, 80, 120, 160)), (1, 0.02, (0, 60)), (2, 0.02, (0, 60))])
def test_cases_of_every_format(gpu, fmt, voxel, frames):
    sc, K, fr = scene_frames(frames=frames, cols=320, rows=240)
    p = dict(num_buckets=1 << 16, num_excess=1 << 16, num_blocks=1 << 16, voxel_size=voxel,
             trunc_dist=float(np.float32(voxel) * np.float32(3.0)), max_new_blocks=1 << 16)
    g, _ = _fuse_both(p, fr, [sc.pose(f) for f in frames], K, fmt=fmt)
    blocks = g.export_blocks()
    print("mesh cases: format %d, %d blocks" % (fmt, len(blocks)), flush=True)
    if voxel == 0.01:
        assert len(blocks) > 2 * 2048  # three chunks of the scan
    want = _cases(blocks, g.read_blocks(blocks)[0])
    meta = g.MeshScene(max_triangles=2_000_000, with_meta=True)[3].cpu().numpy()
    keys = [tuple(r) for r in meta.tolist()]
    assert len(keys) == len(set(keys)) > 1000  # each triangle once: none overwritten
    assert {(x, y, z): c >> 4 for x, y, z, c in keys} == want
    last = {}
    for x, y, z, c in keys:  # a voxel's triangles are numbered 0, 1, ...
        assert c & 15 == last.get((x, y, z), -1) + 1
        last[(x, y, z)] = c & 15


def test_empty_map(gpu):
    g = A.Mapping(num_buckets=64, num_excess=64, num_blocks=64, voxel_size=0.01, trunc_dist=0.03, max_new_blocks=64)
    for _ in range(2):
        v, n, c, meta = g.MeshScene(max_triangles=10, with_meta=True)
        assert v.shape[0] == 0 and g.stats()["n_triangles"] == 0
