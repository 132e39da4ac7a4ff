"""Allocation's two ways of naming a ray's blocks (offsets from the camera's block, and whole keys
for rays that leave their range) and its per-lane queue: the block set is the oracle's for bands of
one to many blocks, near and beyond the offsets' range, and coordinates past the key range are
flagged."""
import numpy as np
import pytest
import torch

from fusion_amd import api as A
from oracle import binding as O
from tests.helpers import rows_set

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("voxel,trunc,shift", [
    (0.02, 3.0, 0.0),      # one or two blocks per ray
    (0.005, 8.0, 0.0),     # a band as long as a block
    (0.002, 100.0, 0.0),   # more blocks per ray than the queue holds
    (0.0005, 40.0, 0.0),   # 500 blocks are 2 m: depths on both sides
    (0.02, 3.0, -3000.0),  # negative block coordinates far from the origin
])
def test_block_set(gpu, voxel, trunc, shift):
    cols, rows = 61, 47
    K = (60.0, 60.0, 30.0, 23.0)
    print("alloc: voxel %g trunc %g shift %g" % (voxel, trunc, shift), flush=True)
    rng = np.random.default_rng(1)
    depth = rng.uniform(0.5, 2.9, (rows // 4 + 1, cols // 4 + 1)).repeat(4, 0).repeat(4, 1)[:rows, :cols].astype(np.float32)
    depth[rng.random(depth.shape) < 0.1] = np.nan
    rgb = np.zeros((rows, cols, 3), np.uint8)
    nm = np.full((rows, cols, 4), np.nan, np.float32)
    pose = np.eye(4)
    pose[:3, 3] = (shift, 0.3, -shift)
    p = dict(num_buckets=1 << 17, num_excess=1 << 17, num_blocks=1 << 17, voxel_size=float(np.float32(voxel)),
             trunc_dist=float(np.float32(voxel) * np.float32(trunc)))
    o = O.Map(**p)
    o.fuse_map_color(depth, rgb, nm, pose, K)
    g = A.Mapping(**p, max_new_blocks=1 << 17)
    g.FuseMapColor(torch.from_numpy(depth).cuda(), torch.from_numpy(rgb).cuda(), torch.from_numpy(nm).cuda(), pose, K)
    ob = o.export_blocks()
    assert len(ob) > 50 and rows_set(g.export_blocks()) == rows_set(ob)
    assert g.stats()["flags"] == 0


@pytest.mark.parametrize("blocks_from_limit", [2, -600])
def test_key_range_is_flagged(gpu, blocks_from_limit):
    """a camera at the key range's end (2^20 blocks): blocks past it are skipped and flagged, by
    rays within the offsets' range and beyond it"""
    voxel = 0.01
    d = torch.full((16, 16), 1.0, dtype=torch.float32, device="cuda")
    pose = np.eye(4)
    pose[2, 3] = ((1 << 20) - blocks_from_limit) * 8 * voxel
    g = A.Mapping(num_buckets=64, num_excess=64, num_blocks=64, voxel_size=voxel, trunc_dist=0.03, max_new_blocks=64)
    g.FuseMapColor(d, torch.zeros((16, 16, 3), dtype=torch.uint8, device="cuda"),
                   torch.full((16, 16, 4), float("nan"), device="cuda"), pose, (20.0, 20.0, 8.0, 8.0))
    assert g.stats()["flags"] & 8 and g.stats()["n_allocated"] == 0


def test_key_range_is_flagged_by_rays_past_a_full_set(gpu):
    """rays spread over a block each per pixel and ten in depth fill the tile's set before any of them
    leaves the key range, so every block past it is one that found no slot"""
    voxel, n = 0.01, 16
    d = torch.full((n, n), 2.5, dtype=torch.float32, device="cuda")
    pose = np.eye(4)
    pose[2, 3] = (1 << 20) * 8 * voxel - 2.8
    g = A.Mapping(num_buckets=1 << 14, num_excess=1 << 13, num_blocks=1 << 14, voxel_size=voxel, trunc_dist=0.72,
                  max_new_blocks=1 << 14)
    print("alloc: full set at the key range's end", flush=True)
    g.FuseMapColor(d, torch.zeros((n, n, 3), dtype=torch.uint8, device="cuda"),
                   torch.full((n, n, 4), float("nan"), device="cuda"), pose, (25.0, 25.0, 7.5, 7.5))
    z = g.export_blocks()[:, 2]
    assert len(z) > 2000 and z.min() < (1 << 20) - 8 and z.max() == (1 << 20) - 1
    assert g.stats()["flags"] == 8


def test_rays_where_a_step_rounds_up(gpu):
    """past 2^23 voxels a march's step of just over half a voxel rounds to a whole one, so the ray ends
    as far again behind its band, beyond the offsets' range; it takes no block of the key range"""
    voxel = 0.01
    pose = np.eye(4)
    pose[:3, :3] = [[0, 0, 1], [0, 1, 0], [-1, 0, 0]]  # looking along x
    pose[0, 3] = ((1 << 20) - 470) * 8 * voxel
    g = A.Mapping(num_buckets=1 << 10, num_excess=1 << 10, num_blocks=1 << 10, voxel_size=voxel, trunc_dist=2.24,
                  depth_max=50.0, max_new_blocks=1 << 10)
    print("alloc: steps that round up", flush=True)
    g.FuseMapColor(torch.full((1, 1), 484 * 8 * voxel, device="cuda"),
                   torch.zeros((1, 1, 3), dtype=torch.uint8, device="cuda"),
                   torch.full((1, 1, 4), float("nan"), device="cuda"), pose, (525.0, 525.0, 0.0, 0.0))
    assert len(g.export_blocks()) == 0 and g.stats()["flags"] == 8
