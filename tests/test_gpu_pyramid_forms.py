"""The pyramid kernels at the edges of their tiles and windows against the CPU oracle, bit for bit.

The filter works on 16x16 tiles, the halvings and the derivative take a wave's whole windows and
its clipped ones apart: images below one tile, one sample over or under a tile, and of odd sizes,
with noise, holes and depths beyond the cutoff.
"""
import numpy as np
import pytest
import torch

from fusion_amd import api as A
from oracle import binding as O
from tests.helpers import mismatch, same_bits

pytestmark = pytest.mark.gpu

SIZES = [(2, 2), (3, 5), (4, 4), (31, 15), (32, 16), (33, 17), (36, 20), (37, 21), (65, 64), (71, 83), (131, 37)]


def _depth(cols, rows):
    rng = np.random.default_rng(cols * 1000 + rows)
    d = (7000 + 900 * rng.standard_normal((rows, cols))).astype(np.uint16)
    d[rng.random((rows, cols)) < 0.1] = 0
    d[rng.random((rows, cols)) < 0.1] = 60000
    return d


@pytest.mark.parametrize("cols,rows", SIZES)
def test_depth_forms_bit_exact(gpu, cols, rows):
    print("depth forms %dx%d" % (cols, rows), flush=True)
    d = _depth(cols, rows)
    raw, f0 = A.FilterDepth(torch.from_numpy(d.view(np.int16)).cuda(), 5000.0, 3.0)
    oraw, of0 = O.filter_depth(d, 5000.0, 3.0)
    assert same_bits(raw.cpu().numpy(), oraw), mismatch(raw.cpu().numpy(), oraw)
    assert same_bits(f0.cpu().numpy(), of0), mismatch(f0.cpu().numpy(), of0)
    for src in (of0, oraw):  # the raw depth has the holes beyond the cutoff
        g = A.PyrDownGauss(torch.from_numpy(src).cuda()).cpu().numpy()
        o = O.pyrdown_gauss(src)
        assert same_bits(g, o), mismatch(g, o)


@pytest.mark.parametrize("cols,rows", SIZES)
def test_image_forms_bit_exact(gpu, cols, rows):
    print("image forms %dx%d" % (cols, rows), flush=True)
    rng = np.random.default_rng(cols * 1000 + rows)
    img = rng.integers(0, 256, size=(rows, cols), dtype=np.uint8)
    img[: rows // 2][rng.random((rows // 2, cols)) < 0.5] = 255
    t = torch.from_numpy(img).cuda()
    if min(cols, rows) >= 4:  # smaller images are refused
        assert np.array_equal(A.PyrDownGaussU8(t).cpu().numpy(), O.pyrdown_u8(img))
    dx, dy = A.ComputeDerivativeImage(t)
    ox, oy = O.derivative_image(img)
    assert np.array_equal(dx.cpu().numpy(), ox)
    assert np.array_equal(dy.cpu().numpy(), oy)


@pytest.mark.parametrize("cols,rows", [(32, 32), (36, 44), (100, 68), (128, 64)])
def test_frame_pyramid_equals_the_single_operations(gpu, cols, rows):
    # a session's frame makes its maps in launches of its own, level by level; the model maps of a
    # frame are those of the raycast before it, halved
    print("frame %dx%d" % (cols, rows), flush=True)
    K = (0.9 * cols, 0.9 * cols, cols / 2 - 0.5, rows / 2 - 0.5)
    rng = np.random.default_rng(cols)
    y, x = np.mgrid[0:rows, 0:cols]
    mp = dict(num_buckets=1 << 14, num_excess=1 << 13, num_blocks=1 << 13, voxel_size=0.02, trunc_dist=0.06,
              max_new_blocks=1 << 14)
    s = A.System(A.system_params(cols=cols, rows=rows, K=K, map=mp))
    bits = lambda t: t.cpu().numpy()
    for k in range(2):
        d = (5000 * (1.2 + 0.002 * x + 0.003 * y) + 5 * rng.standard_normal((rows, cols))).astype(np.uint16)
        d[rng.random((rows, cols)) < 0.02] = 0
        rgb = rng.integers(0, 256, (rows, cols, 3), dtype=np.uint8)
        last = [s.view("model_vmap").clone(), s.view("model_nmap").clone()]
        s.GrabImage(*A.to_device(d, rgb))
        torch.cuda.synchronize()
        raw, f = A.FilterDepth(torch.from_numpy(d.view(np.int16)).cuda(), s.params.depth_scale, s.params.depth_cutoff)
        assert same_bits(bits(s.view("raw")), bits(raw))
        for l in range(3):
            f = A.PyrDownGauss(f) if l else f
            v = A.ComputeVMap(f, *A.level_k(K, l), s.params.depth_cutoff)
            assert same_bits(bits(s.view("depth", l)), bits(f)), l
            assert same_bits(bits(s.view("vmap", l)), bits(v)), l
            assert same_bits(bits(s.view("nmap", l)), bits(A.ComputeNMap(v))), l
        for l in (1, 2):
            if k:
                last = A.ResizeMap(*last)
                assert same_bits(bits(s.view("model_vmap", l)), bits(last[0])), l
                assert same_bits(bits(s.view("model_nmap", l)), bits(last[1])), l
    s.close()
