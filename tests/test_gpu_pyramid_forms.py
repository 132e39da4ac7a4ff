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
