"""Stencils read row by row on the x-fastest layout and inside vdb leaves: volumes
whose rows are as short as a stencil, odd row lengths (rows then start at every
alignment of the element), points on and beyond the faces, every element type.
Linear samples and gradients are bit-identical to the oracle; tricubic samples
are within 1e-5 of the field scale (the bar of test_gpu_dense.py)."""
import numpy as np
import pytest

import oracle as O
import openvkl_amd as vkl
from tests import volumes as V
from tests.test_gpu_dense import assert_same, check_cubic

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

TYPES = [np.uint8, np.int16, np.uint16, np.float16, np.float32, np.float64]


@pytest.mark.parametrize("dtype", TYPES, ids=[np.dtype(t).name for t in TYPES])
@pytest.mark.parametrize("dims", [(2, 2, 2), (4, 4, 4), (5, 7, 6), (33, 3, 9)])
def test_row_stencils(device, dims, dtype):
    rng = np.random.default_rng(11)
    data = rng.uniform(0, 100, dims[::-1]).astype(dtype)
    vol, grid = device.structured_regular(data), O.Grid.dense(data)
    hi = np.array(dims, np.float32) - 1
    pts = np.concatenate([V.uniform_points(4000, (0, 0, 0), hi), V.uniform_points(1000, (-2, -2, -2), hi + 2),
                          rng.integers(-1, 34, (500, 3)).astype(np.float32)]).astype(np.float32)
    d = torch.from_numpy(pts).cuda()
    s = vol.sampler(filter=vkl.VKL_FILTER_LINEAR)
    grid.set_sampler(O.LINEAR)
    assert_same(s.sample(d).cpu().numpy(), grid.sample(pts))
    assert_same(s.gradient(d).cpu().numpy(), grid.gradient(pts))
    s = vol.sampler(filter=vkl.VKL_FILTER_CUBIC)
    grid.set_sampler(O.CUBIC)
    inside = pts[np.isfinite(grid.sample(pts))]
    if len(inside):
        check_cubic(grid, s.sample(torch.from_numpy(inside).cuda()).cpu().numpy(), inside)


@pytest.mark.parametrize("dtype", [np.float16, np.float32], ids=["float16", "float32"])
def test_leaf_rows(device, dtype):
    """Every cell position of a leaf, the ones across its faces among them."""
    rng = np.random.default_rng(12)
    origins = np.array([[0, 0, 0], [8, 0, 0], [0, 8, 0], [8, 8, 8], [24, 0, 0]], np.int32)
    leaves = rng.uniform(0, 1, (len(origins), 512)).astype(dtype)
    n = len(origins)
    kw = dict(packed_dense=[leaves.reshape(-1)])
    level, fmt = np.full(n, 3, np.uint32), np.ones(n, np.uint32)
    vol = device.vdb(level, origins, fmt, **kw)
    grid = O.Grid.vdb(level, origins, fmt, **kw)
    k = np.stack(np.meshgrid(np.arange(33), np.arange(17), np.arange(17), indexing="ij"), -1).reshape(-1, 3)
    pts = (k + rng.uniform(0, 0.999, k.shape)).astype(np.float32)
    d = torch.from_numpy(pts).cuda()
    s = vol.sampler(filter=vkl.VKL_FILTER_LINEAR)
    grid.set_sampler(O.LINEAR)
    assert_same(s.sample(d).cpu().numpy(), grid.sample(pts))
    assert_same(s.gradient(d).cpu().numpy(), grid.gradient(pts))


def test_cell_of_special_coordinates(device):
    """Cells of coordinates where float -> int conversion is special: signed
    zeros and subnormals, halves, integers, the ends of the int range, infinities
    and NaN."""
    big = [2.0 ** 31, -2.0 ** 31, 2147483520.0, -2147483904.0, 3e38, -3e38, np.inf, -np.inf, np.nan]
    small = [0.0, -0.0, 1e-45, -1e-45, 1.2e-38, -1.2e-38, 0.5, -0.5, 1.0, -1.0, 0.99999994, -0.99999994, 2.5, 6.0]
    axis = np.array(big + small, np.float32)
    data = np.random.default_rng(3).uniform(-1, 1, (7, 7, 7)).astype(np.float32)
    kw = dict(origin=(0, 0, 0), background=5.0)
    vol, grid = device.structured_regular(data, **kw), O.Grid.dense(data, **kw)
    pts = np.full((3 * len(axis) + len(axis) ** 2, 3), 2.25, np.float32)
    for a in range(3):
        pts[a * len(axis):(a + 1) * len(axis), a] = axis
    pts[3 * len(axis):, 0], pts[3 * len(axis):, 2] = np.repeat(axis, len(axis)), np.tile(axis, len(axis))
    d = torch.from_numpy(pts).cuda()
    for filt, ofilt in ((vkl.VKL_FILTER_NEAREST, O.NEAREST), (vkl.VKL_FILTER_LINEAR, O.LINEAR)):
        s = vol.sampler(filter=filt)
        grid.set_sampler(ofilt)
        assert_same(s.sample(d).cpu().numpy(), grid.sample(pts))
    assert_same(s.gradient(d).cpu().numpy(), grid.gradient(pts))
