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


@pytest.mark.parametrize("dims", [(2, 2, 2), (4, 4, 4), (5, 7, 6), (33, 3, 9)])
@pytest.mark.parametrize("background", [float("nan"), 37.5])
def test_cubic_rows_at_the_faces(device, dims, background):
    """Tricubic samples and gradients where stencils reach across a face: the
    background enters there as it does in the oracle, NaN included."""
    data = np.random.default_rng(13).uniform(0, 100, dims[::-1]).astype(np.float32)
    vol, grid = device.structured_regular(data, background=background), O.Grid.dense(data, background=background)
    hi = np.array(dims, np.float32) - 1
    pts = np.concatenate([V.uniform_points(4000, (0, 0, 0), hi), V.uniform_points(1000, (-2, -2, -2), hi + 2)])
    d = torch.from_numpy(pts).cuda()
    s = vol.sampler(filter=vkl.VKL_FILTER_CUBIC, gradient_filter=vkl.VKL_FILTER_CUBIC)
    grid.set_sampler(O.CUBIC, gradient_filter=O.CUBIC)
    for gradient in (False, True):
        got = (s.gradient if gradient else s.sample)(d).cpu().numpy()
        want = (grid.gradient if gradient else grid.sample)(pts)
        np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
        if not np.isnan(want).all():
            check_cubic(grid, got, pts, gradient=gradient)


def test_row_offsets_above_2_gib(device):
    """Row offsets are 32-bit byte offsets up to 4 GiB: a uint8 volume of just
    less. The lerps of 8 bytes round 3 times each way, below 255 * 2e-6."""
    nx, ny, nz = 2048, 2048, 1020
    data = torch.randint(0, 256, (nz, ny, nx), dtype=torch.uint8, device="cuda:0",
                         generator=torch.Generator(device="cuda:0").manual_seed(14))
    vol = device.structured_regular(data)
    g = torch.Generator(device="cuda:0").manual_seed(15)
    p = torch.rand((20000, 3), device="cuda:0", generator=g) * torch.tensor([nx - 1.0, ny - 1.0, nz - 1.0], device="cuda:0")
    p[:5000, 2] = (nz - 1.0) - torch.rand(5000, device="cuda:0", generator=g) * 3.0
    i = torch.floor(p).long()
    f = (p - i).double()
    flat, want = data.reshape(-1), 0.0
    for c in range(8):
        k = torch.minimum(i + torch.tensor([c >> 2, (c >> 1) & 1, c & 1], device="cuda:0"),
                          torch.tensor([nx - 1, ny - 1, nz - 1], device="cuda:0"))
        w = [f[:, a] if (c >> (2 - a)) & 1 else 1 - f[:, a] for a in range(3)]
        want = want + w[0] * w[1] * w[2] * flat[(k[:, 2] * ny + k[:, 1]) * nx + k[:, 0]].double()
    assert int(((i[:, 2] * ny + i[:, 1]) * nx).max()) > 1 << 31
    got = vol.sampler(filter=vkl.VKL_FILTER_LINEAR).sample(p.contiguous()).double()
    assert float((got - want).abs().max()) < 1e-3
