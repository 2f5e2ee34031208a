"""Interval and hit iteration where a lane's walk takes its rarer turns: rays
along an axis (zero direction components of both signs) and on cell planes,
leaves beside tiles on every level, undefined voxels inside a march (the NaN
retries), several iso values in one step, plateaus at an iso value, ranges that
end inside a cell, batches of one ray and of a wavefront and one. Bit-identical
to the oracle."""
import numpy as np
import pytest

import oracle as O
import openvkl_amd as vkl
from tests import volumes as V
from tests.test_gpu_iterators import compare_intervals, rays_through

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def dense_pair(device):
    rng = np.random.default_rng(21)
    data = V.procedural((45, 38, 51), lambda x, y, z: np.sin(0.4 * x) * np.cos(0.3 * y) + 0.02 * z)
    data[rng.random(data.shape) < 0.002] = np.nan
    data[10:20, 10:20, 10:20] = 0.25
    return device.structured_regular(data), O.Grid.dense(data)


def tiled_pair(device):
    rng = np.random.default_rng(22)
    k = np.stack(np.meshgrid(*[np.arange(6)] * 3, indexing="ij"), -1).reshape(-1, 3)
    leaf = k[rng.random(len(k)) < 0.4] * 8
    tile2 = np.array([[128, 0, 0], [0, 128, 128]])
    origins = np.concatenate([leaf, tile2, [[4096, 0, 0]]]).astype(np.int32)
    level = np.array([3] * len(leaf) + [2] * len(tile2) + [1], np.uint32)
    fmt = np.array([1] * len(leaf) + [0] * (len(tile2) + 1), np.uint32)
    dense = rng.uniform(0, 1, (len(leaf), 512)).astype(np.float32)
    dense[rng.random(dense.shape) < 0.002] = np.nan
    kw = dict(packed_dense=[dense.reshape(-1)], packed_tile=[np.array([0.4, 0.7, 0.2], np.float32)])
    return device.vdb(level, origins, fmt, **kw), O.Grid.vdb(level, origins, fmt, **kw)


def rays(box, count, seed):
    """Random rays towards the inner 150^3 of the box, and axis-aligned ones,
    some from integer coordinates."""
    lo, hi = np.asarray(box[:3]), np.minimum(np.asarray(box[3:]), np.asarray(box[:3]) + 150)
    org, d = rays_through(np.concatenate([lo, hi]).astype(np.float32), count, seed)
    rng = np.random.default_rng(seed + 1)
    for i in range(0, count, 3):
        axis, sign = rng.integers(3), rng.choice([-1.0, 1.0])
        o = np.floor(lo + rng.random(3) * (hi - lo)) if i % 2 else lo + rng.random(3) * (hi - lo)
        o[axis] = (lo if sign > 0 else hi)[axis] - 3.0 * sign
        org[i], d[i] = o, [0.0, -0.0, 0.0]
        d[i, axis] = sign
    return org, d


@pytest.mark.parametrize("which", ["dense", "tiled"])
@pytest.mark.parametrize("count", [1, 65, 400])
def test_hits(device, which, count):
    vol, grid = (dense_pair if which == "dense" else tiled_pair)(device)
    values = [0.25, 0.4, -0.3, 0.41]
    org, d = rays(grid.bounding_box(), count, 31)
    tr = np.tile(np.array([[2.3, 77.7]], np.float32), (count, 1))
    ctx = vol.sampler().hit_context(values)
    args = [torch.from_numpy(a).cuda() for a in (org, d, tr)]
    out, cnt = ctx.batch(args[0], args[1], t_ranges=args[2], max_per_ray=48)
    out, cnt = out.cpu().numpy(), cnt.cpu().numpy()
    for r in range(count):
        want = grid.hits(org[r], d[r], values, t_range=tr[r], max_out=48)
        assert cnt[r] == len(want), r
        np.testing.assert_array_equal(out[r, :cnt[r]].view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("which", ["dense", "tiled"])
@pytest.mark.parametrize("hint", [0.0, 0.25, 0.5, 1.0])
@pytest.mark.parametrize("ranges", [None, [[0.1, 0.2], [0.6, 0.9]]], ids=["all", "selected"])
def test_intervals(device, which, hint, ranges):
    vol, grid = (dense_pair if which == "dense" else tiled_pair)(device)
    org, d = rays(grid.bounding_box(), 130, 33)
    ctx = vol.sampler().interval_context(hint=hint, value_ranges=ranges)
    out, cnt = ctx.batch(torch.from_numpy(org).cuda(), torch.from_numpy(d).cuda(), max_per_ray=1024)
    compare_intervals((out.cpu().numpy(), cnt.cpu().numpy()), grid, org, d, O.map_depth(hint), value_ranges=ranges,
                      max_per_ray=1024)


@pytest.mark.parametrize("which", ["dense", "tiled"])
@pytest.mark.parametrize("entries", [1, 2, 256, 257, 1024, 1025])
def test_transfer_function_sizes(device, which, entries):
    """Interval rendering and Woodcock tracking with tables on both sides of
    the sizes that are staged in LDS."""
    vol, grid = (dense_pair if which == "dense" else tiled_pair)(device)
    org, d = rays(grid.bounding_box(), 200, 35)
    tf = np.random.default_rng(entries).random((entries, 4), dtype=np.float32)
    tf[:, 3] *= 0.2
    rng = (-0.5, 1.25)
    s = vol.sampler()
    grid.set_sampler(O.LINEAR)
    o, dd, t = (torch.from_numpy(a).cuda() for a in (org, d, tf))
    got, cnt = s.interval_context().ray_march(o, dd, t, rng)
    want, wcnt = grid.ray_march_intervals(org, d, tf, rng)
    np.testing.assert_array_equal(cnt.cpu().numpy().view(np.uint32), wcnt)
    np.testing.assert_array_equal(got.cpu().numpy().view(np.uint32), want.view(np.uint32))
    tr = np.tile(np.array([[0.0, 120.0]], np.float32), (200, 1))
    state = np.stack([np.full(200, 7, np.uint32), np.arange(200, dtype=np.uint32)], 1)
    ev, sm, n = s.woodcock(o, dd, torch.from_numpy(tr).cuda(), torch.from_numpy(state.view(np.int32)).cuda(), 0.5, t, rng)
    wev, wsm, wn = grid.woodcock(org, d, tr, state.copy(), 0.5, tf, rng)[:3]
    for a, b in ((ev, wev), (sm, wsm)):
        a, b = a.cpu().numpy(), np.asarray(b, np.float32)
        assert ((a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b))).all()
    np.testing.assert_array_equal(n.cpu().numpy().view(np.uint32), np.asarray(wn, np.uint32))


def far_rays(box, count, seed):
    """Rays from 150 voxels away through the inside of the box, so that the
    walk's accumulated t differs from the box exit's on many of them."""
    rng = np.random.default_rng(seed)
    lo, hi = np.asarray(box[:3], np.float64), np.asarray(box[3:], np.float64)
    out = rng.standard_normal((count, 3))
    org = (lo + hi) / 2 + 150.0 * out / np.linalg.norm(out, axis=1, keepdims=True)
    d = lo + rng.random((count, 3)) * (hi - lo) - org
    return org.astype(np.float32), (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)


@pytest.mark.parametrize("dims", [(45, 38, 51), (9, 64, 23), (40, 48, 33)])
@pytest.mark.parametrize("cell_centered", [True, False])
def test_intervals_end_at_the_upper_faces(device, dims, cell_centered):
    """Every voxel an interval, upper faces inside an 8^3 block: a walk that
    steps over one has left the volume, in the batch, the plan and the per-ray
    calls."""
    data = np.random.default_rng(41).uniform(0, 1, dims[::-1]).astype(np.float32)
    vol = device.structured_regular(data, cell_centered=cell_centered)
    grid = O.Grid.dense(data, cell_centered=cell_centered)
    org, d = far_rays(grid.bounding_box(), 1000, 42)
    ctx = vol.sampler().interval_context(hint=1.0)
    o, dd = torch.from_numpy(org).cuda(), torch.from_numpy(d).cuda()
    out, cnt = (a.cpu().numpy() for a in ctx.batch(o, dd, max_per_ray=256))
    compare_intervals((out, cnt), grid, org, d, O.map_depth(1.0), max_per_ray=256)
    plan = vkl.RayBatchPlan(device, [(ctx, o, dd, 256)])
    plan.execute()
    torch.cuda.synchronize()
    res, n = plan.results[0].cpu().numpy(), plan.counts[0].cpu().numpy()
    plan.release()
    np.testing.assert_array_equal(n, cnt)
    for r in range(len(org)):
        np.testing.assert_array_equal(res[r, :n[r]].view(np.uint32), out[r, :n[r]].view(np.uint32))
    for r in range(0, len(org), 125):
        np.testing.assert_array_equal(ctx.intervals(org[r], d[r]).view(np.uint32), out[r, :cnt[r]].view(np.uint32))


@pytest.mark.parametrize("which", ["dense", "tiled"])
@pytest.mark.parametrize("hint", [0.5, 1.0])
@pytest.mark.parametrize("count", [1, 2, 3, 9, 40])
def test_many_value_ranges(device, which, hint, count):
    """Selectors of one to many ranges, in any order, overlapping ones among
    them, values below, between and above all of them."""
    vol, grid = (dense_pair if which == "dense" else tiled_pair)(device)
    rng = np.random.default_rng(43 + count)
    lo = rng.uniform(0.05, 0.8, count)
    ranges = np.stack([lo, lo + rng.uniform(0.001, 0.03, count)], 1).astype(np.float32)
    org, d = rays(grid.bounding_box(), 130, 44)
    ctx = vol.sampler().interval_context(hint=hint, value_ranges=ranges)
    out, cnt = ctx.batch(torch.from_numpy(org).cuda(), torch.from_numpy(d).cuda(), max_per_ray=1024)
    compare_intervals((out.cpu().numpy(), cnt.cpu().numpy()), grid, org, d, O.map_depth(hint), value_ranges=ranges,
                      max_per_ray=1024)


@pytest.mark.parametrize("missing", [300, 520])
def test_tables_beside_rays_that_miss(device, missing):
    """Whole wavefronts and workgroups whose rays all miss, which do not stage
    the table, before ones that do, and part-filled last ones."""
    vol, grid = dense_pair(device)
    org, d = rays(grid.bounding_box(), missing + 200, 45)
    d[:missing] = -d[:missing]
    tf = np.random.default_rng(46).random((64, 4), dtype=np.float32)
    tf[:, 3] *= 0.2
    rng = (-0.5, 1.25)
    s = vol.sampler()
    grid.set_sampler(O.LINEAR)
    o, dd, t = (torch.from_numpy(a).cuda() for a in (org, d, tf))
    got, cnt = s.interval_context().ray_march(o, dd, t, rng)
    want, wcnt = grid.ray_march_intervals(org, d, tf, rng)
    assert (wcnt[:missing] == 0).mean() > 0.9 and wcnt[missing:].max() > 0
    np.testing.assert_array_equal(cnt.cpu().numpy().view(np.uint32), wcnt)
    np.testing.assert_array_equal(got.cpu().numpy().view(np.uint32), want.view(np.uint32))
    n = len(org)
    tr = np.tile(np.array([[0.0, 120.0]], np.float32), (n, 1))
    tr[:missing] = [1.0, 0.0]
    state = np.stack([np.full(n, 7, np.uint32), np.arange(n, dtype=np.uint32)], 1)
    ev, sm, k = s.woodcock(o, dd, torch.from_numpy(tr).cuda(), torch.from_numpy(state.view(np.int32)).cuda(), 0.5, t, rng)
    wev, wsm, wk = grid.woodcock(org, d, tr, state.copy(), 0.5, tf, rng)[:3]
    for a, b in ((ev, wev), (sm, wsm)):
        a, b = a.cpu().numpy(), np.asarray(b, np.float32)
        assert ((a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b))).all()
    np.testing.assert_array_equal(k.cpu().numpy().view(np.uint32), np.asarray(wk, np.uint32))
