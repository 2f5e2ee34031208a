"""Performance cases of the sampling and traversal device.

Each case is one call that a program using the device makes, through the
public binding: point samples and gradients of structuredRegular and vdb
volumes, interval and hit iteration of many rays, and the fused renderers.

listed()            the cases that are timed by name
draw(rng)           one more case of the same ranges
prepare(case, seed) volume, sampler / iterator context and inputs on the GPU
run(state)          one pass; returns its outputs
work(case)          compulsory bytes and floating-point operations of a pass
exact(case, seed)   the outputs in binary64 by plain torch, where they have a
                    value that does not depend on where an iteration stops
"""
import ctypes
import math

import numpy as np
import torch

import openvkl_amd as vkl

FILTERS = {"nearest": vkl.VKL_FILTER_NEAREST, "linear": vkl.VKL_FILTER_LINEAR, "cubic": vkl.VKL_FILTER_CUBIC}
ELEMENT = {"u8": (torch.uint8, 1, 100.0, 30.0), "i16": (torch.int16, 2, 400.0, 300.0),
           "f16": (torch.float16, 2, 1.0, 0.4), "f32": (torch.float32, 4, 1.0, 0.4),
           "f64": (torch.float64, 8, 1.0, 0.4)}
DEV = "cuda:0"


def listed():
    return [
        # A picking or probe tool, or one tile of a host renderer: a few
        # thousand points, where the call itself is what counts.
        points("points_tile", (128, 128, 128), "f32", 4096),
        # The reference's own sampling benchmark: random points in a small
        # float volume in the caller's layout.
        points("points_1m", (128, 128, 128), "f32", 1 << 20),
        # Monte Carlo integration over a large volume that was laid out for
        # random points.
        points("points_64m_packed", (512, 512, 512), "f32", 1 << 26, packed=True),
        # Normals of a CT scan (16-bit, odd dimensions, anisotropic voxels) at
        # scattered surface points.
        points("gradients_ct", (413, 379, 211), "i16", (1 << 22) + 3, op="gradient", spacing=(0.75, 0.75, 1.25)),
        # Multi-planar reformatting: a tricubic oblique slice of a half volume.
        points("slice_cubic", (256, 240, 178), "f16", 2048 * 1031, filter="cubic", order="slice"),
        # A simulation with motion blur: four time steps per voxel, a time
        # per sample.
        points("motion_blur", (160, 144, 131), "f32", (1 << 20) + 77, steps=4),
        # Path-tracer collisions inside a sparse cloud.
        vdb("vdb_points", "points", 1024, "f32", count=1 << 23),
        # A renderer's interval traversal of a sparse cloud (empty-space
        # skipping), camera rays.
        vdb("vdb_intervals", "intervals", 1024, "f32", count=640 * 360, hint=0.5),
        # Iso-surface queries of incoherent (secondary) rays in a sparse
        # volume.
        vdb("vdb_hits", "hits", 1024, "f16", count=(1 << 17) + 5),
        # One frame of each volume renderer.
        frame("frame_march", "march", (512, 512, 512), "f32", 1920, 1080),
        frame("frame_hits", "shade", (300, 260, 340), "f32", 1920, 1080),
        frame("frame_woodcock", "woodcock", (384, 511, 400), "f16", 1920, 1080),
    ]


def points(name, dims, dtype, count, filter="linear", op="sample", order="random", packed=False, steps=0,
           spacing=(1.0, 1.0, 1.0)):
    return {"name": name, "kind": "points", "nx": dims[0], "ny": dims[1], "nz": dims[2], "dtype": dtype,
            "count": count, "filter": filter, "op": op, "order": order, "packed": packed, "steps": steps,
            "sx": spacing[0], "sy": spacing[1], "sz": spacing[2]}


def vdb(name, what, res, dtype, count, hint=0.5, filter="linear", op="sample"):
    return {"name": name, "kind": "vdb", "what": what, "res": res, "dtype": dtype, "count": count, "hint": hint,
            "filter": filter, "op": op}


def frame(name, what, dims, dtype, width, height):
    return {"name": name, "kind": "frame", "what": what, "nx": dims[0], "ny": dims[1], "nz": dims[2],
            "dtype": dtype, "width": width, "height": height}


def log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["points", "points", "vdb", "frame"])
    if kind == "points":
        dims = [rng.randint(24, 420) for _ in range(3)]
        kw = {"filter": rng.choice(["nearest", "linear", "linear", "linear", "cubic"]),
              "op": rng.choice(["sample", "sample", "gradient"]), "order": rng.choice(["random", "slice"])}
        if kw["op"] == "gradient" and kw["filter"] == "nearest":
            kw["filter"] = "linear"
        if rng.random() < 0.25:
            dims = [min(d, 200) for d in dims]
            kw.update(steps=rng.randint(2, 5), filter="linear")
        elif kw["filter"] != "cubic" and rng.random() < 0.25:
            kw["packed"] = True
        most = 1 << (22 if kw["filter"] == "cubic" else 24)
        c = points("", dims, rng.choice(sorted(ELEMENT)), log_int(rng, 1000, most), **kw)
    elif kind == "vdb":
        what = rng.choice(["points", "intervals", "hits"])
        most = {"points": 1 << 23, "intervals": 1 << 18, "hits": 1 << 17}[what]
        c = vdb("", what, rng.choice([256, 384, 512, 768, 1024]), rng.choice(["f16", "f32"]),
                log_int(rng, 1000, most), hint=rng.choice([0.0, 0.25, 0.5, 1.0]),
                filter=rng.choice(["nearest", "linear", "linear"]))
        if what == "points":
            c["op"] = rng.choice(["sample", "sample", "gradient"])
            if rng.random() < 0.25:
                c["filter"], c["count"] = "cubic", min(c["count"], 1 << 21)
            if c["op"] == "gradient" and c["filter"] == "nearest":
                c["filter"] = "linear"
    else:
        what = rng.choice(["march", "shade", "woodcock"])
        w = log_int(rng, 160, 1920)
        c = frame("", what, [rng.randint(64, 400) for _ in range(3)], rng.choice(["u8", "i16", "f16", "f32"]), w,
                  rng.randint(max(w // 2, 90), w * 9 // 16 + 20))
    del c["name"]
    return c


# ---- inputs ---------------------------------------------------------------------------

def generator(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def uniform(g, *shape):
    return torch.rand(shape, device=DEV, generator=g)


def grid_field(case, seed):
    """Smooth structure of a few dozen voxels' wavelength plus 2 % noise, as
    simulations and scans hold it: [nz, ny, nx] (with time steps as the last,
    fastest axis) in the case's element type."""
    tdtype, _, mid, amp = ELEMENT[case["dtype"]]
    g = generator(seed)
    phase = (uniform(g, 4, 3) * (2 * math.pi)).cpu()
    freq = (0.04 + 0.16 * uniform(g, 4, 3)).cpu()
    axes = [torch.arange(n, device=DEV, dtype=torch.float32) for n in (case["nx"], case["ny"], case["nz"])]
    f = torch.zeros((case["nz"], case["ny"], case["nx"]), device=DEV)
    for k in range(4):
        wave = [torch.sin(axes[a] * float(freq[k, a]) + float(phase[k, a])) for a in range(3)]
        f += (0.6 ** k) * wave[2][:, None, None] * wave[1][None, :, None] * wave[0][None, None, :]
    f = f * 0.5 + 0.04 * (uniform(g, *f.shape) - 0.5)
    if case.get("steps"):
        t = torch.linspace(0.0, 1.0, case["steps"], device=DEV)
        f = f[..., None] * (1.0 - 0.5 * t) + 0.2 * t
    return (mid + amp * f).to(tdtype).contiguous()


def grid_points(case, seed):
    """[count, 3] object-space points: uniform over the volume, or the raster
    of an oblique slice through it."""
    g = generator(seed + 1)
    n = case["count"]
    ext = torch.tensor([(case["nx"] - 1) * case["sx"], (case["ny"] - 1) * case["sy"], (case["nz"] - 1) * case["sz"]],
                       device=DEV)
    if case["order"] == "random":
        return (uniform(g, n, 3) * (ext * 0.9999)).contiguous()
    width = max(1, int(math.sqrt(n)))
    i = torch.arange(n, device=DEV)
    u, v = (i % width) / width - 0.5, (i // width) / (n // width + 1) - 0.5
    tilt = 0.3 * (uniform(g, 3) - 0.5)
    unit = torch.stack([u + 0.1 * tilt[2] * v, v + tilt[0] * u, tilt[1] * u + tilt[2] * v], 1) * 0.75
    return ((unit + 0.5) * ext).contiguous()


def shell(case, seed):
    """Leaves of a cloudy sphere shell: origins [n, 3] int32 and voxels
    [n, 512] (z fastest), only the 8^3 cells that the shell touches."""
    res = case["res"]
    g = generator(seed)
    radius, width = 0.33 + 0.04 * float(uniform(g, 1)), 10.0 / res
    phase = (uniform(g, 3, 3) * (2 * math.pi)).cpu()
    c = res / 2.0
    mid = torch.arange(res // 8, device=DEV, dtype=torch.float32) * 8 + 4.0 - c
    r = torch.sqrt(mid[:, None, None] ** 2 + mid[None, :, None] ** 2 + mid[None, None, :] ** 2) / res
    origins = (torch.nonzero((r - radius).abs() < width + 7.0 / res) * 8).to(torch.int32)
    l8 = torch.arange(8, device=DEV, dtype=torch.float32)
    local = torch.stack([a.reshape(-1) for a in torch.meshgrid(l8, l8, l8, indexing="ij")], 1)
    tdtype = ELEMENT[case["dtype"]][0]
    leaves = torch.empty((origins.shape[0], 512), device=DEV, dtype=tdtype)
    for a in range(0, origins.shape[0], 1 << 16):
        p = origins[a:a + (1 << 16), None, :].float() + local[None]
        rr = torch.sqrt(((p - c) ** 2).sum(2)) / res
        noise = torch.zeros_like(rr)
        for k in range(3):
            w = torch.sin(p * (0.03 * 2 ** k) + phase[k].to(DEV))
            noise += 0.5 ** k * w[..., 0] * w[..., 1] * w[..., 2]
        leaves[a:a + (1 << 16)] = (torch.clamp(1.0 - (rr - radius).abs() / width, 0.0, 1.0) *
                                   (1.0 + 0.5 * noise)).to(tdtype)
    return origins, leaves


def leaf_points(case, origins, seed):
    g = generator(seed + 1)
    k = torch.randint(0, origins.shape[0], (case["count"],), device=DEV, generator=g)
    return (origins[k].float() + uniform(g, case["count"], 3) * 7.999).contiguous()


def camera(lo, hi, width, height, seed):
    """Row-major pinhole rays of a camera that looks at the box from outside:
    origins, unit directions and ranges clipped to the box (empty: (1, 0))."""
    g = generator(seed + 2)
    a, b = (uniform(g, 2) * 0.8 + 0.3).tolist()
    centre, size = [(l + h) / 2 for l, h in zip(lo, hi)], [h - l for l, h in zip(lo, hi)]
    view = np.array([math.cos(b) * math.sin(a), math.sin(b), math.cos(b) * math.cos(a)])
    eye = np.array(centre) + 1.3 * max(size) * view
    right = np.cross([0.0, 1.0, 0.0], view)
    right /= np.linalg.norm(right)
    up = np.cross(view, right)
    i = torch.arange(width * height, device=DEV)
    u = ((i % width).float() + 0.5) / width - 0.5
    v = (((i // width).float() + 0.5) / height - 0.5) * (height / width)
    to = [torch.tensor(x, device=DEV, dtype=torch.float32) for x in (right, up, -view)]
    d = u[:, None] * to[0] + v[:, None] * to[1] + to[2]
    d = (d / torch.linalg.norm(d, dim=1, keepdim=True)).contiguous()
    o = torch.tensor(eye, device=DEV, dtype=torch.float32).expand(width * height, 3).contiguous()
    t0 = (torch.tensor(lo, device=DEV) - o) / d
    t1 = (torch.tensor(hi, device=DEV) - o) / d
    near, far = torch.minimum(t0, t1).amax(1).clamp(min=0.0), torch.maximum(t0, t1).amin(1)
    hit = far > near
    tr = torch.stack([torch.where(hit, near, torch.ones_like(near)), torch.where(hit, far, torch.zeros_like(far))], 1)
    return o, d, tr.contiguous()


def crossing_rays(lo, hi, count, seed):
    """Incoherent rays: origins on a sphere around the box, towards uniform
    points inside it."""
    g = generator(seed + 2)
    lo, hi = torch.tensor(lo, device=DEV), torch.tensor(hi, device=DEV)
    out = torch.randn((count, 3), device=DEV, generator=g)
    out = out / torch.linalg.norm(out, dim=1, keepdim=True)
    o = (lo + hi) / 2 + out * (hi - lo).amax()
    d = lo + uniform(g, count, 3) * (hi - lo) - o
    return o.contiguous(), (d / torch.linalg.norm(d, dim=1, keepdim=True)).contiguous()


class State:
    """What the program holds between calls; gives the objects back at its end."""

    def __init__(self, case):
        self.case, self.owned = case, []
        self.device = self.own(vkl.Device("hip"))

    def own(self, obj):
        self.owned.append(obj)
        return obj

    def __del__(self):
        for obj in reversed(self.owned):
            obj.release()


MAX_INTERVALS, MAX_HITS = 64, 8


def prepare(case, seed):
    s = State(case)
    if case["kind"] == "vdb":
        origins, leaves = shell(case, seed)
        n = origins.shape[0]
        s.volume = s.own(s.device.vdb(np.full(n, 3, np.uint32), origins.cpu().numpy(), np.ones(n, np.uint32),
                                      packed_dense=[leaves.reshape(-1)]))
        s.sampler = s.own(s.volume.sampler(filter=FILTERS[case["filter"]]))
        if case["what"] == "points":
            s.points = leaf_points(case, origins, seed)
            s.out = torch.zeros((case["count"], 3) if case["op"] == "gradient" else (case["count"],), device=DEV)
            return s
        box = (0.0, 0.0, 0.0), (float(case["res"]),) * 3
        if case["what"] == "intervals":
            height = max(1, int(math.sqrt(case["count"] * 9 / 16)))
            s.org, s.dir, _ = camera(*box, -(-case["count"] // height), height, seed)
            s.org, s.dir = s.org[:case["count"]].contiguous(), s.dir[:case["count"]].contiguous()
            s.context = s.own(s.sampler.interval_context(hint=case["hint"], value_ranges=[[0.05, 10.0]]))
            s.call, slots, width = vkl.lib().vklIterateIntervalsBatch, MAX_INTERVALS, 5
        else:
            s.org, s.dir = crossing_rays(*box, case["count"], seed)
            s.context = s.own(s.sampler.hit_context([0.3, 0.8]))
            s.call, slots, width = vkl.lib().vklIterateHitsBatch, MAX_HITS, 3
        # Slots past a ray's count keep their zeros.
        s.slots = slots
        s.out = torch.zeros((s.org.shape[0], slots, width), device=DEV)
        s.counts = torch.zeros(s.org.shape[0], dtype=torch.int32, device=DEV)
        return s
    voxels = grid_field(case, seed)
    spacing = (case.get("sx", 1.0), case.get("sy", 1.0), case.get("sz", 1.0))
    kw = {}
    if case.get("steps"):
        kw = {"dims": (case["nx"], case["ny"], case["nz"]), "structured_steps": case["steps"]}
        voxels = voxels.reshape(-1)
    s.volume = s.own(s.device.structured_regular(voxels, spacing=spacing, corner_packed=case.get("packed") or None,
                                                 **kw))
    s.sampler = s.own(s.volume.sampler(filter=FILTERS[case.get("filter", "linear")]))
    if case["kind"] == "points":
        s.points = grid_points(case, seed)
        s.times = uniform(generator(seed + 3), case["count"]) if case["steps"] else None
        s.out = torch.zeros((case["count"], 3) if case["op"] == "gradient" else (case["count"],), device=DEV)
        return s
    hi = [float(case[a] - 1) for a in ("nx", "ny", "nz")]
    s.org, s.dir, s.ranges = camera((0.0, 0.0, 0.0), hi, case["width"], case["height"], seed)
    s.value_range = tuple(float(x) for x in s.volume.value_range())
    lo, up = s.value_range
    tf = uniform(generator(seed + 4), 64, 4)
    tf[:, 3] = torch.linspace(0.0, 0.03, 64, device=DEV)
    s.tf = tf
    if case["what"] == "march":
        s.context = s.own(s.sampler.interval_context(value_ranges=[[lo + 0.3 * (up - lo), up]]))
    elif case["what"] == "shade":
        s.context = s.own(s.sampler.hit_context([lo + 0.4 * (up - lo), lo + 0.65 * (up - lo)]))
    else:
        s.sigma = 0.25
        i = torch.arange(case["width"] * case["height"], dtype=torch.int32, device=DEV)
        s.rng = torch.stack([torch.full_like(i, seed & 0x7fffffff), i], 1).contiguous()
    return s


def run(s):
    case = s.case
    if case["kind"] == "points":
        f = s.sampler.gradient if case["op"] == "gradient" else s.sampler.sample
        return f(s.points, out=s.out, times=s.times)
    if case["kind"] == "vdb":
        if case["what"] == "points":
            return (s.sampler.gradient if case["op"] == "gradient" else s.sampler.sample)(s.points, out=s.out)
        s.call(ctypes.byref(s.context.h), s.org.shape[0], s.org.data_ptr(), s.dir.data_ptr(), None, None,
               s.out.data_ptr(), s.slots, s.counts.data_ptr())
        s.device.check()
        return s.out, s.counts
    if case["what"] == "march":
        return s.context.ray_march(s.org, s.dir, s.tf, s.value_range, t_ranges=s.ranges)
    if case["what"] == "shade":
        return s.context.render_hits(s.org, s.dir, s.tf, s.value_range, t_ranges=s.ranges)
    # The generator's states go on from call to call in a renderer; a pass
    # starts from the frame's first ones.
    rng = s.rng.clone()
    event, value, count = s.sampler.woodcock(s.org, s.dir, s.ranges, rng, s.sigma, s.tf, s.value_range)
    return event, value, count, rng


# ---- compulsory work --------------------------------------------------------------------

# Voxels of a stencil and operations of its evaluation.
STENCIL = {"nearest": 1, "linear": 8, "cubic": 64}
FLOPS = {"nearest": 18, "linear": 45, "cubic": 260}


def work(case):
    es = ELEMENT[case["dtype"]][1]
    if case["kind"] == "vdb":
        # Leaves of the shell: its area times its thickness, in 8^3 cells.
        voxels = 4 * math.pi * (0.35 * case["res"]) ** 2 * 34
        n = case["count"]
        if case["what"] == "points":
            read = voxels * -math.expm1(-STENCIL[case["filter"]] * n / voxels)
            grad = case["op"] == "gradient"
            return {"bytes": n * (24 if grad else 16) + read * es, "flops": n * FLOPS[case["filter"]] * (2 if grad else 1)}
        # Mean results per ray (camera rays cross the shell twice, each time
        # through a few cells of the depth that the hint selects), and the
        # value range of each cell that a ray reports.
        cells = {0.0: 1, 0.25: 2, 0.5: 10, 1.0: 48}[case["hint"]] if case["what"] == "intervals" else 0
        each = cells * (20 + 8) + 28 if case["what"] == "intervals" else 2 * (12 + 8 * es) + 28
        return {"bytes": n * each, "flops": n * (60 + 20 * max(cells, 40))}
    voxels = case["nx"] * case["ny"] * case["nz"] * max(case.get("steps", 0), 1)
    if case["kind"] == "points":
        n, taps = case["count"], STENCIL[case["filter"]] * (2 if case["steps"] else 1)
        read = voxels * -math.expm1(-taps * n / voxels)
        grad = case["op"] == "gradient"
        per = (24 if grad else 16) + (4 if case["steps"] else 0)
        return {"bytes": n * per + read * es,
                "flops": n * (FLOPS[case["filter"]] * (2 if grad else 1) + (24 if case["steps"] else 0))}
    rays = case["width"] * case["height"]
    size = (case["nx"] + case["ny"] + case["nz"]) / 3
    if case["what"] == "march":
        return {"bytes": rays * (32 + 20) + voxels * es * 0.6, "flops": rays * 0.3 * size * 80}
    if case["what"] == "shade":
        return {"bytes": rays * (32 + 20) + voxels * es * 0.6, "flops": rays * 0.7 * size * 50}
    return {"bytes": rays * (32 + 16 + 12) + voxels * es * 0.6, "flops": rays * 20 * 120}


# ---- the same outputs in binary64 ---------------------------------------------------------

def catmull_rom(t):
    w = torch.stack([-t ** 3 + 2 * t ** 2 - t, 3 * t ** 3 - 5 * t ** 2 + 2, -3 * t ** 3 + 4 * t ** 2 + t,
                     t ** 3 - t ** 2], 0) * 0.5
    dw = torch.stack([-3 * t ** 2 + 4 * t - 1, 9 * t ** 2 - 10 * t, -9 * t ** 2 + 8 * t + 1, 3 * t ** 2 - 2 * t],
                     0) * 0.5
    return w, dw


def interpolate(p, fetch, filter, op, offset):
    """Sample or index-space gradient at index-space points p (binary64);
    fetch(ix, iy, iz) gives the voxels in binary64."""
    if filter == "nearest":
        i = torch.floor(p + offset).long()
        return fetch(i[:, 0], i[:, 1], i[:, 2])
    i = torch.floor(p).long()
    f = p - i
    if filter == "linear":
        w, dw, first = torch.stack([1 - f, f]), torch.stack([-torch.ones_like(f), torch.ones_like(f)]), 0
    else:
        (w, dw), first = catmull_rom(f), -1
    taps = w.shape[0]
    out = [0.0, 0.0, 0.0] if op == "gradient" else [0.0]
    for a in range(taps):
        for b in range(taps):
            for c in range(taps):
                v = fetch(i[:, 0] + a + first, i[:, 1] + b + first, i[:, 2] + c + first)
                if op == "gradient":
                    out[0] = out[0] + dw[a, :, 0] * w[b, :, 1] * w[c, :, 2] * v
                    out[1] = out[1] + w[a, :, 0] * dw[b, :, 1] * w[c, :, 2] * v
                    out[2] = out[2] + w[a, :, 0] * w[b, :, 1] * dw[c, :, 2] * v
                else:
                    out[0] = out[0] + w[a, :, 0] * w[b, :, 1] * w[c, :, 2] * v
    return torch.stack(out, 1) if op == "gradient" else out[0]


def exact(case, seed):
    # Intervals, hits and renderings are what an iteration with its own
    # partition, stopping rules and draws yields: no value of their own.
    if case["kind"] == "frame" or case["kind"] == "vdb" and case["what"] != "points":
        return None
    nan = torch.tensor(float("nan"), device=DEV, dtype=torch.float64)
    if case["kind"] == "vdb":
        origins, leaves = shell(case, seed)
        pts = leaf_points(case, origins, seed)
        cells = case["res"] // 8
        slot = torch.full((cells, cells, cells), -1, dtype=torch.int64, device=DEV)
        o = (origins // 8).long()
        slot[o[:, 0], o[:, 1], o[:, 2]] = torch.arange(origins.shape[0], device=DEV)
        flat = leaves.reshape(-1)
        size = [int(x) + 8 for x in origins.amax(0)]
        scale, offset = torch.ones(3, device=DEV, dtype=torch.float64), 0.0

        def fetch(x, y, z, rows):
            inside = (x >= 0) & (y >= 0) & (z >= 0) & (x < size[0]) & (y < size[1]) & (z < size[2])
            x, y, z = [c.clamp(0, s - 1) for c, s in zip((x, y, z), size)]
            k = slot[x >> 3, y >> 3, z >> 3]
            v = flat[k.clamp(min=0) * 512 + ((x & 7) << 6) + ((y & 7) << 3) + (z & 7)].double()
            return torch.where(inside, torch.where(k >= 0, v, torch.zeros_like(v)), nan)
    else:
        voxels, pts = grid_field(case, seed), grid_points(case, seed)
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        scale = torch.tensor([case["sx"], case["sy"], case["sz"]], device=DEV, dtype=torch.float32).double()
        offset, flat, steps = 0.5, voxels.reshape(-1), case["steps"]
        times = uniform(generator(seed + 3), case["count"]).double() if steps else None

        def fetch(x, y, z, rows):
            inside = (x >= 0) & (y >= 0) & (z >= 0) & (x < nx) & (y < ny) & (z < nz)
            at = (z.clamp(0, nz - 1) * ny + y.clamp(0, ny - 1)) * nx + x.clamp(0, nx - 1)
            if steps:
                t = times[rows] * (steps - 1)
                k = torch.floor(t).long().clamp(max=steps - 2)
                v = (1 - (t - k)) * flat[at * steps + k].double() + (t - k) * flat[at * steps + k + 1].double()
            else:
                v = flat[at].double()
            return torch.where(inside, v, nan)
    out = []
    for a in range(0, pts.shape[0], 1 << 22):
        rows = slice(a, min(a + (1 << 22), pts.shape[0]))
        r = interpolate(pts[rows].double() / scale, lambda x, y, z: fetch(x, y, z, rows), case["filter"], case["op"],
                        offset)
        out.append(r / scale if case["op"] == "gradient" else r)
    return torch.cat(out)
