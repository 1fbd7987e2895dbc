"""The work that users of the ray-caster have it do, as cases to be timed.

A case is a dict of plain values; prepare() makes what a program holds before
the call, run() is one pass through the public entry points, work() is what
the pass cannot do without and exact() is the same answer from plain torch in
64 bits.  The kinds of case:

  oap       off_axis_projection() of a host dataset, the whole drop-in call:
            upload, cast, read back, normalise
  single    Context.render_noalloc(): one camera on a resident volume, the
            call behind an interactive view
  proj      a prepared Batch of one off-axis projection of a resident volume
  vr        a prepared Batch of one volume render with an 8-Gaussian
            ColorTransferFunction; grey: with grey opacity
  persp     the same through the perspective lens (a ray per pixel)
  iproj     a prepared Batch of one interpolated projection (the sampler of a
            "projection" VolumeSource)
  amr_proj, amr_vr
            the same two calls on an AMR hierarchy: hundreds of small bricks
  serve     the continuous-batching server: a burst of cameras of many image
            sizes, half projections and half volume renders
  snapshot  one frame of a time series: a ResidentVolume from a snapshot's
            cells, one volume render of it, and the volume freed
"""

import math

import numpy as np
import torch

from yt_amd import _lib, data, off_axis_projection, render
from yt_amd.transfer_functions import gaussian_ctf

DEV = "cuda" if torch.cuda.is_available() else "cpu"

# Image sides of the batched workload; servers take any side.
SIDES = (128, 256, 512, 1024)


def listed():
    return [
        # The smallest whole call: yt's plain method on a 64^3 field.
        dict(name="oap_64_256", kind="oap", n=64, r0=256, r1=256, weighted=False, width=1.0),
        # An ordinary one: weighted (temperature by density), an odd field, a wide image.
        dict(name="oap_weighted_odd", kind="oap", n=117, r0=640, r1=401, weighted=True, width=1.3),
        # The shortest call: a thumbnail of a small resident field.
        dict(name="single_64_128", kind="single", n=64, r0=128, r1=128, weighted=False, width=1.0),
        # The 256^3 density-weighted projection at 1024^2.
        dict(name="proj_weighted_256_1024", kind="proj", n=256, split=1, r0=1024, r1=1024, weighted=True, width=1.0),
        # The volume render of a Scene: 8 Gaussians over log10 density.
        dict(name="vr_256_800x600", kind="vr", n=256, split=1, r0=800, r1=600, samples=10, grey=False, width=1.5),
        # Grey opacity: opaque surfaces, as create_scene users set it.
        dict(name="grey_192_512", kind="vr", n=192, split=1, r0=512, r1=512, samples=10, grey=True, width=1.5),
        # A perspective camera outside the domain, an odd image.
        dict(name="persp_160_501x333", kind="persp", n=160, split=1, r0=501, r1=333, samples=10, width=1.0),
        # The smooth projection of a "projection" source.
        dict(name="iproj_256_512", kind="iproj", n=256, split=1, r0=512, r1=512, samples=10, width=1.0),
        # The AMR workload: about 640 grids, 1700 kd-tree bricks.
        dict(name="amr_proj_700x500", kind="amr_proj", n=128, levels=3, r0=700, r1=500, width=1.0),
        dict(name="amr_vr_1024", kind="amr_vr", n=128, levels=3, r0=1024, r1=1024, samples=10, width=1.0),
        # A burst of requests on the 512^3 field in 2^3 bricks.
        dict(name="serve_512_16", kind="serve", n=512, split=2, images=16, smallest=128, largest=1024),
        # One frame of a time series.
        dict(name="snapshot_128_400", kind="snapshot", n=128, r0=400, r1=400, samples=10, width=1.2),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("oap", "single", "proj", "vr", "vr", "persp", "iproj", "amr_proj", "amr_vr", "serve",
                       "snapshot"))
    width = round(rng.uniform(0.6, 1.9), 3)
    size = dict(r0=_log_int(rng, 96, 1024), r1=_log_int(rng, 96, 1024))
    if kind == "oap":
        return dict(kind=kind, n=_log_int(rng, 24, 144), weighted=rng.random() < 0.4, width=width,
                    r0=_log_int(rng, 64, 800), r1=_log_int(rng, 64, 800))
    if kind == "single":
        return dict(kind=kind, n=_log_int(rng, 24, 128), weighted=rng.random() < 0.3, width=width,
                    r0=_log_int(rng, 64, 320), r1=_log_int(rng, 64, 320))
    if kind == "proj":
        return dict(kind=kind, n=_log_int(rng, 48, 288), split=rng.choice((1, 1, 2, 4)),
                    weighted=rng.random() < 0.5, width=width, **size)
    if kind == "vr":
        return dict(kind=kind, n=_log_int(rng, 48, 256), split=rng.choice((1, 1, 2)),
                    samples=rng.choice((10, 10, 10, 5)), grey=rng.random() < 0.4, width=width, **size)
    if kind == "persp":
        return dict(kind=kind, n=_log_int(rng, 48, 192), split=1, samples=10, width=1.0,
                    r0=_log_int(rng, 96, 640), r1=_log_int(rng, 96, 640))
    if kind == "iproj":
        return dict(kind=kind, n=_log_int(rng, 48, 256), split=rng.choice((1, 1, 2)),
                    samples=rng.choice((10, 10, 5)), width=width, **size)
    if kind in ("amr_proj", "amr_vr"):
        c = dict(kind=kind, n=rng.choice((64, 96, 128)), levels=rng.choice((1, 2, 3)), width=width, **size)
        if kind == "amr_vr":
            c["samples"] = 10
        return c
    if kind == "serve":
        return dict(kind=kind, n=rng.choice((128, 192, 256, 384)), split=rng.choice((1, 2)),
                    images=rng.randint(3, 16), smallest=rng.choice((96, 128, 200)),
                    largest=rng.choice((512, 777, 1024)))
    return dict(kind="snapshot", n=_log_int(rng, 48, 144), samples=10, width=width,
                r0=_log_int(rng, 96, 640), r1=_log_int(rng, 96, 640))


# ---------------------------------------------------------------------------
# Inputs

def _lognormal(n, seed, dtype):
    """exp(g) of a Gaussian random field g with P(k) ~ k^-3, mean 0 and
    sigma 1 on an n^3 grid, as a host array."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    w = torch.fft.rfftn(torch.randn((n, n, n), generator=gen, device=DEV, dtype=torch.float32))
    k = torch.fft.fftfreq(n, device=DEV)
    kz = torch.fft.rfftfreq(n, device=DEV)
    k2 = k[:, None, None] ** 2 + k[None, :, None] ** 2 + kz[None, None, :] ** 2
    amp = torch.where(k2 > 0, k2 ** -0.75, torch.zeros_like(k2))
    g = torch.fft.irfftn(w * amp, (n, n, n))
    g = (g - g.mean()) / g.std()
    return torch.exp(g).to(dtype).cpu().numpy()


def _fields(case, seed):
    """density (and temperature where the case weights by density)."""
    f64 = case["kind"] in ("oap", "snapshot", "persp")
    dtype = torch.float64 if f64 else torch.float32
    f = {"density": _lognormal(case["n"], seed, dtype)}
    if case.get("weighted"):
        noise = np.random.default_rng(seed + 1).standard_normal(f["density"].shape, dtype=np.float32)
        f["temperature"] = f["density"] ** 0.6 * np.exp(0.3 * noise).astype(f["density"].dtype)
    return f


def _dataset(case, seed):
    if case["kind"].startswith("amr"):
        hierarchy = data.make_amr_hierarchy(case["n"], case["levels"], seed_density=seed, seed_flag=seed + 1)
        return data.load_amr_grids(hierarchy, [case["n"]] * 3)
    split = case.get("split", 1)
    return data.load_uniform_grid(_fields(case, seed), psize=(split,) * 3 if split > 1 else None)


def _direction(seed):
    """A view direction and a north vector."""
    rng = np.random.default_rng(seed + 2)
    normal = rng.normal(size=3)
    return normal / np.linalg.norm(normal), rng.normal(size=3)


def _bounds(ds):
    lo = min(float(np.log10(g["density"].min())) for g in ds.grids)
    hi = max(float(np.log10(g["density"].max())) for g in ds.grids)
    return lo, hi


def _transfer(ds, grey=False):
    tf = gaussian_ctf(_bounds(ds), n_gauss=8, nbins=256)
    tf.grey_opacity = grey
    return tf


def _perspective(case, seed):
    """A camera two domain widths away that sees the whole domain."""
    normal, north = _direction(seed)
    focus = np.array([0.5, 0.5, 0.5])
    return focus - 2.0 * normal, focus, north, (1.6, 1.6, 2.0)


def _burst(case, seed):
    """(normal, north, side, is volume render) of each request of a burst."""
    rng = np.random.default_rng(seed + 3)
    sides = [s for s in SIDES if case["smallest"] <= s <= case["largest"]]
    sides += [case["smallest"], case["largest"]]
    sides = sorted(set(sides))
    out = []
    for i in range(case["images"]):
        normal = rng.normal(size=3)
        out.append((normal / np.linalg.norm(normal), rng.normal(size=3), sides[i % len(sides)], i % 4 in (1, 2)))
    return out


class Held:
    """What a program keeps between calls; given back when it is dropped."""

    def __init__(self, **kw):
        self.__dict__.update(kw)

    def __del__(self):
        for name in ("batch", "server"):
            if getattr(self, name, None) is not None:
                getattr(self, name).close()
        if getattr(self, "volume", None) is not None:
            self.volume.free()


def prepare(case, seed):
    kind = case["kind"]
    ds = _dataset(case, seed)
    normal, north = _direction(seed)
    center = (0.5, 0.5, 0.5)
    if kind == "oap":
        return Held(kind=kind, ds=ds, item="temperature" if case["weighted"] else "density",
                    weight="density" if case["weighted"] else None, normal=normal, north=north,
                    center=center, width=case["width"], resolution=[case["r0"], case["r1"]])
    ctx = _lib.default_context()
    if kind == "snapshot":
        return Held(kind=kind, ctx=ctx, ds=ds, tf=_transfer(ds), samples=case["samples"], normal=normal,
                    north=north, center=center, width=case["width"], resolution=[case["r0"], case["r1"]])
    if kind == "serve":
        volume = render.ResidentVolume(ctx, ds, proj_fields="density", vr_field="density")
        tf = _lib.TF.from_tf_obj(_transfer(ds))
        specs = []
        for nrm, nth, side, is_vr in _burst(case, seed):
            p = render.camera_params(center, nrm, 1.0, side, nth)
            specs.append(volume.vr_request(p, tf) if is_vr else volume.projection_request(p))
        server = _lib.Server(ctx, max_requests=64, budget_bytes=1 << 30)
        return Held(kind=kind, volume=volume, specs=specs, server=server)
    if kind in ("single", "proj", "amr_proj"):
        weighted = bool(case.get("weighted"))
        volume = render.ResidentVolume(ctx, ds, proj_fields="temperature" if weighted else "density",
                                       weight="density" if weighted else None)
    else:
        # a "projection" source integrates the field itself, not its logarithm
        volume = render.ResidentVolume(ctx, ds, vr_field="density", log_field=kind != "iproj")
    if kind == "persp":
        position, focus, nth, width = _perspective(case, seed)
        p = render.perspective_params(position, focus, width, (case["r0"], case["r1"]), nth)
    else:
        p = render.camera_params(center, normal, case["width"], (case["r0"], case["r1"]), north)
    if kind in ("single", "proj", "amr_proj"):
        spec = volume.projection_request(p)
    elif kind == "iproj":
        spec = volume.interpolated_projection_request(p, n_samples=case["samples"])
    else:
        spec = volume.vr_request(p, _transfer(ds, case.get("grey", False)), n_samples=case["samples"])
    if kind == "single":
        return Held(kind=kind, ctx=ctx, volume=volume, spec=spec)
    batch = _lib.Batch(ctx, [spec], _lib.BATCH_PERSISTENT | _lib.BATCH_GRAPH)
    return Held(kind=kind, volume=volume, batch=batch)


# ---------------------------------------------------------------------------
# One pass

def run(state):
    if state.kind == "oap":
        return off_axis_projection(
            state.ds, state.center, state.normal, state.width, state.resolution, state.item,
            weight=state.weight, north_vector=state.north)
    if state.kind == "single":
        return state.ctx.render_noalloc(state.spec)
    if state.kind == "serve":
        server = state.server
        at, images = {}, [None] * len(state.specs)
        for i, spec in enumerate(state.specs):
            at[server.submit(spec)] = i
        while at:
            for rid in server.wait():
                images[at.pop(rid)] = server.read_planar(rid)
        return images
    if state.kind == "snapshot":
        volume = render.ResidentVolume(state.ctx, state.ds, vr_field="density")
        p = render.camera_params(state.center, state.normal, state.width, state.resolution, state.north)
        image = state.ctx.render_noalloc(volume.vr_request(p, state.tf, n_samples=state.samples))
        volume.free()
        return image
    state.batch.run()
    return state.batch.read_image(0)


# ---------------------------------------------------------------------------
# What a pass cannot do without

def _amr_cells(case):
    blocks = (330, 280, 230)
    return case["n"] ** 3 + sum(min(blocks[i], (case["n"] // 8) ** 3) for i in range(case["levels"])) * 16 ** 3


def work(case):
    """The cells a pass reaches, once each, and the image; operations from
    the mean number of cells a ray of random direction visits."""
    kind, n = case["kind"], case["n"]
    bytes_, flops = 0.0, 0.0
    if kind == "serve":
        images = [(side, side, 1.0, vr) for _, _, side, vr in _burst(case, 0)]
    else:
        images = [(case["r0"], case["r1"], case["width"], kind in ("vr", "persp", "amr_vr", "snapshot"))]
    per_axis = n * (1.0 + 0.3 * case.get("levels", 0))
    cells = _amr_cells(case) if kind.startswith("amr") else n ** 3
    nf = 2 if case.get("weighted") else 1
    samples = case.get("samples", 10)
    seen = {False: 0.0, True: 0.0}
    for r0, r1, width, vr in images:
        scale = (width if kind != "persp" else 1.6) ** 2
        visits = 1.5 * per_axis * r0 * r1 / scale
        visits = min(visits, 1.5 * per_axis * r0 * r1)
        seen[vr] += visits
        if vr:
            flops += visits * (60.0 + 23.0 * samples)
        elif kind == "iproj":
            flops += visits * 60.0
        else:
            flops += visits * 2.0 * nf
        if kind == "serve":
            bytes_ += r0 * r1 * 4.0 * (3 if vr else 1)
        else:
            bytes_ += r0 * r1 * (8.0 if kind == "oap" else 32.0)
    for visits in seen.values():
        if kind in ("oap", "snapshot"):  # the call takes the whole field, whatever the camera sees
            bytes_ += (cells * 8.0 * nf) if visits else 0.0
        else:
            bytes_ += min(float(cells), visits) * 4.0 * nf
    return {"bytes": bytes_, "flops": flops}


# ---------------------------------------------------------------------------
# The same answers in 64 bits, from plain torch

def _basis(normal, north):
    normal = normal / np.linalg.norm(normal)
    north = north / np.linalg.norm(north)
    north = north - np.dot(north, normal) * normal
    east = np.cross(north, normal)
    return east / np.linalg.norm(east), north / np.linalg.norm(north), normal


def _f64(a):
    return torch.as_tensor(np.asarray(a, dtype=np.float64), device=DEV)


def _parallel_rays(normal, north, width, r0, r1):
    """Origins (r0 r1, 3) and the shared direction, t in [0, 1]."""
    east, up, normal = _basis(normal, north)
    px = width * np.arange(r0) / (r0 - 1.0) - width / 2.0
    py = width * np.arange(r1) / (r1 - 1.0) - width / 2.0
    back = np.full(3, 0.5) - 0.5 * width * normal
    pos = px[:, None, None] * east + py[None, :, None] * up + back
    return _f64(pos.reshape(-1, 3)), _f64(np.broadcast_to(normal * width, (r0 * r1, 3)).copy())


def _perspective_rays(case, seed):
    position, focus, north, width = _perspective(case, seed)
    east, up, normal = _basis(focus - position, north)
    r0, r1 = case["r0"], case["r1"]
    reach = np.linalg.norm(position - 0.5) + 0.5 * math.sqrt(3.0)
    x = width[0] * np.linspace(-0.5, 0.5, r0)
    y = width[0] * (r1 / r0) * np.linspace(-0.5, 0.5, r1)
    d = (x[:, None, None] * east + y[None, :, None] * up + normal * width[2]) * (reach / width[2])
    return _f64(np.broadcast_to(position, (r0 * r1, 3)).copy()), _f64(d.reshape(-1, 3))


def _in_extent(normal, north, width, r0, r1, le, re):
    """The pixels that the caster looks at for a box: its bounding rectangle,
    rounded, and a pixel more on each side (lenses.pyx:22-55)."""
    east, up, normal = _basis(normal, north)
    back = np.full(3, 0.5) - 0.5 * width * normal
    corners = np.array([[(le, re)[i][0], (le, re)[j][1], (le, re)[k][2]]
                        for i in (0, 1) for j in (0, 1) for k in (0, 1)])
    keep = []
    for axis, r in ((east, r0), (up, r1)):
        v = corners @ axis
        per = width / r
        a = int(np.rint((v.min() - back @ axis + width / 2.0) / per))
        b = a + int(np.rint((v.max() - v.min()) / per))
        keep.append((min(max(a - 1, 0), r), min(max(b + 1, 0), r)))
    (i0, i1), (j0, j1) = keep
    i = torch.arange(i0, i1, device=DEV)
    j = torch.arange(j0, j1, device=DEV)
    return (i[:, None] * r1 + j[None, :]).reshape(-1)


def _vertices(a):
    """The no-ghost vertex values of cell values: means of 8 cells inside,
    linear extrapolation on the faces."""
    for axis in range(3):
        a = a.movedim(axis, 0)
        first, last = 1.5 * a[:1] - 0.5 * a[1:2], 1.5 * a[-1:] - 0.5 * a[-2:-1]
        a = torch.cat((first, 0.5 * (a[:-1] + a[1:]), last)).movedim(0, axis)
    return a


def _march(pos, direc, le, re, dims, visit):
    """Walks every ray through its box of dims cells; le, re, dims: (3,) or
    one per ray.  visit(index of the rays still inside, enter, exit, cell)."""
    dds = (re - le) / dims
    step = torch.sign(direc)
    inv = torch.where(direc != 0, 1.0 / direc, torch.full_like(direc, float("inf")))
    a, b = (le - pos) * inv, (re - pos) * inv
    still = direc == 0
    a = torch.where(still, torch.full_like(a, -1e30), a)
    b = torch.where(still, torch.full_like(b, 1e30), b)
    t0 = torch.minimum(a, b).amax(1).clamp(min=0.0)
    t1 = torch.maximum(a, b).amin(1).clamp(max=1.0)
    ids = torch.nonzero(t0 < t1).reshape(-1)
    per_ray = dims.dim() == 2
    pick = (lambda v: v[ids]) if per_ray else (lambda v: v)
    lo, dd, nd = pick(le), pick(dds), pick(dims)
    p, d, st, iv, t, end = pos[ids], direc[ids], step[ids], inv[ids], t0[ids], t1[ids]
    cell = torch.floor((p + t[:, None] * d - lo) / dd)
    # A ray that enters through a face starts in the cell on its inner side.
    cell = torch.minimum(cell.clamp(min=0.0), (nd - 1.0).expand_as(cell))
    nxt = torch.where(st != 0, ((cell + (st > 0)) * dd + lo - p) * iv, torch.full_like(p, 1e60))
    dt = torch.where(st != 0, dd * iv.abs(), torch.zeros_like(p))
    while ids.numel():
        tm, axis = nxt.min(1)
        out = torch.minimum(tm, end)
        visit(ids, t, out, cell)
        one = torch.nn.functional.one_hot(axis, 3).to(torch.float64)
        cell = cell + one * st
        nxt = nxt + one * dt
        t = out
        go = (tm < end) & ((cell >= 0) & (cell < nd)).all(1)
        keep = torch.nonzero(go).reshape(-1)
        if keep.numel() < ids.numel():
            ids, p, d, st, t, end = ids[keep], p[keep], d[keep], st[keep], t[keep], end[keep]
            cell, nxt, dt = cell[keep], nxt[keep], dt[keep]
            if per_ray:
                nd = nd[keep]


def _project(pos, direc, boxes):
    """Sums of the fields along the rays; boxes: (le, re, values (nf, n, n, n), ray ids)."""
    nf = boxes[0][2].shape[0]
    total = torch.zeros((pos.shape[0], nf), dtype=torch.float64, device=DEV)
    for le, re, v, ids in boxes:
        dims = torch.tensor(v.shape[1:], dtype=torch.float64, device=DEV)
        flat = v.reshape(nf, -1).t().contiguous()
        part = torch.zeros((ids.numel(), nf), dtype=torch.float64, device=DEV)

        def visit(i, en, ex, cell):
            c = cell.long()
            at = (c[:, 0] * v.shape[2] + c[:, 1]) * v.shape[3] + c[:, 2]
            part[i] += flat[at] * (ex - en)[:, None]

        _march(pos[ids], direc[ids], le, re, dims, visit)
        total[ids] += part
    return total


def _project_many(pos, direc, grids):
    """_project over many small grids at once: a ray per (grid, pixel) pair."""
    flat = torch.cat([v.reshape(-1) for _, _, v, _ in grids])
    base, pair = [], {k: [] for k in ("ids", "grid")}
    at = 0
    for g, (_, _, v, ids) in enumerate(grids):
        base.append(at)
        at += v.numel()
        pair["ids"].append(ids)
        pair["grid"].append(torch.full_like(ids, g))
    ids, grid = torch.cat(pair["ids"]), torch.cat(pair["grid"])
    le = torch.stack([g[0] for g in grids])[grid]
    re = torch.stack([g[1] for g in grids])[grid]
    dims = torch.tensor([g[2].shape for g in grids], dtype=torch.float64, device=DEV)[grid]
    base = torch.tensor(base, device=DEV)[grid]
    part = torch.zeros(ids.numel(), dtype=torch.float64, device=DEV)

    def visit(i, en, ex, cell):
        c, d = cell.long(), dims[i].long()
        part[i] += flat[base[i] + (c[:, 0] * d[:, 1] + c[:, 1]) * d[:, 2] + c[:, 2]] * (ex - en)

    _march(pos[ids], direc[ids], le, re, dims, visit)
    return torch.zeros(pos.shape[0], dtype=torch.float64, device=DEV).index_add_(0, ids, part)


def _samples(pos, direc, box, n, each):
    """each(ray ids, dt, values (rays, n)) for every cell: the trilinear
    values at the cell's n mid-point sub-samples."""
    le, re, v, ids = box
    dims = torch.tensor([s - 1.0 for s in v.shape], dtype=torch.float64, device=DEV)
    dds = (re - le) / dims
    p0, d0 = pos[ids], direc[ids]
    flat = v.reshape(-1)
    s1, s0 = v.shape[2], v.shape[1] * v.shape[2]
    s = torch.arange(n, dtype=torch.float64, device=DEV) + 0.5

    def visit(i, en, ex, cell):
        dt = (ex - en) / n
        tt = en[:, None] + s * dt[:, None]
        x = [((p0[i, a, None] + tt * d0[i, a, None]) - (cell[:, a] * dds[a] + le[a])[:, None]) / dds[a]
             for a in range(3)]
        c = cell.long()
        at = c[:, 0] * s0 + c[:, 1] * s1 + c[:, 2]
        val = 0.0
        for a in (0, 1):
            for b in (0, 1):
                row = at + a * s0 + b * s1
                z = flat[row][:, None] * (1.0 - x[2]) + flat[row + 1][:, None] * x[2]
                val = val + z * ((x[0] if a else 1.0 - x[0]) * (x[1] if b else 1.0 - x[1]))
        each(ids[i], dt, val)

    _march(p0, d0, le, re, dims, visit)


def _composite(pos, direc, boxes, tf, n):
    """rgba of the rays through the boxes, given in the order rays cross them."""
    rgba = torch.zeros((pos.shape[0], 4), dtype=torch.float64, device=DEV)
    b0, b1 = (float(x) for x in tf.x_bounds)
    y = torch.stack([_f64(t.y) for t in tf.funcs], 1)
    dbin = (b1 - b0) / (y.shape[0] - 1)
    slope = (y[1:] - y[:-1]) / dbin

    def each(i, dt, val):
        ok = (val > b0) & (val < b1)
        k = ((val - b0) / dbin).long().clamp(0, y.shape[0] - 2)
        e = y[k] + (val - (b0 + k * dbin))[..., None] * slope[k]
        e = torch.where(ok[..., None], e, torch.zeros_like(e))
        e = torch.cat((e[..., :3] * e[..., 3:], e[..., 3:]), -1) * dt[:, None, None]
        c = rgba[i]
        for s in range(n):
            if tf.grey_opacity:
                c = e[:, s] + (1.0 - e[:, s, 3:]).clamp(min=0.0) * c
            else:
                c = e[:, s] + (1.0 - e[:, s]).clamp(min=0.0) * c
        rgba[i] = c

    for box in boxes:
        _samples(pos, direc, box, n, each)
    if not tf.grey_opacity:
        rgba[:, 3] = 0.0
    return rgba


def _cells(case, ds, grid, mask):
    """The projected fields of a block, child-masked: (fields, n, n, n)."""
    m = _f64(mask)
    if case.get("weighted"):
        w = _f64(grid["density"]) * m
        return torch.stack((_f64(grid["temperature"]) * w, w))
    return (_f64(grid["density"]) * m)[None]


def exact(case, seed):
    kind = case["kind"]
    if kind == "amr_vr":
        return None
    ds = _dataset(case, seed)
    normal, north = _direction(seed)
    if kind == "serve":
        # the projections of a burst, while they are quick
        out, left = [], 4
        for nrm, nth, side, is_vr in _burst(case, seed):
            if is_vr or left == 0:
                out.append(None)
                continue
            left -= 1
            pos, direc = _parallel_rays(nrm, nth, 1.0, side, side)
            boxes = [(_f64(g.LeftEdge), _f64(g.RightEdge), _cells(case, ds, g, m),
                      _in_extent(nrm, nth, 1.0, side, side, g.LeftEdge, g.RightEdge)) for g, m in ds.blocks()]
            out.append(_project(pos, direc, boxes).t().reshape(1, side, side).cpu().numpy())
        return out
    r0, r1 = case["r0"], case["r1"]
    if kind == "persp":
        pos, direc = _perspective_rays(case, seed)
        ids = [torch.arange(r0 * r1, device=DEV)] * len(ds.grids)
    else:
        pos, direc = _parallel_rays(normal, north, case["width"], r0, r1)
        ids = [_in_extent(normal, north, case["width"], r0, r1, g.LeftEdge, g.RightEdge) for g in ds.grids]
    image = torch.zeros((r0 * r1, 4), dtype=torch.float64, device=DEV)
    if kind in ("oap", "single", "proj", "amr_proj"):
        boxes = [(_f64(g.LeftEdge), _f64(g.RightEdge), _cells(case, ds, g, g.child_mask), i)
                 for g, i in zip(ds.grids, ids) if g.child_mask.any()]
        if kind == "amr_proj":
            boxes = [(le, re, v[0], i) for le, re, v, i in boxes]
            image[:, 0] = _project_many(pos, direc, boxes)
        else:
            total = _project(pos, direc, boxes)
            if kind == "oap":
                if case["weighted"]:
                    v = torch.where(total[:, 1] == 0, torch.zeros_like(total[:, 0]), total[:, 0] / total[:, 1])
                else:
                    v = total[:, 0] * case["width"]
                return v.reshape(r0, r1).cpu().numpy()
            image[:, :total.shape[1]] = total
        return image.reshape(r0, r1, 4).cpu().numpy()
    # boxes in the order the rays cross them: the lower side of an axis first where rays go up it
    sign = np.sign(direc[0].cpu().numpy())
    order = sorted(range(len(ds.grids)), key=lambda k: float(np.dot(ds.grids[k].LeftEdge, sign)))
    values = (lambda v: v) if kind == "iproj" else torch.log10
    boxes = [(_f64(ds.grids[k].LeftEdge), _f64(ds.grids[k].RightEdge),
              values(_vertices(_f64(ds.grids[k]["density"]))), ids[k]) for k in order]
    if kind == "iproj":
        total = torch.zeros(r0 * r1, dtype=torch.float64, device=DEV)

        def each(i, dt, val):
            total[i] += val.sum(1) * dt

        for box in boxes:
            _samples(pos, direc, box, case["samples"], each)
        image[:, 0] = total
    else:
        image = _composite(pos, direc, boxes, _transfer(ds, case.get("grey", False)), case["samples"])
    return image.reshape(r0, r1, 4).cpu().numpy()
