"""Performance cases of the renderer: what its users have it do, through the
package's public entry points.

A case names its kind and sizes:

* ``query``    batched closest-hit queries (``Scene.trace_hits`` on host
               arrays, ``Scene.trace_hits_device`` on device buffers);
* ``viewer``   one step of a progressive viewer: a few samples into device
               films, a snapshot, its readback and the display estimate;
* ``render``   samples into films in device or host memory
               (``Scene.render_pt_device`` / ``Scene.render_pt``);
* ``batch``    several jobs of different sizes in one call (``render_batch``);
* ``sppm``     one progressive photon-mapping pass (``Sppm.pass_device``);
* ``guided``   path tracing with the learned guide proposing directions;
* ``gradient`` forward and backward of the guide's network over a minibatch
               (``Guide.gradient``).

Scenes are the package's procedural ones.  Their geometry is fixed; the seed
of a case moves the camera, changes the materials or the layout, and keys the
random streams.
"""
import functools
import math
import os
import tempfile

import numpy as np
import torch

import hastyrenderer_amd as ha
from hastyrenderer_amd import scenes

DEVICE = "cuda:0"


# ---------------------------------------------------------------- cases ----
def listed():
    return [
        # a picking or visibility query of a host program: latency
        dict(name="query_host_1k", kind="query", api="host", subdiv=3, rays=1000),
        # a renderer that only offloads its ray queries: incoherent rays, throughput
        dict(name="query_device_4m", kind="query", api="device", subdiv=4, rays=4194301),
        # the interactive viewer on a small film: one sample, snapshot, readback, estimate
        dict(name="viewer_cornell", kind="viewer", scene="cornell", width=320, height=240, samples=1, depth=8),
        # a thumbnail with every texture feature and a sky, films in host memory
        dict(name="render_textured_host", kind="render", api="host", scene="textured", width=211, height=173,
             samples=8, depth=8),
        # one progressive pass over a large film of odd size
        dict(name="render_grid_1spp", kind="render", api="device", scene="grid", width=1283, height=721, samples=1,
             depth=16),
        # the headline scene (GGX sphere grid, importance-sampled sky, thin lens): a final-quality batch
        dict(name="render_grid_1024", kind="render", api="device", scene="grid", width=1024, height=1024,
             samples=128, depth=16),
        # glass with dispersion and a metal ring in a closed box, area light only, long paths
        dict(name="render_caustic", kind="render", api="device", scene="caustic", width=720, height=405, samples=16,
             depth=30),
        # a render farm's batch: jobs of mixed film sizes, sample counts and triangle counts
        dict(name="batch_cuboids", kind="batch", jobs=6, min_side=96, max_side=400, min_samples=4, max_samples=32,
             min_cuboids=500, max_cuboids=8000),
        # a photon-mapping pass at the reference's parameters
        dict(name="sppm_caustic", kind="sppm", width=960, height=540, depth=16, store=0.5, emit=10.0, radius=0.0,
             fixed=False),
        # the same with a dense photon map and the order-independent int64 flux
        dict(name="sppm_dense_fixed", kind="sppm", width=640, height=360, depth=16, store=4.0, emit=200.0,
             radius=0.1, fixed=True),
        # guided rendering of the metal-ring box with a learned selection
        dict(name="guided_ring", kind="guided", width=384, height=384, samples=8, depth=32),
        # one minibatch of the guide's online training
        dict(name="gradient_64k", kind="gradient", samples=65536),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("query", "query", "viewer", "render", "render", "render", "batch", "sppm", "sppm", "guided",
                       "gradient"))
    if kind == "query":
        api = rng.choice(("host", "device"))
        n = _log(rng, 500, 200000) if api == "host" else _log(rng, 1000, 4000000)
        return dict(kind=kind, api=api, subdiv=rng.choice((3, 4)), rays=n)
    if kind == "viewer":
        return dict(kind=kind, scene=rng.choice(("cornell", "textured")), width=_log(rng, 160, 900),
                    height=_log(rng, 120, 700), samples=rng.choice((1, 1, 2, 4)), depth=rng.choice((4, 8, 16)))
    if kind == "render":
        scene = rng.choice(("grid", "grid", "caustic", "cornell", "textured"))
        w, h = _log(rng, 64, 1400), _log(rng, 48, 1024)
        most = max(1, min(128, 20000000 // (w * h)))
        return dict(kind=kind, api=rng.choice(("device", "device", "host")), scene=scene, width=w, height=h,
                    samples=_log(rng, 1, most), depth=rng.choice((4, 8, 16, 30)))
    if kind == "batch":
        return dict(kind=kind, jobs=rng.randint(2, 9), min_side=rng.randint(40, 120), max_side=rng.randint(200, 420),
                    min_samples=rng.randint(1, 6), max_samples=rng.randint(12, 32), min_cuboids=500,
                    max_cuboids=rng.randint(2000, 8000))
    if kind == "sppm":
        dense = rng.random() < 0.5
        return dict(kind=kind, width=_log(rng, 128, 960), height=_log(rng, 96, 540), depth=rng.choice((8, 16)),
                    store=rng.uniform(1.0, 3.0) if dense else 0.5, emit=rng.uniform(40.0, 120.0) if dense else 10.0,
                    radius=rng.uniform(0.03, 0.1) if dense else 0.0, fixed=rng.random() < 0.5)
    if kind == "guided":
        return dict(kind=kind, width=_log(rng, 100, 500), height=_log(rng, 100, 500), samples=rng.randint(1, 8),
                    depth=rng.choice((8, 16, 32)))
    return dict(kind=kind, samples=_log(rng, 1000, 130000))


# --------------------------------------------------------------- scenes ----
@functools.lru_cache(maxsize=None)
def _grid_desc(subdiv):
    return scenes.write_ggx_grid("", subdiv=subdiv, as_desc=True)


@functools.lru_cache(maxsize=None)
def _caustic_desc():
    # 200,000 triangles in the ring
    return scenes.write_caustic_scene("", n_major=500, n_minor=200, as_desc=True)


def _film(desc, width, height, depth, samples):
    return dict(desc, settings=dict(desc["settings"], width=width, height=height, max_depth=depth,
                                    num_samples=samples))


def _look(desc, position, target):
    p, fwd, right, up = scenes.look_at_frame(position, target)
    return dict(desc, camera=dict(desc["camera"], position=p, forward=fwd, right=right, up=up))


def _scene(case, seed):
    """The scene of a case as a program holds it: loaded, its BVH built."""
    rng = np.random.default_rng(seed)
    name, w, h = case["scene"], case["width"], case["height"]
    depth, samples = case["depth"], max(1, case.get("samples", 1))
    if name == "grid":
        a = rng.uniform(-0.3, 0.3)
        d = _look(_film(_grid_desc(4), w, h, depth, samples), [8.5 * math.sin(a), 4.0, 8.5 * math.cos(a)],
                  [0.0, 0.4, 0.0])
        mats = [dict(m) for m in d["materials"]]
        for m in mats[1:]:
            m["albedo"] = [float(x) for x in rng.uniform(0.2, 1.0, 3)]
        d["materials"] = mats
        return ha.Scene.create(**d)
    if name == "caustic":
        x = rng.uniform(-0.2, 0.2)
        d = _look(_film(_caustic_desc(), w, h, depth, samples), [x, 1.7, 1.95], [0.0, 0.2, -0.2])
        return ha.Scene.create(**d)
    with tempfile.TemporaryDirectory() as folder:
        if name == "textured":
            return ha.Scene(scenes.write_textured_scene(folder, width=w, height=h, spp=samples, max_depth=depth,
                                                        seed=seed))
        return ha.Scene(scenes.write_cornell(os.path.join(folder, "cornell"), width=w, height=h, spp=samples,
                                             max_depth=depth))


def _films(width, height):
    return tuple(torch.zeros((height, width, 3), dtype=torch.float32, device=DEVICE) for _ in range(3))


def _rays(n, seed):
    """Rays of a bounce over the sphere grid: origins in the air between and
    above the spheres, directions uniform over the sphere; a few leave the
    scene."""
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    u = torch.rand((n, 3), generator=g, device=DEVICE)
    o = torch.stack([u[:, 0] * 8.0 - 4.0, u[:, 1] * 1.6 + 0.01, u[:, 2] * 8.0 - 4.0], 1)
    d = torch.randn((n, 3), generator=g, device=DEVICE)
    d = d / d.norm(dim=1, keepdim=True)
    return torch.cat([o, d], 1).contiguous()


# The guide's network: layer widths, and the used part of the padded ones.
_LAYERS = ((80, 64), (64, 64), (64, 64), (64, 64), (64, 48))


def _guide_params(seed):
    """Parameters of a network part-way through training: He-scaled weights,
    small biases, zero where the layout pads (flat, per layer W^T then b)."""
    rng = np.random.default_rng(seed)
    flat = []
    for i, (k, m) in enumerate(_LAYERS):
        used_in, used_out = (78 if i == 0 else k), (40 if i == 4 else m)
        w = np.zeros((m, k), np.float32)
        b = np.zeros(m, np.float32)
        w[:used_out, :used_in] = rng.normal(0.0, math.sqrt((2.0 if i < 4 else 0.5) / used_in), (used_out, used_in))
        b[:used_out] = rng.normal(0.0, 0.05, used_out)
        flat += [w.ravel(), b]
    return np.concatenate(flat).astype(np.float32)


def _guide_samples(n, seed):
    """Training samples as path ends give them: points in the box, normals
    and outgoing directions, incident directions around the normal, and
    weights with a long tail (mean 1)."""
    rng = np.random.default_rng(seed)

    def unit(v):
        return v / np.linalg.norm(v, axis=1, keepdims=True)

    x = rng.uniform([-2.0, 0.0, -2.0], [2.0, 3.0, 2.0], (n, 3))
    nrm = unit(rng.normal(size=(n, 3)))
    wo = unit(nrm + unit(rng.normal(size=(n, 3))) * 0.999)
    wi = unit(nrm + unit(rng.normal(size=(n, 3))) * 0.999)
    f = np.minimum(rng.lognormal(-0.5, 1.0, n), 20.0)
    return np.concatenate([x, nrm, wo, wi, f[:, None]], 1).astype(np.float32)


_BOX_LO = np.array([-2.0, 0.0, -2.0], np.float32)
_BOX_HI = np.array([2.0, 3.0, 2.0], np.float32)


# -------------------------------------------------------------- prepare ----
def prepare(case, seed):
    kind = case["kind"]
    if kind == "query":
        scene = ha.Scene.create(**_film(_grid_desc(case["subdiv"]), 64, 64, 4, 1))
        rays = _rays(case["rays"], seed)
        if case["api"] == "host":
            return dict(kind="query_host", scene=scene, rays=rays.cpu().numpy())
        hits = torch.empty((case["rays"], 8), dtype=torch.int32, device=DEVICE)
        return dict(kind="query_device", scene=scene, rays=rays, hits=hits)
    if kind == "viewer":
        scene = _scene(case, seed)
        films = ha.Films(scene)
        out = tuple(np.zeros((case["height"], case["width"], 3), np.float32) for _ in range(3))
        return dict(kind=kind, scene=scene, films=films, out=out, seed=seed & 0x7FFFFFFF, n=case["samples"], next=0)
    if kind == "render":
        scene = _scene(case, seed)
        st = dict(kind="render_" + case["api"], scene=scene, seed=seed & 0x7FFFFFFF, n=case["samples"])
        if case["api"] == "device":
            st["films"] = _films(case["width"], case["height"])
        return st
    if kind == "batch":
        rng = np.random.default_rng(seed)
        # the sizes belong to the case, the scenes to the seed
        sizes = np.random.default_rng(case["jobs"] * 7919 + case["max_side"])
        jobs, keep = [], []
        for j in range(case["jobs"]):
            side, spp, cuboids = (int(round(math.exp(sizes.uniform(math.log(case["min_" + k]),
                                                                    math.log(case["max_" + k])))))
                                  for k in ("side", "samples", "cuboids"))
            width = side + j % 3  # not all square
            scene = ha.Scene.create(**scenes.cuboid_scene_desc(cuboids, width, side, spp, int(rng.integers(1 << 31))))
            films = ha.DeviceFilms(width, side)
            jobs.append((scene, int(rng.integers(1 << 31)), 0, spp, films))
            keep.append(films)
        return dict(kind=kind, jobs=jobs)
    if kind == "sppm":
        scene = _scene(dict(case, scene="caustic"), seed)
        sp = ha.Sppm(scene, seed & 0x7FFFFFFF, store_fraction=case["store"], emit_fraction=case["emit"],
                     initial_radius=case["radius"], fixed_point_flux=case["fixed"])
        return dict(kind=kind, scene=scene, sppm=sp, films=_films(case["width"], case["height"]), next=0)
    if kind == "guided":
        scene = _scene(dict(case, scene="caustic"), seed)
        guide = ha.Guide(scene, seed=seed & 0x7FFFFFFF)
        guide.set_selection(0.05, 0.9)
        scene.set_guide(guide, fraction=0.5, train_lr=0.0)
        return dict(kind="render_device", scene=scene, guide=guide, seed=seed & 0x7FFFFFFF, n=case["samples"],
                    films=_films(case["width"], case["height"]))
    scene = ha.Scene.create(**_film(_grid_desc(3), 64, 64, 4, 1))
    guide = ha.Guide(scene, seed=0)
    guide.set_box(_BOX_LO, _BOX_HI)
    guide.set_params(_guide_params(seed))
    return dict(kind="gradient", scene=scene, guide=guide, samples=_guide_samples(case["samples"], seed))


# ------------------------------------------------------------------ run ----
def run(st):
    kind = st["kind"]
    if kind == "query_host":
        h = st["scene"].trace_hits(st["rays"])
        return dict(geom=h["geom_id"], prim=h["prim_id"], t=h["t"], u=h["u"], v=h["v"], ng=h["ng"])
    if kind == "query_device":
        hits = st["hits"]
        st["scene"].trace_hits_device(st["rays"].data_ptr(), st["rays"].shape[0], hits.data_ptr())
        return dict(ids=hits[:, :2], values=hits.view(torch.float32)[:, 2:])
    if kind == "viewer":
        films = st["films"]
        films.render(st["seed"], st["next"], st["n"])
        st["next"] = (st["next"] + st["n"]) % 256
        films.snapshot()
        color, normal, albedo, count = films.read(wait=True, out=st["out"])
        return dict(color=color, normal=normal, albedo=albedo, count=count, estimate=ha.Films.estimate([films], 0.5))
    if kind == "render_device":
        for f in st["films"]:
            f.zero_()
        st["scene"].render_pt_device(st["seed"], 0, st["n"], *(f.data_ptr() for f in st["films"]))
        return st["films"]
    if kind == "render_host":
        return st["scene"].render_pt(st["seed"], 0, st["n"])
    if kind == "batch":
        for job in st["jobs"]:
            job[4].zero()
        ha.render_batch(st["jobs"])
        return [job[4].download() for job in st["jobs"]]
    if kind == "sppm":
        st["sppm"].pass_device(st["next"], *(f.data_ptr() for f in st["films"]))
        st["next"] += 1
        return st["films"]
    grad, loss = st["guide"].gradient(st["samples"])
    return dict(gradient=grad, loss=loss)


# ----------------------------------------------------------------- work ----
# Operations of a ray and a path vertex: about 10 four-wide nodes of 4 x 20,
# 3 triangles of 50, and for a vertex the BSDF, the light sample and ten
# random numbers of a ten-round generator.
_RAY_FLOPS = 10 * 4 * 20 + 3 * 50
_VERTEX_FLOPS = 2500
_TRIS = {"grid": 250882, "caustic": 200028, "cornell": 36, "textured": 1320}
_RAYS_PER_PATH = {"grid": 2.7, "caustic": 7.0, "cornell": 6.0, "textured": 3.5}


def _render_work(scene, pixels, samples, tris=None):
    tris = _TRIS[scene] if tris is None else tris
    rays = _RAYS_PER_PATH.get(scene, 6.0) * pixels * samples
    # films read and written, triangles (positions, normals) read once
    return dict(bytes=pixels * 72.0 + tris * 72.0, flops=rays * (_RAY_FLOPS + _VERTEX_FLOPS / 2))


def work(case):
    kind = case["kind"]
    if kind == "query":
        tris = 49 * 20 * 4 ** case["subdiv"] + 2
        return dict(bytes=case["rays"] * 56.0 + tris * 36.0, flops=case["rays"] * float(_RAY_FLOPS))
    if kind in ("viewer", "render"):
        return _render_work(case["scene"], case["width"] * case["height"], case["samples"])
    if kind == "batch":
        side = math.sqrt(case["min_side"] * case["max_side"])
        spp = math.sqrt(case["min_samples"] * case["max_samples"])
        tris = 12 * math.sqrt(case["min_cuboids"] * case["max_cuboids"])
        w = _render_work("cuboids", side * side, spp, tris)
        return {k: v * case["jobs"] for k, v in w.items()}
    if kind == "sppm":
        px = case["width"] * case["height"]
        # emission stops at whichever comes first; about one photon in 30 of this light's is stored
        emitted = min(case["emit"], 30.0 * case["store"]) * px
        w = _render_work("caustic", px, 1)
        # ten planes of statistics read and written, photons written once
        return dict(bytes=w["bytes"] + px * 80.0 + case["store"] * px * 48.0,
                    flops=w["flops"] + emitted * (_RAY_FLOPS + 500.0))
    if kind == "guided":
        w = _render_work("caustic", case["width"] * case["height"], case["samples"])
        queries = 4.0 * case["width"] * case["height"] * case["samples"]
        return dict(bytes=w["bytes"], flops=w["flops"] + queries * 2.0 * sum(k * m for k, m in _LAYERS))
    return dict(bytes=case["samples"] * 52.0 + 4.0 * 2 * sum(k * m + m for k, m in _LAYERS),
                flops=case["samples"] * 6.0 * sum(k * m for k, m in _LAYERS))


def tolerance(case):
    kind = case["kind"]
    if kind == "query":
        return "exact"  # the hit is the same triangle at the same bits whatever the search order
    if kind == "guided":
        # a proposal that differs in the last bits of its FP32 reciprocals and
        # exponentials moves a few paths to other surfaces
        return dict(rel=0.01, max=0.9)
    if kind == "gradient":
        return dict(rel=4e-3, max=0.2)  # BF16 activations and gradients between the layers
    # radiance sums in FP32; every decision of a path is IEEE-exact
    return dict(rel=1e-5, max=1e-3)


# ---------------------------------------------------------------- exact ----
def _exact_query(case, seed):
    d = _grid_desc(case["subdiv"])
    v = torch.from_numpy(d["vertices"]).to(DEVICE).double()
    tri = v[torch.from_numpy(d["vertex_indices"].astype(np.int64)).to(DEVICE)]
    p0, e1, e2 = tri[:, 0], tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
    rays = _rays(case["rays"], seed).double()
    out_t, out_u, out_v, out_n = [], [], [], []
    for r in rays.split(64):
        o, dr = r[:, None, :3], r[:, None, 3:].expand(-1, p0.shape[0], -1)
        pv = torch.linalg.cross(dr, e2[None].expand_as(dr))
        det = (pv * e1).sum(-1)
        s = o - p0
        u = (s * pv).sum(-1) / det
        q = torch.linalg.cross(s, e1[None].expand_as(s))
        w = (dr * q).sum(-1) / det
        t = (e2 * q).sum(-1) / det
        t = torch.where((u >= 0) & (w >= 0) & (u + w <= 1) & (t > 1e-6), t, math.inf)
        best, k = t.min(1)
        hit = torch.isfinite(best)
        n = torch.linalg.cross(e1[k], e2[k])
        n = n / n.norm(dim=1, keepdim=True)
        zero = torch.zeros_like(best)
        pick = torch.arange(len(k), device=DEVICE)
        out_t.append(best)
        out_u.append(torch.where(hit, u[pick, k], zero))
        out_v.append(torch.where(hit, w[pick, k], zero))
        out_n.append(torch.where(hit[:, None], n, torch.zeros_like(n)))
    t, u, w, n = (torch.cat(x) for x in (out_t, out_u, out_v, out_n))
    return dict(geom=None, prim=None, t=t.cpu().numpy(), u=u.cpu().numpy(), v=w.cpu().numpy(), ng=n.cpu().numpy())


def _exact_gradient(case, seed):
    flat = torch.from_numpy(_guide_params(seed)).to(DEVICE).double().requires_grad_(True)
    smp = torch.from_numpy(_guide_samples(case["samples"], seed)).to(DEVICE).double()
    lo, hi = (torch.from_numpy(a).to(DEVICE).double() for a in (_BOX_LO, _BOX_HI))
    x = (smp[:, :3] - lo) / (hi - lo)
    ang = math.pi * x[:, :, None] * 2.0 ** torch.arange(12, device=DEVICE, dtype=torch.float64)
    enc = torch.stack([ang.sin(), ang.cos()], -1).reshape(len(smp), 72)
    h = torch.cat([enc, smp[:, 3:9], torch.zeros((len(smp), 2), device=DEVICE, dtype=torch.float64)], 1)
    at = 0
    for i, (k, m) in enumerate(_LAYERS):
        w = flat[at:at + k * m].view(m, k)
        b = flat[at + k * m:at + k * m + m]
        at += k * m + m
        h = h @ w.t() + b
        if i < 4:
            h = h.relu()
    lobes = h[:, :40].reshape(-1, 8, 5)
    mu = lobes[..., :3] / lobes[..., :3].norm(dim=-1, keepdim=True)
    kappa = lobes[..., 3].clamp(-4.0, 9.0).exp()
    logw = torch.log_softmax(lobes[..., 4], -1)
    cosine = (mu * smp[:, None, 9:12]).sum(-1)
    logv = torch.log(kappa / (2.0 * math.pi * -torch.expm1(-2.0 * kappa))) + kappa * (cosine - 1.0)
    loss = -(smp[:, 12] * torch.logsumexp(logw + logv, -1)).mean()
    loss.backward()
    return dict(gradient=flat.grad.cpu().numpy(), loss=float(loss.detach()))


def exact(case, seed):
    if case["kind"] == "query" and case["api"] == "host" and case["rays"] <= 20000 and case["subdiv"] == 3:
        return _exact_query(case, seed)
    if case["kind"] == "gradient":
        return _exact_gradient(case, seed)
    return None  # images of whole paths, and queries too large to search without a BVH
