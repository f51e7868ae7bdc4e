"""Timed cases of the ray-query library, each through its public entry points.

A case is a dict of plain values.  listed() gives the cases that are timed by
name, draw() more of the same ranges, prepare() what a program holds before
the call (scene, volume, network, rays in device memory), run() one pass, and
exact() the same numbers in 64-bit arithmetic where the outputs have such
values.  Traversal results have none: which triangle a walk ends at depends on
the visit cap and on the rope and slab tolerances, which are defined in
32-bit arithmetic; the same holds for the marches' hit decisions.

Kinds:
  frame    closest hit of a camera's primary rays; with bounce, then one
           diffuse bounce ray per hit (the cooperative kernel for the
           primaries, its refill form for the bounces, as a renderer issues
           them); with shadow, then one any-hit ray per hit towards a light
  objects  three transformed objects, rays in host memory, object ids and
           interpolated hit attributes
  rebuild  kd-tree built on the device from a changed triangle soup, uploaded
           and traced
  chunk    terrain chunk generated at its origin, sphere traced with normals
           and shaded to pixels
  edit     brush edit of a resident volume, then the exact-field march of it
  hybrid   surrogate hybrid trace of a terrain volume
  forward  surrogate network at a set of points
  gradient loss and parameter gradient of one batch of host samples
  fit      a new network fitted to a volume: distance transform, sampling,
           Adam steps
  batch    scenes and terrain tiles traced by one captured graph
"""
from __future__ import annotations

import math

import numpy as np
import torch

import rayengine_amd as re
from rayengine_amd import workloads as W

_CTX = None


def _ctx() -> re.Context:
    """The program's one library context."""
    global _CTX
    if _CTX is None:
        _CTX = re.Context(0)
    return _CTX


def listed():
    return [
        # the smallest call: an icosphere among loose triangles, one picking-sized tile of rays
        {"name": "frame_small", "kind": "frame", "scene": "small", "tris": 6144, "width": 64, "height": 64,
         "bounce": False, "shadow": False},
        # an ordinary directly lit frame at an odd resolution
        {"name": "frame_shadow", "kind": "frame", "scene": "cluster", "tris": 50021, "width": 1001, "height": 563,
         "bounce": False, "shadow": True},
        # the headline: a million triangles, full-HD primaries and their diffuse bounces
        {"name": "frame_bounce", "kind": "frame", "scene": "cluster", "tris": 1 << 20, "width": 1920, "height": 1080,
         "bounce": True, "shadow": False},
        # a host program's query of a scene with moving objects, attributes included
        {"name": "objects_host", "kind": "objects", "tris": 20011, "rays": 100003},
        # geometry changed: the tree is rebuilt before the next frame
        {"name": "rebuild_frame", "kind": "rebuild", "scene": "cluster", "tris": 1 << 18, "leaf": 8, "width": 1280,
         "height": 720},
        # a new terrain chunk comes into view and is drawn
        {"name": "chunk_frame", "kind": "chunk", "dx": 256, "dy": 256, "dz": 256, "width": 1920, "height": 1080},
        # one brush stroke in a terrain editor and the redraw after it, ragged volume
        {"name": "edit_redraw", "kind": "edit", "dx": 203, "dy": 165, "dz": 187, "width": 1280, "height": 720},
        # terrain drawn through its learned distance
        {"name": "hybrid_frame", "kind": "hybrid", "dim": 192, "width": 1280, "height": 720, "steps": 1500},
        # learned distance at a large set of points (a collision or meshing grid)
        {"name": "net_forward", "kind": "forward", "points": 1000003},
        # one small training batch by hand, gradient back on the host
        {"name": "net_gradient", "kind": "gradient", "points": 8192},
        # a network fitted to a new chunk
        {"name": "net_fit", "kind": "fit", "dim": 128, "samples": 1 << 20, "batch": 65536, "steps": 256},
        # many small scenes and tiles in one launch
        {"name": "batch_mixed", "kind": "batch", "scenes": 24, "tiles": 6, "tri_lo": 1000, "tri_hi": 100000,
         "ray_lo": 8000, "ray_hi": 200000, "tile_lo": 64, "tile_hi": 160, "surrogate": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "objects", "rebuild", "chunk", "edit", "hybrid", "forward",
                       "gradient", "fit", "batch"])
    c = {"kind": kind}
    if kind == "frame":
        small = rng.random() < 0.25
        c["scene"] = "small" if small else "cluster"
        c["tris"] = 6144 if small else _log(rng, 2000, 1 << 20)
        c["width"] = _log(rng, 48, 1920)
        c["height"] = max(27, c["width"] * 9 // 16 + rng.randrange(-8, 1))
        c["bounce"] = rng.random() < 0.5
        c["shadow"] = not c["bounce"] and rng.random() < 0.6
    elif kind == "objects":
        c["tris"], c["rays"] = _log(rng, 500, 50000), _log(rng, 1000, 300000)
    elif kind == "rebuild":
        c["scene"], c["tris"], c["leaf"] = "cluster", _log(rng, 2000, 1 << 18), rng.choice([4, 8, 12])
        c["width"] = _log(rng, 48, 1280)
        c["height"] = max(27, c["width"] * 9 // 16)
    elif kind == "chunk":
        for a in ("dx", "dy", "dz"):
            c[a] = _log(rng, 40, 256)
        c["width"] = _log(rng, 160, 1920)
        c["height"] = c["width"] * 9 // 16
    elif kind == "edit":
        for a in ("dx", "dy", "dz"):
            c[a] = _log(rng, 40, 256)
        c["width"] = _log(rng, 160, 1920)
        c["height"] = c["width"] * 9 // 16
    elif kind == "hybrid":
        c["dim"], c["width"], c["steps"] = 8 * rng.randrange(8, 25), _log(rng, 160, 1280), 1500
        c["height"] = c["width"] * 9 // 16
    elif kind == "forward":
        c["points"] = _log(rng, 100, 4000000)
    elif kind == "gradient":
        c["points"] = 64 * _log(rng, 1, 1024)
    elif kind == "fit":
        c["dim"], c["samples"] = 8 * rng.randrange(6, 17), 1 << rng.randrange(16, 21)
        c["batch"], c["steps"] = 64 * _log(rng, 64, 1024), _log(rng, 16, 256)
    else:
        c.update(scenes=rng.randrange(1, 25), tiles=rng.randrange(0, 7), tri_lo=1000,
                 tri_hi=_log(rng, 5000, 100000), ray_lo=_log(rng, 1000, 8000), ray_hi=_log(rng, 10000, 200000),
                 tile_lo=64, tile_hi=160, surrogate=rng.random() < 0.5)
    return c


# ------------------------------------------------------------------ inputs

class _State(dict):
    """What a program holds; library objects are given back with it."""

    def __del__(self):
        try:
            for o in self.get("own", ()):
                o.release()
        except Exception:
            pass


_TILES = {}


def _tile_order(width, height):
    if (width, height) not in _TILES:
        _TILES[width, height] = W.tile_order(width, height)
    return _TILES[width, height]


def _dev(a, dtype=None):
    return torch.as_tensor(np.ascontiguousarray(a, dtype), device="cuda")


def _empty(*shape, dtype=torch.float32):
    return torch.empty(shape, dtype=dtype, device="cuda")


def _seed(seed, salt=0):
    return (int(seed) * 1000003 + salt) & 0x7FFFFFFF


def _soup(case, seed):
    if case["scene"] == "small":
        loose = case["tris"] - 5120
        return np.concatenate([re.icosphere(4, 1.0), re.random_tris(_seed(seed), loose, -2.0, 2.0, 0.02, 0.2)])
    return re.cluster_soup(_seed(seed), case["tris"], 64, -10.0, 10.0, 0.3, -3.0, 0.5)


def _camera(case, soup):
    """The small scene's camera, or one 0.8 units outside a cluster, looking
    through its centre (the cluster fills the view)."""
    if case["scene"] == "small":
        return W.SMALL_CAMERA
    c = soup.reshape(-1, 3, 3).mean(1, dtype=np.float64)
    near = c[np.argmin((c * c).sum(1))]
    for _ in range(2):
        near = c[((c - near) ** 2).sum(1) < 1.0].mean(0)
    out = near / (np.linalg.norm(near) + 1e-9)
    return re.Camera(pos=tuple(near + 0.8 * out), view=tuple(-out))


def _second(case):
    return case["width"] * case["height"] * 9 // 10


def _prepare_frame(case, seed):
    ctx = _ctx()
    soup = _soup(case, seed)
    scene = ctx.upload_scene([re.SceneObject(re.KDTree(soup, ctx=ctx))])
    o, d = re.camera_rays(_camera(case, soup), case["width"], case["height"])
    order = _tile_order(case["width"], case["height"])
    o, d = o[order], d[order]
    n = len(o)
    s = _State(own=[scene], scene=scene, n=n, o=_dev(o), d=_dev(d), prim=_empty(n, dtype=torch.int32), t=_empty(n))
    if case["bounce"] or case["shadow"]:
        prim, t = scene.trace_closest(o, d)
        if case["bounce"]:
            so, sd = re.bounce_rays(soup, o, d, prim, t, _seed(seed, 1))
        else:
            so, sd = W.shadow_rays(soup, o, d, prim, t, W.CLUSTER_LIGHT)
        # one secondary ray per hit, spread evenly over the hits to nine tenths of the pixels: as many rays
        # whatever the share of the view that the seed's cluster fills (95 % or so)
        m = _second(case)
        pick = np.arange(m) * len(so) // m
        s.update(m=m, so=_dev(so[pick]), sd=_dev(sd[pick]))
        if case["bounce"]:
            s.update(sprim=_empty(m, dtype=torch.int32), st=_empty(m))
        else:
            s.update(occ=_empty(m, dtype=torch.uint8))
    return s


def _run_frame(s):
    s["scene"].trace_closest_device(s["o"].data_ptr(), s["d"].data_ptr(), s["n"], s["prim"].data_ptr(),
                                    s["t"].data_ptr(), sync=False)
    out = {"prim": s["prim"], "t": s["t"]}
    if "sprim" in s:
        s["scene"].trace_closest_device(s["so"].data_ptr(), s["sd"].data_ptr(), s["m"], s["sprim"].data_ptr(),
                                        s["st"].data_ptr(), sync=False, variant=5)
        out.update(bounce_prim=s["sprim"], bounce_t=s["st"])
    if "occ" in s:
        s["scene"].occluded_device(s["so"].data_ptr(), s["sd"].data_ptr(), s["m"], s["occ"].data_ptr(), sync=False)
        out.update(occluded=s["occ"])
    return out


def _prepare_objects(case, seed):
    ctx = _ctx()
    rng = np.random.default_rng(_seed(seed, 2))
    k = case["tris"] // 3
    soups = [re.random_tris(_seed(seed, i), k if i else case["tris"] - 2 * k, -2.0, 2.0, 0.05, 0.5) for i in range(3)]
    objs, off = [], 0
    for i, soup in enumerate(soups):
        objs.append(re.SceneObject(re.KDTree(soup), location=tuple(rng.uniform(-1.5, 1.5, 3)),
                                   rotation_y=float(rng.uniform(0, 6.28)), prim_offset=off))
        off += len(soup)
    scene = ctx.upload_scene(objs)
    normals = rng.standard_normal((off, 9)).astype(np.float32)
    uvs = rng.random((off, 6)).astype(np.float32)
    scene.set_attributes(normals, uvs)
    n = case["rays"]
    o = rng.uniform(-6, 6, (n, 3))
    d = rng.uniform(-2, 2, (n, 3)) - o
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return _State(own=[scene], scene=scene, o=o.astype(np.float32), d=d.astype(np.float32))


def _run_objects(s):
    prim, t, obj = s["scene"].trace_closest(s["o"], s["d"], with_obj=True, one_sided=False)
    normal, uv, bary, point = s["scene"].hit_attributes(s["o"], s["d"], prim, obj, one_sided=False)
    return {"prim": prim, "t": t, "obj": obj, "normal": normal, "uv": uv, "bary": bary, "point": point}


def _prepare_rebuild(case, seed):
    soup = _soup(case, seed)
    o, d = re.camera_rays(_camera(case, soup), case["width"], case["height"])
    order = _tile_order(case["width"], case["height"])
    n = len(o)
    return _State(soup=soup, leaf=case["leaf"], n=n, o=_dev(o[order]), d=_dev(d[order]),
                  prim=_empty(n, dtype=torch.int32), t=_empty(n))


def _run_rebuild(s):
    ctx = _ctx()
    scene = ctx.upload_scene([re.SceneObject(re.KDTree(s["soup"], max_leaf_tris=s["leaf"], ctx=ctx))])
    scene.trace_closest_device(s["o"].data_ptr(), s["d"].data_ptr(), s["n"], s["prim"].data_ptr(),
                               s["t"].data_ptr(), sync=False)
    scene.release()
    return {"prim": s["prim"], "t": s["t"]}


def _dims(case):
    return (case["dx"], case["dy"], case["dz"])


def _terrain_rays(case):
    o, d = re.camera_rays(W.TERRAIN_CAMERA, case["width"], case["height"])
    return _dev(o), _dev(d), len(o)


def _prepare_chunk(case, seed):
    dim = _dims(case)
    o, d, n = _terrain_rays(case)
    rng = np.random.default_rng(_seed(seed, 3))
    return _State(dim=dim, spacing=tuple(1.0 / v for v in dim), perm=_seed(seed), n=n, o=o, d=d,
                  origin=(float(rng.integers(-8, 8)), 0.0, float(rng.integers(-8, 8))),
                  width=case["width"], height=case["height"], t=_empty(n), hit=_empty(n, dtype=torch.uint8),
                  steps=_empty(n, dtype=torch.int32), normal=_empty(n, 3), rgba=_empty(n, dtype=torch.int32))


def _run_chunk(s):
    ctx = _ctx()
    vol = ctx.noise_volume(dim=s["dim"], spacing=s["spacing"], seed=s["perm"], origin=s["origin"])
    vol.trace_device(s["o"].data_ptr(), s["d"].data_ptr(), s["n"], s["t"].data_ptr(), s["hit"].data_ptr(),
                     s["steps"].data_ptr(), s["normal"].data_ptr(), sync=False)
    re.frame_shade_device(ctx, s["d"].data_ptr(), s["hit"].data_ptr(), s["normal"].data_ptr(), s["width"],
                          s["height"], s["rgba"].data_ptr(), sync=False)
    vol.release()
    return {k: s[k] for k in ("t", "hit", "steps", "normal", "rgba")}


def _prepare_edit(case, seed):
    dim = _dims(case)
    o, d, n = _terrain_rays(case)
    rng = np.random.default_rng(_seed(seed, 4))
    vol = _ctx().noise_volume(dim=dim, spacing=tuple(1.0 / v for v in dim), seed=_seed(seed))
    c = (float(rng.uniform(0.3, 0.7)), float(rng.uniform(0.3, 0.5)), float(rng.uniform(0.2, 0.6)))
    return _State(own=[vol], vol=vol, n=n, o=o, d=d, center=c, radius=float(rng.uniform(0.08, 0.2)), t=_empty(n),
                  hit=_empty(n, dtype=torch.uint8))


def _run_edit(s):
    r = s["radius"]
    s["vol"].edit("sphere_subtract", center=s["center"], extent=(r, r, r), material=2.0)
    re.hybrid_trace_device(s["vol"], None, s["o"].data_ptr(), s["d"].data_ptr(), s["n"], s["t"].data_ptr(),
                           s["hit"].data_ptr(), sync=False, k_exact=0.05, h_min_voxels=1.0, n_bisect=1)
    return {"t": s["t"], "hit": s["hit"]}


def _fitted(ctx, vol, seed, steps):
    """A network fitted to the volume, as a program would have it at hand."""
    dist = re.distance_volume(vol)
    net = re.Surrogate(ctx, seed=seed)
    net.train(dist, n_samples=1 << 20, batch=65536, steps=steps, seed=seed)
    dist.release()
    return net


def _prepare_hybrid(case, seed):
    ctx = _ctx()
    dm = case["dim"]
    vol = ctx.noise_volume(dim=(dm,) * 3, spacing=(1.0 / dm,) * 3, seed=_seed(seed))
    net = _fitted(ctx, vol, _seed(seed, 5), case["steps"])
    o, d, n = _terrain_rays(case)
    return _State(own=[vol, net], vol=vol, net=net, n=n, o=o, d=d, t=_empty(n), hit=_empty(n, dtype=torch.uint8))


def _run_hybrid(s):
    re.hybrid_trace_device(s["vol"], s["net"], s["o"].data_ptr(), s["d"].data_ptr(), s["n"], s["t"].data_ptr(),
                           s["hit"].data_ptr(), sync=False, tau_voxels=4.0, margin_voxels=1.0, k_exact=0.1, n_bisect=4)
    return {"t": s["t"], "hit": s["hit"]}


# the network: 99 inputs (sin and cos of 2 pi f p for 16 frequencies f = 2^(k/2) per coordinate, then the
# coordinates), four hidden layers of 64 SiLU units, one linear output; parameters flat, layer by layer
_LAYERS = [(64, 99), (64, 64), (64, 64), (64, 64), (1, 64)]


def _weights(seed):
    rng = np.random.default_rng(_seed(seed, 6))
    parts = []
    for fan_out, fan_in in _LAYERS:
        bound = math.sqrt(3.0 / fan_in)
        parts += [rng.uniform(-bound, bound, fan_out * fan_in), rng.uniform(-0.1, 0.1, fan_out)]
    return np.concatenate(parts).astype(np.float32)


def _points(case, seed):
    return np.random.default_rng(_seed(seed, 7)).random((case["points"], 3), np.float32)


def _targets(case, seed):
    """Distances as training meets them: half of them close to the surface."""
    rng = np.random.default_rng(_seed(seed, 8))
    far = rng.uniform(-0.4, 0.6, case["points"])
    near = rng.uniform(-0.01, 0.01, case["points"])
    return np.where(np.arange(case["points"]) % 2 == 0, far, near).astype(np.float32)


def _network64(params, pts):
    x = torch.as_tensor(pts, dtype=torch.float64, device=params.device)
    f = 2.0 ** (torch.arange(16, dtype=torch.float64, device=params.device) / 2)
    a = 2 * math.pi * x[:, :, None] * f
    h = torch.cat([torch.stack([a.sin(), a.cos()], -1).reshape(len(x), 96), x], 1)
    at = 0
    for i, (fan_out, fan_in) in enumerate(_LAYERS):
        w = params[at:at + fan_out * fan_in].reshape(fan_out, fan_in)
        b = params[at + fan_out * fan_in:at + fan_out * (fan_in + 1)]
        at += fan_out * (fan_in + 1)
        h = h @ w.T + b
        if i < 4:
            h = h * torch.sigmoid(h)
    return h[:, 0]


def _prepare_net(case, seed):
    net = re.Surrogate(_ctx())
    net.set_params(_weights(seed))
    pts = _points(case, seed)
    s = _State(own=[net], net=net)
    if case["kind"] == "forward":
        s.update(pts=_dev(pts), n=len(pts), out=_empty(len(pts)))
    else:
        s["samples"] = np.concatenate([pts, _targets(case, seed)[:, None]], 1)
    return s


def _run_forward(s):
    s["net"].forward_device(s["pts"].data_ptr(), s["n"], s["out"].data_ptr(), sync=False)
    return s["out"]


def _run_gradient(s):
    loss, grad = s["net"].batch_step(s["samples"], over_weight=4.0)
    return {"loss": loss, "grad": grad}


def _prepare_fit(case, seed):
    dm = case["dim"]
    vol = _ctx().noise_volume(dim=(dm,) * 3, spacing=(1.0 / dm,) * 3, seed=_seed(seed))
    return _State(own=[vol], vol=vol, seed=_seed(seed, 9), case=case)


def _run_fit(s):
    c = s["case"]
    net = re.Surrogate(_ctx(), seed=s["seed"])
    dist = re.distance_volume(s["vol"])
    loss = net.train(dist, n_samples=c["samples"], batch=min(c["batch"], c["samples"]), steps=c["steps"],
                     seed=s["seed"])
    params, m, v, _ = net.params()
    dist.release()
    net.release()
    return {"loss": loss, "params": params, "m": m, "v": v}


def _spread(lo, hi, n):
    """n sizes log-spaced over [lo, hi]."""
    return [int(round(lo * (hi / lo) ** (i / max(n - 1, 1)))) for i in range(n)]


def _tile_dims(case):
    return [8 * round(v / 8) for v in _spread(case["tile_lo"], case["tile_hi"], case["tiles"])]


def _batch_rays(case):
    scenes = _spread(case["ray_lo"], case["ray_hi"], case["scenes"])
    return scenes, _spread(case["ray_lo"], case["ray_hi"], case["tiles"])[::-1]


def _incoherent(rng, lo, hi, n):
    mid, r = (lo + hi) / 2, 0.75 * np.linalg.norm(hi - lo) + 1e-3
    u = rng.standard_normal((n, 3))
    o = mid + r * u / np.linalg.norm(u, axis=1, keepdims=True)
    d = lo + (hi - lo) * rng.random((n, 3)) - o
    return o.astype(np.float32), (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)


def _prepare_batch(case, seed):
    ctx = _ctx()
    rng = np.random.default_rng(_seed(seed, 10))
    rays_s, rays_t = _batch_rays(case)
    scenes, tiles, os_, ds_, own, at = [], [], [], [], [], 0
    for i, (tris, n) in enumerate(zip(_spread(case["tri_lo"], case["tri_hi"], case["scenes"]), rays_s)):
        soup = re.cluster_soup(_seed(seed, 100 + i), tris, 64, -10.0, 10.0, 0.3, -3.0, 0.5)
        v = soup.reshape(-1, 3).astype(np.float64)
        o, d = _incoherent(rng, v.min(0), v.max(0), n)
        scenes.append((re.KDTree(soup, ctx=ctx), at, n))
        os_.append(o)
        ds_.append(d)
        at += n
    for i, (dm, n) in enumerate(zip(_tile_dims(case), rays_t)):
        vol = ctx.noise_volume(dim=(dm,) * 3, spacing=(1.0 / dm,) * 3, seed=_seed(seed, 200 + i))
        own.append(vol)
        o, d = _incoherent(rng, np.zeros(3), np.ones(3), n)
        mode = (0, 1, 0, 2 if case["surrogate"] else 1)[i % 4]
        if mode == 2:
            own.append(_fitted(ctx, vol, _seed(seed, 300 + i), 300))
            tiles.append((vol, mode, at, n, own[-1]))
        else:
            tiles.append((vol, mode, at, n))
        os_.append(o)
        ds_.append(d)
        at += n
    b = re.Batch(ctx, scenes, tiles, np.concatenate(os_), np.concatenate(ds_),
                 side_share=0.375 if case["surrogate"] else 0.0,
                 march=dict(k_exact=0.05, h_min_voxels=1.0, n_bisect=1),
                 hybrid=dict(tau_voxels=4.0, margin_voxels=1.0, k_exact=0.1, n_bisect=4))
    return _State(own=[b] + own, batch=b)


def _run_batch(s):
    s["batch"].run(sync=False)
    prim, t = s["batch"].results()
    return {"prim": prim, "t": t}


_PREPARE = {"frame": _prepare_frame, "objects": _prepare_objects, "rebuild": _prepare_rebuild, "chunk": _prepare_chunk,
            "edit": _prepare_edit, "hybrid": _prepare_hybrid, "forward": _prepare_net, "gradient": _prepare_net,
            "fit": _prepare_fit, "batch": _prepare_batch}
_RUN = {"frame": _run_frame, "objects": _run_objects, "rebuild": _run_rebuild, "chunk": _run_chunk, "edit": _run_edit,
        "hybrid": _run_hybrid, "forward": _run_forward, "gradient": _run_gradient, "fit": _run_fit,
        "batch": _run_batch}


def prepare(case, seed):
    s = _PREPARE[case["kind"]](case, seed)
    s["kind"] = case["kind"]
    # the inputs were written on torch's stream and are read on the context's
    torch.cuda.synchronize()
    return s


def run(state):
    return _RUN[state["kind"]](state)


# ------------------------------------------------------------------ work

# multiply-adds of one network evaluation, two operations each
_NET_FLOPS = 2 * sum(a * b for a, b in _LAYERS)


def work(case):
    """Bytes: inputs once (rays 24, triangles 36, points 12, grid values 4)
    and results once; operations: network products, and about 350 per voxel
    of noise.  What a walk or a march reads on its way depends on the data
    and is not counted."""
    k = case["kind"]
    if k == "frame":
        n = case["width"] * case["height"]
        m = _second(case)
        return {"bytes": 32 * n + (32 * m if case["bounce"] else 25 * m if case["shadow"] else 0), "flops": 0}
    if k == "objects":
        return {"bytes": case["rays"] * (24 + 12 + 40) + 96 * case["tris"], "flops": 0}
    if k == "rebuild":
        return {"bytes": 36 * case["tris"] + 40 * case["tris"] + 32 * case["width"] * case["height"], "flops": 0}
    if k in ("chunk", "edit"):
        vox, n = case["dx"] * case["dy"] * case["dz"], case["width"] * case["height"]
        if k == "chunk":
            return {"bytes": 4 * vox + n * (24 + 9 + 12 + 4), "flops": 350 * vox}
        return {"bytes": 16 * vox + n * (24 + 5), "flops": 0}
    if k == "hybrid":
        n = case["width"] * case["height"]
        return {"bytes": n * (24 + 5) + 4 * case["dim"] ** 3, "flops": n * _NET_FLOPS}
    if k == "forward":
        return {"bytes": 16 * case["points"], "flops": case["points"] * _NET_FLOPS}
    if k == "gradient":
        return {"bytes": 16 * case["points"] + 4 * 18945, "flops": 3 * case["points"] * _NET_FLOPS}
    if k == "fit":
        b = min(case["batch"], case["samples"])
        return {"bytes": 8 * case["dim"] ** 3 + case["steps"] * (16 * b + 24 * 18945) + 16 * case["samples"],
                "flops": 3 * case["steps"] * b * _NET_FLOPS}
    rays_s, rays_t = _batch_rays(case)
    net = sum(n for i, n in enumerate(rays_t) if case["surrogate"] and i % 4 == 3)
    return {"bytes": 32 * (sum(rays_s) + sum(rays_t)), "flops": net * _NET_FLOPS}


# ------------------------------------------------------------------ exact

def exact(case, seed):
    if case["kind"] not in ("forward", "gradient"):
        return None
    params = torch.as_tensor(_weights(seed), dtype=torch.float64, device="cuda")
    pts = _points(case, seed)
    if case["kind"] == "forward":
        return torch.cat([_network64(params, pts[i:i + (1 << 18)]) for i in range(0, len(pts), 1 << 18)])
    params.requires_grad_(True)
    r = _network64(params, pts) - torch.as_tensor(_targets(case, seed), dtype=torch.float64, device="cuda")
    loss = (torch.where(r > 0, 4.0, 1.0) * r * r).mean()
    loss.backward()
    return {"loss": float(loss.detach()), "grad": params.grad}
