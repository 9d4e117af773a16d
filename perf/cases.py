"""Performance cases: what a renderer built on this package has it do, through its public entry points.

A caller either traces its own ray batches (closest hits, shadow segments, transparent shadows, subsurface
probes, many scenes at once), or hands over whole frames (one render, a render server, the finished film's
EXR file). The listed cases hold one or two sizes of each, from a thousand rays in a room of four thousand
triangles, where launches count, to four million bounce rays through a million triangles. Scenes and rays
are those of the benchmark and the tests (the Cornell room, icospheres on a ground plane, triangle soups),
made from the seed on the GPU.

* ``listed()`` / ``draw(rng)``: the cases; a drawn one has sizes from the same ranges.
* ``prepare(case, seed)``: the built accelerators, scenes and ray batches a program holds before the call.
* ``run(state)``: one call of the path, its whole result.
* ``work(case)``: bytes and operations one call cannot do without.
* ``exact(case, seed)``: closest hits in 64 bits by testing every triangle, where that is quick enough.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from sort_amd import Context, Obvh, Qbvh, film, integrator, scenes, serve
from sort_amd.batch import Pool

FLT_MAX = 3.4028234663852886e38

# What each case stands for:
#   closest_small      a viewport pick or one tile's last rays: 1,000 bounce rays in the Cornell room
#   closest_mid        one tile row's bounce rays, below the batch size that is sorted, on a 4-wide tree
#   closest_bounce     the headline workload: 4,194,304 bounce rays through 2^20 triangles, 8-wide
#   closest_camera     the primary rays of a 1920 x 1080 frame, in pixel order, on a mesh of 150 spheres
#   occluded           shadow segments to an area light, an odd count, through a 300K-triangle soup
#   attenuation        the same with half of the triangles transparent (SORT's transparent shadows)
#   multi              subsurface probes: up to four hits of one material along short segments
#   pool               twelve scenes of uneven size and uneven batches, traced by one launch
#   render_cornell     the small frame: 256 x 256, 16 samples, depth 5 (1M paths)
#   render_spheres     the large frame: 640 x 480, 24 samples, depth 8, 100 spheres (7.4M paths)
#   served             a render server's mix: five requests over three resident scenes, all at once
#   film               the EXR file of a finished 1920 x 1080 frame that lies in HBM


def listed():
    return [
        dict(name="closest_small", kind="closest", scene="cornell", tris=4056, rays=1000, pattern="bounce", width=8),
        dict(name="closest_mid", kind="closest", scene="soup", tris=50021, rays=100003, pattern="bounce", width=4),
        dict(name="closest_bounce", kind="closest", scene="soup", tris=1 << 20, rays=1 << 22, pattern="bounce", width=8),
        dict(name="closest_camera", kind="closest", scene="spheres", tris=768002, rays=1920 * 1080, pattern="camera",
             width=8),
        dict(name="occluded", kind="occluded", scene="soup", tris=300007, rays=1500001, width=8),
        dict(name="attenuation", kind="attenuation", scene="soup", tris=200003, rays=600011, width=8),
        dict(name="multi", kind="multi", scene="soup", tris=200003, rays=500009, width=8),
        dict(name="pool", kind="pool", scenes=12, tris=60000, rays=150000, width=4),
        dict(name="render_cornell", kind="render", scene="cornell", tris=4056, w=256, h=256, spp=16, depth=5, width=8),
        dict(name="render_spheres", kind="render", scene="spheres", tris=512002, w=640, h=480, spp=24, depth=8, width=8),
        dict(name="served", kind="served", scenes=3, tris=60000, requests=5, res=256, spp=8, depth=8, width=4),
        dict(name="film", kind="film", w=1920, h=1080),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["closest", "closest", "occluded", "occluded", "attenuation", "multi", "pool", "render",
                       "render", "served", "film"])
    width = rng.choice([8, 4])
    if kind == "film":
        return dict(kind=kind, w=_logint(rng, 64, 1920), h=_logint(rng, 48, 1080))
    if kind == "served":
        return dict(kind=kind, scenes=rng.randint(1, 4), tris=_logint(rng, 5000, 60000), requests=rng.randint(2, 6),
                    res=_logint(rng, 64, 256), spp=_logint(rng, 2, 8), depth=rng.randint(4, 8), width=width)
    if kind == "pool":
        return dict(kind=kind, scenes=rng.randint(2, 16), tris=_logint(rng, 1000, 60000),
                    rays=_logint(rng, 500, 150000), width=width)
    if kind == "render":
        if rng.random() < 0.5:
            return dict(kind=kind, scene="cornell", tris=4056, w=_logint(rng, 32, 400), h=_logint(rng, 32, 400),
                        spp=_logint(rng, 1, 16), depth=rng.randint(1, 8), width=width)
        return dict(kind=kind, scene="spheres", tris=2 + 5120 * rng.randint(10, 100), w=_logint(rng, 64, 640),
                    h=_logint(rng, 48, 480), spp=_logint(rng, 1, 24), depth=rng.randint(2, 8), width=width)
    rays = _logint(rng, 200, 1500000 if kind != "closest" else 1 << 22)
    scene = rng.choice(["soup", "soup", "cornell", "spheres"]) if kind in ("closest", "occluded") else "soup"
    tris = {"soup": _logint(rng, 2000, 1 << 20 if kind == "closest" else 300000), "cornell": 4056,
            "spheres": 2 + 5120 * rng.randint(5, 150)}[scene]
    c = dict(kind=kind, scene=scene, tris=tris, rays=rays, width=width)
    if kind == "closest":
        c["pattern"] = rng.choice(["bounce", "camera"])
    return c


# ---- inputs ------------------------------------------------------------------------------------------

_CTX = None


def _ctx():
    global _CTX
    if _CTX is None:
        _CTX = Context(0)
    return _CTX


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _unit(v):
    return v / v.norm(dim=-1, keepdim=True)


def _soup(n, g):
    """n triangles, centroids uniform in the unit cube, sizes LogNormal(ln 0.004, 0.5) at 2^20 triangles and
    larger in proportion to the spacing of fewer."""
    c = torch.rand((n, 1, 3), generator=g, device="cuda")
    s = torch.exp(torch.randn((n, 1, 1), generator=g, device="cuda") * 0.5) * (0.004 * ((1 << 20) / n) ** (1 / 3))
    a = _unit(torch.randn((n, 3, 3), generator=g, device="cuda"))
    v = c + s * (a - a.mean(dim=1, keepdim=True))
    pos = v.reshape(-1, 3).cpu().numpy()
    return pos, np.arange(3 * n, dtype=np.uint32).reshape(-1, 3)


_MADE = {}  # the unit sphere and the room, the same for every seed


def _geometry(case, seed):
    """dict(pos, idx, quads, normals, tri_material, materials, quad_radiance, env, camera) of the case's scene."""
    kind, n, g = case.get("scene", "soup"), case["tris"], _gen(seed)
    if kind == "cornell":
        if "cornell" not in _MADE:
            _MADE["cornell"] = scenes.cornell_sphere()
        sc = dict(_MADE["cornell"])
        jit = np.random.default_rng(seed).uniform(-0.02, 0.02, 3)  # each seed looks from another place
        sc["camera"] = dict(sc["camera"], eye=tuple(float(x) for x in np.array([0.5, 0.5, 0.03]) + jit * [1, 1, 0.5]))
        return sc
    if kind == "spheres":
        make = scenes.icosphere
        if "ico" not in _MADE:
            _MADE["ico"] = make(5)
        scenes.icosphere = lambda level=5: _MADE["ico"]
        try:
            return scenes.spheres_scene((n - 2) // 5120, seed=seed)
        finally:
            scenes.icosphere = make
    pos, idx = _soup(n, g)
    u = torch.randint(0, 8, (n,), generator=g, device="cuda").to(torch.int32).cpu().numpy().view(np.uint32)
    I = integrator
    mats = [I.lambert((0.7, 0.7, 0.7)), I.lambert((0.8, 0.3, 0.2)), I.lambert((0.2, 0.6, 0.3)), I.lambert((0.3, 0.4, 0.8)),
            I.ggx((0.9, 0.8, 0.6), 0.2), I.ggx((0.7, 0.7, 0.75), 0.5),
            I.dielectric((1, 1, 1), (1, 1, 1), roughness=0.05, ior=1.5),
            I.dielectric((1, 1, 1), (0.9, 1, 0.9), roughness=0.15, ior=1.5)]
    return dict(pos=pos, idx=idx, quads=[scenes.translate_quad((0.5, 1.3, 0.5), 0.5, facing_down=True)],
                normals=None, tri_material=u, materials=mats, quad_radiance=np.full((1, 3), 8.0, np.float32),
                env=(0.25, 0.3, 0.35), camera=dict(eye=(0.5, 0.5, -1.5), target=(0.5, 0.5, 0.5), up=(0, 1, 0),
                                                   fov_y_deg=40.0))


def _accel(case, geo, quads=True):
    cls = Obvh if case["width"] == 8 else Qbvh
    return cls(_ctx()).build(geo["pos"], geo["idx"], geo["quads"] if quads else None)


def _camera_rays(cam, n):
    """n primary rays through the pixel centres of a 16:9 frame, row by row."""
    w = max(1, int(round(math.sqrt(n * 16 / 9))))
    h = -(-n // w)
    e = torch.tensor(cam["eye"], device="cuda", dtype=torch.float32)
    f = _unit(torch.tensor(cam["target"], device="cuda", dtype=torch.float32) - e)
    r = _unit(torch.linalg.cross(f, torch.tensor([0.0, 1.0, 0.0], device="cuda")))
    u = torch.linalg.cross(r, f)
    i = torch.arange(n, device="cuda")
    th = math.tan(math.radians(cam["fov_y_deg"]) * 0.5)
    x = ((i % w).float() + 0.5) / w * 2 - 1
    y = 1 - (torch.div(i, w, rounding_mode="floor").float() + 0.5) / h * 2
    d = _unit(f + (x * th * w / h)[:, None] * r + (y * th)[:, None] * u)
    return _rays(e.expand(n, 3), 0.0, d, FLT_MAX)


def _rays(o, tmin, d, tmax):
    out = torch.empty((o.shape[0], 8), device="cuda")
    out[:, 0:3] = o
    out[:, 3] = tmin
    out[:, 4:7] = d
    out[:, 7] = tmax
    return out


def _surface_points(acc, geo, n, g):
    """n random points that the scene's camera sees, and their normals facing it."""
    cam = _camera_rays(geo["camera"], 1 << 18)
    hits = acc.get_intersect(cam)
    prim = hits.view(torch.int32)[:, 1].long()
    ok = torch.nonzero((prim >= 0) & (prim < len(geo["idx"]))).flatten()
    pick = ok[torch.randint(0, ok.numel(), (n,), generator=g, device="cuda")]
    d = cam[pick, 4:7]
    p = cam[pick, 0:3] + hits[pick, 0:1] * d
    idx = torch.from_numpy(geo["idx"].view(np.int32)).cuda().long()[prim[pick]]
    pos = torch.from_numpy(geo["pos"]).cuda()
    v = pos[idx]
    nrm = torch.linalg.cross(v[:, 2] - v[:, 0], v[:, 1] - v[:, 0])
    nrm = nrm / nrm.norm(dim=1, keepdim=True).clamp_min(1e-20)
    return p, torch.where((nrm * d).sum(1, keepdim=True) > 0, -nrm, nrm), d


def _bounce_rays(acc, geo, n, g):
    """Cosine-distributed rays leaving random visible points, as a path's next vertex casts them."""
    p, nrm, _ = _surface_points(acc, geo, n, g)
    d = nrm + _unit(torch.randn((n, 3), generator=g, device="cuda"))
    return _rays(p, 1e-4, _unit(d + 1e-6 * nrm), FLT_MAX)


def _shadow_rays(acc, geo, n, g):
    """Segments from random visible points to random points of the scene's first area light."""
    p, _, _ = _surface_points(acc, geo, n, g)
    q = geo["quads"][0]
    c = torch.tensor(np.asarray(q["mat"], np.float32).reshape(4, 4)[:3, 3].copy(), device="cuda")
    u = (torch.rand((n, 2), generator=g, device="cuda") - 0.5) * float(q["size_x"])
    v = c + torch.stack([u[:, 0], torch.zeros_like(u[:, 0]), u[:, 1]], 1) - p
    ln = v.norm(dim=1)
    return _rays(p, 0.01, v / ln[:, None], ln - 0.01)


def _pool_sizes(case):
    """(triangles, rays) of each scene of a pool: LogNormal factors around the case's sizes, up to four times."""
    rs = np.random.default_rng(case["tris"] + case["rays"])
    f = np.minimum(np.exp(rs.normal(0.0, 0.8, (case["scenes"], 2))), 4.0)
    return [(max(64, int(case["tris"] * a)), max(64, int(case["rays"] * b))) for a, b in f]


def prepare(case, seed):
    kind, g = case["kind"], _gen(seed + 1)
    if kind == "film":
        img = torch.exp(torch.randn((case["h"], case["w"], 3), generator=g, device="cuda") * 1.5 - 1.0)
        return dict(kind=kind, film=img)
    if kind == "pool":
        accs, rays, ids = [], [], []
        for i, (tris, n) in enumerate(_pool_sizes(case)):
            geo = _geometry(dict(case, tris=tris), seed * 100 + i)
            acc = _accel(case, geo, quads=False)
            accs.append(acc)
            rays.append(_bounce_rays(acc, geo, n, g))
            ids.append(torch.full((n,), i, dtype=torch.int32, device="cuda"))
        return dict(kind=kind, pool=Pool(_ctx(), accs), rays=torch.cat(rays), ids=torch.cat(ids))
    if kind == "served":
        srv = serve.Server(_ctx(), hbm_budget=16 << 30, wave_paths=1 << 21)
        rs, reqs, sids = np.random.default_rng(seed), [], []
        for i in range(case["scenes"]):
            geo = _geometry(case, seed * 100 + i)
            sids.append(srv.add_scene(_accel(case, geo), geo["materials"], tri_material=geo["tri_material"],
                                      quad_radiance=geo["quad_radiance"], env_radiance=geo["env"]))
        for i in range(case["requests"]):
            f = (1, 2, 1, 1, 2, 1)[i % 6]
            reqs.append((sids[i % len(sids)], serve.random_camera(rs), case["res"] * f, case["res"] * f,
                         max(1, case["spp"] // f), case["depth"], seed * 1000 + i))
        return dict(kind=kind, server=srv, requests=reqs)
    geo = _geometry(case, seed)
    acc = _accel(case, geo)
    if kind == "render":
        pt = integrator.PathTracing(acc, geo["materials"], tri_material=geo["tri_material"], normals=geo["normals"],
                                    quad_radiance=geo["quad_radiance"], env_radiance=geo["env"],
                                    max_recursive_depth=case["depth"])
        return dict(kind=kind, pt=pt, acc=acc, cam=integrator.camera(**geo["camera"]), w=case["w"], h=case["h"],
                    spp=case["spp"], seed=seed)
    n, st = case["rays"], dict(kind=kind, acc=acc)
    if kind == "closest":
        st["rays"] = _camera_rays(geo["camera"], n) if case["pattern"] == "camera" else _bounce_rays(acc, geo, n, g)
    elif kind == "multi":
        p, _, d = _surface_points(acc, geo, n, g)
        d = _unit(d + 0.3 * torch.randn((n, 3), generator=g, device="cuda"))
        st["rays"] = _rays(p - 0.02 * d, 0.0, d, 0.04)
        st["tri_mat"] = torch.from_numpy((geo["tri_material"] & 3).view(np.int32)).cuda()
        first = acc.get_intersect(st["rays"]).view(torch.int32)[:, 1].long()
        hit = (first >= 0) & (first < len(geo["idx"]))
        st["ray_mat"] = torch.where(hit, st["tri_mat"][torch.where(hit, first, 0)], 0).to(torch.int32).contiguous()
    else:
        st["rays"] = _shadow_rays(acc, geo, n, g)
        if kind == "attenuation":
            tr = torch.rand((len(geo["idx"]) + 1, 4), generator=g, device="cuda")
            tr[:, :3] = 0.2 + 0.8 * tr[:, :3]
            tr[:, 3] = (tr[:, 3] < 0.5).float()
            st["tr"] = tr.contiguous()
    return st


# ---- one pass ----------------------------------------------------------------------------------------

def _hits(h):
    return {"t": h[..., 0], "prim": h.view(torch.int32)[..., 1], "uv": h[..., 2:]}


def run(st):
    kind = st["kind"]
    if kind == "closest":
        return _hits(st["acc"].get_intersect(st["rays"]))
    if kind == "occluded":
        return st["acc"].is_occluded(st["rays"])
    if kind == "attenuation":
        return st["acc"].attenuation(st["rays"], st["tr"])
    if kind == "multi":
        h, c = st["acc"].multi(st["rays"], st["ray_mat"], st["tri_mat"])
        return dict(_hits(h), count=c)
    if kind == "pool":
        return _hits(st["pool"].trace(st["rays"], st["ids"]))
    if kind == "render":
        return st["pt"].render(st["cam"], st["w"], st["h"], st["spp"], seed=st["seed"])
    if kind == "served":
        srv, out = st["server"], []
        rids = [srv.submit(*r) for r in st["requests"]]
        for rid in rids:
            srv.wait(rid)
            out.append(srv.result(rid))
            srv.release(rid)
        return out
    return np.frombuffer(film.encode_exr(st["film"]), np.uint8)


# ---- what one pass cannot do without -----------------------------------------------------------------

# A ray reads 32 bytes and writes its record; a tree holds at least nine floats and an id per triangle and is
# read once; a ray tests eight boxes (three subtractions and products, two comparisons per plane pair) on each
# level of an 8-wide tree and one triangle.
def _ray_flops(tris):
    return 8 * 18 * max(1.0, math.log(max(tris, 8), 8)) + 50


def work(case):
    kind = case["kind"]
    if kind == "film":
        return {"bytes": case["w"] * case["h"] * 18.0, "flops": 0.0}
    if kind == "pool":
        sizes = _pool_sizes(case)
        return {"bytes": float(sum(52 * n + 40 * t for t, n in sizes)),
                "flops": sum(n * _ray_flops(t) for t, n in sizes)}
    if kind in ("render", "served"):
        if kind == "render":
            pix, paths = case["w"] * case["h"], case["w"] * case["h"] * case["spp"]
        else:
            fs = [(1, 2, 1, 1, 2, 1)[i % 6] for i in range(case["requests"])]
            pix = sum((case["res"] * f) ** 2 for f in fs)
            paths = sum((case["res"] * f) ** 2 * max(1, case["spp"] // f) for f in fs)
        # at least a camera ray and, for half of the paths, one shadow ray
        return {"bytes": 12.0 * pix + 40.0 * case["tris"] * case.get("scenes" if kind == "served" else "", 1),
                "flops": 1.5 * paths * _ray_flops(case["tris"])}
    out = {"closest": 16, "occluded": 1, "attenuation": 16, "multi": 72}[kind]
    table = {"attenuation": 16, "multi": 4}.get(kind, 0)
    return {"bytes": float((32 + out) * case["rays"] + (40 + table) * case["tris"]),
            "flops": case["rays"] * _ray_flops(case["tris"])}


def exact(case, seed):
    """Closest hits against every triangle and quad light in 64 bits; the primitive of a tie is not fixed."""
    if case["kind"] != "closest" or case["rays"] * case["tris"] > 6e9:
        return None
    geo = _geometry(case, seed)
    rays = prepare(case, seed)["rays"].double()
    pos = torch.from_numpy(geo["pos"]).cuda().double()
    v = pos[torch.from_numpy(geo["idx"].view(np.int32)).cuda().long()]
    p0, e1, e2 = v[:, 0], v[:, 1] - v[:, 0], v[:, 2] - v[:, 0]
    nrm = torch.linalg.cross(e1, e2)
    n = rays.shape[0]
    t = torch.full((n,), FLT_MAX, dtype=torch.float64, device="cuda")
    uv = torch.zeros((n, 2), dtype=torch.float64, device="cuda")
    step = max(1, int(4e7) // case["tris"])
    for a in range(0, n, step):
        r = rays[a:a + step]
        o, lo, d, hi = r[:, 0:3], r[:, 3:4], r[:, 4:7], r[:, 7:8]
        # with s = p0 - o: t = s.n / d.n, u = (s x d).e2 / d.n, v = -(s x d).e1 / d.n, as sums of products
        det = d @ nrm.T
        m = torch.linalg.cross(o, d)
        tt = ((p0 * nrm).sum(1) - o @ nrm.T) / det
        # (s x d).e = p0.(d x e) - (o x d).e = d.(e x p0) - (o x d).e
        uu = (d @ torch.linalg.cross(e2, p0).T - m @ e2.T) / det
        vv = -(d @ torch.linalg.cross(e1, p0).T - m @ e1.T) / det
        bad = ~((uu >= 0) & (vv >= 0) & (uu + vv <= 1) & (tt > lo) & (tt <= hi))
        tt = tt.masked_fill(bad, math.inf)
        best, at = tt.min(dim=1)
        k = torch.nonzero(torch.isfinite(best)).flatten()
        t[a + k] = best[k]
        uv[a + k, 0] = uu[k, at[k]]
        uv[a + k, 1] = vv[k, at[k]]
    for q in geo["quads"]:
        inv = torch.tensor(np.asarray(q["inv"], np.float64).reshape(4, 4), device="cuda")
        o = rays[:, 0:3] @ inv[:3, :3].T + inv[:3, 3]
        d = rays[:, 4:7] @ inv[:3, :3].T
        tq = -o[:, 1] / d[:, 1]
        x, z = o[:, 0] + tq * d[:, 0], o[:, 2] + tq * d[:, 2]
        ok = ((x.abs() <= q["size_x"] / 2) & (z.abs() <= q["size_y"] / 2) & (tq > rays[:, 3]) & (tq <= rays[:, 7]) &
              (tq <= t))
        t = torch.where(ok, tq, t)
        uv = torch.where(ok[:, None], torch.zeros_like(uv), uv)
    return {"t": t, "prim": None, "uv": uv}
