"""Closest and any hit through the walk tree against the oracle, bit for bit, where its candidates and
the Fast-BVH's rules are hardest to keep together: equal hits (doubled triangles, coplanar overlaps,
rays through shared vertices and edges), leaf boxes without thickness, rays along the axes, scenes far
from the origin, origins far from the scene, directions and windows at the edge of what the walk tree
takes, trees of one to a few records, and depth-limited leaves of hundreds of primitives."""
import numpy as np
import pytest
import torch

from oracle.oracle import OracleBvh
from sort_amd import MISS, Obvh, Qbvh, batch, scenes

pytestmark = pytest.mark.gpu

FLT_MAX = np.float32(3.4028234663852886e38)


def _doubled(g):
    """A soup, every triangle again as it is, turned around, or starting at another vertex."""
    pos, _ = scenes.soup(1500, seed=5)
    t = pos.reshape(-1, 3, 3) * np.float32(1.0)
    c = t.mean(axis=1, keepdims=True)
    t = (c + (t - c) * np.float32(8.0)).astype(np.float32)
    order = np.array([[0, 1, 2], [0, 2, 1], [1, 2, 0]])[g.integers(0, 3, len(t))]
    t = np.concatenate([t, np.take_along_axis(t, order[:, :, None], axis=1)])
    return scenes.tris_to_mesh(list(t[g.permutation(len(t))])), None


def _grid(g, n=24, axis=2):
    """Two parallel sheets of axis-aligned squares with shared corners at multiples of 1/n."""
    tris = []
    for z in (0.25, 0.75):
        for i in range(n):
            for j in range(n):
                p = [(i / n, j / n, z), ((i + 1) / n, j / n, z), ((i + 1) / n, (j + 1) / n, z), (i / n, (j + 1) / n, z)]
                p = [tuple(np.roll(q, axis - 2)) for q in p]
                tris += [np.array([p[0], p[1], p[2]], np.float32), np.array([p[0], p[2], p[3]], np.float32)]
    return scenes.tris_to_mesh(tris), None


def _overlap(g):
    """Coplanar triangles of all sizes on one plane, over one another, with quad lights on it too."""
    t = g.uniform(0.0, 1.0, (600, 3, 3)).astype(np.float32)
    t[:, 1:] = t[:, :1] + (t[:, 1:] - np.float32(0.5)) * np.exp(g.uniform(-4, 0, (600, 1, 1))).astype(np.float32)
    t[:, :, 1] = np.float32(0.5)
    quads = [scenes.translate_quad((float(x), 0.5, float(z)), 0.2) for x, z in g.uniform(0.2, 0.8, (4, 2))]
    return scenes.tris_to_mesh(list(t)), quads


def _rays(g, n, mesh):
    """Random rays, rays along the axes, and rays aimed at vertices and edge midpoints."""
    pos = mesh[0]
    lo, hi = pos.min(axis=0), pos.max(axis=0)
    ext = np.float32(max(float((hi - lo).max()), 1e-3))
    o = (lo + (hi - lo) * g.uniform(-0.4, 1.4, (n, 3)) + ext * g.normal(0, 0.3, (n, 3))).astype(np.float32)
    d = g.normal(size=(n, 3)).astype(np.float32)
    k = np.arange(n)
    v = pos[g.integers(0, len(pos), n)]
    w = pos[(g.integers(0, len(pos) // 3, n) * 3)[:, None] + np.array([0, 1])].mean(axis=1).astype(np.float32)
    d = np.where((k % 4 == 1)[:, None], v - o, np.where((k % 4 == 2)[:, None], w - o, d)).astype(np.float32)
    ax = k % 4 == 3
    d[ax] = 0
    d[ax, k[ax] // 4 % 3] = np.where(k[ax] // 12 % 2, 1.0, -1.0)
    on = ax & (k % 8 == 7)  # through a vertex, along an axis
    o[on] = (v - 2 * ext * d)[on]
    d[k % 16 == 5] *= np.float32(3.0)
    return o, d


SCENES = {"doubled": _doubled, "grid z": _grid, "grid x": lambda g: _grid(g, axis=0), "overlap": _overlap}


def _check(acc, ob, rays, label):
    print(f"[walk] {label} width={acc.width} rays={len(rays)}", flush=True)
    d = torch.from_numpy(np.ascontiguousarray(rays)).cuda()
    hits, occ = acc.get_intersect(d).cpu().numpy(), acc.is_occluded(d).cpu().numpy()
    ref, ref_occ = ob.closest(rays, threads=16), ob.occluded(rays, threads=16)
    bad = np.nonzero(np.any(hits.view(np.uint32) != ref.view(np.uint32), axis=1))[0]
    assert bad.size == 0, f"{label}: {bad.size} closest differ, ray {rays[bad[0]]}: {hits[bad[0]]} {ref[bad[0]]}"
    assert np.array_equal(occ, ref_occ), label
    try:  # small batches give four lanes to a ray; with 8 LDS entries every ray has one
        batch.set_tuning(acc.ctx, lds_entries=8)
        lanes, lanes_occ = acc.get_intersect(d).cpu().numpy(), acc.is_occluded(d).cpu().numpy()
    finally:
        batch.set_tuning(acc.ctx)
    assert np.array_equal(lanes.view(np.uint32), hits.view(np.uint32)) and np.array_equal(lanes_occ, occ), label
    acc.check_errors()
    return hits


def _build(ctx, width, mesh, quads, **kw):
    acc = (Obvh if width == 8 else Qbvh)(ctx, **kw).build(mesh[0], mesh[1], quads)
    return acc, OracleBvh(mesh[0], mesh[1], quads, width=width, max_depth=kw.get("max_node_depth", 28),
                          max_leaf=kw.get("max_pri_in_leaf", 16))


@pytest.mark.parametrize("width", [8, 4])
@pytest.mark.parametrize("scene", list(SCENES))
def test_ties_flat_boxes_and_axis_rays(gpu_ctx, width, scene):
    g = np.random.default_rng(len(scene) + width)
    mesh, quads = SCENES[scene](g)
    for kw in ({}, {"max_node_depth": 3}, {"max_pri_in_leaf": 1}):
        acc, ob = _build(gpu_ctx, width, mesh, quads, **kw)
        o, d = _rays(g, 12000, mesh)
        hits = _check(acc, ob, scenes.make_rays(o, d, 0.0, FLT_MAX), f"{scene} {kw}")
        assert np.mean(hits[:, 1].view(np.uint32) != MISS) > 0.1
        tmin = g.uniform(0, 0.5, len(o)).astype(np.float32)
        _check(acc, ob, scenes.make_rays(o, d, tmin, tmin + g.uniform(0, 1, len(o)).astype(np.float32)), "windowed")


@pytest.mark.parametrize("width", [8, 4])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 8, 9, 16, 17, 33])
def test_few_triangles(gpu_ctx, width, n):
    g = np.random.default_rng(n)
    mesh = scenes.tris_to_mesh(list(g.uniform(0, 1, (n, 3, 3)).astype(np.float32)))
    acc, ob = _build(gpu_ctx, width, mesh, [scenes.translate_quad((0.5, 1.2, 0.5), 0.5)] if n % 2 else None)
    _check(acc, ob, scenes.make_rays(*_rays(g, 3000, mesh), 0.0, FLT_MAX), f"{n} triangles")


@pytest.mark.parametrize("shift,scale,away", [(0.0, 1.0, 50.0), (1000.0, 1.0, 0.0), (3e4, 1.0, 0.0), (0.0, 1e-4, 0.0),
                                              (0.0, 1e6, 0.0), (0.0, 1.0, 1e5), (0.0, 1e9, 0.0)])
def test_far_scenes_and_origins(gpu_ctx, shift, scale, away):
    """A scene past the origin by more than 4,096 times its size has no walk tree, and an origin as far
    out leaves it; short of that both use it."""
    g = np.random.default_rng(9)
    pos, idx = scenes.soup(3000, seed=8)
    t = pos.reshape(-1, 3, 3)
    c = t.mean(axis=1, keepdims=True)
    t = ((c + (t - c) * 10) * scale + shift).astype(np.float32)
    mesh = scenes.tris_to_mesh(list(t))
    acc, ob = _build(gpu_ctx, 8, mesh, None)
    o, d = _rays(g, 8000, mesh)
    if away:
        target = mesh[0][g.integers(0, len(mesh[0]), len(o))]
        d = (target - o).astype(np.float32)
        d /= np.linalg.norm(d, axis=1, keepdims=True)
        o = (target - np.float32(away) * d).astype(np.float32)
    _check(acc, ob, scenes.make_rays(o, d, 0.0, FLT_MAX), f"shift {shift} scale {scale} away {away}")


@pytest.mark.parametrize("lds", [8, 16])
def test_windows_directions_and_pool(gpu_ctx, lds):
    """Negative, infinite and empty windows, directions from 1e-14 to 1e14 long, zero and near-zero
    components, mixed among ordinary rays; the same rays against three scenes of a pool at once."""
    g = np.random.default_rng(3)
    pos, idx = scenes.soup(4000, seed=21)
    t = pos.reshape(-1, 3, 3)
    c = t.mean(axis=1, keepdims=True)
    mesh = scenes.tris_to_mesh(list((c + (t - c) * 6).astype(np.float32)))
    acc, ob = _build(gpu_ctx, 8, mesh, None)
    o, d = _rays(g, 16384, mesh)
    k = np.arange(len(o))
    r = scenes.make_rays(o, d, 0.0, FLT_MAX)
    r[k % 16 == 0, 3] = np.float32(-0.5)
    r[k % 16 == 1, 3] = np.float32(-2.0)
    r[k % 16 == 2, 7] = np.inf
    r[k % 16 == 3, 7] = np.float32(-1.0)
    r[k % 16 == 4, 3] = np.float32(-0.0)
    r[k % 16 == 6, 4:7] *= np.float32(1e-14)
    r[k % 16 == 8, 4:7] *= np.float32(1e14)
    r[k % 16 == 9, 4:7] *= np.float32(1e-4)
    r[k % 16 == 10, 4] = np.float32(2e-6)
    r[k % 16 == 11, 5:7] *= np.float32(1e-7)
    try:
        batch.set_tuning(gpu_ctx, lds_entries=lds)
        hits = _check(acc, ob, r, f"windows lds {lds}")
        batch.set_tuning(gpu_ctx, lds_entries=lds)
        accs = [acc] + [Obvh(gpu_ctx).build(*scenes.soup(n, seed=n)) for n in (700, 40)]
        pool = batch.Pool(gpu_ctx, accs)
        sid = (k % 3).astype(np.int32)
        got = pool.trace(torch.from_numpy(r).cuda(), torch.from_numpy(sid).cuda()).cpu().numpy()
        pool.check_errors()
    finally:
        batch.set_tuning(gpu_ctx)
    assert np.array_equal(got[sid == 0].view(np.uint32), hits[sid == 0].view(np.uint32))
    for i in (1, 2):
        one = accs[i].get_intersect(torch.from_numpy(r).cuda()).cpu().numpy()
        assert np.array_equal(got[sid == i].view(np.uint32), one[sid == i].view(np.uint32))
    pool.close()


@pytest.mark.parametrize("quads", [False, True])
@pytest.mark.parametrize("width", [8, 4])
def test_vertices_with_a_nan_coordinate(gpu_ctx, width, quads):
    """Such a triangle is never hit; its neighbours in the tree are, as if it were not there."""
    g = np.random.default_rng(11)
    t = g.uniform(0.0, 1.0, (3000, 1, 3)) + g.normal(0.0, 0.03, (3000, 3, 3))
    t = t.astype(np.float32)
    bad = np.arange(0, len(t), 4)
    rays = _rays(g, 12000, (t.reshape(-1, 3), None))
    t[bad, bad // 4 % 3, bad // 12 % 3] = np.nan
    mesh = scenes.tris_to_mesh(list(t))
    acc, ob = _build(gpu_ctx, width, mesh, [scenes.translate_quad((0.5, 1.2, 0.5), 0.5)] if quads else None)
    hits = _check(acc, ob, scenes.make_rays(*rays, 0.0, FLT_MAX), f"nan quads={quads}")
    prim = hits[:, 1].view(np.uint32)
    assert np.mean(prim != MISS) > 0.1 and not np.isin(prim, bad).any()


@pytest.mark.parametrize("n", [700, 40000])
def test_windows_of_one_float(gpu_ctx, n):
    """Windows that hold a known hit's distance and no other number: the boxes on the way to it start at tmin,
    and a stack entry, whose last two bits name its slot, may not be taken for one past tmax."""
    g = np.random.default_rng(n)
    t = g.uniform(0.0, 1.0, (n, 1, 3)) + g.normal(0.0, 0.5 * n ** (-1 / 3), (n, 3, 3))
    mesh = scenes.tris_to_mesh(list(t.astype(np.float32)))
    acc, ob = _build(gpu_ctx, 8, mesh, None)
    o, d = _rays(g, 20000, mesh)
    hits = ob.closest(scenes.make_rays(o, d, 0.0, FLT_MAX), threads=16)
    at = hits[:, 0][hits[:, 1].view(np.uint32) != MISS]
    o, d = o[hits[:, 1].view(np.uint32) != MISS], d[hits[:, 1].view(np.uint32) != MISS]
    for ulps in (1, 2, 3):
        lo = (at.view(np.uint32) - np.uint32(ulps)).view(np.float32)
        rays = scenes.make_rays(o, d, lo, at)
        found = _check(acc, ob, rays, f"{ulps} ulps, {n} triangles")
        assert np.mean(found[:, 1].view(np.uint32) != MISS) > 0.5


def _sheets(n):
    """Two parallel tilted sheets of n x n squares, and a function for points of the first one's plane."""
    c, a, b = np.array([0.1, 0.05, 0.2]), np.array([0.9, 0.31, -0.17]), np.array([-0.23, 0.77, 0.41])
    up = np.cross(a, b) / np.linalg.norm(np.cross(a, b))
    at = lambda i, j, k: (c + a * i / n + b * j / n + 0.25 * k * up).astype(np.float32)
    tris = []
    for k in (0, 1):
        for i in range(n):
            for j in range(n):
                p = [at(i, j, k), at(i + 1, j, k), at(i + 1, j + 1, k), at(i, j + 1, k)]
                tris += [np.stack(p[:3]), np.stack([p[0], p[2], p[3]])]
    return scenes.tris_to_mesh(tris), lambda x, y, off: (c + x[:, None] * a + y[:, None] * b + off[:, None] * up).astype(np.float32)


@pytest.mark.parametrize("width", [8, 4])
@pytest.mark.parametrize("n", [4, 16, 48])
def test_rays_in_the_plane_of_a_tilted_sheet(gpu_ctx, width, n):
    """Edge-on, the triangle test accepts rays far beside a triangle; every such hit of the Fast-BVH has to be
    there, in the lanes' form, the quads', through a pool, and with windows."""
    g = np.random.default_rng(n)
    mesh, point = _sheets(n)
    acc, ob = _build(gpu_ctx, width, mesh, None)
    m = 30000
    for off in (0.0, 1e-6, 1e-5):
        o, e = (point(g.uniform(-0.2, 1.2, m), g.uniform(-0.2, 1.2, m), g.uniform(-off, off, m)) for _ in range(2))
        o[::3] = mesh[0][g.integers(0, len(mesh[0]) // 2, len(o[::3]))]
        rays = scenes.make_rays(o, (e - o).astype(np.float32), 0.0, FLT_MAX)
        hits = _check(acc, ob, rays, f"sheet {n} off {off}")
        tmin = g.uniform(0, 0.5, m).astype(np.float32)
        _check(acc, ob, scenes.make_rays(o, (e - o).astype(np.float32), tmin, tmin + np.float32(0.3)), "windowed")
        pool = batch.Pool(gpu_ctx, [acc, acc])
        got = pool.trace(torch.from_numpy(rays).cuda(), torch.from_numpy((np.arange(m) % 2).astype(np.int32)).cuda()).cpu().numpy()
        assert np.array_equal(got.view(np.uint32), hits.view(np.uint32))
        pool.close()


@pytest.mark.parametrize("width", [8, 4])
@pytest.mark.parametrize("tiny", [3e-6, 1e-6, 1e-7, 1e-19])
def test_tiny_triangles_and_needles_among_others(gpu_ctx, width, tiny):
    """Half of the triangles at the size of the arithmetic's rounding (or the whole scene below underflow),
    a tenth of the others long needles; rays at vertices and along the needles."""
    g = np.random.default_rng(int(-np.log10(tiny)))
    n = 4000
    size = np.where(np.arange(n) % 2, 0.2, max(tiny, 1e-7))[:, None, None] * np.ones((n, 1, 3))
    size[np.arange(n) % 20 == 1] = [1e-6, 1e-6, 0.4]
    t = (g.uniform(0, 1, (n, 1, 3)) + g.uniform(-0.5, 0.5, (n, 3, 3)) * size) * (tiny if tiny < 1e-10 else 1.0)
    mesh = scenes.tris_to_mesh(list(t.astype(np.float32)))
    acc, ob = _build(gpu_ctx, width, mesh, None)
    o, d = _rays(g, 40000, mesh)
    k = np.arange(len(o))
    needle = mesh[0].reshape(-1, 3, 3)[g.integers(0, n // 20, len(o)) * 20 + 1]
    along = (needle[:, 1] - needle[:, 0]) * np.float32(1.0)
    o = np.where((k % 3 == 0)[:, None], needle[:, 0] - 2 * along, o).astype(np.float32)
    d = np.where((k % 3 == 0)[:, None], along, d).astype(np.float32)
    if tiny > 1e-10:
        d /= np.maximum(np.linalg.norm(d, axis=1, keepdims=True), 1e-20).astype(np.float32)
    _check(acc, ob, scenes.make_rays(o, d, 0.0, FLT_MAX), f"tiny {tiny}")


def test_directions_below_the_slab_clamp(gpu_ctx):
    """The Fast-BVH steps through its boxes along a direction of no component below 1e-5: rays with smaller
    ones, of several lengths, in a flat scene and a soup."""
    g = np.random.default_rng(17)
    for mesh in (_sheets(16)[0], scenes.tris_to_mesh(list((g.uniform(0, 1, (4000, 1, 3)) + g.uniform(-0.05, 0.05, (4000, 3, 3))).astype(np.float32)))):
        acc, ob = _build(gpu_ctx, 8, mesh, None)
        o, d = _rays(g, 32000, mesh)
        k = np.arange(len(o))
        d[k, k % 3] = g.uniform(-1.2e-5, 1.2e-5, len(o))
        d[k % 5 == 0] *= np.float32(1e-3)
        d[k % 5 == 1, 0] = 0.0
        d[k % 7 == 2] *= np.float32(30.0)
        o[k % 2 == 0] = (mesh[0][g.integers(0, len(mesh[0]), len(o))] - 0.7 * d)[k % 2 == 0]
        _check(acc, ob, scenes.make_rays(o, d.astype(np.float32), 0.0, FLT_MAX), "clamped directions")


def test_pool_in_which_one_scene_has_no_walk_tree(gpu_ctx):
    """A scene past the origin by more than 4,096 times its size has none; the pool's rays then all take the
    Fast-BVH, closest and any hit, with the results that each scene gives alone."""
    g = np.random.default_rng(23)
    accs, rays = [], []
    for n, shift in ((3000, 0.0), (2000, 3e4), (500, 0.0)):
        t = g.uniform(0, 1, (n, 1, 3)) + g.uniform(-0.1, 0.1, (n, 3, 3)) + shift
        mesh = scenes.tris_to_mesh(list(t.astype(np.float32)))
        accs.append(_build(gpu_ctx, 8, mesh, None)[0])
        rays.append(scenes.make_rays(*_rays(g, 5000, mesh), 0.0, FLT_MAX))
    pool = batch.Pool(gpu_ctx, accs)
    sid = np.repeat(np.arange(3), 5000).astype(np.int32)
    d, ids = torch.from_numpy(np.concatenate(rays)).cuda(), torch.from_numpy(sid).cuda()
    hits, occ = pool.trace(d, ids).cpu().numpy(), pool.trace(d, ids, any_hit=True).cpu().numpy()
    pool.check_errors()
    for i, acc in enumerate(accs):
        one = torch.from_numpy(rays[i]).cuda()
        assert np.array_equal(hits[sid == i].view(np.uint32), acc.get_intersect(one).cpu().numpy().view(np.uint32))
        assert np.array_equal(occ[sid == i], acc.is_occluded(one).cpu().numpy())
    pool.close()


@pytest.mark.parametrize("wrong", [0.0, 1e-5, 0.05])
def test_turned_quads(gpu_ctx, wrong):
    """Quad lights turned and scaled any way among triangles, hit head-on, along their planes and at their edges;
    with an inverse that is off by rounding, by 1e-5 and by more than a walk tree is built for."""
    g = np.random.default_rng(29)
    quads = []
    for _ in range(12):
        q, _ = np.linalg.qr(g.normal(size=(3, 3)))
        m = np.eye(4)
        m[:3, :3] = q * np.exp(g.uniform(-1, 1))
        m[:3, 3] = g.uniform(0, 1, 3)
        inv = np.linalg.inv(m)
        inv[:3] += wrong * g.uniform(-1, 1, (3, 4))
        quads.append(dict(mat=m.astype(np.float32).ravel(), inv=inv.astype(np.float32).ravel(), size_x=0.3, size_y=0.2))
    t = g.uniform(0, 1, (600, 1, 3)) + g.uniform(-0.05, 0.05, (600, 3, 3))
    mesh = scenes.tris_to_mesh(list(t.astype(np.float32)))
    acc, ob = _build(gpu_ctx, 8, mesh, quads)
    n = 24000
    k = np.arange(n)
    mats = np.stack([np.asarray(q["mat"], np.float64).reshape(4, 4) for q in quads])[k % 12]
    local = np.stack([g.uniform(-0.2, 0.2, n), np.zeros(n), g.uniform(-0.15, 0.15, n)], 1)
    local[k % 5 == 1, 0] = 0.15
    at = np.einsum("nij,nj->ni", mats[:, :3, :3], local) + mats[:, :3, 3]
    d = g.normal(size=(n, 3))
    flat = k % 3 == 0  # along the quad's plane, or within 1e-6 of it
    side = np.stack([g.normal(size=n), g.choice([0.0, 1e-6, 1e-3], n), g.normal(size=n)], 1)
    d[flat] = np.einsum("nij,nj->ni", mats[:, :3, :3], side)[flat]
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    o = at - d * g.uniform(0.01, 2.0, (n, 1))
    hits = _check(acc, ob, scenes.make_rays(o.astype(np.float32), d.astype(np.float32), 0.0, FLT_MAX), f"quads off by {wrong}")
    prim = hits[:, 1].view(np.uint32)
    assert np.mean((prim >= 600) & (prim != MISS)) > 0.1
