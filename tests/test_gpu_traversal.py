"""Closest-hit and visibility casting on the GPU vs the CPU oracle.

Hit triangle ids, t and barycentrics must be bit-identical for identical rays
(Moller-Trumbore as Ray.hpp:121-167; closest-t, then smaller triangle index).
"""
import math

import numpy as np
import pytest

from mray_amd import abi, scenes
from oracle import refcpu

pytestmark = pytest.mark.gpu


def _random_rays(n, seed, origin_scale=2.0):
    rng = np.random.default_rng(seed)
    o = rng.uniform(-origin_scale, origin_scale, size=(n, 3))
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    rays = np.zeros((n, 8), np.float32)
    rays[:, 0:3] = o
    rays[:, 3] = 1e-4
    rays[:, 4:7] = d
    rays[:, 7] = 3.4e38
    # a few short rays and axis-aligned directions
    rays[: n // 10, 7] = rng.uniform(0.1, 2.0, size=n // 10)
    rays[n // 10: n // 10 + 6, 4:7] = np.array([[1, 0, 0], [-1, 0, 0], [0, 1, 0], [0, -1, 0],
                                                [0, 0, 1], [0, 0, -1]], np.float32)
    return rays


def _compare(acc, oscene, rays, brute):
    import torch
    d = torch.from_numpy(rays).cuda()
    prim, t, bary = acc.cast_closest(d)
    prim = prim.cpu().numpy().view(np.uint32)
    t = t.cpu().numpy()
    bary = bary.cpu().numpy()
    rp, rt, rb = oscene.cast_closest(rays, brute=brute)
    hit = rp != abi.INVALID_PRIM
    print(f"rays={len(rays)} hits={int(hit.sum())}", flush=True)
    assert np.array_equal(prim, rp)
    assert np.array_equal(t.view(np.uint32), rt.view(np.uint32))
    assert np.array_equal(bary[hit].view(np.uint32), rb[hit].view(np.uint32))
    vis = acc.cast_visibility(d).cpu().numpy()
    rvis = oscene.cast_visibility(rays)
    assert np.array_equal(vis.astype(np.uint32), rvis)
    # any-hit agrees with closest hit
    assert np.array_equal(vis == 1, ~hit)


@pytest.mark.parametrize("builder,width", [("sah", 4), ("lbvh", 4), ("sah", 8), ("lbvh", 8)])
def test_closest_soup_vs_bruteforce(torch_gpu, builder, width):
    from mray_amd import native
    s = scenes.random_triangles(3000, seed=9)
    acc = native.Accel(s, builder=builder, width=width)
    _compare(acc, refcpu.OracleScene(s), _random_rays(20000, 1), brute=True)


@pytest.mark.parametrize("builder,width", [("sah", 4), ("lbvh", 4), ("sah", 8)])
def test_closest_soup_large(torch_gpu, builder, width):
    from mray_amd import native
    s = scenes.random_triangles(200000, seed=4)
    acc = native.Accel(s, builder=builder, width=width)
    _compare(acc, refcpu.OracleScene(s), _random_rays(100000, 2), brute=False)


def test_primary_rays_cornell(torch_gpu):
    """Primary camera rays of the Cornell workload (identical rays, from the oracle)."""
    from mray_amd import native
    s = scenes.cornell()
    acc = native.Accel(s)
    o = refcpu.OracleScene(s)
    params = abi.render_params(256, 256, 1)
    rays, _ = o.camera_rays(params, 256 * 256)
    _compare(acc, o, rays, brute=True)


@pytest.mark.parametrize("builder,width", [("sah", 4), ("lbvh", 4), ("sah", 8)])
def test_primary_rays_terrain(torch_gpu, builder, width):
    from mray_amd import native
    s = scenes.terrain_spheres(grid=256, spheres=300, width=320, height=180)
    acc = native.Accel(s, builder=builder, width=width)
    o = refcpu.OracleScene(s)
    params = abi.render_params(320, 180, 1)
    rays, _ = o.camera_rays(params, 320 * 180)
    _compare(acc, o, rays, brute=False)


def test_single_triangle_and_edges(torch_gpu):
    """One-triangle scene (single-leaf LBVH case) and rays through edges/vertices."""
    from mray_amd import native
    pos = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0]], np.float32)
    s = scenes.Scene(positions=pos, tbn=scenes.quat_world_to_tangent(np.tile([[0, 0, 1.0]], (3, 1))),
                     indices=np.array([[0, 1, 2]], np.uint32),
                     surface_keys=np.zeros(1, np.uint32), cull=np.zeros(1, np.uint8),
                     materials=[{"type": abi.MAT_LAMBERT, "albedo": (0.5, 0.5, 0.5)}],
                     light_tris=np.zeros(0, np.uint32), light_radiance=np.zeros((0, 3), np.float32),
                     light_two_sided=np.zeros(0, np.uint8),
                     camera={"position": (0, 0, 2), "gaze": (0, 0, 0), "up": (0, 1, 0),
                             "fov": (math.radians(40),) * 2, "nearFar": (0.01, 100.0)})
    acc = native.Accel(s)
    xs = np.linspace(-0.25, 1.25, 61, dtype=np.float32)
    g = np.array([[x, y] for x in xs for y in xs], np.float32)
    rays = np.zeros((len(g), 8), np.float32)
    rays[:, 0:2] = g
    rays[:, 2] = 1.0
    rays[:, 3] = 0.0
    rays[:, 6] = -1.0
    rays[:, 7] = 10.0
    _compare(acc, refcpu.OracleScene(s), rays, brute=True)


@pytest.mark.parametrize("width", [4, 8])
def test_rays_in_box_planes(torch_gpu, width):
    """Axis-parallel rays (+0 and -0 direction components) whose origins lie
    on the BVH box planes of a grid of axis-aligned quads."""
    from mray_amd import native
    pos, idx = [], []
    for i in range(4):
        for j in range(4):
            b = len(pos)
            x0, y0 = i / 4, j / 4
            pos += [[x0, y0, 0], [x0 + 0.25, y0, 0], [x0 + 0.25, y0 + 0.25, 0], [x0, y0 + 0.25, 0]]
            idx += [[b, b + 1, b + 2], [b, b + 2, b + 3]]
    pos = np.array(pos, np.float32)
    idx = np.array(idx, np.uint32)
    n = len(idx)
    s = scenes.Scene(positions=pos, tbn=np.tile(np.array([[1, 0, 0, 0]], np.float32), (len(pos), 1)),
                     indices=idx, surface_keys=np.zeros(n, np.uint32), cull=np.zeros(n, np.uint8),
                     materials=[{"type": abi.MAT_LAMBERT, "albedo": (1, 1, 1)}],
                     light_tris=np.zeros(0, np.uint32), light_radiance=np.zeros((0, 3), np.float32),
                     light_two_sided=np.zeros(0, np.uint8),
                     camera={"position": (0, 0, 1), "gaze": (0, 0, 0), "up": (0, 1, 0),
                             "fov": (1.0, 1.0), "nearFar": (0.1, 10.0)})
    acc = native.Accel(s, width=width)
    o = refcpu.OracleScene(s)
    g = np.arange(0, 17, dtype=np.float32) / 16
    xy = np.array([[x, y] for x in g for y in g], np.float32)
    rays = np.zeros((len(xy), 8), np.float32)
    rays[:, 0:2] = xy
    rays[:, 2] = 1.0
    rays[:, 6] = -1.0
    rays[:, 7] = 10.0
    neg = rays.copy()
    neg[:, 4] = -0.0
    neg[:, 5] = -0.0
    for r in (rays, neg):
        _compare(acc, o, r, brute=True)


def _plane_stack(n_planes):
    """n_planes parallel squares [-1, 1]^2 at z = k / n_planes, two triangles
    each: every box of the tree spans the whole square, so a ray along +z
    enters every child of every node it visits."""
    pos, idx = [], []
    for k in range(n_planes):
        z = k / n_planes
        b = len(pos)
        pos += [[-1, -1, z], [1, -1, z], [1, 1, z], [-1, 1, z]]
        idx += [[b, b + 1, b + 2], [b, b + 2, b + 3]]
    pos = np.array(pos, np.float32)
    idx = np.array(idx, np.uint32)
    n = len(idx)
    return scenes.Scene(positions=pos, tbn=np.tile(np.array([[1, 0, 0, 0]], np.float32), (len(pos), 1)),
                        indices=idx, surface_keys=np.zeros(n, np.uint32), cull=np.zeros(n, np.uint8),
                        materials=[{"type": abi.MAT_LAMBERT, "albedo": (1, 1, 1)}],
                        light_tris=np.zeros(0, np.uint32), light_radiance=np.zeros((0, 3), np.float32),
                        light_two_sided=np.zeros(0, np.uint8),
                        camera={"position": (0, 0, -2), "gaze": (0, 0, 0), "up": (0, 1, 0),
                                "fov": (1.0, 1.0), "nearFar": (0.1, 10.0)})


def _first_descent_depth(nodes, x, y):
    """Stack depth of a +z ray at (x, y) when its near-first walk of the
    4-wide tree reaches its first leaf: every node pushes its hit inner
    children but the nearest (words 0-23: lo/hi x, y, z of the 4 children,
    24-27: child words, leaf flag 0x80000000)."""
    node, depth = 0, 0
    while True:
        w = nodes[node]
        inner = []
        for k in range(4):
            lx, hx = w[0 + k].view(np.float32), w[4 + k].view(np.float32)
            ly, hy = w[8 + k].view(np.float32), w[12 + k].view(np.float32)
            lz = w[16 + k].view(np.float32)
            c = int(w[24 + k])
            if not (lx <= x <= hx and ly <= y <= hy) or (c & 0x80000000):
                continue
            inner.append((float(lz), c))
        if not inner:
            return depth
        inner.sort()
        depth += len(inner) - 1
        node = inner[0][1]


@pytest.mark.parametrize("builder", ["sah", "lbvh"])
def test_deep_stack_spills_past_lds(torch_gpu, builder):
    """A walk whose stack outgrows the 12 LDS levels: the deeper entries go
    to the lane's global spill area, and waves mix lanes on either side of
    the boundary.  Hits, t, barycentrics and visibility equal brute force."""
    from mray_amd import native
    s = _plane_stack(4096)
    acc = native.Accel(s, builder=builder, width=4)
    nodes, _ = acc.read_wide()
    depth = _first_descent_depth(nodes, np.float32(0.1), np.float32(-0.2))
    print(f"{builder}: {len(nodes)} nodes, first-descent stack depth {depth}", flush=True)
    assert depth > 12
    rng = np.random.default_rng(3)
    n = 4096
    rays = np.zeros((n, 8), np.float32)
    # +z rays from below (deep stacks), oblique rays and rays from between
    # the planes (shallow stacks) interleaved within every wave
    rays[:, 0:2] = rng.uniform(-0.9, 0.9, size=(n, 2))
    rays[:, 2] = -1.0
    rays[:, 6] = 1.0
    odd = np.arange(n) % 3 == 1
    d = rng.normal(size=(int(odd.sum()), 3))
    d[:, 2] = np.abs(d[:, 2]) + 0.2
    rays[odd, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    mid = np.arange(n) % 3 == 2
    rays[mid, 2] = rng.uniform(0.0, 1.0, size=int(mid.sum()))
    rays[mid, 6] = -1.0
    rays[:, 3] = 1e-4
    rays[:, 7] = 3.4e38
    _compare(acc, refcpu.OracleScene(s), rays, brute=True)


@pytest.mark.parametrize("cells,offset,flat", [(24, 0.0, True), (96, 0.0, True), (96, 1000.0, False), (96, -3e4, True),
                                               (200, 0.0, False)])
def test_node_kinds_equal_brute_force(torch_gpu, cells, offset, flat):
    """Small trees are walked on exact boxes, larger ones (over 4096 nodes) on
    boxes quantised to 8 bits: both equal brute force for axis-parallel rays
    (+0 and -0) that start on box planes, rays along edges and random rays, on
    flat and bumpy grids, near the origin and far from it."""
    from mray_amd import native
    rng = np.random.default_rng(cells)
    g = np.arange(cells + 1, dtype=np.float32) / cells + np.float32(offset)
    x, y = np.meshgrid(g, g, indexing="ij")
    z = np.zeros_like(x) if flat else (0.05 * rng.random(x.shape)).astype(np.float32)
    pos = np.stack([x, y, z], -1).reshape(-1, 3).astype(np.float32)
    i, j = np.meshgrid(np.arange(cells), np.arange(cells), indexing="ij")
    v = (i * (cells + 1) + j).reshape(-1)
    idx = np.concatenate([np.stack([v, v + cells + 1, v + cells + 2], 1),
                          np.stack([v, v + cells + 2, v + 1], 1)]).astype(np.uint32)
    n = len(idx)
    s = scenes.Scene(positions=pos, tbn=np.tile(np.array([[1, 0, 0, 0]], np.float32), (len(pos), 1)),
                     indices=idx, surface_keys=np.zeros(n, np.uint32), cull=np.zeros(n, np.uint8),
                     materials=[{"type": abi.MAT_LAMBERT, "albedo": (1, 1, 1)}],
                     light_tris=np.zeros(0, np.uint32), light_radiance=np.zeros((0, 3), np.float32),
                     light_two_sided=np.zeros(0, np.uint8),
                     camera={"position": (0, 0, 1), "gaze": (0, 0, 0), "up": (0, 1, 0),
                             "fov": (1.0, 1.0), "nearFar": (0.1, 10.0)})
    acc = native.Accel(s)
    print(f"{n} triangles, {acc.info()['wide_nodes']} nodes, offset {offset}", flush=True)
    assert (acc.info()["wide_nodes"] > 4096) == (cells > 24)
    down = np.zeros((400, 8), np.float32)
    down[:, 0:2] = g[rng.integers(0, cells + 1, (400, 2))]     # on vertices and planes
    down[200:, 0] += np.float32(0.3 / cells)
    down[:, 2] = 1.0
    down[:, 6] = -1.0
    down[:, 7] = 10.0
    down[::2, 4:6] = -0.0
    slant = np.zeros((400, 8), np.float32)
    slant[:, 0:3] = rng.uniform(-0.5, 1.5, (400, 3)) + [offset, offset, 0.6]
    to = np.stack([g[rng.integers(0, cells + 1, 400)], g[rng.integers(0, cells + 1, 400)], np.zeros(400)], 1)
    slant[:, 4:7] = to - slant[:, 0:3]                         # through vertices
    slant[::3, 5] = 0.0
    slant[::7, 4] = 1e-35
    slant[:, 7] = 1e6
    along = np.zeros((100, 8), np.float32)                     # in the grid's plane
    along[:, 0:3] = np.stack([np.full(100, offset - 0.25), g[rng.integers(0, cells + 1, 100)],
                              rng.choice([0.0, 0.01], 100)], 1)
    along[:, 4] = 1.0
    along[:, 7] = 100.0
    _compare(acc, refcpu.OracleScene(s), np.concatenate([down, slant, along]).astype(np.float32), brute=True)
    acc.close()


def _lit_grid(cells, extent):
    """A flat grid over [-extent, extent]^2 at z = 0, every triangle a
    two-sided light of its own, and a camera straight above it whose opening
    angle is so small that all its rays are exactly axis-parallel."""
    g = (np.arange(cells + 1, dtype=np.float64) / cells * 2 - 1) * extent
    x, y = np.meshgrid(g, g, indexing="ij")
    pos = np.stack([x, y, np.zeros_like(x)], -1).reshape(-1, 3).astype(np.float32)
    i, j = np.meshgrid(np.arange(cells), np.arange(cells), indexing="ij")
    v = (i * (cells + 1) + j).reshape(-1)
    idx = np.concatenate([np.stack([v, v + cells + 1, v + cells + 2], 1),
                          np.stack([v, v + cells + 2, v + 1], 1)]).astype(np.uint32)
    n = len(idx)
    key = (np.arange(n) | abi.LIGHT_FLAG).astype(np.uint32)
    rad = np.random.default_rng(n).uniform(0.5, 2.0, size=(n, 3)).astype(np.float32)
    at = (0.1 * extent, -0.23 * extent)
    return scenes.Scene(positions=pos, tbn=np.tile(np.array([[1, 0, 0, 0]], np.float32), (len(pos), 1)),
                        indices=idx, surface_keys=key, cull=np.zeros(n, np.uint8),
                        materials=[{"type": abi.MAT_LAMBERT, "albedo": (1, 1, 1)}],
                        light_tris=np.arange(n, dtype=np.uint32), light_radiance=rad,
                        light_two_sided=np.ones(n, np.uint8),
                        camera={"position": at + (0.5 * extent,), "gaze": at + (0.0,), "up": (0, 1, 0),
                                "fov": (1e-25, 1e-25), "nearFar": (0.01 * extent, 10.0 * extent)})


@pytest.mark.parametrize("cells", [24, 96])
@pytest.mark.parametrize("extent", [1e3, 4e7, 1e8, 1e10])
def test_axis_parallel_rays_in_large_scenes(torch_gpu, extent, cells):
    """Axis-parallel rays (+0, -0 and tiny components) and directions that are
    far from unit length over scenes of large extent, on exact and on quantised
    nodes: equal to brute force."""
    from mray_amd import native
    s = _lit_grid(cells, extent)
    acc = native.Accel(s)
    assert (acc.info()["wide_nodes"] > 4096) == (cells > 24)
    rng = np.random.default_rng(cells)
    g = s.positions[:, 0]
    rays = np.zeros((600, 8), np.float32)
    rays[:, 0:2] = rng.choice(g, (600, 2))                       # on vertices and planes
    rays[200:, 0:2] = rng.uniform(-1.2 * extent, 1.2 * extent, (400, 2))
    rays[:, 2] = 0.5 * extent
    rays[:, 6] = -1.0
    rays[:, 7] = 3.4e38
    rays[::2, 4:6] = -0.0
    rays[1::5, 4] = 1e-36
    # direction lengths of 1e-9 and 1e9: t grows and shrinks with them
    rays[100:150, 4:7] *= np.float32(1e-9)
    rays[150:200, 4:7] *= np.float32(1e9)
    rays[5::60, 4:7] = 0.0                                       # no direction: no hit
    along = rays[:100].copy()                                    # across the grid, above and in its plane
    along[:, 0] = -1.5 * extent
    along[:, 2] = 0.0
    along[:, 4:7] = (1.0, 0.0, -0.0)
    _compare(acc, refcpu.OracleScene(s), np.concatenate([rays, along]), brute=True)
    acc.close()


@pytest.mark.parametrize("kind", ["one", "lane_refill", "batch"])
@pytest.mark.parametrize("extent", [1e3, 1e9])
def test_renders_of_large_scenes(torch_gpu, extent, kind):
    """Renders whose camera rays are exactly axis-parallel, over a small tree
    of large extent: every path reaches the light below the camera, as in the
    oracle (batch and lane-refill walks take quantised nodes at any size)."""
    from mray_amd import native
    s = _lit_grid(16, extent)
    params = abi.render_params(8, 8, 4, rr=(4, 4), mode=abi.SAMPLE_PURE, seed=3,
                               flags=abi.RENDER_LANE_REFILL if kind == "lane_refill" else 0)
    acc = native.Accel(s)
    if kind == "batch":
        b = native.BatchScene([acc])
        r = native.BatchRenderer(b, [{"scene": 0, "width": 8, "height": 8, "spp": 4}], params)
    else:
        r = native.Renderer(acc, params)
    st = r.render_all()
    film = r.film()
    film = film[0] if kind == "batch" else film
    r.close()
    ref, rst = refcpu.OracleScene(s).render(params)
    img, rimg = film[:3] / film[3], ref[:3] / ref[3]
    print(f"{kind} extent {extent:g}: {st['dead_paths']} paths, image {img.min():.3f}..{img.max():.3f}", flush=True)
    assert st["dead_paths"] == rst["dead_paths"] == 256
    assert rimg.min() >= 0.49
    assert np.allclose(img, rimg, rtol=1e-5)
    acc.close()


def _exact_visits(nodes, rays):
    """Nodes of the 4-wide tree (words 0-23: lo/hi x, y, z of the 4 children,
    24-27: child words) that rays without a hit enter, in float64."""
    lo = np.stack([nodes[:, 8 * a: 8 * a + 4].view(np.float32) for a in range(3)], 2).astype(np.float64)
    hi = np.stack([nodes[:, 8 * a + 4: 8 * a + 8].view(np.float32) for a in range(3)], 2).astype(np.float64)
    child = nodes[:, 24:28]
    inner = (child & 0x80000000) == 0
    total = 0
    for r in rays.astype(np.float64):
        live = np.array([0])
        while len(live):
            total += len(live)
            with np.errstate(divide="ignore", over="ignore", invalid="ignore"):
                a, b = (lo[live] - r[0:3]) / r[4:7], (hi[live] - r[0:3]) / r[4:7]
            near = np.minimum(a, b).max(axis=2)
            far = np.maximum(a, b).min(axis=2)
            live = child[live][(np.maximum(near, r[3]) <= np.minimum(far, r[7])) & inner[live]]
    return total


@pytest.mark.parametrize("cells,flags", [(16, 0), (16, abi.RENDER_LANE_REFILL), (96, 0), (96, abi.RENDER_LANE_REFILL)])
def test_counters_are_the_timed_walk_s(torch_gpu, cells, flags):
    """Counted nodes are those the uncounted kernels visit: on small trees the
    exact boxes' (counted here in float64 over rays that only meet culled
    triangles), on larger ones the quantised boxes', which are a little looser."""
    from mray_amd import native
    s = _lit_grid(cells, 1.0)
    rng = np.random.default_rng(cells)
    s.positions[:, 2] = 0.8 / cells * rng.random(len(s.positions)).astype(np.float32)
    s.indices = s.indices[:, ::-1].copy()                        # facing away from the camera
    s.surface_keys = np.zeros(len(s.indices), np.uint32)
    s.light_tris, s.light_radiance = s.light_tris[:0], s.light_radiance[:0]
    s.light_two_sided = s.light_two_sided[:0]
    s.cull = np.ones(len(s.indices), np.uint8)
    s.camera = {"position": (0.13, -0.2, 1.5), "gaze": (0.0, 0.1, 0.0), "up": (0, 1, 0), "fov": (1.0, 1.0),
                "nearFar": (0.01, 100.0)}
    params = abi.render_params(24, 24, 1, rr=(4, 4), mode=abi.SAMPLE_PURE, seed=1, flags=flags)
    o = refcpu.OracleScene(s)
    rays, _ = o.camera_rays(params, 24 * 24)
    assert np.all(o.cast_closest(rays, brute=True)[0] == abi.INVALID_PRIM)
    acc = native.Accel(s)
    nodes, _ = acc.read_wide()
    ref = _exact_visits(nodes, rays)
    ctr = acc.cast_closest(torch_gpu.from_numpy(rays).cuda(), count_visits=True)[3].cpu().numpy()
    r = native.Renderer(acc, params)
    r.set_measurement(counting=True)
    st = r.render_all()
    r.close()
    print(f"{len(nodes)} nodes: exact {ref}, cast {ctr[0]}, render {st['node_visits']}", flush=True)
    assert st["ext_rays"] == 576 and st["node_visits"] == ctr[0]
    if len(nodes) <= 4096:
        assert ctr[0] == ref
    else:
        assert ref < ctr[0] < 1.2 * ref
    # a direction's length changes t and nothing else: by a power of two, the
    # walk is the same to the bit, with an axis it is parallel to as well
    visits = []
    for scale in (1.0, 2.0 ** -13, 2.0 ** 13, 2.0 ** -40):
        r = rays.copy()
        r[:, 4] = 0.0
        r[::2, 5] = -0.0
        r[:, 3] = 0.0
        r[:, 4:7] *= np.float32(scale)
        r[:, 7] = 3.4e38
        visits.append(int(acc.cast_closest(torch_gpu.from_numpy(r).cuda(), count_visits=True)[3][0]))
    assert visits[0] > 576 and len(set(visits)) == 1, visits
    acc.close()


@pytest.mark.parametrize("builder", ["sah", "lbvh"])
def test_deep_stack_on_exact_nodes(torch_gpu, builder):
    """As test_deep_stack_spills_past_lds, over few enough planes for exact
    nodes, past the 10 LDS levels of these walks."""
    from mray_amd import native
    s = _plane_stack(1400)
    acc = native.Accel(s, builder=builder, width=4)
    nodes, _ = acc.read_wide()
    depth = _first_descent_depth(nodes, np.float32(0.1), np.float32(-0.2))
    print(f"{builder}: {len(nodes)} nodes, first-descent stack depth {depth}", flush=True)
    assert len(nodes) <= 4096 and depth > 12
    rng = np.random.default_rng(4)
    rays = np.zeros((2000, 8), np.float32)
    rays[:, 0:2] = rng.uniform(-0.9, 0.9, size=(2000, 2))
    rays[:, 2] = np.where(np.arange(2000) % 3 == 2, rng.uniform(0.0, 1.0, size=2000), -1.0)
    d = rng.normal(size=(2000, 3))
    d[:, 2] = np.abs(d[:, 2]) + 0.2
    d[::2] = (0.0, -0.0, 1.0)
    rays[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    rays[:, 3] = 1e-4
    rays[:, 7] = 3.4e38
    _compare(acc, refcpu.OracleScene(s), rays, brute=True)
    acc.close()
