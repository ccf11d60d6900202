"""LBVH build on the GPU vs the CPU oracle: bit-exact integer and box outputs.

Reference: KCGenMortonCode (AcceleratorLBVH.cu:96-168), the CUB pair sort
(AcceleratorLBVH.hpp:828-838), KCConstructLBVHInternalNodes
(AcceleratorLBVH.cu:170-299) and KCUnionLBVHBoundingBoxes (:301-435).
"""
import numpy as np
import pytest

from mray_amd import scenes
from oracle import refcpu

pytestmark = pytest.mark.gpu


def _scenes():
    return [scenes.cornell(), scenes.random_triangles(20000, seed=3),
            scenes.terrain_spheres(grid=96, spheres=40, width=64, height=36)]


@pytest.mark.parametrize("idx", [0, 1, 2])
def test_accel_lbvh_matches_oracle(torch_gpu, idx):
    from mray_amd import native
    scene = _scenes()[idx]
    print(f"scene {scene.name} tris={scene.triangle_count}", flush=True)
    acc = native.Accel(scene)
    codes, order, nodes, boxes = acc.read_lbvh()
    o = refcpu.OracleScene(scene)
    rcodes, rorder, rnodes, rboxes, _ = o.lbvh()
    assert np.array_equal(codes, rcodes), "Morton codes differ"
    assert np.array_equal(order, rorder), "sorted leaf order differs"
    assert np.array_equal(nodes, rnodes), "Karras topology differs"
    assert np.array_equal(boxes.view(np.uint32), rboxes.view(np.uint32)), "node boxes differ"
    info = acc.info()
    assert info["triangles"] == scene.triangle_count
    acc.close()


def test_stage_morton_codes(torch_gpu):
    from mray_amd import native
    torch = torch_gpu
    rng = np.random.default_rng(11)
    for n in (1, 7, 1000, 300001):
        centers = rng.uniform(-3.0, 5.0, size=(n, 3)).astype(np.float32)
        # include points on the box faces and corners
        centers[: min(n, 4)] = np.array([[-3, -3, -3], [5, 5, 5], [-3, 5, 1], [5, -3, 0]],
                                        np.float32)[: min(n, 4)]
        box = np.array([-3, -3, -3, 5, 5, 5.5], np.float32)
        d_c = torch.from_numpy(centers).cuda()
        d_b = torch.from_numpy(box).cuda()
        g63 = native.morton63(d_c, d_b).cpu().numpy().view(np.uint64)
        g30 = native.morton30(d_c, d_b).cpu().numpy().view(np.uint32)
        assert np.array_equal(g63, refcpu.morton63_codes(centers, box))
        assert np.array_equal(g30, refcpu.morton30_codes(centers, box))


def test_stage_centers_aabbs_reduce(torch_gpu):
    from mray_amd import native
    torch = torch_gpu
    s = scenes.random_triangles(5000, seed=5)
    d_pos = torch.from_numpy(s.positions).cuda()
    d_idx = torch.from_numpy(s.indices.astype(np.int32)).cuda()
    c, a = native.prim_centers_aabbs(d_pos, d_idx)
    rc, ra = refcpu.prim_centers_aabbs(s.positions, s.indices)
    assert np.array_equal(c.cpu().numpy().view(np.uint32), rc.view(np.uint32))
    assert np.array_equal(a.cpu().numpy().view(np.uint32), ra.view(np.uint32))
    box = native.reduce_aabb(a).cpu().numpy()
    assert np.array_equal(box, np.concatenate([ra[:, :3].min(0), ra[:, 3:].max(0)]))


@pytest.mark.parametrize("n", [1, 2, 4095, 4096, 4097, 250000])
def test_stage_radix_sort_stable(torch_gpu, n):
    from mray_amd import native
    torch = torch_gpu
    rng = np.random.default_rng(n)
    keys = rng.integers(0, 1 << 63, size=n, dtype=np.uint64)
    keys[::3] = keys[0]                     # many duplicates: stability matters
    keys[1::7] = np.uint64((1 << 63) - 1)
    vals = np.arange(n, dtype=np.uint32)
    dk = torch.from_numpy(keys.view(np.int64).copy()).cuda()
    dv = torch.from_numpy(vals.view(np.int32).copy()).cuda()
    native.radix_sort_u64_u32(dk, dv)
    gk = dk.cpu().numpy().view(np.uint64)
    gv = dv.cpu().numpy().view(np.uint32)
    order = np.argsort(keys, kind="stable")
    assert np.array_equal(gk, keys[order])
    assert np.array_equal(gv, vals[order])


def _lbvh_inputs(codes, seed):
    rng = np.random.default_rng(seed)
    n = len(codes)
    order = rng.permutation(n).astype(np.uint32)
    lo = rng.uniform(-1, 0, size=(n, 3)).astype(np.float32)
    aabbs = np.concatenate([lo, lo + 0.1], axis=1).astype(np.float32)
    return order, aabbs


def _gpu_lbvh(codes, order, aabbs):
    import torch
    from mray_amd import native
    nodes, boxes = native.lbvh_build(torch.from_numpy(codes.view(np.int64).copy()).cuda(),
                                     torch.from_numpy(order.view(np.int32).copy()).cuda(),
                                     torch.from_numpy(aabbs).cuda())
    return nodes.cpu().numpy().view(np.uint32), boxes.cpu().numpy()


def test_stage_lbvh_build_duplicate_runs(torch_gpu):
    """63-bit codes with long runs of equal codes (index-XOR fallback of Delta)."""
    rng = np.random.default_rng(2)
    n = 5000
    codes = rng.integers(0, 1 << 63, size=n, dtype=np.uint64)
    codes[100:700] = codes[100]
    codes[2000:2003] = codes[2000]
    codes = np.sort(codes)
    order, aabbs = _lbvh_inputs(codes, 3)
    assert refcpu.lbvh_tree_valid(codes, order)
    nodes, boxes = _gpu_lbvh(codes, order, aabbs)
    rnodes, rboxes = refcpu.lbvh_from_sorted(codes, order, aabbs)
    assert np.array_equal(nodes, rnodes)
    assert np.array_equal(boxes, rboxes)


def test_stage_lbvh_build_degenerate_codes(torch_gpu):
    """Codes that differ only in low bits next to equal-code runs: the
    reference's Delta yields a malformed tree.  The kernels stay in bounds and
    produce the same (malformed) child links as the oracle; parent links and
    box values of a malformed tree are order-dependent and not compared."""
    rng = np.random.default_rng(2)
    n = 3000
    codes = np.sort(rng.integers(0, 64, size=n).astype(np.uint64))
    order, aabbs = _lbvh_inputs(codes, 4)
    assert not refcpu.lbvh_tree_valid(codes, order)
    assert refcpu.lbvh_tree_valid(codes, order, strict=True)
    nodes, _ = _gpu_lbvh(codes, order, aabbs)
    rnodes, _ = refcpu.lbvh_from_sorted(codes, order, aabbs)
    # children are written by their own node's thread (deterministic); in a
    # malformed tree several nodes claim one child, so parent words race
    assert np.array_equal(nodes[:, :2], rnodes[:, :2])


def _canonical(nodes, prims):
    """The 4-wide tree as nested tuples from the root: each slot's box bits
    and either its leaf word or its subtree (node numbering removed)."""
    out = []
    stack = [0]
    seen = 0
    while stack:
        v = stack.pop()
        seen += 1
        w = nodes[v]
        row = [tuple(w[:24].tolist())]
        for k in range(4):
            c = int(w[24 + k])
            if c == 0xFFFFFFFF or c & 0x80000000:
                row.append(c)
            else:
                row.append("node")
                stack.append(c)
        out.append(tuple(row))
    return out, seen


@pytest.mark.parametrize("idx", [0, 1, 2, 3])
def test_device_collapse_is_host_collapse(torch_gpu, idx):
    """The LBVH builder's 4-wide tree and triangle soup built on the GPU
    (collapse.hip) against the same collapse on the host: the same nodes in
    the same depth-first order of their children, the same leaf words and
    the same soup."""
    from mray_amd import native
    scene = (_scenes() + [scenes.random_triangles(300001, seed=9)])[idx]
    dev = native.Accel(scene, builder="lbvh")
    host = native.Accel(scene, builder="lbvh", host_collapse=True)
    dn, dp = dev.read_wide()
    hn, hp = host.read_wide()
    di, hi = dev.info(), host.info()
    dev.close()
    host.close()
    print(f"scene {scene.name}: {scene.triangle_count} tris, wide nodes {di['wide_nodes']}", flush=True)
    assert di["wide_nodes"] == hi["wide_nodes"] == len(dn) == len(hn)
    assert np.array_equal(dp, hp)
    assert np.array_equal(np.sort(dp), np.arange(scene.triangle_count, dtype=np.uint32))
    cd, nd = _canonical(dn, dp)
    ch, nh = _canonical(hn, hp)
    assert nd == nh == len(dn)
    assert cd == ch


@pytest.mark.parametrize("noalloc,n", [(a, n) for a in (False, True) for n in
                                       (63, 64, 65, 1023, 4097, 12287, 12288, 12289, 16385, 524287, 524288, 600001,
                                        1048576)] + [(False, 2097151), (False, 2097152), (False, 2100001)])
def test_stage_radix_sort_forms(torch_gpu, n, noalloc):
    """Both sort forms around their limits: one workgroup up to 12288 pairs,
    then tiles of 1024, from 2^19 of 2048 and from 2^21 of 3072; ties
    everywhere, keys with the top bit set."""
    from mray_amd import native
    torch = torch_gpu
    rng = np.random.default_rng(n)
    keys = rng.integers(0, 1 << 64, size=n, dtype=np.uint64)
    keys[::3] &= np.uint64(0xFF00000000000003)      # long runs of equal keys
    vals = rng.permutation(n).astype(np.uint32)
    dk = torch.from_numpy(keys.view(np.int64).copy()).cuda()
    dv = torch.from_numpy(vals.view(np.int32).copy()).cuda()
    (native.radix_sort_u64_u32_noalloc if noalloc else native.radix_sort_u64_u32)(dk, dv)
    order = np.argsort(keys, kind="stable")
    assert np.array_equal(dk.cpu().numpy().view(np.uint64), keys[order])
    assert np.array_equal(dv.cpu().numpy().view(np.uint32), vals[order])


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 16, 17, 64, 65, 255, 256, 257, 1024, 1025, 4097, 65537])
def test_stage_lbvh_boxes_at_level_edges(torch_gpu, n):
    """Node boxes from the leaf-order levels (groups of 4, 16, 64, ...) where
    a level is full, one short and one over; equal to the climb's, bit for
    bit, since min and max do not depend on the order."""
    rng = np.random.default_rng(n)
    codes = np.unique(rng.integers(0, 1 << 63, size=n + 8, dtype=np.uint64))[:n]
    order, aabbs = _lbvh_inputs(codes, n + 1)
    nodes, boxes = _gpu_lbvh(codes, order, aabbs)
    rnodes, rboxes = refcpu.lbvh_from_sorted(codes, order, aabbs)
    assert np.array_equal(nodes, rnodes)
    assert np.array_equal(boxes.view(np.uint32), rboxes.view(np.uint32))


def test_malformed_reference_tree_is_rebuilt(torch_gpu):
    """A scene whose triangle centres share few Morton codes in long runs (the
    reference's Delta gives a malformed tree for them) builds with the strict
    tie-break, as the device-side check of the first tree demands; hits equal
    brute force."""
    from mray_amd import abi, native
    rng = np.random.default_rng(8)
    n = 3000
    # centres on 64 neighbouring cells of the 2^21 grid, spread by two far triangles
    cell = rng.integers(0, 4, size=(n, 3)).astype(np.float64) * 2.0 ** -21 * 1.00000001
    tri = rng.uniform(-1e-3, 1e-3, size=(n, 3, 3))
    tri -= tri.mean(axis=1, keepdims=True)
    tri += cell[:, None, :]
    tri[0] += 0.999
    pos = tri.reshape(-1, 3).astype(np.float32)
    s = scenes.random_triangles(n, seed=4)
    s.positions, s.indices = pos, np.arange(3 * n, dtype=np.uint32).reshape(-1, 3)
    s.tbn = np.tile(np.array([[1, 0, 0, 0]], np.float32), (3 * n, 1))
    o = refcpu.OracleScene(s)
    codes, order, nodes, _, _ = o.lbvh()
    print("distinct codes", len(np.unique(codes)), "reference tree valid",
          refcpu.lbvh_tree_valid(np.sort(codes), order), flush=True)
    assert not refcpu.lbvh_tree_valid(np.sort(codes), order)
    acc = native.Accel(s, builder="lbvh")
    _, gorder, gnodes, gboxes = acc.read_lbvh()
    rays = np.zeros((500, 8), np.float32)
    rays[:, 0:3] = rng.uniform(-2e-3, 2e-3, size=(500, 3)) + [0, 0, 1]
    rays[:, 6] = -1.0
    rays[:, 7] = 10.0
    prim, t, _ = acc.cast_closest(torch_gpu.from_numpy(rays).cuda())
    rp, rt, _ = o.cast_closest(rays, brute=True)
    assert (rp != abi.INVALID_PRIM).sum() > 100
    assert np.array_equal(prim.cpu().numpy().view(np.uint32), rp)
    assert np.array_equal(t.cpu().numpy(), rt)
    # the tree handed out is well formed: each node's children name it as parent
    inner = gnodes[:, :2][gnodes[:, :2] < 0x80000000]
    assert np.array_equal(np.sort(inner), np.arange(1, n - 1))
    leaves = gnodes[:, :2][gnodes[:, :2] >= 0x80000000] & 0x7FFFFFFF
    assert np.array_equal(np.sort(leaves), np.arange(n))
    acc.close()


@pytest.mark.parametrize("cap", [1 << 19, (1 << 21) + 1])
def test_sort_workspace_of_a_larger_count(torch_gpu, cap):
    """One workspace, sized for `cap` pairs, sorts counts on either side of
    the steps where tiles grow (more tiles just below them)."""
    from mray_amd import native
    torch = torch_gpu
    L = native.lib()
    nb = L.mray_radix_sort_temp_bytes(cap)
    tmp = torch.empty(nb, dtype=torch.uint8, device="cuda")
    rng = np.random.default_rng(cap)
    for n in (cap, cap - 1, cap - 2, (1 << 19) - 1, 504065):
        keys = rng.integers(0, 1 << 64, size=n, dtype=np.uint64)
        dk = torch.from_numpy(keys.view(np.int64).copy()).cuda()
        dv = torch.arange(n, dtype=torch.int32, device="cuda")
        native.check(L.mray_radix_sort_u64_u32(native._ptr(dk), native._ptr(dv), n, native._ptr(tmp), nb,
                                               native._stream()))
        order = np.argsort(keys, kind="stable")
        assert np.array_equal(dk.cpu().numpy().view(np.uint64), keys[order])
        assert np.array_equal(dv.cpu().numpy().view(np.uint32), order.astype(np.uint32))
