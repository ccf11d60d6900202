"""Host checks of the traversal trees (tests/cpp/bvh_check.cpp, built from the
library's own sah.cpp / bvh4.cpp): SAH tree validity, leaf coverage of the
4-wide and compressed 8-wide trees, conservative 8-bit box decoding, and a
host walk of the compressed tree against brute force; and of the one-level
walks' box tests (tests/cpp/slab_check.cpp, from the kernels' headers)."""
import os
import subprocess

import numpy as np
import pytest

from mray_amd import scenes

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CHECK = os.path.join(ROOT, "tests", "cpp", "bvh_check")


@pytest.mark.parametrize("name", ["soup", "terrain", "cornell", "flat_grid"])
def test_trees(tmp_path, name):
    if not os.path.exists(CHECK):
        pytest.fail("tests/cpp/bvh_check is not built; run __graft_entry__.build()")
    if name == "soup":
        s = scenes.random_triangles(6000, seed=3)
    elif name == "terrain":
        s = scenes.terrain_spheres(grid=96, spheres=60, width=64, height=36)
    elif name == "cornell":
        s = scenes.cornell()
    else:
        s = None
    if s is not None:
        tri = np.asarray(s.positions, np.float32)[np.asarray(s.indices)].reshape(-1, 9)
    else:
        # axis-aligned flat quads: zero-extent boxes on one axis everywhere
        q = []
        for i in range(20):
            for j in range(20):
                x0, y0 = i / 20, j / 20
                a, b, c, d = [x0, y0, 0], [x0 + .05, y0, 0], [x0 + .05, y0 + .05, 0], [x0, y0 + .05, 0]
                q += [a + b + c, a + c + d]
        tri = np.array(q, np.float32)
    path = str(tmp_path / "soup.bin")
    with open(path, "wb") as f:
        f.write(np.array([len(tri)], np.uint32).tobytes())
        f.write(tri.astype(np.float32).tobytes())
    r = subprocess.run([CHECK, path], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout + r.stderr


SLAB = os.path.join(ROOT, "tests", "cpp", "slab_check")


@pytest.mark.parametrize("extent,offset,scale,t_max",
                         [(e, 0.0, 1.0, 3.4e38) for e in (1e-3, 1.0, 1e4, 4e7, 1e8, 1e10, 1e12, 1e15, 1e20)] +
                         [(1.0, o, 1.0, 3.4e38) for o in (1e-3, 1e4, -3e5)] +
                         [(1e4, 1e3, m, 3.4e38) for m in (1e6, 1e-3, 1e-9, 1e-12, 1e-20)] +
                         [(1.0, 0.5, 1.0, 0.7), (1e-3, 0.0, 1e-3, 1.0), (1e9, 0.0, 1e9, 1.0)])
def test_slab_tests_are_conservative(extent, offset, scale, t_max):
    """The box tests of the one-level walks, on exact and on quantised boxes
    (compiled from the kernels' headers), against intervals in long double:
    no box whose interval is not empty is missed, for axis-parallel rays (+0,
    -0 and tiny components) that start inside, on planes or outside, at node
    extents from 1e-3 to 1e20, far from the origin, and with directions of any
    length; boxes a ray passes by clearly are missed."""
    if not os.path.exists(SLAB):
        pytest.fail("tests/cpp/slab_check is not built; run __graft_entry__.build()")
    r = subprocess.run([SLAB, str(extent), str(offset), str(scale), str(t_max), "5", "20000"],
                       capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout + r.stderr
