"""Renders whose slot pools outgrow the resident waves (about 393 K slots) or
the fused refill (4096 blocks of 256 slots), against the oracle.

Below about 393 K slots every wave's work is its own chunk by position; above,
the rest is handed out by counters, first of the wave's own part of the list and
then of the parts that still hold chunks.  Up to 4096 slot blocks the refill sums
the blocks' counts itself, above it scans them in a launch of its own.  A chunk
handed out twice or never would change a path's state and with it the pixel: the
films agree pixel by pixel up to the order of their float additions, and the
counts of paths and rays are equal.
"""
import numpy as np
import pytest

from mray_amd import abi, scenes
from oracle import refcpu

pytestmark = pytest.mark.gpu


def _same_film(film, ref):
    # at most 4 samples a pixel: three additions of one rounding each.  Against
    # the pixel's largest channel: a spectral path's colour comes of a 3 x 3
    # matrix (entries up to 3.3) whose rows cancel, up to 10 roundings of it.
    assert np.max(np.abs(film[3] - ref[3]) / np.maximum(ref[3], 1e-3)) < 1e-5
    scale = np.maximum(np.abs(ref[:3]).max(axis=0), 1e-3)
    assert np.max(np.abs(film[:3] - ref[:3]) / scale) < 1e-5


@pytest.mark.parametrize("slots", [393216, 393217, 400000, 614401, 1048576, 1048577])
def test_slot_pools_match_oracle(torch_gpu, slots):
    from mray_amd import native
    # 842,800 or 1,806,000 paths: slots are refilled
    w, h, spp = (700, 301, 4) if slots < 700000 else (1500, 301, 4)
    s = scenes.cornell(aspect=w / h)
    p = abi.render_params(w, h, spp, rr=(3, 3), seed=2, max_ray_count=slots)
    acc = native.Accel(s)
    r = native.Renderer(acc, p)
    for turn in range(2):                                # the second frame on used counters
        if turn:
            r.reset()
        st = r.render_all()
        film = r.film()
        ref, rst = refcpu.OracleScene(s).render(p)
        print(f"{slots} slots ({-(-slots // 256)} blocks): {st['dead_paths']} paths, {st['ext_rays']} rays", flush=True)
        for k in ("dead_paths", "ext_rays"):   # (the GPU casts no shadow rays that carry nothing)
            assert st[k] == rst[k], k
        _same_film(film, ref)
    r.close()
    acc.close()


def test_large_spectral_terrain_matches_oracle(torch_gpu):
    """Quantised nodes, uneven walks (waves that finish early take other
    parts' chunks), one sample of every pixel at once: 2400 slot blocks."""
    from mray_amd import native
    w, h = 1024, 600
    s = scenes.terrain_spheres(grid=96, spheres=60, width=w, height=h)
    p = abi.render_params(w, h, 1, rr=(4, 4), seed=5, spectral=True)
    refcpu.spectral_load(native.spectral_tables())
    acc = native.Accel(s)
    r = native.Renderer(acc, p)
    st = r.render_all()
    film = r.film()
    r.close()
    acc.close()
    ref, rst = refcpu.OracleScene(s).render(p)
    print(f"terrain: {st['ext_rays']} rays, {st['shadow_rays']} shadow rays", flush=True)
    for k in ("dead_paths", "ext_rays"):
        assert st[k] == rst[k], k
    _same_film(film, ref)


def test_large_batch_matches_oracle(torch_gpu):
    from mray_amd import native
    scs = [scenes.cornell(aspect=8 / 5), scenes.cornell(aspect=1.0, tess=6, seed=9)]
    views = [{"scene": 0, "width": 800, "height": 500, "spp": 2}, {"scene": 1, "width": 333, "height": 401, "spp": 3}]
    p = abi.render_params(1, 1, 1, rr=(3, 3), seed=6, max_ray_count=600000)
    accs = [native.Accel(s) for s in scs]
    b = native.BatchScene(accs)
    r = native.BatchRenderer(b, views, p)
    st = r.render_all()
    films = r.film()
    r.close()
    b.close()
    refs, rst = refcpu.render_batch([refcpu.OracleScene(s) for s in scs], views, p)
    for k in ("dead_paths", "ext_rays"):
        assert st[k] == rst[k], k
    for f, o in zip(films, refs):
        _same_film(f, o)
