"""Radiance-cache queries on several streams and from several caches: the
workspace of the split encoding belongs to the GPU, one area per stream."""
import ctypes
import gc

import numpy as np
import pytest

from tests.test_gpu_nrc import _records

pytestmark = pytest.mark.gpu


def _infer(nrc, rec, n, out, stream=None, count=None):
    from mray_amd import native
    native.check(native.lib().mray_nrc_infer(nrc.h, native._ptr(rec), 0 if count is not None else n,
                                             native._ptr(count) if count is not None else None, native._ptr(out),
                                             ctypes.c_void_p(stream.cuda_stream) if stream else None))


def test_caches_share_query_memory(torch_gpu):
    """The query workspace belongs to the GPU and not to each cache: 24 small
    caches, as a batch renderer attaches them, hold a few MiB each at most.
    Queries of several caches on more streams than there are areas, in
    changing sizes and with no waits between, answer as the one-kernel form;
    the last cache's end gives the memory back."""
    from mray_amd import native
    torch = torch_gpu
    gc.collect()                                         # caches that earlier tests left
    first = native.Nrc(levels=3, log2_table=12, max_batch=64, seed=99)
    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    caches = [native.Nrc(levels=3, log2_table=12, max_batch=64, seed=k) for k in range(24)]
    held = free0 - torch.cuda.mem_get_info()[0]
    print(f"24 more caches hold {held / 2**20:.1f} MiB", flush=True)
    # each about 15 allocations of at most 96 KiB; the driver rounds a
    # size class up to 2 MiB
    assert held < 24 * (8 << 20)
    rng = np.random.default_rng(5)
    rec = torch.from_numpy(_records(rng, 131073)).cuda()
    sizes = (100, 4096, 4097, 70000, 33, 20000, 131072, 131073)
    one = {}
    for k in range(6):
        for n in sizes:
            count = torch.tensor([n], dtype=torch.int32, device="cuda")
            one[k, n] = torch.empty((n, 3), device="cuda")
            _infer(caches[k], rec, n, one[k, n], count=count)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(6)]
    got = {}
    for turn in range(3):
        for k, s in enumerate(streams):
            for n in sizes:
                got[turn, k, n] = torch.zeros((n, 3), device="cuda")
    torch.cuda.synchronize()
    for (turn, k, n), out in got.items():
        _infer(caches[k], rec, n, out, stream=streams[(k + turn) % 6])
    torch.cuda.synchronize()
    for (turn, k, n), out in got.items():
        assert torch.equal(out, one[k, n]), (turn, k, n)
    for c in caches:
        c.close()
    del got, one
    before = torch.cuda.mem_get_info()[0]
    first.close()
    assert torch.cuda.mem_get_info()[0] - before >= 32 << 20


def test_queries_on_two_streams_overlap(torch_gpu):
    """A short query on one stream does not wait for another stream's long
    ones (on one of four streams at least: two streams may share a hardware
    queue)."""
    from mray_amd import native
    torch = torch_gpu
    nrc = native.Nrc(levels=16, log2_table=16, max_batch=64, seed=1)
    rec = torch.rand((1 << 19, 11), device="cuda")
    long, short = torch.empty((1 << 19, 3), device="cuda"), torch.empty((4, 512, 3), device="cuda")
    streams = [torch.cuda.Stream() for _ in range(5)]
    for k in range(5):                                   # areas allocated, kernels loaded
        _infer(nrc, rec, 512, short[k % 4], stream=streams[k])
    torch.cuda.synchronize()
    early = []
    for k in range(4):
        done = [torch.cuda.Event() for _ in range(2)]
        for _ in range(100):                             # tens of ms
            _infer(nrc, rec, 1 << 19, long, stream=streams[0])
        done[0].record(streams[0])
        _infer(nrc, rec, 512, short[k], stream=streams[1 + k])
        done[1].record(streams[1 + k])
        done[1].synchronize()
        early.append(not done[0].query())
        torch.cuda.synchronize()
    print("finished before the long queries:", early, flush=True)
    assert any(early)
    nrc.close()
