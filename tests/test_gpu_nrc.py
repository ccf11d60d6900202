"""Neural radiance cache kernels vs the CPU oracle (oracle/nrc_ref.py).

Forward: the GPU's hash encoding + bf16-MFMA MLP against the oracle's
bf16-emulating forward on the same fp32 master parameters (the grid enters as
its fp16 copy).  Backward: every weight gradient and the grid gradient of the
relative L2 loss against the oracle's analytic gradients (themselves pinned by
finite differences in test_oracle_nrc.py).  Adam: one step against the
closed-form update on the GPU's own gradients.  Tolerances reflect bf16
operands with fp32 accumulation in a different order than the oracle's.
"""
import numpy as np
import pytest

from mray_amd import abi
from oracle import nrc_ref as N

pytestmark = pytest.mark.gpu


def _records(rng, n):
    rec = np.zeros((n, 11), np.float32)
    rec[:, 0:3] = rng.uniform(0.0, 1.0, size=(n, 3))
    rec[:, 3:8] = rng.uniform(0.0, 1.0, size=(n, 5))
    rec[:, 8:11] = rng.uniform(0.0, 1.0, size=(n, 3))
    return rec


def _oracle_weights(w):
    return [w[l] for l in range(5)] + [w[5][:, :N.OUT_PAD]]


def _rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-30))


@pytest.fixture(scope="module")
def nrc(torch_gpu):
    from mray_amd import native
    n = native.Nrc(max_batch=4096, seed=3)
    # larger grid values than the default init so the encoding matters
    rng = np.random.default_rng(11)
    n.write(abi.NRC_GRID, rng.uniform(-0.5, 0.5, size=(n.grid_params,)).astype(np.float32))
    yield n
    n.close()


def test_forward_matches_oracle(nrc, torch_gpu):
    torch = torch_gpu
    rng = np.random.default_rng(0)
    rec = _records(rng, 1000)                       # not a multiple of 32: tail tile
    out = nrc.infer(torch.from_numpy(rec).cuda()).cpu().numpy()
    w = nrc.read(abi.NRC_WEIGHTS)
    grid = N.f16(nrc.read(abi.NRC_GRID))
    x, _ = N.encode_inputs(rec, grid, N.level_scale())
    y, _ = N.forward(x, _oracle_weights(w), mixed=True)
    e = _rel(out, y)
    print(f"forward rel err {e:.3e}, |y| {np.abs(y).mean():.3e}", flush=True)
    assert np.isfinite(out).all()
    assert e < 2e-2


def test_backward_matches_oracle(nrc, torch_gpu):
    torch = torch_gpu
    rng = np.random.default_rng(1)
    B = 512
    rec = _records(rng, B)
    tgt = rng.uniform(0.0, 2.0, size=(B, 3)).astype(np.float32)
    nrc.zero_grads()
    nrc.backward(torch.from_numpy(rec).cuda(), torch.from_numpy(tgt).cuda())
    loss = nrc.loss()
    wg = nrc.read(abi.NRC_WEIGHT_GRADS)
    gg = nrc.read(abi.NRC_GRID_GRADS)
    w = nrc.read(abi.NRC_WEIGHTS)
    grid = N.f16(nrc.read(abi.NRC_GRID))
    x, aux = N.encode_inputs(rec, grid, N.level_scale())
    y, acts = N.forward(x, _oracle_weights(w), mixed=True)
    ref_loss, dy = N.loss_grad(y, tgt, B)
    grads, dx = N.backward(dy, acts, _oracle_weights(w), mixed=True)
    print(f"loss gpu {loss:.6f} cpu {ref_loss:.6f}", flush=True)
    assert loss == pytest.approx(ref_loss, rel=2e-2)
    for l in range(6):
        g_gpu = wg[l] if l < 5 else wg[5][:, :3]
        g_ref = grads[l] if l < 5 else grads[5][:, :3]
        e = _rel(g_gpu, g_ref)
        print(f"layer {l}: rel err {e:.3e}", flush=True)
        assert e < 5e-2
    assert np.all(wg[5][:, 3:] == 0.0)
    ref_gg = N.grid_grad(dx, aux, grid.shape)
    e = _rel(gg, ref_gg)
    print(f"grid grad rel err {e:.3e}", flush=True)
    assert e < 5e-2
    nrc.zero_grads()


def test_adam_step(nrc, torch_gpu):
    torch = torch_gpu
    rng = np.random.default_rng(2)
    B = 256
    rec = _records(rng, B)
    tgt = rng.uniform(0.0, 1.0, size=(B, 3)).astype(np.float32)
    from mray_amd import native
    fresh = native.Nrc(max_batch=1024, seed=5)
    w0 = fresh.read(abi.NRC_WEIGHTS).astype(np.float64)
    fresh.backward(torch.from_numpy(rec).cuda(), torch.from_numpy(tgt).cuda())
    g = fresh.read(abi.NRC_WEIGHT_GRADS).astype(np.float64)
    fresh.adam()
    w1 = fresh.read(abi.NRC_WEIGHTS).astype(np.float64)
    # first Adam step: w - lr * g / (|g| + eps) elementwise (bias-corrected)
    p, _, _ = N.adam(w0, g, np.zeros_like(g), np.zeros_like(g), 1, lr=1e-2)
    touched = g != 0
    assert touched.sum() > 1000
    assert np.allclose(w1[touched], p[touched], rtol=1e-5, atol=1e-7)
    assert np.all(fresh.read(abi.NRC_WEIGHT_GRADS) == 0.0)     # cleared for the next step
    fresh.close()


def test_training_reduces_loss(torch_gpu):
    """Online training on a smooth radiance-like field: the relative L2 loss
    falls by an order of magnitude within 300 Adam steps."""
    torch = torch_gpu
    from mray_amd import native
    nrc = native.Nrc(max_batch=4096, seed=7)
    rng = np.random.default_rng(3)

    def field(r):
        p = r[:, 0:3]
        base = 0.5 + 0.4 * np.sin(6.0 * p[:, 0]) * np.cos(4.0 * p[:, 2])
        return (base[:, None] * (0.3 + r[:, 8:11])).astype(np.float32)
    losses = []
    for step in range(300):
        rec = _records(rng, 4096)
        tgt = field(rec)
        nrc.train(torch.from_numpy(rec).cuda(), torch.from_numpy(tgt).cuda())
        if step % 50 == 0 or step == 299:
            losses.append(nrc.loss())
    print("losses", losses, flush=True)
    test = _records(rng, 2048)
    pred = nrc.infer(torch.from_numpy(test).cuda()).cpu().numpy()
    ref = field(test)
    rel = float(np.mean((pred - ref) ** 2 / (ref ** 2 + 0.01)))
    print(f"held-out relMSE {rel:.3e}", flush=True)
    assert losses[-1] < 0.1 * losses[0]
    assert rel < 0.02
    nrc.close()


def test_lazy_grid_adam(torch_gpu):
    """MRAY_NRC_LAZY_ADAM: over two steps, grid entries with a zero gradient in
    a step keep parameter (and moments); entries with one follow Adam with
    their own moments.  Checked against the oracle's Adam applied entrywise
    under the same masks.  The MLP stays dense (as test_adam_step)."""
    torch = torch_gpu
    from mray_amd import native
    rng = np.random.default_rng(11)
    n = native.Nrc(max_batch=1024, seed=7, lazy_adam=True)
    m = v = None
    touched_before = None
    for step in (1, 2):
        p = n.read(abi.NRC_GRID).astype(np.float64)
        if m is None:
            m, v = np.zeros_like(p), np.zeros_like(p)
        rec = _records(rng, 128)
        tgt = rng.uniform(0.0, 1.0, size=(128, 3)).astype(np.float32)
        n.backward(torch.from_numpy(rec).cuda(), torch.from_numpy(tgt).cuda())
        g = n.read(abi.NRC_GRID_GRADS).astype(np.float64)
        n.adam()
        got = n.read(abi.NRC_GRID).astype(np.float64)
        touched = g != 0
        assert touched.sum() > 1000 and (~touched).sum() > 1000
        p2, m2, v2 = N.adam(p, g, m, v, step, lr=1e-2)
        assert np.array_equal(got[~touched], p[~touched])       # not written at all
        assert np.allclose(got[touched], p2[touched], rtol=1e-5, atol=1e-7)
        m = np.where(touched, m2, m)
        v = np.where(touched, v2, v)
        if touched_before is not None:
            # entries with momentum from step 1 but no gradient now stay put,
            # where dense Adam would still move them
            idle = touched_before & ~touched
            assert idle.sum() > 100
        touched_before = touched
    assert np.all(n.read(abi.NRC_GRID_GRADS) == 0.0)
    n.close()


@pytest.mark.parametrize("levels,log2_table", [(1, 12), (6, 14), (16, 15)])
def test_infer_forms_agree(torch_gpu, levels, log2_table):
    """Queries encoded in a pass of their own (the count known on the host,
    chunks of 2^19) answer exactly as in the one-kernel form (the count read
    on the device), at the counts where a tile, a block and the chunk change."""
    import ctypes
    from mray_amd import native
    torch = torch_gpu
    nrc = native.Nrc(levels=levels, log2_table=log2_table, max_batch=32, seed=levels)
    rng = np.random.default_rng(levels)
    nrc.write(abi.NRC_GRID, rng.uniform(-0.5, 0.5, size=(nrc.grid_params,)).astype(np.float32))
    rec = _records(rng, 600000)
    rec[:64, 0:3] = rng.integers(0, 2, size=(64, 3))       # corners of the box
    d = torch.from_numpy(rec).cuda()
    for n in (1, 31, 32, 33, 255, 256, 257, 511, 513, 524288, 524289, 600000):
        one = torch.full((n + 1, 3), -7.0, device="cuda")
        count = torch.tensor([n], dtype=torch.int32, device="cuda")
        native.check(native.lib().mray_nrc_infer(nrc.h, ctypes.c_void_p(d.data_ptr()), 0,
                                                 ctypes.c_void_p(count.data_ptr()),
                                                 ctypes.c_void_p(one.data_ptr()), None))
        assert torch.equal(nrc.infer(d[:n].contiguous()), one[:n]), n
        assert torch.all(one[n:] == -7.0)
    nrc.close()


@pytest.mark.parametrize("lazy", [False, True])
@pytest.mark.parametrize("levels,log2_table,count", [(1, 10, 32), (5, 13, 992), (16, 14, 1024), (16, 16, 4128)])
def test_train_is_backward_then_adam(torch_gpu, levels, log2_table, count, lazy):
    """A training step (gradients applied where they are formed) against the
    separate passes: the weights equal bit for bit (their sums have one
    order); the grid's sums are LDS or global atomics, whose order moves a
    gradient by rounding and, where it cancels to nothing, Adam's normalised
    step by up to twice the rate.  Gradients pending from an earlier backward
    pass are applied as well, and nothing is left pending."""
    from mray_amd import native
    torch = torch_gpu
    rng = np.random.default_rng(count)
    rec = [torch.from_numpy(_records(rng, count)).cuda() for _ in range(3)]
    tgt = [torch.from_numpy(rng.uniform(0, 2, size=(count, 3)).astype(np.float32)).cuda() for _ in range(3)]
    caches = [native.Nrc(levels=levels, log2_table=log2_table, max_batch=count, seed=4, lazy_adam=lazy)
              for _ in range(2)]
    init = rng.uniform(-0.3, 0.3, size=(caches[0].grid_params,)).astype(np.float32)
    for c in caches:
        c.write(abi.NRC_GRID, init)
    a, b = caches
    a.train(rec[0], tgt[0])
    a.backward(rec[1], tgt[1])
    a.train(rec[2], tgt[2])
    b.backward(rec[0], tgt[0])
    b.adam()
    b.backward(rec[1], tgt[1])
    b.backward(rec[2], tgt[2])
    b.adam()
    wa, wb = a.read(abi.NRC_WEIGHTS), b.read(abi.NRC_WEIGHTS)
    ga, gb = a.read(abi.NRC_GRID), b.read(abi.NRC_GRID)
    moved = np.abs(ga.reshape(-1) - init) > 0
    off = np.abs(ga - gb)
    print(f"weights off {np.abs(wa - wb).max():.2e}, grid off {off.max():.2e}, "
          f"over 1e-4: {np.mean(off > 1e-4):.2e}, moved {moved.mean():.3f}", flush=True)
    # the second step's inputs differ by the grid's rounding: one bf16 ulp of
    # an activation here and there
    assert _rel(wa, wb) < 1e-4
    assert moved.sum() > 8 * levels and np.mean(off > 1e-4) < 1e-3 and off.max() <= 4.1e-2
    for c in caches:
        assert np.all(c.read(abi.NRC_WEIGHT_GRADS) == 0.0) and np.all(c.read(abi.NRC_GRID_GRADS) == 0.0)
        c.close()


@pytest.mark.parametrize("levels,log2_table,count", [(5, 13, 992), (16, 16, 4128)])
def test_captured_backward_leaves_gradients_pending(torch_gpu, levels, log2_table, count):
    """A backward pass captured in a graph leaves gradients pending at every
    replay, whatever the host called since: the next training step applies
    them, and the loss read back is the replayed batch's."""
    from mray_amd import native
    torch = torch_gpu
    rng = np.random.default_rng(levels)
    rec = [torch.from_numpy(_records(rng, count)).cuda() for _ in range(3)]
    tgt = [torch.from_numpy(rng.uniform(0, 2, size=(count, 3)).astype(np.float32)).cuda() for _ in range(3)]
    a, b = (native.Nrc(levels=levels, log2_table=log2_table, max_batch=count, seed=4) for _ in range(2))
    init = rng.uniform(-0.3, 0.3, size=(a.grid_params,)).astype(np.float32)
    for c in (a, b):
        c.write(abi.NRC_GRID, init)
        c.train(rec[0], tgt[0])                    # kernels loaded before the capture
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        native.check(native.lib().mray_nrc_backward(a.h, native._ptr(rec[1]), native._ptr(tgt[1]), count,
                                                    native._stream()))
    for step in range(3):                          # replays between the program's own calls
        a.train(rec[2], tgt[2])
        g.replay()
        b.train(rec[2], tgt[2])
        b.backward(rec[1], tgt[1])
        la, lb = a.loss(), b.loss()
        assert la == pytest.approx(lb, rel=1e-3)
        if step == 1:
            for c in (a, b):
                c.zero_grads()
        if step == 2:
            a.backward(rec[0][:32].contiguous(), tgt[0][:32].contiguous())
            b.backward(rec[0][:32].contiguous(), tgt[0][:32].contiguous())
            for c in (a, b):
                c.adam()
            # Adam has run since, from the host's view nothing is pending
            g.replay()
            b.backward(rec[1], tgt[1])
            assert a.loss() == pytest.approx(b.loss(), rel=1e-3)
    # b's reference: the same gradients, applied by the separate passes
    a.train(rec[0], tgt[0])
    b.backward(rec[0], tgt[0])
    b.adam()
    wa, wb = a.read(abi.NRC_WEIGHTS), b.read(abi.NRC_WEIGHTS)
    off = np.abs(a.read(abi.NRC_GRID) - b.read(abi.NRC_GRID))
    print(f"weights off {np.abs(wa - wb).max():.2e}, grid off {off.max():.2e}", flush=True)
    # as in test_train_is_backward_then_adam, over six steps
    assert _rel(wa, wb) < 1e-3
    assert np.mean(off > 1e-3) < 1e-2
    for c in (a, b):
        assert np.all(c.read(abi.NRC_WEIGHT_GRADS) == 0.0) and np.all(c.read(abi.NRC_GRID_GRADS) == 0.0)
        c.close()
