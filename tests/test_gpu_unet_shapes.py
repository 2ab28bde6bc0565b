"""The network's kernels at the grids where their tiles can go wrong: columns
that end inside a 16-pixel tile and inside an 8-pixel group at every level, an
odd number of rows and a single column at the coarsest level, one sample of a
larger batch after a full one (stale samples must not count), and sizes on
both sides of a forward block's rule and of the pixel slices. Against the numpy oracle with the tolerances of
test_gpu_unet.py (forward 2e-2, gradients as one vector by relative L2 5e-2:
bf16 steps of 2^-8 that different fp32 orders flip); a second run must give the
same bits."""
import importlib
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "oracle"))
import unet_oracle as U  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,h,w", [(1, 8, 8), (1, 16, 24), (2, 8, 40), (3, 24, 56), (1, 40, 104),
                                   (2, 32, 128)])
def test_network_at_ragged_grids(gpu, n, h, w):
    ws = importlib.import_module("gamera-cube_amd.warm_start")
    print(f"network {n} x {h} x {w}", flush=True)
    rng = np.random.default_rng(100 * h + w)
    params = U.init_params(h + w)
    for k in params:
        if k.endswith(".b"):
            params[k][...] = (0.05 * rng.standard_normal(params[k].shape)).astype(np.float32)
    names = [a + s for a, _, _, _ in U.LAYERS for s in (".w", ".b")] + ["head.w", "head.b"]
    net = ws.WarmStartNet(h, w, n + 1, seed=0)
    net.set_params(np.concatenate([params[k].ravel() for k in names]))
    full = rng.standard_normal((n + 1, h, w, U.IN_CHANNELS)).astype(np.float32)
    net.gradients(full, rng.standard_normal((n + 1, h, w)).astype(np.float32))
    x = rng.standard_normal((n, h, w, U.IN_CHANNELS)).astype(np.float32)
    target = rng.standard_normal((n, h, w)).astype(np.float32)
    out = net.forward(x)
    ref, acts = U.forward(params, x)
    assert np.linalg.norm(out - ref) <= 2e-2 * np.linalg.norm(ref)
    loss = net.gradients(x, target)
    got = net.grads()
    ref_loss, g_out = U.loss_and_grad_out(ref, target)
    want = U.backward(params, acts, g_out)
    flat = np.concatenate([np.asarray(want[k]).ravel() for k in names])
    err = np.linalg.norm(got - flat) / np.linalg.norm(flat)
    print(f"  gradients rel L2 {err:.2e}", flush=True)
    assert abs(loss - ref_loss) <= 1e-2 * ref_loss
    assert err <= 5e-2
    assert net.gradients(x, target) == pytest.approx(loss, rel=1e-6)
    assert np.array_equal(net.grads(), got)


@pytest.mark.parametrize("n", [15, 16, 17, 25])
def test_large_batches_match_single_samples(gpu, n):
    """Around the size from which features are uploaded in chunks (16 samples
    of 64 x 128 are 16 MiB; 17 and 25 end inside a chunk): every sample gives
    the bits it gives by itself, and parameters come back as they went."""
    ws = importlib.import_module("gamera-cube_amd.warm_start")
    print(f"batch of {n}", flush=True)
    rng = np.random.default_rng(n)
    net = ws.WarmStartNet(64, 128, n, seed=3)
    params = rng.standard_normal(net.param_count).astype(np.float32) * 0.02
    net.set_params(params)
    assert np.array_equal(net.params(), params)
    x = rng.standard_normal((n, 64, 128, 32)).astype(np.float32)
    out = net.forward(x)
    for k in (0, n // 2, n - 1):
        assert np.array_equal(net.forward(x[k:k + 1])[0], out[k])
