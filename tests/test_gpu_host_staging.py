"""Host-pointer calls through the pinned staging memory and above its
limit (512 KB a direction): the same results as the device-pointer calls,
which copy nothing, at array sizes around the 16-byte pieces, the 256-byte
regions and the limit. Marked gpu."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_parity import make_trainer

pytestmark = pytest.mark.gpu

ENC = dict(n_levels=8, n_features_per_level=2, log2_hashmap_size=14, base_resolution=8.0,
           per_level_scale=1.5)
NET = dict(n_neurons=32, n_hidden_layers=1)


@pytest.mark.parametrize("dims,m,n", [
    (3, 1, 1), (2, 3, 21), (3, 3, 64), (3, 3, 65), (4, 16, 4096),
    (4, 4, 32768),   # inputs exactly the limit
    (4, 4, 32769),   # one point above it
    (3, 16, 8191), (3, 16, 8193)])  # outputs on either side of the limit
def test_host_calls_match_device_calls(dims, m, n):
    import torch
    print(f"staging {dims}D M{m} n{n}", flush=True)
    rng = np.random.default_rng(n)
    x = rng.random((n, dims), dtype=np.float32)
    y = rng.random((n, m), dtype=np.float32)
    kw = dict(batch=max(n, 2), hash_range=0.5)
    with make_trainer(dims, m, ENC, NET, **kw) as a, make_trainer(dims, m, ENC, NET, **kw) as b:
        for seed in range(2):  # the second call finds the first one's bytes in the staging memory
            dx = torch.from_numpy(x).cuda()
            out = torch.full((n, m), np.nan, device="cuda")
            torch.cuda.synchronize()
            a.inference_device(dx.data_ptr(), out.data_ptr(), n)
            a.synchronize()
            assert np.array_equal(a.inference(x), out.cpu().numpy())
            assert np.allclose(a.forward_for_training(x), out.cpu().numpy(), rtol=1e-4, atol=1e-5)
            jo, jac = a.evaluate_with_gradient(x)
            assert jac.shape == (n, m, dims) and np.isfinite(jac).all()
            assert np.allclose(jo, out.cpu().numpy(), rtol=1e-4, atol=1e-5)
            dy, loss = torch.from_numpy(y).cuda(), torch.zeros(1, device="cuda")
            torch.cuda.synchronize()
            host = a.training_step(x, y)
            b.training_step_device(dx.data_ptr(), dy.data_ptr(), n, loss.data_ptr())
            b.synchronize()
            # the same kernels on the same bytes; this shape's weight gradients
            # add through LDS atomics, so later losses may differ by their order
            assert host == pytest.approx(float(loss[0]), rel=1e-6 if seed == 0 else 1e-4)
            x = x[::-1].copy()
            y = y[::-1].copy()


def test_two_threads_share_the_staging_memory():
    """One call at a time holds the context's staging memory; a call of another
    thread meanwhile copies without it. Each thread's trainer keeps its own
    results."""
    import threading
    rng = np.random.default_rng(5)
    xs = [rng.random((900 + 700 * k, 3), dtype=np.float32) for k in range(2)]
    trs = [make_trainer(3, 2, ENC, NET, seed=k + 1, hash_range=0.5) for k in range(2)]
    want = [tr.inference(x) for tr, x in zip(trs, xs)]
    bad = []

    def work(k):
        for _ in range(60):
            if not np.array_equal(trs[k].inference(xs[k]), want[k]):
                bad.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for tr in trs:
        tr.close()
    assert not bad
