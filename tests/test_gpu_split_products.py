"""The layer-wise path's wide products on split bf16 operands
(layer_split_kernel.hpp) at widths, depths and batch sizes off its 64-row,
64- and 128-column, 32-K tiles, against the oracle, and their error against 64
bits beside that of the fp32 arithmetic they replace. Marked gpu."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_parity import make_trainer, omodel, rel_tensor

pytestmark = pytest.mark.gpu

ENC = dict(n_levels=8, n_features_per_level=2, log2_hashmap_size=12, base_resolution=8.0,
           per_level_scale=1.5)


@pytest.mark.parametrize("width,layers,m,n", [
    (96, 2, 2, 1), (100, 2, 17, 63), (132, 2, 3, 65), (192, 3, 20, 33), (260, 2, 2, 64),
    (512, 2, 1, 31), (128, 3, 4, 129)])
def test_outputs_and_gradients_match_oracle(oracle, width, layers, m, n):
    """Outputs 1e-5 of |ref| + rms, MLP gradients 1e-5 of the largest: the
    repository's fp32 bars (batches small enough to keep clear of ReLU
    kinks)."""
    print(f"split products w{width}x{layers} M{m} n{n}", flush=True)
    rng = np.random.default_rng(width + n)
    with make_trainer(3, m, ENC, dict(n_neurons=width, n_hidden_layers=layers),
                      hash_range=0.5, batch=max(n, 2)) as tr:
        hw, mw = tr.get_weights()
        pos = rng.random((n, 3), dtype=np.float32)
        g = rng.normal(0, 1.0, (n, m)).astype(np.float32)
        ref = oracle.forward(omodel(oracle, tr), hw, mw, pos)
        tol = 1e-5 * (np.abs(ref) + np.sqrt((ref.astype(np.float64) ** 2).mean()))
        assert np.all(np.abs(tr.inference(pos) - ref) <= tol)
        tr.zero_gradients()
        tr.backward_accumulate(pos, g)
        _, gm = tr.debug_gradients()
        _, ogm, _, _, _ = oracle.forward_backward(omodel(oracle, tr), hw, mw, pos, d_out=g)
        assert rel_tensor(gm, ogm) <= 1e-5


@pytest.mark.parametrize("width,n", [(128, 70001), (256, 40000), (96, 3000)])
def test_forward_error_against_64_bits(width, n):
    """Both tile widths (128 columns from four blocks a CU on): the 2-norm error
    against 64 bits stays below that of the fp32 MFMA tiles at the same shape
    and inputs (2.6e-7, 4.3e-7, 2.1e-7; the split products 1.8e-7, 2.5e-7,
    1.5e-7). Bound: per layer K / 32 roundings of the accumulator at 2^-24, a
    random walk of sqrt(8) * 6e-8 = 1.7e-7 at K = 256 and once more for bias
    and output, over three layers in quadrature below 4e-7."""
    print(f"split products error w{width} n{n}", flush=True)
    rng = np.random.default_rng(width)
    with make_trainer(3, 4, ENC, dict(n_neurons=width, n_hidden_layers=3), hash_range=0.5,
                      batch=1024) as tr:
        _, mw = tr.get_weights()
        pos = rng.random((n, 3), dtype=np.float32)
        out = tr.inference(pos)
        x = tr.debug_encode(pos).astype(np.float64)
        at, sizes = 0, [16, width, width, width, 4]
        for i, (a, b) in enumerate(zip(sizes, sizes[1:])):
            x = x @ mw[at:at + a * b].reshape(a, b).astype(np.float64) + mw[at + a * b:at + a * b + b]
            at += a * b + b
            if i < 3:
                x = np.maximum(x, 0)
        assert np.linalg.norm(out - x) <= 4e-7 * np.linalg.norm(x)
