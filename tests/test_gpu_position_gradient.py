"""The position gradient kernel (grad_kernel.hpp: one thread per point and
level, levels rounded up to a power of two) at level counts, feature counts
and batch sizes off its block shape, against the oracle. Marked gpu.

Tolerance: the fp32 outputs' 1e-5 of |ref| + rms; the batches are small so
that no point lies within rounding of a ReLU kink (a few thousand
pre-activations against an fp32 ulp of ~1e-7)."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_parity import make_trainer, omodel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,levels,feats,n", [
    (2, 1, 2, 1), (3, 1, 4, 257), (3, 5, 2, 33), (2, 17, 1, 15), (3, 32, 2, 9), (4, 32, 4, 8),
    (4, 3, 1, 85), (2, 16, 4, 17), (3, 12, 4, 16), (4, 16, 2, 31), (3, 31, 1, 7)])
def test_position_gradient_matches_oracle(oracle, dims, levels, feats, n):
    print(f"position gradient {dims}D L{levels} F{feats} n{n}", flush=True)
    enc = dict(n_levels=levels, n_features_per_level=feats, log2_hashmap_size=14,
               base_resolution=4.0, per_level_scale=1.2)
    rng = np.random.default_rng(levels * 100 + n)
    with make_trainer(dims, 2, enc, dict(n_neurons=24, n_hidden_layers=1), hash_range=0.5) as tr:
        hw, mw = tr.get_weights()
        pos = rng.random((n, dims), dtype=np.float32)
        out, jac = tr.evaluate_with_gradient(pos)
        oout, ojac = oracle.evaluate_with_gradient(omodel(oracle, tr), hw, mw, pos)
        for got, ref in ((out, oout), (jac, ojac)):
            tol = 1e-5 * (np.abs(ref) + np.sqrt((ref.astype(np.float64) ** 2).mean()))
            assert np.all(np.abs(got - ref) <= tol), float(np.abs(got - ref).max())
