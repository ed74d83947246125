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


@pytest.mark.parametrize("width,n,bound", [
    (128, 70001, 2.2e-7), (256, 40000, 3.3e-7), (96, 3000, 1.8e-7)])
def test_forward_error_against_64_bits(width, n, bound):
    """Both tile widths (128 columns from four blocks a CU on): the 2-norm error
    against 64 bits stays below that of the fp32 MFMA tiles at the same shape
    and inputs (2.6e-7, 4.3e-7, 2.1e-7; the split products 1.8e-7, 2.5e-7,
    1.5e-7). Bounds halfway between the two, so that neither the fp32 tiles nor
    split products as inexact as them pass; K / 32 roundings of the accumulator
    at 2^-24, a random walk of sqrt(8) * 6e-8 = 1.7e-7 a layer at K = 256, lie
    below."""
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
        assert np.linalg.norm(out - x) <= bound * np.linalg.norm(x)


# (width, points): 128-column tiles in the delta, dx and (256 wide) weight-
# gradient products, over many chunks of the batch; 64-column ones and few
# chunks. Bounds of the split products' dW1, db1 and, through dx, the table,
# halfway between their errors (3.5e-7, 4.4e-7, 3.5e-6; 2.2e-7, 2.2e-7, 2.6e-6;
# 1.7e-7, 1.9e-7, 3.7e-6) and the fp32 MFMA tiles' (9.8e-7, 8.9e-7, 5.2e-6;
# 5.7e-7, 4.6e-7, 3.8e-6; 4.4e-7, 4.4e-7, 5.2e-6)
@pytest.mark.parametrize("width,n,dw1,db1,table", [
    (256, 66001, 6.5e-7, 6.5e-7, 4.3e-6), (128, 70001, 4e-7, 3.4e-7, 3.2e-6),
    (256, 3001, 3e-7, 3.1e-7, 4.4e-6)])
def test_gradient_error_against_64_bits(width, n, dw1, db1, table):
    """Weight, bias and table gradients of a step's backward against 64 bits on
    the same features, with pre-activations kept away from 0 by the biases (no
    ReLU mask that a rounding decides). The first and last layers' products are
    fp32 ones in both (2.3e-7 to 1.2e-6): below twice the largest. Of the
    table's error most is the fixed point's truncation, which an ulp of d can
    move."""
    torch = pytest.importorskip("torch")
    print(f"split gradients error w{width} n{n}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(width + n)
    enc = dict(n_levels=16, n_features_per_level=2, log2_hashmap_size=12, base_resolution=8.0,
               per_level_scale=1.3)
    sizes = [32, width, width, 4]
    rng = np.random.default_rng(n)
    with make_trainer(3, 4, enc, dict(n_neurons=width, n_hidden_layers=2), hash_range=0.5,
                      batch=n) as tr:
        hw, mw = (w.copy() for w in tr.get_weights())
        at, spans = 0, []
        for i, (a, b) in enumerate(zip(sizes, sizes[1:])):
            spans.append((at, at + a * b, at + a * b + b))
            if i < 2:
                mw[spans[-1][1]:spans[-1][2]] = np.where(np.arange(b) % 2, 4.0, -4.0) * (1 + 7 * i)
            at = spans[-1][2]
        tr.set_initial_weights(hw, mw)
        pos = rng.random((n, 3), dtype=np.float32)
        dout = rng.normal(0, 1.0, (n, 4)).astype(np.float32)
        feats, idx, wts = tr.debug_encode(pos, with_corners=True)
        tr.zero_gradients()
        tr.backward_accumulate(pos, dout)
        gh, gm = tr.debug_gradients()
        w = [torch.from_numpy(mw[p:q].reshape(a, b)).cuda().double()
             for (p, q, _), a, b in zip(spans, sizes, sizes[1:])]
        bias = [torch.from_numpy(mw[q:r]).cuda().double() for _, q, r in spans]
        acts = [torch.from_numpy(feats).cuda().double()]
        for i in range(2):
            z = acts[-1] @ w[i] + bias[i]
            assert float(z.abs().min()) > 1e-4
            acts.append(z.relu())
        d, errors = torch.from_numpy(dout).cuda().double(), {}
        for i in (2, 1, 0):
            p, q, r = spans[i]
            for key, lo, hi, want in ((f"dW{i}", p, q, (acts[i].T @ d).flatten()),
                                      (f"db{i}", q, r, d.sum(0))):
                got = torch.from_numpy(gm[lo:hi]).cuda().double()
                errors[key] = float((got - want).norm() / want.norm())
            d = d @ w[i].T.contiguous()
            if i:
                d *= acts[i] > 0
        # the table's fixed point: every contribution times 65536, truncated
        want = torch.zeros(16, 1 << 12, 2, dtype=torch.float64, device="cuda")
        ci, cw = torch.from_numpy(idx.astype(np.int64)).cuda(), torch.from_numpy(wts).cuda().double()
        for lv in range(16):
            for c in range(8):
                want[lv].index_add_(0, ci[:, lv, c], torch.trunc(
                    d[:, 2 * lv:2 * lv + 2] * cw[:, lv, c, None] * 65536))
        got = torch.from_numpy(gh.astype(np.float64)).cuda().view_as(want)
        errors["table"] = float((got - want).norm() / want.norm())
        print(" ".join(f"{k} {v:.2e}" for k, v in errors.items()), flush=True)
        bounds = {"dW1": dw1, "db1": db1, "table": table}
        for key, error in errors.items():
            assert error <= bounds.get(key, 2.4e-6), (key, error)


def _forward64(mw, sizes, x):
    """The MLP in 64 bits with the path's ReLU (a NaN gives 0)."""
    at, acts = 0, [x]
    for i, (a, b) in enumerate(zip(sizes, sizes[1:])):
        w = mw[at:at + a * b].reshape(a, b).astype(np.float64)
        x = x @ w + mw[at + a * b:at + a * b + b]
        at += a * b + b
        if i < len(sizes) - 2:
            x = np.where(x > 0, x, 0.0)
        acts.append(x)
    return acts


def _same(got, want, tol):
    """Equal where infinite or NaN, within tol of |want| + rms elsewhere."""
    got, want = np.asarray(got, np.float64), np.asarray(want, np.float64)
    kinds = (np.isnan, np.isposinf, np.isneginf)
    for kind in kinds:
        assert np.array_equal(kind(got), kind(want)), kind.__name__
    fin = np.isfinite(want)
    if fin.any():
        rms = np.sqrt((want[fin] ** 2).mean())
        assert np.all(np.abs(got[fin] - want[fin]) <= tol * (np.abs(want[fin]) + rms))


# an infinite entry of W_0 makes a hidden unit's activations infinite; one of
# W_1 is itself an operand of the split product
@pytest.mark.parametrize("layer,value", [
    (0, np.inf), (1, np.inf), (1, -np.inf), (1, 3.4e38), (1, -3.4e38)])
@pytest.mark.parametrize("width,n", [(256, 200), (96, 65)])
def test_values_without_bf16_parts(width, n, layer, value):
    """Infinities and finite values above bf16's largest (3.39e38) keep their
    fp32 meaning: outputs and weight gradients are infinite, NaN and finite
    where 64 bits says so, and a step over infinite outputs reports a loss that
    is not finite. The finite rest within 1e-5, the repository's fp32 bar."""
    print(f"split products without parts w{width} layer {layer} {value}", flush=True)
    rng = np.random.default_rng(width + layer)
    sizes = [16, width, width, 2]
    at = [0, 17 * width, (17 + width + 1) * width]
    with make_trainer(3, 2, ENC, dict(n_neurons=width, n_hidden_layers=2), hash_range=0.5,
                      batch=n) as tr, np.errstate(all="ignore"):
        hw, mw = (w.copy() for w in tr.get_weights())
        hw = np.abs(hw)  # positive features: an infinite W_0[0][unit] reaches every point
        if np.isfinite(value):
            hw *= np.float32(1e-3)  # hidden activations below 1, so that 3.4e38 times them is finite
        tr.set_initial_weights(hw, mw)
        pos = rng.random((n, 3), dtype=np.float32)
        feats = tr.debug_encode(pos).astype(np.float64)
        unit = int(np.argmax((_forward64(mw, sizes, feats)[1] > 0).sum(0)))
        if layer == 0:
            mw[unit] = value
            row = at[1] + unit * width  # W_1's row of that unit: values whose lower parts are 0
            mw[row:row + width] = np.where(rng.random(width) < 0.5, 0.25, -0.25)
        else:
            mw[at[1] + unit * width + 3] = value
        tr.set_initial_weights(hw, mw)
        acts = _forward64(mw, sizes, feats)
        if np.isfinite(value):
            assert np.abs(acts[2]).max() < 3.4e38
        _same(tr.inference(pos), acts[-1], 1e-5)
        if np.isfinite(value):
            return
        d = rng.normal(0, 1.0, (n, 2)).astype(np.float32)
        tr.zero_gradients()
        tr.backward_accumulate(pos, d)
        _, gm = tr.debug_gradients()
        want, d = [], d.astype(np.float64)
        for i in (2, 1, 0):
            a, b = sizes[i], sizes[i + 1]
            want.append(np.concatenate([(acts[i].T @ d).ravel(), d.sum(0)]))
            d = d @ mw[at[i]:at[i] + a * b].reshape(a, b).astype(np.float64).T
            if i:
                d = np.where(acts[i] > 0, d, 0.0)
        _same(gm, np.concatenate(want[::-1]), 1e-5)
        finite = np.isfinite(acts[-1]).all()
        assert finite == (value < 0)
        assert np.isfinite(tr.training_step(pos, np.zeros((n, 2), np.float32))) == finite
