"""Which batches the training passes put in Morton order, at the sizes on
either side of which the rule changes, and what the sorted ones compute,
against the oracle. Marked gpu."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_parity import (GEOMS, _compact_2d, away_from_relu_kinks, make_trainer, omodel,
                             rel_tensor)

pytestmark = pytest.mark.gpu


# the smallest sorted batch of the plans whose separate hash-grid backward
# merges runs of lanes on one entry, for host-pointer and device-pointer steps
@pytest.mark.parametrize("dims,feats,host,n", [
    (3, 1, True, 4097), (3, 1, False, 1025), (2, 1, True, 1025), (2, 1, False, 33),
    (3, 4, True, 33), (3, 4, False, 33), (2, 4, True, 33), (4, 2, True, 8193), (4, 2, False, 8193)])
def test_sorted_steps_do_not_depend_on_the_row_order(dims, feats, host, n):
    """The sort is stable, so a batch and its sorted copy take the same order: the
    same loss and weights to the bit (unsorted, the two would add their weight
    gradients in different orders)."""
    torch = pytest.importorskip("torch")
    print(f"row order {dims}D F{feats} {'host' if host else 'device'} n{n}", flush=True)
    rng = np.random.default_rng(n + feats)
    enc = dict(n_levels=8, n_features_per_level=feats, log2_hashmap_size=14, base_resolution=16.0,
               per_level_scale=1.5)
    pos = rng.random((n, dims), dtype=np.float32)
    tgt = rng.random((n, 3), dtype=np.float32)
    got = []
    for turn in range(2):
        with make_trainer(dims, 3, enc, dict(n_neurons=64, n_hidden_layers=2), batch=n,
                          hash_range=0.5) as tr:
            order = tr.debug_morton_sort(pos)[1] if turn else np.arange(n)
            x, y = pos[order], tgt[order]
            if host:
                loss = tr.training_step(x, y)
            else:
                dx, dy = torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda()
                out = torch.zeros(1, device="cuda")
                torch.cuda.synchronize()
                tr.training_step_device(dx.data_ptr(), dy.data_ptr(), n, out.data_ptr())
                tr.synchronize()
                loss = float(out[0])
            got.append((loss, *tr.get_weights()))
    assert got[0][0] == got[1][0]
    assert np.array_equal(got[0][1], got[1][1]) and np.array_equal(got[0][2], got[1][2])


# above the sizes from which batches of every plan are sorted (2^15 points in
# 2D, 2^17 - 1 else), and of a separate hash-grid backward (3d_f1, 4d_f2)
@pytest.mark.parametrize("name,n", [("2d_f2", 34001), ("3d_f2", 138001), ("3d_f1", 4301),
                                    ("4d_f2", 8701)])
def test_sorted_backward_matches_oracle(oracle, name, n):
    """backward_accumulate over a sorted batch (and forward_for_training, in the
    caller's row order): the fp32 bars of the small batches. Output gradients
    of 2^-7 keep a truncation that an ulp of d moves as rare as there."""
    d, enc, net, m_out = GEOMS[name]
    print(f"sorted backward {name} n{n}", flush=True)
    rng = np.random.default_rng(n)
    with make_trainer(d, m_out, enc, net, hash_range=0.5, batch=n) as tr:
        hw, mw = tr.get_weights()
        pos = away_from_relu_kinks(oracle, tr, hw, mw, rng.random((n, d), dtype=np.float32))
        assert len(pos) > 0.95 * n
        g = rng.normal(0, 2.0 ** -7, (len(pos), m_out)).astype(np.float32)
        ref = oracle.forward(omodel(oracle, tr), hw, mw, pos)
        tol = 1e-5 * (np.abs(ref) + np.sqrt((ref.astype(np.float64) ** 2).mean()))
        assert np.all(np.abs(tr.forward_for_training(pos) - ref) <= tol)
        tr.zero_gradients()
        tr.backward_accumulate(pos, g)
        gh, gm = tr.debug_gradients()
        ogh, ogm, omask, _, _ = oracle.forward_backward(omodel(oracle, tr), hw, mw, pos, d_out=g)
        assert np.array_equal(tr.debug_active_mask(), omask)
        assert rel_tensor(gm, ogm) <= 1e-5
        diff = np.abs(gh.astype(np.int64) - ogh.astype(np.int64))
        assert (diff == 0).mean() > 0.99 and diff.max() <= 16, int(diff.max())


@pytest.mark.parametrize("dims", [2, 3, 4])
def test_one_block_sort(oracle, dims):
    """Batches up to 8192 points are sorted by one kernel: codes and a stable
    order at the sizes around its waves' and instances' shares, with repeated
    points, points outside the domain and (4D, whose codes repeat) long ties."""
    rng = np.random.default_rng(dims)
    enc = dict(n_levels=2, n_features_per_level=2, log2_hashmap_size=10, base_resolution=4.0,
               per_level_scale=2.0)
    with make_trainer(dims, 1, enc, dict(n_neurons=32, n_hidden_layers=1), batch=8193) as tr:
        for n in (2, 63, 65, 256, 257, 511, 1023, 1024, 1025, 2047, 2048, 2049, 4095, 4096, 4097, 6000, 8191, 8192, 8193):
            print(f"one-block sort {dims}D n{n}", flush=True)
            pos = rng.random((n, dims), dtype=np.float32) * np.float32(2.4) - np.float32(1.2)
            pos[n // 2:] = pos[rng.integers(0, n - n // 2, n - n // 2)]
            codes, perm = tr.debug_morton_sort(pos)
            want = oracle.morton_codes(pos, dims)
            assert np.array_equal(codes, _compact_2d(want) if dims == 2 else want)
            assert np.array_equal(perm, np.argsort(codes, kind="stable"))
