"""The visit flags of large fused steps come from the batch's positions
(visit_kernel.hpp) and their hash-grid backward adds only what does not
truncate to 0 (hash_scatter_nonzero_kernel): both against what the corners and
the split path (flags stored by the backward) say. Marked gpu."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_parity import make_trainer
from tiny_metal_nn import OptimizerStateBlob

pytestmark = pytest.mark.gpu

PZ = 805459861

# dims, features, log2 table, levels, n: the pass's smallest batch at T = 2^19
# and one point to either side (131071 takes the other route), 1, 2 and 4 ranges
# of 2^20 entries, the smallest table, feature counts without a fused backward
SHAPES = [
    (3, 2, 19, 4, 131071), (3, 2, 19, 4, 131072), (3, 2, 19, 4, 131073), (3, 2, 10, 16, 524289),
    (3, 4, 21, 2, 262144), (3, 1, 15, 5, 262145), (2, 2, 21, 3, 262144), (4, 2, 22, 2, 262147),
    (4, 4, 16, 8, 131072),
]


def _moments(tr, value):
    sec = [np.full(k, value, np.float32) for k in
           (tr.hash_param_count, tr.hash_param_count, tr.mlp_param_count, tr.mlp_param_count)]
    return OptimizerStateBlob(1, 10, b"".join(
        np.array([4 * s.size], "<u4").tobytes() + s.tobytes() for s in sec))


def _m_of(tr):
    blob = tr.export_optimizer_state().payload
    return np.frombuffer(blob, np.float32, tr.hash_param_count, 4)


def _positions(dims, n, rng):
    pos = rng.random((n, dims), dtype=np.float32)
    pos[: n // 4] = pos[: n // 4] * np.float32(0.02) + np.float32(0.4)  # many points a cell
    pos[0] = 0.0
    pos[1] = 1.0
    pos[2] = -0.37
    # x cells ending in 20 one bits at resolution 16: x and x + 1 lie in
    # different ranges of a table above 2^20 entries
    pos[3, 0] = 65535.96875
    pos[4] = 65535.96875
    return pos


@pytest.mark.parametrize("dims,feats,log2t,levels,n", SHAPES)
def test_visited_entries_are_the_corners(dims, feats, log2t, levels, n):
    print(f"visited set {dims}D F{feats} T2^{log2t} L{levels} n{n}", flush=True)
    rng = np.random.default_rng(n + dims)
    pos = _positions(dims, n, rng)
    tgt = rng.random((n, 2), dtype=np.float32)
    enc = dict(n_levels=levels, n_features_per_level=feats, log2_hashmap_size=log2t,
               base_resolution=16.0, per_level_scale=2.0)
    with make_trainer(dims, 2, enc, dict(n_neurons=64, n_hidden_layers=1), loss="L2",
                      precision="fp16", batch=n, hash_range=0.5) as tr:
        want = np.zeros((levels, 1 << log2t), bool)
        for at in range(0, n, 1 << 16):
            _, idx, _ = tr.debug_encode(pos[at:at + (1 << 16)], with_corners=True)
            for lv in range(levels):
                want[lv, idx[:, lv].ravel()] = True
                if dims == 2:
                    want[lv, idx[:, lv].ravel() ^ (PZ & ((1 << log2t) - 1))] = True
        for _ in range(2):  # the second step's flags start from a buffer the first one cleared
            tr.import_optimizer_state(_moments(tr, 1.0))
            tr.training_step(pos, tgt)
            moved = (_m_of(tr) != 1.0).reshape(levels, 1 << log2t, feats).all(axis=2)
            assert np.array_equal(moved, want)


# the last two: level slices above 8 MB, where the split path's backward goes
# level by level
@pytest.mark.parametrize("dims,feats,log2t,levels,n,base", [
    (3, 2, 14, 16, 524288, 16.0), (3, 4, 17, 8, 262149, 16.0), (4, 2, 16, 8, 131073, 16.0),
    (3, 1, 15, 5, 262201, 16.0), (3, 4, 21, 2, 262145, 128.0), (4, 2, 22, 2, 131073, 64.0)])
def test_gradients_match_the_split_path(dims, feats, log2t, levels, n, base):
    """One fused step against forward_for_training, backward_accumulate (which
    stores its flags in the backward) and adam_step: first moments within 16
    fixed-point units times 1 - beta1, as the parity tests allow for an ulp of
    d that moves a truncation, and exact on 99% of the entries."""
    print(f"split parity {dims}D F{feats} T2^{log2t} L{levels} n{n}", flush=True)
    rng = np.random.default_rng(n)
    pos = _positions(dims, n, rng)
    tgt = rng.random((n, 2), dtype=np.float32) * np.float32(200.0)  # large gradients
    enc = dict(n_levels=levels, n_features_per_level=feats, log2_hashmap_size=log2t,
               base_resolution=base, per_level_scale=1.5)
    args = (dims, 2, enc, dict(n_neurons=64, n_hidden_layers=1))
    kw = dict(loss="L2", precision="fp32", batch=n, hash_range=0.5)
    with make_trainer(*args, **kw) as a, make_trainer(*args, **kw) as b:
        a.import_optimizer_state(_moments(a, 0.0))
        b.import_optimizer_state(_moments(b, 0.0))
        a.training_step(pos, tgt)
        out = b.forward_for_training(pos)
        b.zero_gradients()
        b.backward_accumulate(pos, (np.float32(2) * (out - tgt)) * np.float32(1.0 / n))
        b.adam_step()
        ma, mb = _m_of(a), _m_of(b)
        assert np.count_nonzero(mb) > mb.size // 20
        assert np.abs(ma - mb).max() <= 16 * 0.1 / 65536 + 1e-6 * np.abs(mb).max()
        assert np.mean(ma != mb) <= 0.01


def test_trainers_of_different_table_sizes():
    """A trainer whose visit pass takes 128 KB of LDS steps after one with a
    smaller table was created (both launch the same kernel), and the smaller
    one after it."""
    rng = np.random.default_rng(4)
    n = 1 << 18
    pos, tgt = rng.random((n, 3), dtype=np.float32), rng.random((n, 1), dtype=np.float32)
    net = dict(n_neurons=32, n_hidden_layers=1)

    def enc(log2t):
        return dict(n_levels=2, n_features_per_level=2, log2_hashmap_size=log2t,
                    base_resolution=256.0, per_level_scale=2.0)

    print("two table sizes", flush=True)
    with make_trainer(3, 1, enc(20), net, batch=n) as large, \
            make_trainer(3, 1, enc(10), net, batch=n) as small:
        for tr, log2t in ((large, 20), (small, 10), (large, 20)):
            tr.import_optimizer_state(_moments(tr, 1.0))
            tr.training_step(pos, tgt)
            want = np.zeros((2, 1 << log2t), bool)
            _, idx, _ = tr.debug_encode(pos, with_corners=True)
            for lv in range(2):
                want[lv, idx[:, lv].ravel()] = True
            moved = (_m_of(tr) != 1.0).reshape(2, 1 << log2t, 2).all(axis=2)
            assert np.array_equal(moved, want)


def test_a_failed_step_leaves_no_visit_flags():
    """A step that cannot allocate its activations (2^25 points times 8 layers of
    512: 550 GB) fails after its visit pass was enqueued: the error is reported
    once, and the next step moves the moments of its own corners only."""
    torch = pytest.importorskip("torch")
    from tiny_metal_nn._lib import TmnnError
    n, log2t, levels = 1 << 17, 19, 2
    big = 1 << 25
    assert big * 512 * 8 * 4 > torch.cuda.get_device_properties(0).total_memory
    print("failed step with a visit pass", flush=True)
    rng = np.random.default_rng(9)
    enc = dict(n_levels=levels, n_features_per_level=2, log2_hashmap_size=log2t,
               base_resolution=64.0, per_level_scale=2.0)
    with make_trainer(3, 1, enc, dict(n_neurons=512, n_hidden_layers=8), batch=big,
                      hash_range=0.5) as tr:
        tr.import_optimizer_state(_moments(tr, 1.0))
        x = torch.rand(big, 3, device="cuda")
        y = torch.zeros(big, 1, device="cuda")
        torch.cuda.synchronize()
        with pytest.raises(TmnnError, match="out of memory"):
            tr.training_step_device(x.data_ptr(), y.data_ptr(), big)
        assert tr.step() == 10
        del x, y
        pos = rng.random((n, 3), dtype=np.float32) * np.float32(0.25)
        tr.training_step(pos, np.zeros((n, 1), np.float32))
        want = np.zeros((levels, 1 << log2t), bool)
        _, idx, _ = tr.debug_encode(pos, with_corners=True)
        for lv in range(levels):
            want[lv, idx[:, lv].ravel()] = True
        assert 0.01 < want.mean() < 0.9
        moved = (_m_of(tr) != 1.0).reshape(levels, 1 << log2t, 2).all(axis=2)
        assert np.array_equal(moved, want)


@pytest.mark.parametrize("dims,log2t,n", [(3, 19, 131072), (4, 16, 131072)])
def test_steps_enqueued_back_to_back(dims, log2t, n):
    """Steps without a wait between them, an allocation-free one (whose visit
    pass runs on the main stream) among them, over batches in different
    places: weights and moments equal, to the bit, those of a trainer that is
    waited for after every step. Needs a step's pass after the last finish
    kernel cleared the flags, and its finish kernel after its pass."""
    torch = pytest.importorskip("torch")
    print(f"back to back {dims}D T2^{log2t}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(dims)
    batches = []
    for i in range(6):
        x = torch.rand(n, dims, device="cuda", generator=g)
        x[:, 0] = (x[:, 0] + i) / 6
        batches.append((x.contiguous(), torch.rand(n, 2, device="cuda", generator=g)))
    torch.cuda.synchronize()
    enc = dict(n_levels=8, n_features_per_level=2, log2_hashmap_size=log2t, base_resolution=16.0,
               per_level_scale=1.5)
    got = []
    for wait in (True, False):
        with make_trainer(dims, 2, enc, dict(n_neurons=64, n_hidden_layers=2), loss="L2",
                          batch=n, hash_range=0.5) as tr:
            tr.import_optimizer_state(_moments(tr, 1.0))
            for i, (x, y) in enumerate(batches):
                step = tr.training_step_device_noalloc if i == 3 else tr.training_step_device
                step(x.data_ptr(), y.data_ptr(), n)
                if wait:
                    tr.synchronize()
            got.append((*tr.get_weights(), _m_of(tr).copy()))
    for a, b in zip(*got):
        assert np.array_equal(a, b)
