"""The work that a user of this framework has it do, as cases that can be
measured: training steps, inference, Jacobians and split (accumulated)
training over neural fields of 2 to 4 dimensions, each through the public
`tiny_metal_nn.Trainer`, from calls of a few thousand points on host arrays
to batches of 2^20 points on device memory.

A field is resumed rather than new: its table, MLP and Adam moments come from
the seed with the magnitudes that a training run leaves behind, and a training
state holds a few batches that its steps take in turn. `exact` restates the
same math in 64-bit torch: cells are chosen in the path's own 32-bit
arithmetic (which corner a point takes is a definition, not a rounding), and
the hash gradients keep the path's fixed point (a contribution times 65536,
truncated).
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "tiny-metal-nn_amd"))

from tiny_metal_nn import OptimizerStateBlob, Trainer  # noqa: E402

DEVICE = "cuda:0"
STEP = 100  # steps already taken by a resumed field
POOL = 3  # batches of a training or inference state, taken in turn
LR, BETA1, BETA2, EPS = 1e-2, 0.9, 0.99, 1e-15


def _case(name, do, host, dims, levels, features, log2_table, base, scale, width, layers,
          outputs, precision, loss, n):
    return {"name": name, "do": do, "host": host, "dims": dims, "levels": levels,
            "features": features, "log2_table": log2_table, "base": base, "scale": scale,
            "width": width, "layers": layers, "outputs": outputs, "precision": precision,
            "loss": loss, "n": n}


def listed():
    return [
        # a viewer or a collision query: one small evaluation on host arrays
        # (the default encoding, 64-wide, T = 2^19, 4096 points)
        _case("query_4096", "infer", True, 3, 16, 2, 19, 16.0, 1.447, 64, 2, 1, "fp32", "L2", 4096),
        # surface normals of the same field: outputs and Jacobian
        _case("normals_4096", "jacobian", True, 3, 16, 2, 19, 16.0, 1.447, 64, 2, 1, "fp32", "L2",
              4096),
        # the small signed-distance example: a 16-wide MLP, host arrays, 4096
        # points a step, the loss read back on every step
        _case("sphere_step", "step", True, 3, 4, 2, 14, 16.0, 1.5, 16, 1, 1, "fp32", "L2", 4096),
        # a caller with its own loss: forward, gradient of the outputs handed
        # back, Adam; host arrays, a ragged batch
        _case("own_loss", "accumulate", True, 3, 16, 2, 19, 16.0, 1.447, 64, 2, 3, "fp32", "L2",
              30011),
        # one 256 x 256 tile of a fitted image
        _case("image_infer", "infer", False, 2, 16, 2, 15, 16.0, 1.5, 64, 2, 3, "fp32", "L2",
              1 << 16),
        # image fitting, the flagship step
        _case("image_step", "step", False, 2, 16, 2, 15, 16.0, 1.5, 64, 2, 3, "fp16", "RelativeL2",
              1 << 18),
        # the same field trained in 32 bits (the default precision), ragged
        _case("image_step_fp32", "step", False, 2, 16, 2, 15, 16.0, 1.5, 64, 2, 3, "fp32",
              "RelativeL2", 199999),
        # a radiance-like 3D field: training, and a ragged full-frame query
        _case("nerf_step", "step", False, 3, 16, 2, 19, 16.0, 1.381913, 64, 1, 16, "fp16", "L2",
              1 << 20),
        _case("nerf_infer", "infer", False, 3, 16, 2, 19, 16.0, 1.381913, 64, 1, 16, "fp32", "L2",
              1000003),
        # a large signed-distance field: four features a level, 2^21 entries
        _case("sdf_step", "step", False, 3, 16, 4, 21, 16.0, 1.5, 64, 3, 1, "fp16", "L1", 1 << 19),
        # a space-time field with a 128-wide MLP, the largest step
        _case("dynamic_step", "step", False, 4, 16, 2, 22, 8.0, 1.4, 128, 4, 4, "fp16", "L2",
              1 << 20),
        # an MLP wider than the fused kernels hold
        _case("wide_step", "step", False, 3, 8, 2, 14, 8.0, 2.0, 256, 2, 4, "fp32", "L2", 1 << 16),
    ]


def draw(rng):
    do = rng.choice(["step"] * 5 + ["infer"] * 3 + ["jacobian", "accumulate"])
    levels, features = rng.choice([(4, 2), (8, 2), (16, 2), (16, 2), (16, 2), (8, 4), (16, 4)])
    width = rng.choice([16, 32, 64, 64, 64, 128, 256])
    top = 15 if do == "jacobian" else 17 if width >= 128 else 19
    n = int(round(2.0 ** rng.uniform(10, top)))
    case = _case(None, do, do in ("jacobian", "accumulate") or n < 8192, rng.choice([2, 3, 3, 4]),
                 levels, features, rng.randint(14, 19), rng.choice([8.0, 16.0]),
                 rng.choice([1.381913, 1.4, 1.447, 1.5, 2.0]) if levels <= 8 else
                 rng.choice([1.381913, 1.4, 1.447, 1.5]),
                 width, rng.randint(1, 4), rng.choice([1, 3, 4, 16]),
                 rng.choice(["fp16", "fp32"]) if do in ("step", "accumulate") else "fp32",
                 rng.choice(["L2", "L1", "RelativeL2"]) if do == "step" else "L2", n)
    del case["name"]
    return case


# ---- inputs ------------------------------------------------------------------


def _counts(case):
    table = case["levels"] << case["log2_table"]
    sizes = [case["levels"] * case["features"]] + [case["width"]] * case["layers"] + [case["outputs"]]
    return table * case["features"], sum((a + 1) * b for a, b in zip(sizes, sizes[1:])), sizes


def _config(case):
    return {"encoding": {"n_levels": case["levels"], "n_features_per_level": case["features"],
                         "log2_hashmap_size": case["log2_table"], "base_resolution": case["base"],
                         "per_level_scale": case["scale"]},
            "network": {"n_neurons": case["width"], "n_hidden_layers": case["layers"]},
            "loss": {"otype": case["loss"]},
            "optimizer": {"otype": "Adam", "learning_rate": LR, "beta1": BETA1, "beta2": BETA2,
                          "epsilon": EPS},
            "batch_size": case["n"], "mi355x": {"precision": case["precision"]}}


def _inputs(case, seed):
    """The field's weights and moments [table | MLP] and the pool of batches,
    32-bit, on the GPU: all from the seed."""
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    n, d, m = case["n"], case["dims"], case["outputs"]
    nh, nm, sizes = _counts(case)

    def uniform(*shape):
        return torch.rand(*shape, device=DEVICE, generator=g)

    def normal(*shape):
        return torch.randn(*shape, device=DEVICE, generator=g)

    weights = torch.empty(nh + nm, device=DEVICE)
    torch.randn(nh, device=DEVICE, generator=g, out=weights[:nh])
    weights[:nh] *= 0.1  # a trained table; MLP uniform in its fan-in, with biases
    at = nh
    for a, b in zip(sizes, sizes[1:]):
        weights[at:at + a * b] = (uniform(a * b) * 2 - 1) * math.sqrt(6.0 / a)
        weights[at + a * b:at + a * b + b] = (uniform(b) * 2 - 1) * 0.1
        at += a * b + b
    moments = None
    if case["do"] in ("step", "accumulate"):
        moments = [torch.empty(nh + nm, device=DEVICE) for _ in range(2)]
        for lo, hi, s in ((0, nh, 3e-5), (nh, nh + nm, 1e-3)):
            torch.randn(hi - lo, device=DEVICE, generator=g, out=moments[0][lo:hi])
            moments[0][lo:hi] *= s
            torch.rand(hi - lo, device=DEVICE, generator=g, out=moments[1][lo:hi])
            moments[1][lo:hi].add_(0.5).mul_((3 * s) ** 2)
    freq, phase = torch.rand(m, 4, d, device=DEVICE, generator=g) * 8 - 4, uniform(m, 4) * 6.2831853
    centre, radius = 0.25 + 0.5 * uniform(8, 3), 0.05 + 0.2 * uniform(8)
    pool = []
    for _ in range(POOL):
        x = uniform(n, d)
        if d == 3:  # half of a 3D batch lies near surfaces
            k = torch.randint(0, 8, (n // 2,), device=DEVICE, generator=g)
            way = torch.nn.functional.normalize(normal(n // 2, 3), dim=1)
            x[:n // 2] = centre[k] + way * (radius[k] + 0.02 * uniform(n // 2) - 0.01)[:, None]
            x.clamp_(0.0, 0.999999)
        y = torch.zeros(n, m, device=DEVICE)
        for j in range(4):
            y += 0.5 + 0.5 * torch.sin(2 * math.pi * (x @ freq[:, j].T) + phase[:, j])
        y /= 4
        if case["do"] == "accumulate":  # the caller's d loss / d output
            y = (normal(n, m) * 2 / n).contiguous()
        pool.append((x.contiguous(), y))
    return weights, moments, pool


class _View:
    """A trainer's device buffer as torch sees it. A tensor made from it holds
    it, and it holds the trainer, whose end would free the buffer."""

    def __init__(self, trainer, role):
        buffer = trainer.runtime_buffer(role)
        self.trainer = trainer
        self.__cuda_array_interface__ = {"shape": (buffer["bytes"] // 4,), "typestr": "<f4",
                                         "data": (buffer["device_ptr"], False), "version": 2}


class State:
    def __init__(self, case, seed):
        weights, moments, pool = _inputs(case, seed)
        nh = _counts(case)[0]
        self.case, self.at = case, 0
        self.trainer = Trainer.from_config(_config(case), n_input=case["dims"],
                                           n_output=case["outputs"])
        host = weights.cpu().numpy()
        self.trainer.set_initial_weights(host[:nh], host[nh:])
        if moments is not None:
            sections = [q[a:b] for a, b in ((0, nh), (nh, None)) for q in moments]
            total = sum(4 + 4 * q.numel() for q in sections)
            payload, to = np.empty(total, np.uint8), 0
            for q in sections:  # [u32 bytes][fp32], m and v of the table, then of the MLP
                payload[to:to + 4] = np.array([4 * q.numel()], "<u4").view(np.uint8)
                torch.from_numpy(payload[to + 4:to + 4 + 4 * q.numel()].view(np.float32)).copy_(q)
                to += 4 + 4 * q.numel()
            self.trainer.import_optimizer_state(OptimizerStateBlob(1, STEP, payload))
            self.field = {key: torch.as_tensor(_View(self.trainer, role), device=DEVICE)
                          for key, role in (("weights", "FusedWeights"), ("m", "FusedFirstMoment"),
                                            ("v", "FusedSecondMoment"))}
        self.pool = [tuple(t.cpu().numpy() for t in b) for b in pool] if case["host"] else pool
        self.loss = torch.zeros(1, device=DEVICE)
        self.out = torch.empty(case["n"], case["outputs"], device=DEVICE)
        torch.cuda.synchronize()  # device calls read inputs that are complete

    def batch(self):
        self.at += 1
        return self.pool[(self.at - 1) % len(self.pool)]


def prepare(case, seed):
    return State(case, seed)


def run(state):
    case, trainer, n = state.case, state.trainer, state.case["n"]
    x, y = state.batch()
    if case["do"] == "infer":
        if case["host"]:
            return trainer.inference(x)
        trainer.inference_device(x.data_ptr(), state.out.data_ptr(), n)
        return state.out
    if case["do"] == "jacobian":
        return trainer.evaluate_with_gradient(x)
    if case["do"] == "accumulate":
        trainer.zero_gradients()
        out = trainer.forward_for_training(x)
        trainer.backward_accumulate(x, y)
        trainer.adam_step()
        return {"out": out, **state.field}
    if case["host"]:
        return {"loss": trainer.training_step(x, y), **state.field}
    trainer.training_step_device(x.data_ptr(), y.data_ptr(), n, state.loss.data_ptr())
    return {"loss": state.loss, **state.field}


# ---- what a pass cannot do without --------------------------------------------


def work(case):
    n, d, corners = case["n"], case["dims"], 1 << case["dims"]
    nh, nm, sizes = _counts(case)
    table = 1 << case["log2_table"]
    touched = 0  # table floats that a batch can reach
    for r in _resolutions(case):
        touched += int(min(n * corners, table, (r + 1) ** d)) * case["features"]
    mlp = 2 * n * sum(a * b for a, b in zip(sizes, sizes[1:]))
    encode = 2 * n * corners * nh // table
    if case["do"] == "infer":
        return {"bytes": 4 * (n * (d + case["outputs"]) + touched + nm), "flops": mlp + encode}
    if case["do"] == "jacobian":
        return {"bytes": 4 * (n * (d + case["outputs"] * (1 + d)) + touched + nm),
                "flops": mlp * (1 + case["outputs"]) + encode * (1 + d * case["outputs"])}
    # weights and both moments read and written, targets (or output gradients)
    # read, and where the split calls return the outputs, those written
    rows = d + case["outputs"] * (2 if case["do"] == "accumulate" else 1)
    return {"bytes": 4 * n * rows + 24 * (touched + nm), "flops": 3 * mlp + 2 * encode}


def tolerance(case):
    # Measured against `exact` over the listed cases and six drawn ones: outputs
    # 1.4e-7 to 3.5e-7, Jacobians 1.8e-7 to 2.1e-7, moments and weights after a
    # 32-bit step up to 1.2e-5 and after a 16-bit one up to 2.1e-4. The largest
    # single difference is wider where a rounding can decide: a contribution
    # that truncates to the next 2^-16, or a unit at its ReLU kink (which also
    # moves a Jacobian row by that unit's whole part).
    if case["do"] == "infer":
        return {"rel": 2e-6, "max": 1e-4}
    if case["do"] == "jacobian":
        return {"rel": 1e-3, "max": 0.5}
    return {"rel": 1e-4 if case["precision"] == "fp32" else 1e-3, "max": 0.3}


# ---- the same in 64 bits --------------------------------------------------------


def _resolutions(case):
    r, s = np.float32("%.6f" % case["base"]), np.float32("%.6f" % case["scale"])
    out = []
    for _ in range(case["levels"]):
        out.append(float(r))
        r = np.float32(r * s)
    return out


def _cells(case, x, r):
    """Per corner of x's cells at resolution r: table entries, weights, and the
    weights' derivatives along each axis of the cell."""
    d, primes = case["dims"], (1, 2654435761, 805459861, 56711039)
    s = x * torch.tensor(r, dtype=torch.float32, device=x.device)
    low = torch.floor(s)
    frac, low = (s - low).double(), low.to(torch.int64)
    mask = (1 << case["log2_table"]) - 1
    for k in range(1 << d):
        entry = torch.zeros_like(low[:, 0])
        w, slopes = torch.ones_like(frac[:, 0]), []
        for a in range(d):
            bit = k >> a & 1
            entry ^= (low[:, a] + bit) * primes[a]
            w = w * (frac[:, a] if bit else 1 - frac[:, a])
        for b in range(d):
            s = torch.ones_like(w)
            for a in range(d):
                bit = k >> a & 1
                s = s * ((1.0 if bit else -1.0) if a == b else frac[:, a] if bit else 1 - frac[:, a])
            slopes.append(s)
        yield entry & mask, w, slopes


def _layers(case, weights):
    sizes, at, out = _counts(case)[2], _counts(case)[0], []
    for a, b in zip(sizes, sizes[1:]):
        out.append((weights[at:at + a * b].view(a, b), weights[at + a * b:at + a * b + b], at))
        at += a * b + b
    return out


def _forward(case, table, layers, x):
    feats = []
    for level, r in enumerate(_resolutions(case)):
        feats.append(sum(table[level][entry] * w[:, None] for entry, w, _ in _cells(case, x, r)))
    acts = [torch.cat(feats, 1)]
    for i, (w, b, _) in enumerate(layers):
        h = acts[-1] @ w + b
        acts.append(h.relu() if i + 1 < len(layers) else h)
    return acts


def _loss(case, out, y):
    r = out - y
    if case["loss"] == "L1":
        return r.abs().sum(), r.sign()
    if case["loss"] == "RelativeL2":
        den = out * out + 0.01
        return (r * r / den).sum(), 2 * r / den
    return (r * r).sum(), 2 * r


def exact(case, seed):
    weights, moments, pool = _inputs(case, seed)
    x, y = pool[0]
    del pool
    n, d, m, feats = case["n"], case["dims"], case["outputs"], case["features"]
    nh = _counts(case)[0]
    w64 = weights.double()
    table = w64[:nh].view(case["levels"], -1, feats)
    layers = _layers(case, w64)
    train = case["do"] in ("step", "accumulate")
    outs, jacs, loss = [], [], 0.0
    grad = torch.zeros_like(w64) if train else None
    seen = torch.zeros(table.shape[:2], dtype=torch.bool, device=DEVICE) if train else None
    for at in range(0, n, 1 << 16):
        xs, ys = x[at:at + (1 << 16)], y[at:at + (1 << 16)].double()
        acts = _forward(case, table, layers, xs)
        outs.append(acts[-1])
        if case["do"] == "infer":
            continue
        if case["do"] == "jacobian":
            jac = torch.zeros(xs.shape[0], m, d, dtype=torch.float64, device=DEVICE)
            for o in range(m):
                g = torch.zeros_like(acts[-1])
                g[:, o] = 1
                for i in range(len(layers) - 1, -1, -1):
                    g = g @ layers[i][0].T
                    if i:
                        g = g * (acts[i] > 0)
                for level, r in enumerate(_resolutions(case)):
                    gl = g[:, level * feats:(level + 1) * feats]
                    for entry, _, slopes in _cells(case, xs, r):
                        q = (table[level][entry] * gl).sum(1)
                        for a in range(d):
                            jac[:, o, a] += q * slopes[a] * r
            jacs.append(jac)
            continue
        if case["do"] == "accumulate":
            g = ys
        else:
            part, g = _loss(case, acts[-1], ys)
            loss, g = loss + part, g / n
        for i in range(len(layers) - 1, -1, -1):
            w, b, to = layers[i]
            grad[to:to + w.numel()] += (acts[i].T @ g).reshape(-1)
            grad[to + w.numel():to + w.numel() + b.numel()] += g.sum(0)
            g = g @ w.T
            if i:
                g = g * (acts[i] > 0)
        table_grad = grad[:nh].view_as(table)
        for level, r in enumerate(_resolutions(case)):
            gl = g[:, level * feats:(level + 1) * feats]
            for entry, w, _ in _cells(case, xs, r):
                table_grad[level].index_add_(0, entry, torch.trunc(gl * w[:, None] * 65536) / 65536)
                seen[level][entry] = True
                if d == 2:  # a 2D point is (x, y, 0): the plane above counts as visited
                    seen[level][entry ^ (805459861 & ((1 << case["log2_table"]) - 1))] = True
    out = torch.cat(outs)
    if case["do"] == "infer":
        return out
    if case["do"] == "jacobian":
        return out, torch.cat(jacs)
    m1, m2 = (q.double() for q in moments)
    m1 = BETA1 * m1 + (1 - BETA1) * grad
    m2 = BETA2 * m2 + (1 - BETA2) * grad * grad
    t = STEP + 1
    new = w64 - LR * (m1 / (1 - BETA1 ** t)) / ((m2 / (1 - BETA2 ** t)).sqrt() + EPS)
    got = {"weights": new, "m": m1, "v": m2}
    kept = seen.view(-1, 1).expand(-1, feats).reshape(-1)  # Adam moves the visited entries only
    for key, old in (("weights", weights), ("m", moments[0]), ("v", moments[1])):
        got[key][:nh] = torch.where(kept, got[key][:nh], old[:nh].double())
    if case["do"] == "accumulate":
        return {"out": out, **got}
    return {"loss": (loss / n).reshape(1) if not case["host"] else float(loss / n), **got}
