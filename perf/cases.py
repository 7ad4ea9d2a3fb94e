"""Performance cases of the grouped fixed-fan-in (FFI) layer, through its public entry points.

Five kinds of call, each what a program that trains or serves an FFI layer makes:
  "step"    FFITrainStep.step: forward, both backwards and the SR-SGD update on
            preallocated buffers, with the grad of the logits handed in (bf16);
  "bce"     FFITrainStep.step_bce: the same step with the sparse BCE loss and its
            gradient computed from COO labels in the forward (bf16);
  "layer"   GroupFixedFanIn forward, autograd backward and SRSgd.step, as a program
            written for the reference's API runs them (bf16, fp16, and fp32 layers);
  "infer"   ops.group_ffi_mul without gradients (evaluation, serving);
  "rewire"  GroupFixedFanIn.rewire / GroupFixedFanInReal.rewire.
Sizes: B batch rows, D input features, O labels, G labels per group, F fan-in.
Learning rates are those of the mean loss (0.05): the grads here are of the sum
over the batch, so lr is divided by B and repeated passes train stably.
"""
import math

import torch

from haste_amd import ops
from haste_amd.optim_sr import SRSgd
from haste_amd.rewire import GroupFixedFanIn, GroupFixedFanInReal
from haste_amd.step import FFITrainStep

LR, WD = 0.05, 1e-4
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def listed():
    return [
        # a small output layer: four launches of a few microseconds, latency counts
        dict(name="step_4k", kind="step", B=64, D=768, O=4096, G=32, F=32),
        # the headline training step (131,073 labels: a last group of one label)
        dict(name="step_131k", kind="step", B=512, D=768, O=131073, G=64, F=128),
        # a large output space at a smaller fan-in
        dict(name="step_670k", kind="step", B=512, D=768, O=670091, G=64, F=64),
        # a wide penultimate layer after a ReLU, small groups, the largest fan-in
        dict(name="step_wide", kind="step", B=256, D=4096, O=500000, G=32, F=256, relu=True),
        # the largest layer trained on one GPU: 6 GB of logits
        dict(name="step_3m", kind="step", B=1024, D=768, O=3000000, G=128, F=128),
        # the training loop's own step from sparse labels, no logits written
        dict(name="bce_131k", kind="bce", B=512, D=768, O=131073, G=64, F=128, pos=5),
        # the reference's API at the headline size: autograd's [B, O] grad, odd row pitch
        dict(name="layer_bf16", kind="layer", dtype="bf16", B=512, D=768, O=131073, G=64, F=128,
             momentum=0.0),
        # the same API with mixed precision off
        dict(name="layer_f32", kind="layer", dtype="f32", B=256, D=768, O=131073, G=32, F=64,
             momentum=0.0),
        # a small fp16 layer at ragged sizes, with momentum
        dict(name="layer_f16", kind="layer", dtype="f16", B=70, D=1000, O=20011, G=16, F=48,
             momentum=0.9),
        # evaluation of a short last batch: the weights are most of the traffic
        dict(name="infer_bf16", kind="infer", dtype="bf16", B=24, D=768, O=131073, G=64, F=128),
        # prune 15 % per group, regrow unused indices from zero
        dict(name="rewire_670k", kind="rewire", variant="group", B=1, D=768, O=670091, G=64, F=64),
        # the application's variant: prune 15 % of the whole layer, random restart
        dict(name="rewire_app", kind="rewire", variant="app", B=1, D=768, O=131073, G=64, F=128),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same kinds: sizes over their whole range, odd ones among
    them, with no more than half the largest listed case's logits or products."""
    kind = rng.choice(["step", "step", "bce", "layer", "layer", "infer", "rewire"])
    while True:
        c = dict(kind=kind, B=_log(rng, 8, 1024), D=_log(rng, 300, 4096), O=_log(rng, 1000, 1200000),
                 G=rng.choice([16, 32, 64, 128]), F=16 * rng.randint(1, 16))
        if kind in ("step", "bce") and rng.random() < 0.5:
            c["B"] = max(8, c["B"] // 8 * 8)      # training batches are mostly round
        if c["F"] > c["D"] // 2 or c["B"] * c["O"] > 2 ** 28 or c["B"] * c["O"] * c["F"] > 2 ** 35:
            continue
        if kind == "bce":
            c["pos"] = rng.randint(1, 10)
        if kind in ("layer", "infer"):
            c["dtype"] = rng.choice(["bf16", "bf16", "f16", "f32"])
        if kind == "layer":
            c["momentum"] = rng.choice([0.0, 0.9])
        if kind == "rewire":
            c["B"], c["variant"] = 1, rng.choice(["group", "app"])
        return c


# ---------------------------------------------------------------- inputs

def _gen(seed, n):
    return torch.Generator(device="cuda").manual_seed(seed * 16 + n)


def _indices(c, seed):
    """[groups, F] feature indices: distinct within a group for the step kinds; drawn
    with replacement, as the layer's constructor draws them, for the layer kinds."""
    gc, g = -(-c["O"] // c["G"]), _gen(seed, 0)
    if c["kind"] in ("step", "bce"):
        return torch.cat([torch.rand(min(4096, gc - i), c["D"], generator=g, device="cuda")
                          .argsort(1)[:, :c["F"]].to(torch.int32) for i in range(0, gc, 4096)])
    return torch.randint(c["D"], (gc, c["F"]), generator=g, device="cuda", dtype=torch.int32)


def _tensors(c, seed):
    """(x [B, D], W [O, F], bias [O]) of the layer's own initial distributions."""
    dt = DTYPES[c.get("dtype", "bf16")]
    x = torch.randn(c["B"], c["D"], generator=_gen(seed, 1), device="cuda")
    if c.get("relu"):
        x = x.relu_()
    W = torch.rand(c["O"], c["F"], generator=_gen(seed, 2), device="cuda")
    W = W.mul_(2).sub_(1).mul_(1 / math.sqrt(c["F"]))
    bias = torch.randn(c["O"], generator=_gen(seed, 3), device="cuda").mul_(0.1)
    return x.to(dt), W.to(dt), bias.to(dt)


def _positives(c, seed, per_row):
    """COO [nnz, 2] int32 (row, label): per_row per row, labels skewed to the front."""
    u = torch.rand(c["B"] * per_row, generator=_gen(seed, 4), device="cuda", dtype=torch.float64)
    lab = (c["O"] ** u).long().clamp_(1, c["O"]) - 1
    row = torch.arange(c["B"], device="cuda").repeat_interleave(per_row)
    return torch.stack([row, lab], 1).to(torch.int32)


def _dY(c, seed, ld):
    """sigmoid(z) - y in a [B, ld] buffer, z distributed as the initial logits are."""
    dt = DTYPES[c.get("dtype", "bf16")]
    dY = torch.zeros(c["B"], ld, dtype=dt, device="cuda")
    g = _gen(seed, 5)
    for r in range(0, c["B"], 128):
        z = torch.randn(min(128, c["B"] - r), c["O"], generator=g, device="cuda").mul_(0.58)
        dY[r:r + 128, :c["O"]] = z.sigmoid_()
    p = _positives(c, seed, 5).long()
    dY[p[:, 0], p[:, 1]] = -0.5
    return dY


def _layer(c, seed):
    cls = GroupFixedFanInReal if c.get("variant") == "app" else GroupFixedFanIn
    mode = "random" if c.get("variant") == "app" else "zero"
    kw = {} if c.get("variant") == "app" else {"regrow_mode": "unused"}
    layer = cls(c["D"], c["O"], c["F"], dtype=DTYPES[c.get("dtype", "bf16")], device="cuda",
                group_size=c["G"], prune_mode="fraction", rewire_fraction=0.15, init_mode=mode, **kw)
    x, W, bias = _tensors(c, seed)
    with torch.no_grad():
        layer.weights.copy_(W)
        layer.bias.copy_(bias)
    layer.group_locations = _indices(c, seed)
    return layer, x


def prepare(case, seed):
    c = case
    s = {"case": c, "seed": seed}
    if c["kind"] in ("step", "bce"):
        x, W, bias = _tensors(c, seed)
        s["x"] = x
        s["step"] = FFITrainStep(W, bias, _indices(c, seed), c["B"], c["D"], c["G"],
                                 lr=LR / c["B"], weight_decay=WD, seed=42)
        if c["kind"] == "bce":
            s["labels"] = _positives(c, seed, c["pos"])
        else:
            s["dY"] = _dY(c, seed, s["step"].ldo)
    elif c["kind"] == "layer":
        s["layer"], x = _layer(c, seed)
        s["x"] = x.requires_grad_(True)
        s["dY"] = _dY(c, seed, c["O"])
        s["opt"] = SRSgd(s["layer"].parameters(), lr=LR / c["B"], weight_decay=WD,
                         momentum=c["momentum"], seed=42)
    elif c["kind"] == "infer":
        s["x"], s["W"], s["bias"] = _tensors(c, seed)
        s["idx"] = _indices(c, seed)
    else:
        s["layer"], _ = _layer(c, seed)
    return s


# ---------------------------------------------------------------- one pass

def run(s):
    c = s["case"]
    if c["kind"] == "step":
        st = s["step"]
        st.step(s["x"], s["dY"], st.ldo)
        return {"logits": st.logits, "dx": st.dX, "w": st.W, "bias": st.bias}
    if c["kind"] == "bce":
        st = s["step"]
        loss = st.step_bce(s["x"], s["labels"])
        return {"loss": loss, "dy": st.dY_buf[:, :c["O"]], "dx": st.dX, "w": st.W, "bias": st.bias}
    if c["kind"] == "layer":
        layer, x, opt = s["layer"], s["x"], s["opt"]
        opt.zero_grad()
        x.grad = None
        logits = layer(x)
        logits.backward(s["dY"])
        opt.step()
        w, b = layer.weights, layer.bias
        out = {"logits": logits.detach(), "dx": x.grad, "dw": w.grad, "dbias": b.grad,
               "w": w.detach(), "bias": b.detach()}
        if c["momentum"]:
            out["mw"], out["mb"] = opt.state[w]["momentum_buf"], opt.state[b]["momentum_buf"]
        return out
    if c["kind"] == "infer":
        with torch.no_grad():
            return ops.group_ffi_mul(s["x"], s["W"], s["idx"], s["bias"], gsize=c["G"])
    layer = s["layer"]
    layer.rewire(seed=s["seed"])
    return {"w": layer.weights.detach(), "idx": layer.group_locations}


# ---------------------------------------------------------------- what it cannot do without

def work(case):
    c = case
    B, D, O, F = c["B"], c["D"], c["O"], c["F"]
    e = {"bf16": 2, "f16": 2, "f32": 4}[c.get("dtype", "bf16")]
    idx, x, w, b, z = 4 * -(-O // c["G"]) * F, e * B * D, e * O * F, e * O, e * B * O
    if c["kind"] == "step":      # x, dY, W, bias, idx in; logits, dX, W, bias out
        return {"bytes": 2 * x + 2 * z + 2 * w + 2 * b + idx, "flops": 6 * B * O * F}
    if c["kind"] == "bce":       # x, W, bias, idx, labels in; dY, dX, W, bias out
        return {"bytes": 2 * x + z + 2 * w + 2 * b + idx + 8 * B * c["pos"], "flops": 6 * B * O * F}
    if c["kind"] == "layer":     # also dW, dbias out, and the fp32 momenta in and out
        m = 8 * (O * F + O) if c["momentum"] else 0
        return {"bytes": 2 * x + 2 * z + 3 * w + 3 * b + idx + m, "flops": 6 * B * O * F}
    if c["kind"] == "infer":
        return {"bytes": x + z + w + b + idx, "flops": 2 * B * O * F}
    return {"bytes": 2 * w + 2 * idx, "flops": O * F}


# ---------------------------------------------------------------- tolerances

def tolerance(case):
    """Rewire is a contract on bits.  The others are about four times the error seen
    against 64-bit sums (of the norm, largest): 2.4e-3, 7.8e-3 for bf16 results (one unit
    in the last place: stochastic rounding; the weights of a trained fp16 layer are
    rounded so too), 2.1e-4, 4.9e-4 for fp16 logits, and 3.0e-4, 1.7e-3 for fp32
    layers, which multiply fp16-rounded operands."""
    if case["kind"] == "rewire":
        return "exact"
    if case.get("dtype") == "f32":
        return {"rel": 1.2e-3, "max": 7e-3}
    if case.get("dtype") == "f16" and case["kind"] == "infer":
        return {"rel": 1e-3, "max": 2e-3}
    return {"rel": 1e-2, "max": 3.2e-2}


# ---------------------------------------------------------------- 64 bits

def _groups(c, W, idx):
    """Weights as [groups, G, F] in blocks of groups, with their index rows."""
    gc, G, F = idx.shape[0], c["G"], c["F"]
    step = max(1, 2 ** 27 // (max(G, F) * max(c["B"], F)))
    for g0 in range(0, gc, step):
        g1 = min(gc, g0 + step)
        Wg = torch.zeros((g1 - g0) * G, F, dtype=torch.float64, device=W.device)
        rows = W[g0 * G:min(g1 * G, c["O"])]
        Wg[:rows.shape[0]] = rows.double()
        yield g0 * G, min(g1 * G, c["O"]), Wg.view(-1, G, F), idx[g0:g1].long()


def _logits64(c, x, W, bias, idx):
    z = torch.empty(c["B"], c["O"], dtype=torch.float64, device=x.device)
    xT = x.double().t().contiguous()
    for l0, l1, Wg, ig in _groups(c, W, idx):
        z[:, l0:l1] = torch.bmm(Wg, xT[ig]).flatten(0, 1)[:l1 - l0].t()
    return z.add_(bias.double())


def _grads64(c, x, W, idx, dY):
    xd = x.double().t().contiguous()
    dxT = torch.zeros(c["D"], c["B"], dtype=torch.float64, device=x.device)
    dW = torch.empty(c["O"], c["F"], dtype=torch.float64, device=x.device)
    for l0, l1, Wg, ig in _groups(c, W, idx):
        dg = torch.zeros(Wg.shape[0] * c["G"], c["B"], dtype=torch.float64, device=x.device)
        dg[:l1 - l0] = dY[:, l0:l1].t().double()
        dg = dg.view(-1, c["G"], c["B"])
        dxT.index_add_(0, ig.reshape(-1), torch.bmm(Wg.transpose(1, 2).contiguous(), dg).flatten(0, 1))
        dW[l0:l1] = torch.bmm(dg, xd[ig].transpose(1, 2).contiguous()).flatten(0, 1)[:l1 - l0]
    return dxT.t(), dW, dY.double().sum(0)


def _sgd64(c, p, g):
    return p.double() - LR / c["B"] * (g + WD * p.double())


def exact(case, seed):
    """The same results from 64-bit sums, unrounded (stochastic rounding is of these)."""
    c = case
    if c["kind"] == "rewire" or c["B"] * c["O"] > 2 ** 29:
        return None
    x, W, bias = _tensors(c, seed)
    idx = _indices(c, seed)
    z = _logits64(c, x, W, bias, idx)
    if c["kind"] == "infer":
        return z
    if c["kind"] == "bce":
        y = torch.zeros_like(z)
        p = _positives(c, seed, c["pos"]).long()
        y[p[:, 0], p[:, 1]] = 1.0
        loss = (z.clamp(min=0) - y * z + torch.log1p(torch.exp(-z.abs()))).sum()
        dY = torch.sigmoid(z) - y
        del y
    else:
        dY = _dY(c, seed, c["O"])
    dx, dW, db = _grads64(c, x, W, idx, dY)
    w, b = _sgd64(c, W, dW), _sgd64(c, bias, db)
    if c["kind"] == "step":
        return {"logits": z, "dx": dx, "w": w, "bias": b}
    if c["kind"] == "bce":
        return {"loss": loss, "dy": dY, "dx": dx, "w": w, "bias": b}
    out = {"logits": z, "dx": dx, "dw": dW, "dbias": db, "w": w, "bias": b}
    if c["momentum"]:
        out["mw"], out["mb"] = dW + WD * W.double(), db + WD * bias.double()
    return out
