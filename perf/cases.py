"""The work a user of this framework has it do, as cases that can be timed and compared.

Five kinds of work, each through public entry points:

  "infer"    Network.forward / Network.predict on host images: serving one request, scoring a test set;
  "layer"    layer.compute_activation + layer.train_step on host arrays: a caller with a training loop of its own;
  "fit"      Network.fit on a data set in host memory: the example script's flow, hidden layer then classifier;
  "epoch"    one epoch of the backend object (train_epoch) on a data set that is resident on the GPU;
  "step"     one training step of a layer through the C entry points on device buffers (forward pass, traces,
             weights, bias, mask; in double precision with rewiring);
  "rewire"   the mask rewiring of one hypercolumn (sb_update_mask) on device buffers.

Sizes are those of the example script's presets (784 and 27648 inputs, 15 x 200 hidden units), of bench.py's
workloads (1568 -> 30 x 100, 1568 -> 100 x 100 in double precision, 55296 -> 200 x 100) and of the tests, with odd
ones among them.  Single-precision epochs are first epochs, which do not rewire: over a trajectory the rewired
mask of single precision depends on the order of sums (near-ties of scores), so rewiring is compared in double
precision and, on equal inputs, by itself.
"""
import ctypes
import math

import numpy as np
import torch

from streambrain_amd import _capi

# hyper-parameters of the example script's MNIST preset
TAUPDT, PMIN, KHALF, TAUBDT = 0.006908854922437549, 0.06195283356566607, -139.02586632856327, 0.02218100432360414
CLASSIFIER_TAUPDT = 0.0007449780036161324
CLASSES = 10


def listed():
    return [
        # serving: class probabilities of one image from the example script's network
        {"name": "infer_one", "kind": "infer", "what": "forward", "dtype": "f32", "inputs": 784, "hyper": 15,
         "mini": 200, "density": 0.1, "batch": 1, "samples": 1},
        # scoring the test set: 10000 images, as the example script does after training
        {"name": "infer_test_set", "kind": "infer", "what": "predict", "dtype": "f32", "inputs": 784, "hyper": 15,
         "mini": 200, "density": 0.1, "batch": 128, "samples": 10000},
        # the smallest training calls: a small layer of the tests, driven batch by batch from Python
        {"name": "layer_small", "kind": "layer", "dtype": "f64", "inputs": 100, "hyper": 4, "mini": 12,
         "density": 0.3, "batch": 32, "samples": 250},
        # the example script's flow on a part of its data: an epoch of the hidden layer, two of the classifier
        {"name": "fit_script", "kind": "fit", "dtype": "f32", "inputs": 784, "hyper": 15, "mini": 200,
         "density": 0.1, "batch": 128, "samples": 20000, "classifier_epochs": 2},
        # bench.py's headline layer, one epoch
        {"name": "epoch_headline", "kind": "epoch", "dtype": "f32", "inputs": 1568, "hyper": 30, "mini": 100,
         "density": 0.1, "batch": 128, "samples": 60000, "epoch": 0},
        # the example script in double precision, an epoch with rewiring, ragged last batch
        {"name": "epoch_double", "kind": "epoch", "dtype": "f64", "inputs": 784, "hyper": 15, "mini": 200,
         "density": 0.1, "batch": 128, "samples": 10000, "epoch": 1},
        # odd sizes: no row is a whole number of vectors, no batch a whole number of blocks, every connection present
        {"name": "epoch_odd", "kind": "epoch", "dtype": "f32", "inputs": 1003, "hyper": 13, "mini": 67,
         "density": 1.0, "batch": 100, "samples": 5030, "epoch": 0},
        # the headline layer without a mask, step by step on device buffers
        {"name": "step_dense", "kind": "step", "dtype": "f32", "inputs": 1568, "hyper": 30, "mini": 100,
         "density": 1.0, "batch": 128},
        # the example script's STL-10 layer
        {"name": "step_stl10", "kind": "step", "dtype": "f32", "inputs": 27648, "hyper": 15, "mini": 200,
         "density": 0.57, "batch": 128},
        # bench.py's double-precision layer, rewiring step
        {"name": "step_wide_double", "kind": "step", "dtype": "f64", "inputs": 1568, "hyper": 100, "mini": 100,
         "density": 0.1, "batch": 512},
        # the largest layer that is compared: bench.py's STL-10 shape
        {"name": "step_largest", "kind": "step", "dtype": "f32", "inputs": 55296, "hyper": 200, "mini": 100,
         "density": 0.05, "batch": 256},
        # rewiring one hypercolumn of the example script's STL-10 layer
        {"name": "rewire_stl10", "kind": "rewire", "dtype": "f32", "inputs": 27648, "hyper": 15, "mini": 200,
         "density": 0.57},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _shape(rng, max_synapses, dtype):
    """A layer of the ranges above with at most max_synapses connections."""
    while True:
        n = _log_int(rng, 96, 55296)
        mini = rng.choice([10, 12, 50, 64, 67, 100, 100, 101, 128, 200, 200])
        hyper = _log_int(rng, 3, 200)
        if 8 * hyper * mini * n > max_synapses // 64 and hyper * mini * n <= max_synapses and hyper * mini > 32:
            return {"dtype": dtype, "inputs": n, "hyper": hyper, "mini": mini,
                    "density": round(rng.choice([0.05, 0.1, 0.1, 0.3, 0.57, 1.0]), 2)}


def draw(rng):
    kind = rng.choice(["infer", "layer", "fit", "epoch", "epoch", "step", "step", "step", "rewire"])
    dtype = rng.choice(["f32", "f32", "f64"])
    if kind == "infer":
        samples = _log_int(rng, 1, 10000)
        return {"kind": kind, "what": rng.choice(["forward", "predict"]), **_shape(rng, 8_000_000, dtype),
                "inputs": _log_int(rng, 100, 3000), "hyper": _log_int(rng, 4, 30),
                "batch": min(samples, rng.choice([1, 32, 100, 128, 512])) if samples <= 512 else rng.choice([100, 128, 512]),
                "samples": samples}
    if kind == "layer":
        batch = _log_int(rng, 8, 200)
        return {"kind": kind, **_shape(rng, 1_000_000, dtype), "batch": batch, "samples": rng.randint(2 * batch, 10 * batch)}
    if kind == "fit":
        return {"kind": kind, **_shape(rng, 3_000_000, dtype), "inputs": rng.choice([784, 1568, 1003]),
                "hyper": _log_int(rng, 4, 15), "batch": rng.choice([64, 100, 128, 256]),
                "samples": _log_int(rng, 4000, 20000), "classifier_epochs": rng.choice([1, 2])}
    if kind == "epoch":
        return {"kind": kind, **_shape(rng, 8_000_000, dtype), "inputs": _log_int(rng, 100, 2000),
                "hyper": _log_int(rng, 4, 30), "batch": rng.choice([32, 64, 100, 128, 256]),
                "samples": _log_int(rng, 2000, 20000), "epoch": 1 if dtype == "f64" else 0}
    if kind == "step":
        return {"kind": kind, **_shape(rng, 1_000_000_000 if dtype == "f32" else 60_000_000, dtype),
                "batch": rng.choice([32, 77, 100, 128, 128, 256, 300])}
    return {"kind": kind, **_shape(rng, 400_000_000, dtype)}


# ------------------------------------------------------------------------------------------------- inputs
def _np_type(case):
    return np.float32 if case["dtype"] == "f32" else np.float64


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


STYLES = 200  # distinct kinds of image, 20 of each class (style % 10)


def _styles(g, n):
    """Prototypes of the styles and the mean input of each: a fifth to a half of the pixels on, some never.  An even
    number of inputs beyond 1000 is coded as (x, 1 - x), pixels first, as bench.py does."""
    pixels = n // 2 if n % 2 == 0 and n > 1000 else n
    dark = 0.02 if n > 20000 else 0.6  # photographs have no background
    proto = torch.rand(STYLES, pixels, generator=g, device="cuda")
    proto = proto * (proto > dark) * (torch.rand(pixels, generator=g, device="cuda") < 0.9)
    mean = 0.6 * proto
    return proto, torch.cat([mean, 1 - mean], 1) if pixels < n else mean


def _data(g, proto, rows, n, dtype):
    """Images (a prototype of a random style, each pixel dimmed or dropped at random) and their one-hot classes."""
    style = torch.randint(0, STYLES, (rows,), generator=g, device="cuda")
    px = torch.rand(rows, proto.shape[1], generator=g, device="cuda").mul_(0.5).add_(0.5).mul_(proto[style])
    px *= torch.rand(rows, proto.shape[1], generator=g, device="cuda") < 0.8
    x = torch.cat([px, 1 - px], 1) if proto.shape[1] < n else px
    return x.to(dtype).contiguous(), torch.nn.functional.one_hot(style % CLASSES, CLASSES).to(dtype)


def _traces(g, mean, of_unit, cj, t, learned=0.97):
    """Ci, Cj, Cij of a layer in the middle of its training: unit j has specialised on inputs like mean[of_unit[j]]."""
    ci = mean.mean(0)
    jitter = torch.rand(mean.shape[1], of_unit.shape[0], generator=g, device="cuda").mul_(0.2).add_(0.9)
    cij = jitter.mul_((learned * mean + (1 - learned) * ci).t()[:, of_unit]).mul_(cj)
    return ci.to(t), cj.to(t), cij.to(t)


def _weights(ci, cj, cij, cthr):
    w = (cij.clamp(min=cthr ** 4) / ci.clamp(min=cthr)[:, None]).div_(cj.clamp(min=cthr)).log_()
    w[ci < cthr] = 0
    return w


def _hidden_traces(g, mean, hyper, mini, t):
    """Column c of every hypercolumn stands for style c."""
    cj = torch.rand(hyper * mini, generator=g, device="cuda").add_(0.5).div_(mini)
    return _traces(g, mean, torch.arange(hyper * mini, device="cuda") % mini % STYLES, cj, t)


def _network(case, seed, g, mean, t):
    """The example script's network, a structural-plasticity layer and a dense layer of 10, in mid-training."""
    from streambrain_amd.backend import hip_backend
    np.random.seed(seed % (1 << 31))
    dtype, mini, hidden = _np_type(case), case["mini"], case["hyper"] * case["mini"]
    scale = math.sqrt(case["batch"] / 128)
    net = hip_backend.Network(dtype)
    layers = [hip_backend.StructuralPlasticityLayer(case["inputs"], case["hyper"], mini, TAUPDT * scale, KHALF, PMIN,
                                                    TAUBDT, case["density"], 16, (1, 1 / mini, 1 / mini), dtype),
              hip_backend.DenseLayer(hidden, 1, CLASSES, CLASSIFIER_TAUPDT * scale,
                                     (1 / mini, 1 / CLASSES, 1 / mini / CLASSES), dtype)]
    active = torch.nn.functional.one_hot(torch.arange(hidden, device="cuda") % mini % CLASSES, CLASSES).t() / mini * CLASSES
    cj = torch.full((CLASSES,), 1 / CLASSES, device="cuda")
    for layer, (ci, cj, cij) in ((layers[0], _hidden_traces(g, mean, case["hyper"], mini, t)),
                                 (layers[1], _traces(g, active, torch.arange(CLASSES, device="cuda"), cj, t, 0.1))):
        w = _weights(ci, cj, cij, layer.taupdt / 2).cpu().numpy()
        if layer is layers[0]:
            w *= np.repeat(layer.wmask, mini, axis=1)
        layer.Ci, layer.Cj, layer.Cij, layer.weights = ci.cpu().numpy(), cj.cpu().numpy(), cij.cpu().numpy(), w
        layer.bias = cj.log().cpu().numpy()
        net.add_layer(layer)
    return net, layers


def _device_state(case, seed):
    """A layer in the middle of its training as device buffers, its weights formed from the traces under the mask."""
    g = _generator(seed)
    t = torch.float32 if case["dtype"] == "f32" else torch.float64
    n, hyper, mini = case["inputs"], case["hyper"], case["mini"]
    m = hyper * mini
    s = {"case": case}
    s["wmask"] = (torch.rand(n, hyper, generator=g, device="cuda") < case["density"]).to(torch.uint8)
    proto, mean = _styles(g, n)
    s["Ci"], s["Cj"], s["Cij"] = _hidden_traces(g, mean, hyper, mini, t)
    s["kbi"] = 0.5 + torch.rand(m, generator=g, device="cuda").to(t)
    s["bias"] = s["kbi"] * s["Cj"].log()
    s["W"] = _weights(s["Ci"], s["Cj"], s["Cij"], TAUPDT / 2)
    s["W"].view(n, hyper, mini).mul_(s["wmask"][:, :, None])
    return s, g, proto, t


def _step_state(case, seed):
    """_device_state and a batch of images."""
    s, g, proto, t = _device_state(case, seed)
    s["x"], _ = _data(g, proto, case["batch"], case["inputs"], t)
    return s


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("infer", "layer", "fit", "epoch"):
        g, t = _generator(seed), torch.float32 if case["dtype"] == "f32" else torch.float64
        proto, mean = _styles(g, case["inputs"])
        net, layers = _network(case, seed, g, mean, t)
        x, y = (a.cpu().numpy() for a in _data(g, proto, case["samples"], case["inputs"], t))
        s = {"case": case, "net": net, "layers": layers, "seed": seed % (1 << 31)}
        if kind == "layer":
            b = case["batch"]
            return {**s, "x": [x[k:k + b] for k in range(0, case["samples"], b)]}
        if kind != "epoch":
            return {**s, "x": x, "y": y}
        net.net.initiate_training(x, y)
        rng = np.random.default_rng(seed)
        return {**s, "perm": rng.permutation(case["samples"]), "hc_perm": rng.permutation(case["hyper"])}
    _capi.init()
    if kind == "rewire":
        return _device_state(case, seed)[0]
    n, hyper, mini, b = case["inputs"], case["hyper"], case["mini"], case["batch"]
    s, t = _step_state(case, seed), torch.float32 if case["dtype"] == "f32" else torch.float64
    s["act"] = torch.empty(b, hyper * mini, device="cuda", dtype=t)
    # a sparse layer of a shape the row-list kernel takes is run over its connected rows
    s["sparse"] = case["density"] <= 0.7 and mini % (4 if case["dtype"] == "f32" else 2) == 0 and mini <= 200
    if s["sparse"]:
        most = int(s["wmask"].sum(0, dtype=torch.int64).max())
        s["cap"] = (most + 15) // 16 * 16 + 16
        s["rows"] = torch.empty(hyper, s["cap"], device="cuda", dtype=torch.int32)
        s["row_cnt"] = torch.empty(hyper, device="cuda", dtype=torch.int32)
        s["x_blocked"] = torch.empty((b + 15) // 16 * 16 * n, device="cuda", dtype=t)
        torch.cuda.current_stream().synchronize()
        _capi.check(_capi.lib().sb_mask_rows(s["rows"].data_ptr(), s["row_cnt"].data_ptr(), s["wmask"].data_ptr(), n,
                                             hyper, s["cap"]))
    return s


# --------------------------------------------------------------------------------------------------- work
def _layer_state(layer):
    """What a program reads back after training, as a checkpoint does."""
    return {name: getattr(layer, name) for name in type(layer)._all_names}


def _step(s):
    """One training step of the layer: forward pass of the batch, then the fused step."""
    case, lib, sfx = s["case"], _capi.lib(), "_" + s["case"]["dtype"]
    n, hyper, mini, b = case["inputs"], case["hyper"], case["mini"], case["batch"]
    p = {k: v.data_ptr() for k, v in s.items() if isinstance(v, torch.Tensor)}
    if s["sparse"]:
        _capi.check(getattr(lib, "sb_rows_in_blocks" + sfx)(p["x_blocked"], p["x"], b, n))
        _capi.check(getattr(lib, "sb_compute_activation_rows" + sfx)(
            p["act"], p["x"], p["W"], p["bias"], p["rows"], p["row_cnt"], s["cap"], b, n, hyper, mini, p["x_blocked"]))
    else:
        _capi.check(getattr(lib, "sb_compute_activation" + sfx)(p["act"], p["x"], p["W"], p["bias"], b, n, hyper, mini))
    rewired = hyper // 2 if case["dtype"] == "f64" else -1
    _capi.check(getattr(lib, "sb_plastic_train_step" + sfx)(
        p["W"], p["bias"], p["Ci"], p["Cj"], p["Cij"], p["kbi"], p["wmask"], p["x"], p["act"], b, n, hyper, mini, TAUPDT,
        KHALF, PMIN, TAUBDT, rewired))
    if rewired >= 0 and s["sparse"]:
        _capi.check(lib.sb_mask_rows(p["rows"], p["row_cnt"], p["wmask"], n, hyper, s["cap"]))
    return {k: s[k] for k in ("act", "W", "bias", "Ci", "Cj", "Cij", "kbi", "wmask")}


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "infer":
        return getattr(s["net"], case["what"])(s["x"], case["batch"])
    if kind == "layer":
        layer = s["layers"][0]
        for x in s["x"]:
            act = layer.compute_activation(x)
            layer.train_step(x, act)
        return {"act": act, **_layer_state(layer)}
    if kind == "fit":
        np.random.seed(s["seed"])
        s["net"].fit(s["x"], s["y"], case["batch"], [(0, 1), (1, case["classifier_epochs"])])
        return [_layer_state(layer) for layer in s["layers"]]
    if kind == "epoch":
        s["net"].net.train_epoch(0, case["batch"], s["perm"], s["hc_perm"], case["epoch"])
        return _layer_state(s["layers"][0])
    if kind == "step":
        return _step(s)
    f = getattr(_capi.lib(), "sb_update_mask_" + case["dtype"])
    _capi.check(f(s["wmask"].data_ptr(), s["W"].data_ptr(), s["Ci"].data_ptr(), s["Cj"].data_ptr(), s["Cij"].data_ptr(),
                  TAUPDT / 2, case["inputs"], case["hyper"], case["mini"], case["hyper"] // 2, 16))
    return s["wmask"]


def work(case):
    """What a pass cannot do without.  Every training step reads the batch, the traces and the connected weights and
    writes the traces and the connected weights (the "step" entry point all weights: the caller does not vouch for
    zeros under the mask); an epoch reads its data set twice and writes it once, its order being new."""
    e = 4 if case["dtype"] == "f32" else 8
    n, m = case["inputs"], case["hyper"] * case["mini"]
    kind, live = case["kind"], case["density"] * n * m
    if kind == "rewire":
        return {"bytes": e * (2 * n * case["mini"] + n + case["mini"]) + 2 * n, "flops": 8 * n * case["mini"]}
    b = case["batch"]
    step_bytes = e * (b * (2 * n + 2 * m) + 2 * n * m + 2 * live + 6 * m + 2 * n)
    step_flops = 2 * b * (live + n * m)
    if kind == "step":
        return {"bytes": step_bytes + e * (n * m - live), "flops": step_flops}
    out = m * CLASSES
    if kind == "infer":
        s = case["samples"]
        return {"bytes": e * (s * n + live + out) + s * (4 if case["what"] == "predict" else e * CLASSES),
                "flops": 2 * s * (live + out)}
    steps = -(-case["samples"] // b)
    total = {"bytes": steps * step_bytes + e * (case["samples"] * n + 2 * n * m), "flops": steps * step_flops}
    if kind == "fit":
        k = case["classifier_epochs"]
        total["bytes"] += e * case["samples"] * (2 * n + (2 + k) * m) + steps * k * 3 * e * out
        total["flops"] += 2 * case["samples"] * (live + k * out)
    return total


def tolerance(case):
    """Single precision: four times what the same pass in double precision differs by (2.3e-5 / 1.5e-3 at worst: the
    softmax of logits that are sums of 16000 terms; weights after 469 steps, which a batch on the edge between two units
    moves).  Double precision: the same headroom over the rounding unit."""
    if case["kind"] == "rewire":
        return "exact"
    if case["dtype"] == "f32":
        return {"rel": 1e-4, "max": 6e-3, "differ": 1e-3}
    return {"rel": 2e-13, "max": 1.2e-11, "differ": 0.0}


# -------------------------------------------------------------------------------------- results in 64 bits
def _softmax_units(logits, mini):
    return torch.softmax(logits.view(logits.shape[0], -1, mini), 2).view_as(logits)


def _exact_step(s, x, tau, khalf, pmin, taubdt, mini):
    """One training step on the state `s` (doubles, updated in place): activations, traces, bias, weights, mask."""
    act = _softmax_units(x @ s["W"] + s["bias"], mini)
    cthr = tau / 2
    for name, batch_mean in (("Ci", x.mean(0)), ("Cj", act.mean(0))):
        s[name] = (s[name] * (1 - tau) + tau * batch_mean).clamp_(min=0)
    s["Cij"].mul_(1 - tau).add_(x.t() @ act, alpha=tau / x.shape[0]).clamp_(min=0)
    p4 = pmin / 4
    k = 1 + (khalf - 1) * p4 * p4 / (s["Cj"] - p4) ** 2
    k[(s["Cj"] < p4) | (k < khalf)] = khalf
    s["kbi"] = (1 - taubdt) * s["kbi"] + taubdt * k
    s["bias"] = s["kbi"] * torch.where(s["Cj"] < cthr, 2 * cthr, s["Cj"]).log()
    s["W"] = _weights(s["Ci"], s["Cj"], s["Cij"], cthr)
    s["W"][:, s["Cj"] < cthr] = 0
    s["W"].view(x.shape[1], -1, mini).mul_(s["wmask"][:, :, None])
    return act


def exact(case, seed):
    """None: whole numbers (the class, the mask), weights of a step that rewires, and epochs, over which the
    rounding of one step moves single samples of the next ones."""
    kind, dtype = case["kind"], _np_type(case)
    tau, khalf, pmin, taubdt = (float(dtype(v)) for v in (TAUPDT, KHALF, PMIN, TAUBDT))
    if kind == "step":
        s = {k: v.double() if isinstance(v, torch.Tensor) and v.is_floating_point() else v
             for k, v in _step_state(case, seed).items()}
        act = _exact_step(s, s["x"], tau, khalf, pmin, taubdt, case["mini"])
        rewires = case["dtype"] == "f64"
        return {"act": act, **{k: s[k] for k in ("bias", "Ci", "Cj", "Cij", "kbi")},
                "W": None if rewires else s["W"], "wmask": None}
    if kind == "layer" or (kind == "infer" and case["what"] == "forward"):
        p = prepare(case, seed)
        states = [{"W" if k == "weights" else k: torch.from_numpy(np.array(v)).double().cuda()
                   for k, v in _layer_state(layer).items()} for layer in p["layers"]]
        if kind == "infer":
            x = torch.from_numpy(p["x"]).double().cuda()
            for layer, s in zip(p["layers"], states):
                x = _softmax_units(x @ s["W"] + s["bias"], layer.minicolumns)
            return x
        s, tau = states[0], float(dtype(p["layers"][0].taupdt))
        for x in p["x"]:
            act = _exact_step(s, torch.from_numpy(x).double().cuda(), tau, khalf, pmin, taubdt, case["mini"])
        return {"act": act, "weights": s["W"], **{k: s[k] for k in ("bias", "Ci", "Cj", "Cij", "kbi")}, "wmask": None}
    return None
