"""The work that programs built on this package have it do, as cases that can be timed and
compared: matrix products through `cudeep_amd.ops` on torch tensors, and multi-layer perceptrons
and convolutions through `cudeep_amd.cuDeep.nn`, forward only and forward plus backward.

A case is a dict of plain values; `prepare` makes its inputs (and the model that a program would
keep), `run` is one pass, `exact` the same result in 64 bits from plain torch.
"""
import math

import torch

from cudeep_amd import cuDeep, ops
from cudeep_amd import _lib as L

ACTS = {"none": L.EPI_NONE, "relu": L.EPI_RELU, "gelu": L.EPI_GELU}
PRECS = {"fp32": L.PREC_FP32, "tf32": L.PREC_TF32MODE, "tf32x4": L.PREC_TF32MODE4}
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}


def gemm(m, n, k, prec, ta=False, tb=False, bias=False, act="none", **more):
    return {"kind": "gemm", "m": m, "n": n, "k": k, "prec": prec, "ta": ta, "tb": tb,
            "bias": bias, "act": act, **more}


def mlp(batch, fin, hidden, fout, prec, train, act="relu", **more):
    return {"kind": "mlp", "batch": batch, "fin": fin, "hidden": hidden, "fout": fout,
            "prec": prec, "train": train, "act": act, **more}


def conv(batch, cin, cout, h, w, k, stride, pad, prec, train, dx=True, **more):
    return {"kind": "conv", "batch": batch, "cin": cin, "cout": cout, "h": h, "w": w, "k": k,
            "stride": stride, "pad": pad, "prec": prec, "train": train, "dx": dx, **more}


def listed():
    return [
        # the small product of an interactive program: launch and latency count
        gemm(512, 512, 512, "fp32", name="gemm_fp32_512"),
        # the benchmark's large single-precision product
        gemm(4096, 4096, 4096, "fp32", name="gemm_fp32_4096"),
        # the default (TF32) mode's mid-size product
        gemm(2048, 2048, 2048, "tf32", name="gemm_tf32_2048"),
        # a layer x W^T + b with an activation whose sizes are no multiples of anything
        gemm(1021, 765, 1533, "fp32", tb=True, bias=True, act="gelu", name="linear_fp32_ragged"),
        # a 16-bit feed-forward layer on 2000 tokens
        gemm(2000, 3072, 768, "bf16", tb=True, bias=True, act="gelu", name="linear_bf16_tokens"),
        # double precision, as used to check gradients and in scientific code
        gemm(1024, 1000, 1200, "f64", name="gemm_f64_1000"),
        # one training step of the benchmark's perceptron in the default mode (the input's
        # gradient too, as inside a larger network)
        mlp(8192, 784, 256, 10, "tf32", True, name="mlp_train_8192"),
        # the same perceptron answering a small batch: the smallest call of all
        mlp(64, 784, 256, 10, "fp32", False, name="mlp_infer_64"),
        # one training step of the benchmark's 3x3 layer in single precision
        conv(32, 64, 64, 56, 56, 3, 1, 1, "fp32", True, name="conv3x3_train"),
        # a deeper 3x3 layer at inference on a few images, default mode
        conv(4, 128, 128, 28, 28, 3, 1, 1, "tf32", False, name="conv3x3_infer"),
        # the first layer of an image network: large filter, stride 2, three channels, no
        # gradient for the images
        conv(16, 3, 64, 224, 224, 7, 2, 3, "fp32", True, dx=False, name="conv7x7s2_train"),
        # a 1x1 layer that narrows the channels, training, default mode
        conv(16, 256, 64, 56, 56, 1, 1, 0, "tf32", True, name="conv1x1_train"),
    ]


def _log_int(rng, lo, hi):
    """An integer spread evenly over the logarithm; every second one rounded to a multiple of 8
    or 64, as layer sizes mostly are."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    step = rng.choice([1, 1, 8, 64])
    return max(lo, min(hi, (v + step // 2) // step * step))


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "mlp", "conv", "conv"])
    if kind == "gemm":
        prec = rng.choice(["fp32", "fp32", "tf32", "tf32", "tf32x4", "bf16", "f16", "f64"])
        top = 1200 if prec == "f64" else 3072
        plain = prec == "f64"   # the double-precision entry point has no bias or activation
        return gemm(_log_int(rng, 32, top), _log_int(rng, 32, top), _log_int(rng, 32, top), prec,
                    ta=rng.random() < 0.3, tb=rng.random() < 0.5,
                    bias=not plain and rng.random() < 0.5,
                    act="none" if plain else rng.choice(["none", "relu", "gelu"]))
    if kind == "mlp":
        return mlp(_log_int(rng, 16, 8192), _log_int(rng, 32, 1024), _log_int(rng, 32, 1024),
                   _log_int(rng, 8, 512), rng.choice(["fp32", "tf32"]), rng.random() < 0.6,
                   act=rng.choice(["relu", "relu", "gelu"]))
    k = rng.choice([1, 3, 3, 3, 5, 7])
    stride = rng.choice([1, 1, 1, 2])
    side = rng.choice([7, 13, 14, 28, 31, 56, 60, 112])
    cin, cout = _log_int(rng, 3, 256), _log_int(rng, 16, 256)
    batch, train = _log_int(rng, 1, 32), rng.random() < 0.6
    case = conv(batch, cin, cout, side, side, k, stride, k // 2, rng.choice(["fp32", "tf32"]),
                train, dx=cin > 4)
    while case["batch"] > 1 and work(case)["flops"] > 2.0e10:
        case["batch"] = (case["batch"] + 1) // 2
    return case


# ---- inputs --------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _inputs(case, seed):
    """All inputs of a case as float32 (float64) tensors on the GPU, from the seed alone:
    activations ~ N(0, 1) (after a ReLU inside a convolutional network), weights scaled by their
    fan-in, output gradients of the size a mean loss gives."""
    g = _gen(seed)

    def rnd(*shape, scale=1.0, dtype=torch.float32):
        return torch.randn(shape, device="cuda", generator=g, dtype=dtype) * scale

    if case["kind"] == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        dt = torch.float64 if case["prec"] == "f64" else torch.float32
        a = rnd(*((k, m) if case["ta"] else (m, k)), dtype=dt)
        b = rnd(*((n, k) if case["tb"] else (k, n)), scale=k ** -0.5, dtype=dt)
        bias = rnd(n, scale=0.1) if case["bias"] else None
        if case["prec"] in ("bf16", "f16"):
            a, b = a.to(DTYPES[case["prec"]]), b.to(DTYPES[case["prec"]])
        return {"a": a, "b": b, "bias": bias}
    if case["kind"] == "mlp":
        n, fi, h, fo = case["batch"], case["fin"], case["hidden"], case["fout"]
        return {"x": rnd(n, fi), "w1": rnd(h, fi, scale=(2.0 / fi) ** 0.5), "b1": rnd(h, scale=0.1),
                "w2": rnd(fo, h, scale=h ** -0.5), "b2": rnd(fo, scale=0.1),
                "dy": rnd(n, fo, scale=1.0 / n)}
    n, ci, co, k = case["batch"], case["cin"], case["cout"], case["k"]
    oh, ow = _out(case)
    x = rnd(n, ci, case["h"], case["w"])
    if ci > 4:
        x = x.relu()
    return {"x": x, "w": rnd(co, ci, k, k, scale=(2.0 / (ci * k * k)) ** 0.5),
            "b": rnd(co, scale=0.1), "dy": rnd(n, co, oh, ow, scale=1.0 / n)}


def _out(case):
    return tuple((s + 2 * case["pad"] - case["k"]) // case["stride"] + 1
                 for s in (case["h"], case["w"]))


def _tensor(t, grad=False):
    return cuDeep.Tensor.from_numpy(t.cpu().numpy(), requires_grad=grad)


def prepare(case, seed):
    v = _inputs(case, seed)
    if case["kind"] == "gemm":
        v["case"] = case
        return v
    cuDeep.set_matmul_precision(case["prec"])
    nn = cuDeep.nn
    if case["kind"] == "mlp":
        act = nn.ReLU() if case["act"] == "relu" else nn.GELU()
        model = nn.Sequential(nn.Linear(case["fin"], case["hidden"]), act,
                              nn.Linear(case["hidden"], case["fout"]))
        names = {"0.weight": "w1", "0.bias": "b1", "2.weight": "w2", "2.bias": "b2"}
        dx = True
    else:
        model = nn.Conv2d(case["cin"], case["cout"], case["k"], stride=case["stride"],
                          padding=case["pad"])
        names = {"weight": "w", "bias": "b"}
        dx = case["dx"]
    model.load_state_dict({name: v[key].cpu().numpy() for name, key in names.items()})
    return {"case": case, "model": model, "x": _tensor(v["x"], case["train"] and dx),
            "dy": _tensor(v["dy"]) if case["train"] else None}


# ---- one pass ------------------------------------------------------------------------------

class _Shared:
    """A cuDeep tensor's memory as torch sees it (no copy; keeps the tensor alive)."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.__cuda_array_interface__ = {
            "shape": tuple(tensor.shape()), "typestr": "<f4", "strides": None, "version": 2,
            "data": (tensor._data.data_ptr(), False)}


def _torch(tensor):
    return torch.as_tensor(_Shared(tensor), device="cuda")


def run(state):
    case = state["case"]
    if case["kind"] == "gemm":
        prec, a, b = case["prec"], state["a"], state["b"]
        if prec == "f64":
            return ops.dgemm(a, b, case["ta"], case["tb"])
        if prec == "fp32" and not (case["ta"] or case["tb"] or case["bias"]) \
                and case["act"] == "none":
            return ops.sgemm(a, b)
        more = {"transA": case["ta"], "transB": case["tb"], "bias": state["bias"],
                "bias_mode": L.BIAS_COL if case["bias"] else L.BIAS_NONE,
                "epilogue": ACTS[case["act"]]}
        if prec in PRECS:
            return ops.gemm(a, b, precision=PRECS[prec], **more)
        return ops.gemm16(a, b, **more)
    model, x = state["model"], state["x"]
    if not case["train"]:
        with cuDeep.no_grad():
            return _torch(model(x))
    model.zero_grad()
    x.grad = None
    y = model(x)
    y.backward(state["dy"])
    out = {"y": _torch(y)}
    if x.requires_grad:
        out["x"] = _torch(x.grad)
    for name, p in model.named_parameters():
        out[name] = _torch(p.grad)
    return out


# ---- what a pass cannot do without ---------------------------------------------------------

def work(case):
    if case["kind"] == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        es = {"bf16": 2, "f16": 2, "f64": 8}.get(case["prec"], 4)
        eo = 8 if case["prec"] == "f64" else 4
        return {"bytes": es * (m * k + k * n) + eo * m * n + (4 * n if case["bias"] else 0),
                "flops": 2.0 * m * n * k}
    if case["kind"] == "mlp":
        n, fi, h, fo = case["batch"], case["fin"], case["hidden"], case["fout"]
        weights, flops = fi * h + h + h * fo + fo, 2.0 * n * (fi * h + h * fo)
        if case["train"]:   # in: x, dy, weights; out: y, dx, the weights' gradients
            return {"bytes": 4.0 * (2 * n * fi + 2 * n * fo + 2 * weights), "flops": 3 * flops}
        return {"bytes": 4.0 * (n * fi + n * fo + weights), "flops": flops}
    n, ci, co, k = case["batch"], case["cin"], case["cout"], case["k"]
    oh, ow = _out(case)
    x, y, weights = n * ci * case["h"] * case["w"], n * co * oh * ow, co * ci * k * k + co
    flops = 2.0 * n * co * oh * ow * ci * k * k
    if case["train"]:
        return {"bytes": 4.0 * ((2 if case["dx"] else 1) * x + 2 * y + 2 * weights),
                "flops": (3 if case["dx"] else 2) * flops}
    return {"bytes": 4.0 * (x + y + weights), "flops": flops}


def _gated(case):
    """Whether the case's gradients pass a ReLU: pre-activations within rounding of zero fall on
    either side of it, and each that does changes a whole row of the gradients (a handful of the
    2 million of the largest case in the default mode, about 2e-3 of the gradients' norm)."""
    return case["kind"] == "mlp" and case["train"] and case["act"] == "relu"


def tolerance(case):
    """About four times the errors measured against `exact` over these ranges: 1.1e-6 in single
    precision (1.4e-6 through the Winograd transforms), 4e-6 to 7e-6 in the default mode's split
    products, 4e-5 where those run inside the Winograd transforms (3x3, stride 1), 2e-7 to 5e-7
    for 16-bit operands with sums in 32 bits, 1e-15 in double precision."""
    if case["prec"] == "f64":
        return {"rel": 5e-15}
    if case["prec"] in ("bf16", "f16"):
        return {"rel": 2e-6}
    if _gated(case):
        return {"rel": 8e-3, "max": 0.9}
    if case["prec"] == "fp32":
        return {"rel": 5e-6}
    wino = case["kind"] == "conv" and case["k"] == 3 and case["stride"] == 1
    return {"rel": 1.6e-4 if wino else 2.5e-5}


# ---- the same in 64 bits -------------------------------------------------------------------

def _act(z, act):
    if act == "relu":
        return z.relu()
    return torch.nn.functional.gelu(z, approximate="tanh") if act == "gelu" else z


def exact(case, seed):
    v = {k: t.double() if t is not None else None for k, t in _inputs(case, seed).items()}
    if case["kind"] == "gemm":
        a = v["a"].t() if case["ta"] else v["a"]
        b = v["b"].t() if case["tb"] else v["b"]
        z = torch.mm(a.contiguous(), b.contiguous())
        if v["bias"] is not None:
            z = z + v["bias"]
        return _act(z, case["act"])
    if case["kind"] == "mlp":
        z = v["x"] @ v["w1"].t().contiguous() + v["b1"]
        h = _act(z, case["act"])
        y = h @ v["w2"].t().contiguous() + v["b2"]
        if not case["train"]:
            return y
        dh = v["dy"] @ v["w2"]
        if case["act"] == "relu":
            dz = dh * (z > 0)
        else:
            zz = z.detach().requires_grad_(True)
            dz = torch.autograd.grad(_act(zz, "gelu"), zz, dh)[0]
        out = {"y": y, "x": dz @ v["w1"], "0.weight": dz.t().contiguous() @ v["x"],
               "0.bias": dz.sum(0), "2.weight": v["dy"].t().contiguous() @ h,
               "2.bias": v["dy"].sum(0)}
        if _gated(case):   # decided by the sign of values within rounding of zero
            out.update({"x": None, "0.weight": None, "0.bias": None})
        return out
    n, ci, co, k = case["batch"], case["cin"], case["cout"], case["k"]
    oh, ow = _out(case)
    geom = {"kernel_size": (k, k), "padding": case["pad"], "stride": case["stride"]}
    wm = v["w"].reshape(co, -1)
    y = torch.empty((n, co, oh, ow), device="cuda", dtype=torch.float64)
    dx, dw = torch.empty_like(v["x"]), torch.zeros_like(wm)
    for i in range(n):   # one image at a time: the columns in 64 bits stay small
        col = torch.nn.functional.unfold(v["x"][i:i + 1], **geom)[0]
        y[i] = (wm @ col + v["b"][:, None]).reshape(co, oh, ow)
        if case["train"]:
            dy = v["dy"][i].reshape(co, -1)
            dw += dy @ col.t().contiguous()
            if case["dx"]:
                dx[i] = torch.nn.functional.fold((wm.t().contiguous() @ dy)[None],
                                                 (case["h"], case["w"]), **geom)[0]
    if not case["train"]:
        return y
    out = {"y": y, "weight": dw.reshape(v["w"].shape), "bias": v["dy"].sum((0, 2, 3))}
    if case["dx"]:
        out["x"] = dx
    return out
