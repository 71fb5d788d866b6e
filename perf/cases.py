"""The work whose time is measured: bound queries as a program that uses the package issues
them, each through a public entry point, from one input on a small network to the largest
domain batch.

A case is a dict of plain values.  ``entry`` names what is called:

* ``crown``      ``run_crown_ibp_mlp`` (IBP, then CROWN on the margin specs), as a serving loop
                 calls it: the query captured once (``CapturedQuery``), each pass copying the
                 new inputs in and replaying it
* ``crown_all``  ``run_crown_all_intermediate`` (every pre-activation bound by CROWN)
* ``alpha``      ``run_alpha_crown_from_crown_init``, captured like ``crown``
* ``bab``        ``evaluate_domain_batch`` (beta-CROWN of a frontier's domains), captured
* ``grad``       ``lower_bound_gradients`` (one evaluation and its reverse pass)
* ``region``     ``HipFusedCrownExecutor.run`` on one ReLU -> Linear region
* ``ibp``        ``HipTaskExecutor.run_ibp`` (interval bounds of a whole test batch)

Networks have Kaiming-uniform weights and small random biases, inputs are uniform in [0, 1],
specs are the margins of a random label against every other class.
"""

from __future__ import annotations

import math
from typing import Dict, List, Tuple

import torch

from boundflow_amd import alpha_beta, bab, crown, fused_crown, task_executor
from boundflow_amd.graphs import CapturedQuery
from boundflow_amd.ir import BFTaskModule, BoundTask, TaskKind, TaskOp, default_storage_plan
from boundflow_amd.spec import InputSpec

EPS_F32 = torch.finfo(torch.float32).eps


def listed() -> List[dict]:
    return [
        # one input checked by itself (an interactive query): launches and latency alone
        {"name": "mlp_one", "entry": "crown", "net": "mlp", "batch": 1, "inputs": 784, "width": 256, "depth": 2,
         "classes": 10, "ball": "box", "eps": 2.0 / 255.0},
        # a batch of images through a deep MLP with every layer's bounds refined: the largest query
        {"name": "mlp_layers", "entry": "crown_all", "net": "mlp", "batch": 256, "inputs": 784, "width": 500,
         "depth": 6, "classes": 10, "ball": "linf", "eps": 0.015},
        # many input boxes of a narrow controller-sized network, whose widths are no multiple of four
        {"name": "mlp_narrow", "entry": "crown_all", "net": "mlp", "batch": 1000, "inputs": 5, "width": 50,
         "depth": 6, "classes": 5, "ball": "box", "eps": 0.05},
        # a test batch of 32 x 32 colour images through the strided CNN
        {"name": "cnn", "entry": "crown", "net": "cnn", "batch": 128, "size": 32, "colours": 3, "channels": 16,
         "hidden": 100, "classes": 10, "ball": "linf", "eps": 2.0 / 255.0},
        # grey 28 x 28 images: maps of 14 x 14 and 7 x 7, a batch that fills no power of two
        {"name": "cnn_grey", "entry": "crown", "net": "cnn", "batch": 50, "size": 28, "colours": 1, "channels": 16,
         "hidden": 100, "classes": 10, "ball": "linf", "eps": 0.02},
        # slopes optimised per input on the CNN: 20 bound and gradient passes
        {"name": "cnn_alpha", "entry": "alpha", "net": "cnn", "batch": 32, "size": 32, "colours": 3, "channels": 16,
         "hidden": 100, "classes": 10, "ball": "linf", "eps": 8.0 / 255.0, "steps": 20},
        # one round of a wide branch-and-bound frontier: 4096 split domains of one input, 10 steps
        {"name": "bab_batch", "entry": "bab", "net": "mlp", "batch": 4096, "inputs": 784, "width": 256, "depth": 4,
         "classes": 10, "ball": "linf", "eps": 0.03, "steps": 10},
        # one bound and its reverse pass (slopes and split multipliers) for 1500 domains
        {"name": "bab_grad", "entry": "grad", "net": "mlp", "batch": 1500, "inputs": 784, "width": 256, "depth": 4,
         "classes": 10, "ball": "linf", "eps": 0.03},
        # residual MLP: the backward over a DAG, a batch of ordinary size
        {"name": "residual_mlp", "entry": "crown", "net": "resmlp", "batch": 256, "inputs": 784, "width": 256,
         "hidden": 512, "blocks": 4, "classes": 10, "ball": "linf", "eps": 0.002},
        # residual CNN of 3 x 3 convolutions at stride 1
        {"name": "residual_cnn", "entry": "crown", "net": "rescnn", "batch": 32, "size": 16, "colours": 3,
         "channels": 12, "blocks": 3, "classes": 10, "ball": "linf", "eps": 0.002},
        # one fused region as a planner that owns the backward hands it over: many specs, few domains
        {"name": "region", "entry": "region", "batch": 8, "specs": 257, "inputs": 1024, "width": 512},
        # interval bounds of a whole test set's batch (encoding only, no backward)
        {"name": "ibp_batch", "entry": "ibp", "net": "cnn", "batch": 2048, "size": 32, "colours": 3, "channels": 16,
         "hidden": 100, "classes": 10, "ball": "linf", "eps": 2.0 / 255.0},
    ]


def _size(rng, lo: int, hi: int) -> int:
    """A size spread over the logarithm of its range; half of them a multiple of 8, as widths often are."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5 and n >= 8:
        n = n // 8 * 8
    return max(lo, min(hi, n))


def draw(rng) -> dict:
    entry = rng.choice(["crown", "crown", "crown", "crown", "crown_all", "crown_all", "alpha", "bab", "grad",
                        "region", "ibp"])
    eps = rng.choice([0.01, 0.015, 2.0 / 255.0, 0.02])
    if entry == "region":
        return {"entry": "region", "batch": _size(rng, 1, 16), "specs": _size(rng, 9, 257),
                "inputs": _size(rng, 64, 1024), "width": _size(rng, 64, 512)}
    net = {"crown": rng.choice(["mlp", "mlp", "cnn", "resmlp", "rescnn"]), "crown_all": "mlp", "alpha": "cnn",
           "bab": "mlp", "grad": "mlp", "ibp": rng.choice(["mlp", "cnn"])}[entry]
    case = {"entry": entry, "net": net, "classes": 10, "eps": eps,
            "ball": rng.choice(["linf", "box", "l2"]) if entry == "crown" and net == "mlp" else "linf"}
    if net == "mlp":
        case.update({"inputs": rng.choice([784, 784, _size(rng, 5, 784)]), "depth": rng.randint(2, 6),
                     "width": _size(rng, 50, 500), "batch": _size(rng, 1, 256)})
        if entry == "crown_all":
            case.update({"batch": _size(rng, 16, 200), "ball": rng.choice(["linf", "box"])})
        elif entry == "ibp":
            case["batch"] = _size(rng, 256, 4096)
        elif entry in ("bab", "grad"):
            case.update({"batch": _size(rng, 256, 2048), "width": _size(rng, 64, 256), "depth": rng.randint(2, 4),
                         "eps": 0.03})
        if entry == "bab":
            case["steps"] = rng.randint(2, 10)
    elif net == "cnn":
        size, colours = rng.choice([(32, 3), (28, 1)])
        case.update({"size": size, "colours": colours, "channels": rng.choice([8, 16]), "hidden": _size(rng, 50, 256),
                     "batch": _size(rng, 4, 128)})
        if entry == "alpha":
            case.update({"batch": _size(rng, 4, 32), "steps": rng.randint(3, 20)})
        elif entry == "ibp":
            case["batch"] = _size(rng, 256, 2048)
    elif net == "resmlp":
        case.update({"inputs": 784, "width": _size(rng, 64, 256), "hidden": _size(rng, 64, 512),
                     "blocks": rng.randint(1, 4), "batch": _size(rng, 8, 256), "eps": 0.002})
    else:
        case.update({"size": rng.choice([8, 12, 16]), "colours": 3, "channels": rng.choice([8, 12, 16]),
                     "blocks": rng.randint(1, 3), "batch": _size(rng, 4, 32), "eps": 0.002})
    return case


# ---------------------------------------------------------------------------
# Networks and inputs


def _net(case: dict, gen: torch.Generator, dev) -> Tuple[List[TaskOp], Dict[str, torch.Tensor]]:
    ops: List[TaskOp] = []
    params: Dict[str, torch.Tensor] = {}

    def weights(name, shape):
        fan_in = math.prod(shape[1:])
        bound = math.sqrt(6.0 / fan_in)
        params["W_" + name] = (torch.rand(shape, generator=gen, device=dev) * 2.0 - 1.0) * bound
        params["b_" + name] = torch.randn(shape[0], generator=gen, device=dev) * 0.01
        return ["W_" + name, "b_" + name]

    def linear(x, name, n_in, n_out, out=None):
        out = out or "h_" + name
        ops.append(TaskOp("linear", name, [x] + weights(name, (n_out, n_in)), [out]))
        return out

    def conv(x, name, c_in, c_out, kernel, stride, pad):
        ops.append(TaskOp("conv2d", name, [x] + weights(name, (c_out, c_in, kernel, kernel)), ["h_" + name],
                          {"stride": stride, "padding": pad, "dilation": 1, "groups": 1}))
        return "h_" + name

    def relu(x):
        ops.append(TaskOp("relu", "relu_" + x, [x], ["r_" + x]))
        return "r_" + x

    def flatten(x):
        ops.append(TaskOp("flatten", "flatten", [x], ["flat"], {"start_dim": 1, "end_dim": -1}))
        return "flat"

    def add(x, y, name):
        ops.append(TaskOp("add", name, [x, y], ["s_" + name]))
        return "s_" + name

    x = "input"
    if case["net"] == "mlp":
        n = case["inputs"]
        for i in range(case["depth"]):
            x, n = relu(linear(x, f"l{i}", n, case["width"])), case["width"]
    elif case["net"] == "cnn":
        c, s = case["channels"], case["size"]
        x = relu(conv(x, "c0", case["colours"], c, 4, 2, 1))
        x = relu(conv(x, "c1", c, 2 * c, 4, 2, 1))
        n = 2 * c * (s // 4) ** 2
        x, n = relu(linear(flatten(x), "l0", n, case["hidden"])), case["hidden"]
    elif case["net"] == "resmlp":
        n = case["width"]
        x = relu(linear(x, "stem", case["inputs"], n))
        for i in range(case["blocks"]):
            y = linear(relu(linear(x, f"a{i}", n, case["hidden"])), f"b{i}", case["hidden"], n)
            x = relu(add(x, y, f"add{i}"))
    else:
        c = case["channels"]
        x = relu(conv(x, "stem", case["colours"], c, 3, 1, 1))
        for i in range(case["blocks"]):
            y = conv(relu(conv(x, f"a{i}", c, c, 3, 1, 1)), f"b{i}", c, c, 3, 1, 1)
            x = relu(add(x, y, f"add{i}"))
        x, n = flatten(x), c * case["size"] ** 2
    linear(x, "head", n, case["classes"], "out")
    return ops, params


def _in_shape(case: dict) -> Tuple[int, ...]:
    return (case["inputs"],) if case["net"] in ("mlp", "resmlp") else (case["colours"], case["size"], case["size"])


def _eps(case: dict) -> float:
    return float(torch.tensor(case["eps"], dtype=torch.float32))


def _inputs(case: dict, seed: int, dev) -> dict:
    """Everything a case's call is given, from the seed alone."""
    gen = torch.Generator(device=dev).manual_seed(seed)
    rand = lambda *shape: torch.rand(shape, generator=gen, device=dev)   # noqa: E731
    if case["entry"] == "region":
        D, S, N, P = case["batch"], case["specs"], case["inputs"], case["width"]
        lo = rand(D, N) * -1.0 + 0.3          # about a third of the ReLUs stable
        hi = lo + rand(D, N) * 1.2
        slope = (hi / (hi - lo).clamp_min(EPS_F32)).clamp(0.0, 1.0)
        amb = ((lo < 0) & (hi > 0)).float()
        act = (lo >= 0).float()
        return {"A_u": torch.randn(D, S, N, generator=gen, device=dev), "A_l": torch.randn(D, S, N, generator=gen, device=dev),
                "alpha_u": amb * slope + act, "beta_u": amb * slope * -lo, "alpha_l": amb * (slope > 0.5).float() + act,
                "beta_l": torch.zeros(D, N, device=dev), "weight": (rand(N, P) * 2.0 - 1.0) * math.sqrt(6.0 / P),
                "bias": torch.randn(N, generator=gen, device=dev) * 0.01}
    ops, params = _net(case, gen, dev)
    B, classes = case["batch"], case["classes"]
    one = case["entry"] in ("bab", "grad")   # every domain is a part of one input's set
    x = rand(1 if one else B, *_in_shape(case)).expand(B, *_in_shape(case)).contiguous()
    label = torch.randint(0, classes, (1 if one else B,), generator=gen, device=dev).expand(B)
    eye = torch.eye(classes, device=dev)
    other = torch.arange(classes - 1, device=dev)[None, :]
    other = other + (other >= label[:, None])          # every class but the label, in order
    C = (eye[label][:, None, :] - eye[other]).contiguous()
    given = {"ops": ops, "params": params, "x": x, "C": C}
    if one:
        given["splits"], given["alpha"], given["beta"] = {}, {}, {}
        box = _ibp(ops, params, x[:1], x[:1] - case["eps"], x[:1] + case["eps"])
        names = [op.inputs[0] for op in ops if op.op_type == "relu"]
        amb = torch.cat([((box[n][0] < 0) & (box[n][1] > 0)).flatten() for n in names])
        # 1 to 12 splits a domain on ambiguous neurons (a gradient query: of the first layer alone,
        # where no set of splits empties a box)
        if case["entry"] == "grad":
            amb[case["width"]:] = False
        score = torch.where(amb, rand(B, amb.numel()), torch.full((), -1.0, device=dev))
        pick = score.topk(12, dim=1)
        count = torch.randint(1, 13, (B, 1), generator=gen, device=dev)
        keep = (torch.arange(12, device=dev)[None, :] < count) & (pick.values > 0)
        sign = (torch.randint(0, 2, (B, 12), generator=gen, device=dev) * 2 - 1) * keep
        flat = torch.zeros(B, amb.numel(), dtype=torch.int64, device=dev).scatter_(1, pick.indices, sign).to(torch.int8)
        for i, n in enumerate(names):
            w = case["width"]
            given["splits"][n] = flat[:, i * w:(i + 1) * w].contiguous()
            given["alpha"][n] = rand(B, w)
            given["beta"][n] = rand(B, w) * 0.1 * (given["splits"][n] != 0)
    return given


def _spec(case: dict, x: torch.Tensor) -> InputSpec:
    e = _eps(case)
    if case["ball"] == "box":
        return InputSpec.box(value_name="input", lower=(x - e).clamp(0.0, 1.0), upper=(x + e).clamp(0.0, 1.0))
    make = InputSpec.l2 if case["ball"] == "l2" else InputSpec.linf
    return make(value_name="input", center=x, eps=e)


def _module(ops: List[TaskOp], params: Dict[str, torch.Tensor]) -> BFTaskModule:
    task = BoundTask(task_id="t0", kind=TaskKind.INTERVAL_IBP, ops=ops, input_values=["input"], output_values=["out"],
                     params=list(params))
    return BFTaskModule(tasks=[task], entry_task_id="t0", bindings={"params": params},
                        storage_plan=default_storage_plan(["input"] + [op.outputs[0] for op in ops]))


# ---------------------------------------------------------------------------
# One pass


def prepare(case: dict, seed: int) -> dict:
    dev = torch.device("cuda:0")
    g = _inputs(case, seed, dev)
    if case["entry"] == "region":
        N, P = case["inputs"], case["width"]
        req = fused_crown.FusedReluAffineRequest(kind="linear", input_shape=(P,), output_shape=(N,), attrs={},
                                                 **{k: g[k] for k in ("A_u", "A_l", "alpha_u", "alpha_l", "beta_u",
                                                                      "beta_l", "weight", "bias")})
        return {"entry": "region", "executor": fused_crown.HipFusedCrownExecutor(), "request": req}
    state = {"entry": case["entry"], "module": _module(g["ops"], g["params"]), "spec": _spec(case, g["x"]), "C": g["C"],
             "splits": g.get("splits"), "alpha": g.get("alpha"), "beta": g.get("beta"), "steps": case.get("steps")}
    if case["entry"] in ("crown", "alpha", "bab"):
        # the serving loop's captured query, and the buffers its inputs are copied into
        m, steps = state["module"], case.get("steps")
        held, C = _spec(case, torch.rand_like(g["x"])), torch.zeros_like(g["C"])
        held_splits = None if g.get("splits") is None else {n: torch.zeros_like(s) for n, s in g["splits"].items()}
        call = {"crown": lambda: crown.run_crown_ibp_mlp(m, held, linear_spec_C=C),
                "alpha": lambda: alpha_beta.run_alpha_crown_from_crown_init(m, held, linear_spec_C=C, steps=steps)[0],
                "bab": lambda: bab.evaluate_domain_batch(m, held, linear_spec_C=C, relu_split_state=held_splits,
                                                         steps=steps)}[case["entry"]]
        pairs = [(held.center, state["spec"].center), (C, g["C"])]
        if case["ball"] == "box":
            pairs += [(held.perturbation.lower, state["spec"].perturbation.lower),
                      (held.perturbation.upper, state["spec"].perturbation.upper)]
        if held_splits is not None:
            pairs += [(held_splits[n], g["splits"][n]) for n in held_splits]
        state.update({"query": CapturedQuery(call), "pairs": pairs})
    return state


def run(state: dict):
    entry = state["entry"]
    if entry == "region":
        r = state["executor"].run(state["request"])
        return {"A_u": r.A_prev_u, "A_l": r.A_prev_l, "b_u": r.bias_delta_u, "b_l": r.bias_delta_l}
    if entry == "crown_all":
        final, pre = crown.run_crown_all_intermediate(state["module"], state["spec"], linear_spec_C=state["C"])
        return {"lower": final.lower, "upper": final.upper, "pre_lower": [p.lower for p in pre.values()],
                "pre_upper": [p.upper for p in pre.values()]}
    if entry == "grad":
        b, ga, gb = alpha_beta.lower_bound_gradients(state["module"], state["spec"], linear_spec_C=state["C"],
                                                     relu_alpha=state["alpha"], relu_beta=state["beta"],
                                                     relu_split_state=state["splits"])
        return {"lower": b.lower, "upper": b.upper, "alpha": list(ga.values()), "beta": list(gb.values())}
    if entry == "ibp":
        b = task_executor.HipTaskExecutor().run_ibp(state["module"], state["spec"])
        return {"lower": b.lower, "upper": b.upper}
    for held, new in state["pairs"]:
        held.copy_(new)
    out = state["query"]()
    if entry == "bab":
        # (the optimised parameters themselves are no stable numbers: an Adam trajectory divides by the
        # root of each element's own gradient history, so rounding alone moves single elements)
        return {k: out[k] for k in ("status", "lower", "upper", "branch_layer", "branch_neuron")}
    return {"lower": out.lower, "upper": out.upper}


# ---------------------------------------------------------------------------
# What a pass cannot do without


def _shapes(case: dict) -> List[Tuple[str, int, int, int]]:
    """(op name, inputs, outputs, multiply-adds a row) of every affine op, in order."""
    out = []
    if case["net"] == "mlp":
        dims = [case["inputs"]] + [case["width"]] * case["depth"] + [case["classes"]]
        out = [("l", a, b, a * b) for a, b in zip(dims, dims[1:])]
    elif case["net"] == "resmlp":
        n, h = case["width"], case["hidden"]
        out = [("l", case["inputs"], n, case["inputs"] * n)]
        out += [("l", a, b, a * b) for _ in range(case["blocks"]) for a, b in ((n, h), (h, n))]
        out += [("l", n, case["classes"], n * case["classes"])]
    elif case["net"] == "cnn":
        c, s = case["channels"], case["size"]
        h1, h2 = s // 2, s // 4
        out = [("c", case["colours"] * s * s, c * h1 * h1, c * h1 * h1 * case["colours"] * 16),
               ("c", c * h1 * h1, 2 * c * h2 * h2, 2 * c * h2 * h2 * c * 16),
               ("l", 2 * c * h2 * h2, case["hidden"], 2 * c * h2 * h2 * case["hidden"]),
               ("l", case["hidden"], case["classes"], case["hidden"] * case["classes"])]
    else:
        c, n = case["channels"], case["channels"] * case["size"] ** 2
        out = [("c", case["colours"] * case["size"] ** 2, n, n * case["colours"] * 9)]
        out += [("c", n, n, n * c * 9)] * (2 * case["blocks"])
        out += [("l", n, case["classes"], n * case["classes"])]
    return out


def _weight_values(case: dict) -> int:
    if case["net"] == "cnn":
        c = case["channels"]
        return (case["colours"] * c + 2 * c * c) * 16 + 3 * c + sum(m + o for k, _, o, m in _shapes(case) if k == "l")
    if case["net"] == "rescnn":
        c = case["channels"]
        return (case["colours"] + 2 * case["blocks"] * c) * c * 9 + sum(m + o for k, _, o, m in _shapes(case) if k == "l")
    return sum(m + o for _, _, o, m in _shapes(case))


def work(case: dict) -> dict:
    B = case["batch"]
    if case["entry"] == "region":
        M, N, P = B * case["specs"], case["inputs"], case["width"]
        return {"bytes": 4.0 * (2 * M * (N + P + 1) + 4 * B * N + N * P + N), "flops": 4.0 * M * N * P}
    layers = _shapes(case)
    macs = sum(m for _, _, _, m in layers)
    classes, n_in = case["classes"], layers[0][1]
    S = classes - 1
    inputs = 4.0 * (_weight_values(case) + B * n_in * (2 if case["ball"] == "box" else 1))
    specs, bounds = 4.0 * B * S * classes, 8.0 * B * S
    ibp = 4.0 * B * macs                                  # center and radius products
    hidden = [o for _, _, o, _ in layers[:-1]]
    if case["entry"] == "ibp":
        return {"bytes": inputs + 8.0 * B * classes, "flops": ibp}
    row = 2.0 * macs                                      # one coefficient row of one bound through the network
    if case["entry"] == "crown":
        return {"bytes": inputs + specs + bounds, "flops": ibp + 2.0 * B * S * row}
    if case["entry"] == "crown_all":
        # C = I at each hidden layer after the first: its rows pass the layers below it (the first of
        # them as the weight itself), for both bounds
        below = [2.0 * sum(m for _, _, _, m in layers[:i]) for i in range(1, len(layers) - 1)]
        refine = sum(2.0 * B * n * f for n, f in zip(hidden[1:], below))
        return {"bytes": inputs + specs + bounds + 8.0 * B * sum(hidden), "flops": ibp + refine + 2.0 * B * S * row}
    neurons = sum(hidden)
    if case["entry"] == "grad":
        # both bounds, and the reverse pass of the lower one
        return {"bytes": inputs + specs + bounds + B * neurons * (4.0 * 4 + 1.0), "flops": ibp + 3.0 * B * S * row}
    # steps + 1 lower bounds, steps reverse passes, one upper bound
    passes = 2 * case["steps"] + 2
    splits = 1.0 * B * neurons if case["entry"] == "bab" else 0.0
    return {"bytes": inputs + specs + bounds + splits, "flops": ibp + passes * B * S * row}


# Four times what the same query gives when the network's hidden units are permuted (the function
# unchanged, every sum in another order), over listed and drawn cases:
# * sums alone (crown, ibp; region, whose random rows cancel more);
# * crown_all: a refined bound within rounding of zero makes its ReLU stable or not, which moves the
#   lower slope from 0 to 1 and with it that one input's later bounds (seen in one run of 25);
# * alpha, bab: single elements of an Adam trajectory part where rounding decides a gradient's sign;
# * grad: a coefficient within rounding of zero takes either slope of its ReLU.
TOLERANCE = {"crown": {"rel": 1e-6, "max": 5e-6}, "ibp": {"rel": 1e-6, "max": 5e-6},
             "region": {"rel": 3e-6, "max": 2e-5}, "crown_all": {"rel": 3e-2, "max": 0.4},
             "alpha": {"rel": 1e-4, "max": 1e-2}, "bab": {"rel": 2e-4, "max": 1e-2},
             "grad": {"rel": 3e-3, "max": 0.25}}


def tolerance(case: dict):
    return TOLERANCE[case["entry"]]


# ---------------------------------------------------------------------------
# The same numbers in 64 bits, without the package's code


def _affine(op, params, x, weight=None, bias=True):
    w = params[op.inputs[1]] if weight is None else weight
    b = params[op.inputs[2]] if bias else None
    if op.op_type == "linear":
        y = x.reshape(x.shape[0], -1) @ w.t()
        return y if b is None else y + b
    return torch.nn.functional.conv2d(x, w, b, stride=op.attrs["stride"], padding=op.attrs["padding"])


def _ibp(ops, params, x, lo, hi, ball="linf", eps=0.0, splits=None):
    """Boxes of every value; the box a ReLU reads is the split one."""
    box = {"input": (lo, hi)}
    for op in ops:
        l, u = box[op.inputs[0]]
        t = op.op_type
        if t in ("linear", "conv2d"):
            w = params[op.inputs[1]]
            if ball == "l2" and op.inputs[0] == "input":
                mid, rad = _affine(op, params, x), eps * w.norm(dim=1)[None, :]
            else:
                mid, rad = _affine(op, params, (l + u) / 2), _affine(op, params, (u - l) / 2, w.abs(), False)
            l, u = mid - rad, mid + rad
            s = None if splits is None else splits.get(op.outputs[0])
            if s is not None:
                l, u = torch.where(s > 0, l.clamp_min(0), l), torch.where(s < 0, u.clamp_max(0), u)
        elif t == "relu":
            l, u = l.clamp_min(0), u.clamp_min(0)
        elif t == "add":
            l2, u2 = box[op.inputs[1]]
            l, u = l + l2, u + u2
        else:
            l, u = l.flatten(1), u.flatten(1)
        box[op.outputs[0]] = (l, u)
    return box


def _backward(ops, params, box, C, out, x, lo, hi, lower, ball="linf", eps=0.0, alpha=None, add=None):
    """One CROWN bound of C against value ``out``: rows [B, S, n] pushed back to the input."""
    B, S = C.shape[:2]
    M = B * S
    adj = {out: C.reshape(M, -1)}
    b = torch.zeros(M, dtype=C.dtype, device=C.device)
    per_row = lambda v: v.reshape(B, -1).repeat_interleave(S, dim=0)   # noqa: E731

    def give(name, a):
        adj[name] = adj[name] + a if name in adj else a

    for op in reversed(ops):
        a = adj.pop(op.outputs[0], None)
        if a is None:
            continue
        src, t = op.inputs[0], op.op_type
        if t == "linear":
            b = b + a @ params[op.inputs[2]]
            give(src, a @ params[op.inputs[1]])
        elif t == "conv2d":
            w = params[op.inputs[1]]
            rows = a.reshape((M,) + tuple(box[op.outputs[0]][0].shape[1:]))
            b = b + rows.sum(dim=(2, 3)) @ params[op.inputs[2]]
            g = torch.nn.grad.conv2d_input((M,) + tuple(box[src][0].shape[1:]), w, rows, stride=op.attrs["stride"],
                                           padding=op.attrs["padding"])
            give(src, g.reshape(M, -1))
        elif t == "relu":
            l, u = box[src]
            pos, neg = l >= 0, u <= 0
            chord = u / (u - l).clamp_min(EPS_F32)
            amb = ~(pos | neg)
            au = torch.where(amb, chord, (pos & ~neg).to(l.dtype))
            bu = torch.where(amb, -l * chord, torch.zeros_like(l))
            low = torch.zeros_like(l) if alpha is None else alpha[src].reshape(l.shape).clamp(0, 1)
            al = torch.where(amb, low, (pos & ~neg).to(l.dtype))
            au, bu, al = per_row(au), per_row(bu), per_row(al)
            take_u = (a < 0) if lower else (a >= 0)
            b = b + torch.where(take_u, a * bu, torch.zeros_like(a)).sum(dim=1)
            a = a * torch.where(take_u, au, al)
            if add is not None and src in add:
                a = a + per_row(add[src])
            give(src, a)
        elif t == "add":
            give(op.inputs[0], a)
            give(op.inputs[1], a)
        else:
            give(src, a)
    a = adj["input"]
    mid, rad = per_row((lo + hi) / 2), per_row((hi - lo) / 2)
    if ball == "l2":
        mid = per_row(x)
        spread = eps * a.norm(dim=1)
    else:
        spread = (a.abs() * rad).sum(dim=1)
    v = (a * mid).sum(dim=1) + b
    return (v - spread if lower else v + spread).reshape(B, S)


def exact(case: dict, seed: int):
    if case["entry"] in ("alpha", "bab"):
        return None        # the end of an optimisation has no exact value: its branches depend on rounding
    g = _inputs(case, seed, torch.device("cuda:0"))
    d = lambda t: t.double()   # noqa: E731
    if case["entry"] == "region":
        sel = lambda A, p, q: torch.where(A >= 0, d(p)[:, None, :], d(q)[:, None, :])   # noqa: E731
        W, bias, out = d(g["weight"]), d(g["bias"]), {}
        for side, (p, q) in (("u", ("u", "l")), ("l", ("l", "u"))):
            A = d(g["A_" + side])
            relaxed = A * sel(A, g["alpha_" + p], g["alpha_" + q])
            out["b_" + side] = (A * sel(A, g["beta_" + p], g["beta_" + q])).sum(-1) + relaxed @ bias
            out["A_" + side] = relaxed @ W
        return out
    # convolutions in 64 bits run on the host
    to = (lambda t: t.double()) if case["net"] in ("mlp", "resmlp") else (lambda t: t.double().cpu())
    spec = _spec(case, g["x"])
    ops, params, C = g["ops"], {n: to(p) for n, p in g["params"].items()}, to(g["C"])
    x, eps, ball = to(spec.center), _eps(case), case["ball"]
    if ball == "box":
        lo, hi = to(spec.perturbation.lower), to(spec.perturbation.upper)
    else:
        lo, hi = x - eps, x + eps
    splits = None
    if g.get("splits") is not None:
        splits = {n: to(s) for n, s in g["splits"].items()}
    box = _ibp(ops, params, x, lo, hi, ball, eps, splits)
    if case["entry"] == "ibp":
        return {"lower": box["out"][0], "upper": box["out"][1]}

    def bound(C, out, lower, **more):
        # a few domains at a time where a row is long
        step = max(1, (1 << 27) // (C.shape[1] * max(int(v[0][0].numel()) for v in box.values())))
        parts = []
        for i in range(0, C.shape[0], step):
            at = slice(i, i + step)
            cut = {k: {n: v[at] for n, v in m.items()} for k, m in more.items()}
            parts.append(_backward(ops, params, {n: (l[at], u[at]) for n, (l, u) in box.items()}, C[at], out, x[at],
                                   lo[at], hi[at], lower, ball, eps, **cut))
        return torch.cat(parts)

    if case["entry"] == "grad":
        # (the gradients jump where a coefficient crosses zero, so single elements have no number that
        # another rounding would give again)
        add = {n: -d(g["beta"][n]) * s for n, s in splits.items()}
        alpha = {n: d(v) for n, v in g["alpha"].items()}
        return {"lower": bound(C, "out", True, alpha=alpha, add=add), "upper": bound(C, "out", False, alpha=alpha),
                "alpha": None, "beta": None}
    if case["entry"] == "crown_all":
        names = [op.inputs[0] for op in ops if op.op_type == "relu"]
        # (up to the third ReLU: what follows also hangs on which refined bounds rounding puts past zero)
        known = names[:3]
        for n in known[1:]:
            w = box[n][0].shape[1]
            eye = torch.eye(w, dtype=C.dtype, device=C.device).expand(x.shape[0], w, w)
            l, u = bound(eye, n, True), bound(eye, n, False)
            box[n] = (torch.maximum(box[n][0], l), torch.minimum(box[n][1], u))
        return {"lower": None, "upper": None, "pre_lower": [box[n][0] if n in known else None for n in names],
                "pre_upper": [box[n][1] if n in known else None for n in names]}
    return {"lower": bound(C, "out", True), "upper": bound(C, "out", False)}
