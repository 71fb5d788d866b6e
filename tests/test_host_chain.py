"""The chain that ends at an inner pre-activation is the parsed one, cut short."""

import dataclasses

import pytest
import torch

from boundflow_amd import workloads as wl
from boundflow_amd.crown import parse_chain


@pytest.mark.parametrize("arch", ["mlp", "cnn"])
def test_cut_chain_is_the_parsed_one(arch):
    g = torch.Generator().manual_seed(1)
    w = _workload(arch, g)
    full = parse_chain(w.module, w.spec)
    names = list(full.relu_names)
    assert len(names) >= 2
    for name in names:
        want, got = parse_chain(w.module, w.spec, name), full.until(name)
        assert got.relu_names == want.relu_names and got.output_value == want.output_value
        assert len(got.layers) == len(want.layers)
        for a, b in zip(got.layers, want.layers):
            for f in dataclasses.fields(a):
                # (whether a ReLU reads the last layer is the one thing a cut parse does not see)
                if f.name != "relu_input_of_consumer":
                    x, y = getattr(a, f.name), getattr(b, f.name)
                    assert x is y if torch.is_tensor(x) else x == y


def _workload(arch, g):
    from boundflow_amd.ir import BFTaskModule, BoundTask, TaskKind, TaskOp
    from boundflow_amd.spec import InputSpec
    if arch == "mlp":
        x = torch.rand(2, 7, generator=g)
        params = {f"W{i}": torch.randn(5, 7 if i == 0 else 5, generator=g) for i in range(4)}
        ops = []
        cur = "input"
        for i in range(4):
            ops.append(TaskOp("linear", f"l{i}", [cur, f"W{i}"], [f"h{i}"]))
            if i < 3:
                ops.append(TaskOp("relu", f"r{i}", [f"h{i}"], [f"a{i}"]))
            cur = f"a{i}"
        out = "h3"
    else:
        x = torch.rand(2, 1, 6, 6, generator=g)
        params = {"K": torch.randn(2, 1, 3, 3, generator=g), "b": torch.randn(2, generator=g),
                  "W1": torch.randn(5, 72, generator=g), "W2": torch.randn(3, 5, generator=g)}
        ops = [TaskOp("conv2d", "c", ["input", "K", "b"], ["h0"], attrs={"padding": 1}),
               TaskOp("relu", "r0", ["h0"], ["a0"]), TaskOp("flatten", "f", ["a0"], ["f0"]),
               TaskOp("linear", "l1", ["f0", "W1"], ["h1"]), TaskOp("relu", "r1", ["h1"], ["a1"]),
               TaskOp("linear", "l2", ["a1", "W2"], ["out"])]
        out = "out"
    task = BoundTask(task_id="t0", kind=TaskKind.INTERVAL_IBP, ops=ops, input_values=["input"], output_values=[out])
    module = BFTaskModule(tasks=[task], entry_task_id="t0", bindings={"params": params})
    return wl.Workload(arch, module, InputSpec.linf(value_name="input", center=x, eps=0.05), None, torch.zeros(2))
