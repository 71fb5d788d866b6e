"""The kept bias maps of a DAG backward, on the CPU with the library's calls left out: a captured
query's maps are remade for their own layer's shape when a bias changes in place."""

import pytest
import torch

from boundflow_amd import _lib, crown
from boundflow_amd import crown_dag as dag
from boundflow_amd.ir import BFTaskModule, BoundTask, TaskKind, TaskOp
from boundflow_amd.spec import InputSpec


@pytest.fixture
def no_calls(monkeypatch):
    monkeypatch.setattr(_lib, "call", lambda name, *args: 0)
    monkeypatch.setattr(_lib, "stream_handle", lambda stream=None: None)


def _net():
    """conv -> relu -> conv read by a relu and an add (so no ReLU pass takes its bias) -> conv -> add ->
    linear; the conv outputs differ in shape."""
    conv = lambda name, x, stride: TaskOp("conv2d", name, [x, "W" + name, "b" + name], ["h" + name],   # noqa: E731
                                          {"stride": stride, "padding": 1})
    ops = [conv("1", "input", 1), TaskOp("relu", "r1", ["h1"], ["a1"]), conv("2", "a1", 2),
           TaskOp("relu", "r2", ["h2"], ["a2"]), conv("3", "a2", 1), TaskOp("add", "add", ["h2", "h3"], ["s"]),
           TaskOp("flatten", "flat", ["s"], ["f"]), TaskOp("linear", "head", ["f", "Wh"], ["out"])]
    g = torch.Generator().manual_seed(7)
    rand = lambda *s: torch.randn(*s, generator=g)   # noqa: E731
    params = {"W1": rand(4, 1, 3, 3), "b1": rand(4), "W2": rand(8, 4, 3, 3), "b2": rand(8), "W3": rand(8, 8, 3, 3),
              "b3": rand(8), "Wh": rand(3, 8 * 4 * 4)}
    task = BoundTask(task_id="t0", kind=TaskKind.INTERVAL_IBP, ops=ops, input_values=["input"], output_values=["out"])
    shapes = {"input": (1, 8, 8), "h1": (4, 8, 8), "a1": (4, 8, 8), "h2": (8, 4, 4), "a2": (8, 4, 4), "h3": (8, 4, 4),
              "s": (8, 4, 4), "f": (128,), "out": (3,)}
    return BFTaskModule(tasks=[task], entry_task_id="t0", bindings={"params": params}), params, shapes


def test_a_kept_conv_bias_map_is_remade_for_its_own_layer(no_calls):
    module, params, shapes = _net()
    B = 2
    spec = InputSpec.linf(value_name="input", center=torch.zeros(B, 1, 8, 8), eps=0.1)
    box = lambda name: dag.IntervalState(lower=-torch.ones(B, *shapes[name]), upper=torch.ones(B, *shapes[name]))  # noqa: E731
    trace = dag.DagTrace(interval_env={}, relu_pre={n: box(n) for n in ("h1", "h2")}, shapes=shapes, batch=B)
    with crown.derived_scope() as memo:
        dag.crown_backward_dag(module, spec, trace)
    kept = {key: entry for key, entry in memo.items() if "bias" in key[0]}
    assert len(kept) == 3                        # h1's in its ReLU's pass, h2's and h3's in passes of their own
    for name in ("b1", "b2", "b3"):
        params[name].add_(1.0)
    assert crown.refresh_scope(memo) == 3
    for key in kept:
        (bias,), _versions, (out, _stream, _event), _make = memo[key]
        Co, Ho, Wo = next(shapes["h" + n[1:]] for n in ("b1", "b2", "b3") if params[n] is bias)
        assert torch.equal(out, bias.reshape(Co, 1, 1).expand(Co, Ho, Wo).reshape(-1))
