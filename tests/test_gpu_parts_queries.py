"""Packed weights in whole queries: a weight changed in place is packed again (eager and captured), a
launch record times the contraction and not its packing, and the forms of the packed entry points that
single queries seldom take."""

import pytest
import torch

from boundflow_amd import _lib, profiling
from boundflow_amd import alpha_beta as hab
from boundflow_amd import crown as hc
from boundflow_amd import fused_crown as fc
from boundflow_amd import graphs
from boundflow_amd import workloads as wl
from boundflow_amd.spec import InputSpec
from tests.gpu_util import announce, contraction_tol, device
from tests.test_gemm_parts import gen, pack

pytestmark = pytest.mark.gpu


def _mlp(dev, batch, seed=0, dims=(100, 128, 112, 128, 10)):
    g = torch.Generator().manual_seed(seed)
    module = wl.build_mlp(list(dims), gen=g)
    spec = InputSpec.linf(value_name="input", center=torch.rand(batch, dims[0], generator=g), eps=0.02)
    labels = torch.randint(0, dims[-1], (batch,), generator=g)
    return wl.to_device(wl.Workload("mlp", module, spec, wl.margin_spec(labels), labels), dev)


def _grad(wd):
    trace = hc.forward_ibp_trace(wd.module, wd.spec)
    alpha = hab.alpha_from_crown(trace)
    b, ga, _gb = hab.lower_bound_gradients(wd.module, wd.spec, linear_spec_C=wd.C, relu_alpha=alpha)
    return [b.lower, b.upper, *ga.values()]


def _crown(wd):
    b = hc.run_crown_ibp_mlp(wd.module, wd.spec, linear_spec_C=wd.C)
    return [b.lower, b.upper]


def _weights(wd):
    return [p for p in wd.module.params.values() if p.dim() == 2]


def _copy(wd):
    """The same workload with weights of its own, none of them packed yet."""
    fresh = {n: p.clone() for n, p in wd.module.params.items()}
    module = type(wd.module)(tasks=wd.module.tasks, entry_task_id=wd.module.entry_task_id,
                             bindings={"params": fresh}, storage_plan=wd.module.storage_plan)
    return wl.Workload(wd.name, module, wd.spec, wd.C, wd.labels)


# rows of the packed stores alone, and of the relaxation epilogue
@pytest.mark.parametrize("batch", [64, 1200])
@pytest.mark.parametrize("query", [_crown, _grad])
def test_a_weight_changed_in_place_is_packed_again(batch, query):
    dev = device()
    announce(f"packed weights changed in place, batch {batch}, {query.__name__}")
    wd = _mlp(dev, batch)
    before = [t.clone() for t in query(wd)]
    assert any(hc._kept(tag, (w,)) is not None for w in _weights(wd) for tag in hc._PARTS.values())
    for w in _weights(wd):
        w.mul_(1.25)
    got, want = query(wd), query(_copy(wd))
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert not torch.equal(got[0], before[0])


@pytest.mark.parametrize("batch", [64, 1200])
def test_a_captured_query_follows_its_weights(batch):
    dev = device()
    announce(f"captured query on packed weights, batch {batch}")
    wd = _mlp(dev, batch)
    cap = graphs.CapturedQuery(lambda: _crown(wd))
    assert any(key[0] in hc._PARTS.values() for key in cap._derived)
    for rep in range(4):
        out = [t.clone() for t in cap()]
        want = _crown(_copy(wd))       # eager work, and packing, between the replays
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, want)), f"replay {rep}"
        for w in _weights(wd)[rep % 2::2]:
            w.mul_(0.75)


def _region(dev):
    D, S, N, P = 8, 257, 100, 96
    g = torch.Generator().manual_seed(5)
    r = lambda *s: torch.rand(*s, generator=g).to(dev)   # noqa: E731
    req = fc.FusedReluAffineRequest(kind="linear", input_shape=(P,), output_shape=(N,), attrs={}, A_u=r(D, S, N) - 0.5,
                                    A_l=r(D, S, N) - 0.5, alpha_u=r(D, N), alpha_l=r(D, N), beta_u=r(D, N),
                                    beta_l=r(D, N), weight=r(N, P) - 0.5, bias=r(N))
    return fc.HipFusedCrownExecutor().run(req)


@pytest.mark.parametrize("query", ["crown", "crown_large", "grad", "dag", "dag_grad", "region"])
def test_a_launch_record_is_not_its_packing(query, monkeypatch):
    """The first query on fresh weights: no packing call falls to a bracketed launch."""
    dev = device()
    announce(f"launch records of a first query: {query}")
    calls, call = [], _lib.call

    def watch(name, *args):
        calls.append((name, None if profiling._pending is None or profiling._pending[3] else profiling._pending[0]))
        return call(name, *args)

    dag = lambda: wl.to_device(wl.make_dag("residual_mlp", batch=64, n_in=48, hidden=64, blocks=2), dev)   # noqa: E731
    run = {"crown": lambda w: _crown(w), "crown_large": lambda w: _crown(w), "grad": lambda w: _grad(w),
           "dag": lambda w: _crown(w), "dag_grad": lambda w: _grad(w), "region": lambda w: _region(dev)}[query]
    wd = dag() if query.startswith("dag") else _mlp(dev, 1200 if query == "crown_large" else 64)
    monkeypatch.setattr(_lib, "call", watch)
    timer = profiling.LaunchTimer()
    with profiling.timing(timer):
        run(wd)
    torch.cuda.synchronize()
    packs = [pending for name, pending in calls if name == "bf_gemm_pack_parts"]
    assert packs and all(p is None for p in packs), packs
    assert any(name.endswith("_parts") for name in timer.summary())


@pytest.mark.parametrize("stride0", [False, True])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("D,S,N,P", [(64, 40, 100, 129), (700, 9, 50, 64)])
def test_packed_region_without_relaxation(D, S, N, P, bias, stride0):
    """bf_crown_linear_parts with its bias rows, on rows per domain and on rows every domain shares."""
    dev = device()
    M = D * S
    announce(f"bf_crown_linear_parts D={D} S={S} N={N} P={P} bias={bias} stride0={stride0}")
    g = gen(D, S, N, P, bias, stride0)
    rows = S if stride0 else M
    A, W = {q: torch.randn(rows, N, generator=g) for q in "ul"}, torch.randn(N, P, generator=g)
    b_in, bv = {q: torch.randn(M, generator=g) for q in "ul"}, torch.randn(N, generator=g)
    Ad, bd, bvd = {q: t.to(dev) for q, t in A.items()}, {q: t.to(dev) for q, t in b_in.items()}, bv.to(dev)
    out, b_out = {q: torch.empty(M, P, device=dev) for q in "ul"}, {q: torch.empty(M, device=dev) for q in "ul"}
    Wd = pack(W.to(dev), False)
    p = _lib.ptr
    _lib.call("bf_crown_linear_parts", p(Ad["u"]), p(Ad["l"]), 0 if stride0 else S * N, D, S, N, p(Wd), P,
              p(bvd if bias else None), p(bd["u"]), p(bd["l"]), p(out["u"]), p(out["l"]), p(b_out["u"]), p(b_out["l"]),
              _lib.stream_handle())
    torch.cuda.synchronize()
    for q in "ul":
        full = A[q].repeat(D, 1) if stride0 else A[q]
        err = (out[q].cpu().double() - full.double() @ W.double()).abs()
        assert bool((err <= contraction_tol(full, W, N) + 1e-30).all())
        add = full.double() @ bv.double() if bias else torch.zeros(M, dtype=torch.float64)
        size = full.double().abs() @ bv.double().abs() if bias else torch.zeros(M, dtype=torch.float64)
        err = (b_out[q].cpu().double() - (b_in[q].double() + add)).abs()
        # (N + 1 roundings of at most the sum of the terms' sizes)
        assert bool((err <= (N + 1) * 2.0 ** -24 * (size + b_in[q].double().abs()) + 1e-30).all())


def test_several_weights_in_one_launch():
    """More weights than one launch takes (16), of every remainder, both layouts, rows past their end."""
    dev = device()
    announce("packing 19 weights")
    g = gen(19)
    sizes = [(1 + 13 * i, 16 + 7 * (i % 5) + i, i % 2, 3 * (i % 3)) for i in range(19)]   # N, K, layout, row padding
    ws = [(torch.randn(N, K + pad, generator=g) if t else torch.randn(K, N + pad, generator=g)).to(dev)
          for N, K, t, pad in sizes]
    L = _lib.load()
    outs = [torch.full((int(L.bf_gemm_parts_floats(N, K)),), float("nan"), device=dev) for N, K, _t, _p in sizes]
    _lib.call("bf_gemm_pack_parts", len(ws), _lib.ptr_array(ws), _lib.i64_array([w.shape[1] for w in ws]),
              _lib.i32_array([t for _n, _k, t, _p in sizes]), _lib.i64_array([s[0] for s in sizes]),
              _lib.i64_array([s[1] for s in sizes]), _lib.ptr_array(outs), _lib.stream_handle())
    for (N, K, t, _pad), w, out in zip(sizes, ws, outs):
        dense = (w[:, :K] if t else w[:, :N]).contiguous()
        assert torch.equal(out.view(torch.int32), pack(dense, bool(t)).view(torch.int32)), (N, K, t)
