"""The relaxation pass over rows whose length is no multiple of four and that come many to a domain
(each lane keeps its domain's operands over 16 rows): against float64, on one lane's worth of columns
past and short of a register of them, a shared coefficient and one per domain, either bound alone."""

import pytest
import torch

from boundflow_amd import _lib
from tests.gpu_util import announce, device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,S,K,shared,sides", [(64, 16, 63, True, "ul"), (61, 17, 65, False, "ul"), (40, 50, 50, True, "l"),
                                                (70, 16, 129, False, "u"), (30, 35, 257, True, "ul"), (33, 33, 510, False, "ul")])
@pytest.mark.parametrize("extras", [True, False])
def test_many_rows_per_domain_match_fp64(D, S, K, shared, sides, extras):
    dev = device()
    M = D * S
    announce(f"relaxation pass D={D} S={S} K={K} shared={shared} sides={sides} extras={extras}")
    g = torch.Generator().manual_seed(D + 3 * S + 7 * K + extras)
    A = {q: torch.randn(S if shared else M, K, generator=g) for q in sides}
    lo = torch.randn(D, K, generator=g)
    hi = lo + torch.rand(D, K, generator=g) * 2
    alpha = torch.rand(D, K, generator=g) if extras else None
    add = torch.randn(D, K, generator=g) if extras else None
    cen = torch.randn(D, K, generator=g) if extras else None
    bias, b0 = torch.randn(K, generator=g), torch.randn(M, generator=g)
    table = torch.empty(D, K, 4, device=dev)
    d = lambda t: None if t is None else t.to(dev)   # noqa: E731
    lo_d, hi_d, al_d, add_d, cen_d, bias_d, b0_d = (d(t) for t in (lo, hi, alpha, add, cen, bias, b0))
    _lib.call("bf_relu_relax_table", _lib.ptr(lo_d), _lib.ptr(hi_d), _lib.ptr(al_d), K, D, K, _lib.ptr(table),
              _lib.stream_handle())
    A_d = {q: d(A[q]) for q in sides}
    out = {q: torch.empty(M, K, device=dev) for q in sides}
    bo = {q: torch.empty(M, device=dev) for q in sides}
    co = {q: torch.empty(M, device=dev) for q in sides} if extras else {}
    p = lambda m, q: _lib.ptr(m.get(q))   # noqa: E731
    _lib.call("bf_crown_relu_relax_lu", p(A_d, "u"), p(A_d, "l"), 0 if shared else S * K, D, S, K, _lib.ptr(lo_d),
              _lib.ptr(hi_d), _lib.ptr(al_d), K, _lib.ptr(add_d), K, _lib.ptr(bias_d), _lib.ptr(cen_d), _lib.ptr(b0_d),
              _lib.ptr(b0_d), p(out, "u"), p(out, "l"), p(bo, "u"), p(bo, "l"), p(co, "u"), p(co, "l"),
              _lib.stream_handle())
    torch.cuda.synchronize()
    dom = torch.arange(M) // S
    tab = table.cpu().double()[dom]
    for q in sides:
        a = (A[q].repeat(D, 1) if shared else A[q]).double()
        take_u = a < 0 if q == "l" else a >= 0
        nxt = a * torch.where(take_u, tab[..., 0], tab[..., 2])
        beta = a * torch.where(take_u, tab[..., 1], tab[..., 3])
        if q == "l" and extras:
            nxt = nxt + add.double()[dom]
        err = (out[q].cpu().double() - nxt).abs()
        assert bool((err <= 2.0 ** -22 * (nxt.abs() + (add.double().abs()[dom] if extras else 0.0)) + 1e-30).all())
        sums = [(bo[q], b0.double() + beta.sum(1) + (nxt * bias.double()).sum(1),
                 b0.double().abs() + beta.abs().sum(1) + (nxt * bias.double()).abs().sum(1))]
        if extras:
            sums.append((co[q], (nxt * cen.double()[dom]).sum(1), (nxt * cen.double()[dom]).abs().sum(1)))
        for got, want, size in sums:
            err = (got.cpu().double() - want).abs()
            assert bool((err <= (K + 8) * 2.0 ** -23 * size + 1e-30).all()), float((err / size).max())


@pytest.mark.parametrize("D,S,K,sides", [(1, 1, 1, "ul"), (3, 5, 20, "ul"), (2, 7, 255, "l"), (4, 9, 256, "ul"),
                                         (2, 3, 516, "u"), (1030, 9, 64, "ul"), (70, 16, 63, "ul")])
@pytest.mark.parametrize("one", [True, False])
def test_sum_of_two_coefficients_matches_the_summed_one(D, S, K, sides, one):
    """The pass that adds a second coefficient and its bias rows as it reads them: the coefficients bit
    for bit those of the pass over the sum, the bias rows within the rounding of their own sums; one
    tensor for both bounds and one each."""
    dev = device()
    M = D * S
    announce(f"relaxation of a sum D={D} S={S} K={K} sides={sides} one={one}")
    g = torch.Generator().manual_seed(D + 3 * S + 7 * K + one)
    r = lambda *shape: torch.randn(*shape, generator=g).to(dev)   # noqa: E731
    A, A2, b, b2 = ({q: r(M, *cols) for q in sides} for cols in ((K,), (K,), (), ()))
    if one:
        A, A2 = ({q: m[sides[0]] for q in sides} for m in (A, A2))
    lo, kbias, alpha = r(D, K), r(K), torch.rand(D, K, generator=g).to(dev)
    hi = lo + torch.rand(D, K, generator=g).to(dev) * 2
    out, want = ({q: torch.empty(M, K, device=dev) for q in sides} for _ in range(2))
    bo, bw = ({q: torch.empty(M, device=dev) for q in sides} for _ in range(2))
    p = lambda m, q: _lib.ptr(m.get(q))   # noqa: E731
    tail = (_lib.ptr(lo), _lib.ptr(hi), _lib.ptr(alpha), K, None, 0, _lib.ptr(kbias))
    _lib.call("bf_crown_relu_relax_sum_lu", p(A, "u"), p(A, "l"), p(A2, "u"), p(A2, "l"), D, S, K, *tail, p(b, "u"),
              p(b, "l"), p(b2, "u"), p(b2, "l"), p(out, "u"), p(out, "l"), p(bo, "u"), p(bo, "l"), _lib.stream_handle())
    added, b_added = {q: A[q] + A2[q] for q in sides}, {q: b[q] + b2[q] for q in sides}
    _lib.call("bf_crown_relu_relax_lu", p(added, "u"), p(added, "l"), S * K, D, S, K, *tail, None, p(b_added, "u"),
              p(b_added, "l"), p(want, "u"), p(want, "l"), p(bw, "u"), p(bw, "l"), None, None, _lib.stream_handle())
    torch.cuda.synchronize()
    for q in sides:
        assert torch.equal(out[q], want[q])
        # |beta| <= |A'| |lower|-like terms: both sides sum the same addends, in another order at most
        size = b[q].abs() + b2[q].abs() + (added[q].abs() * (kbias.abs() + 3 * (1 + lo.abs().repeat_interleave(S, 0)))).sum(1)
        assert bool(((bo[q] - bw[q]).abs() <= 2 * (K + 8) * 2.0 ** -24 * size).all())


@pytest.mark.parametrize("D,S,K,sides", [(3, 5, 20, "ul"), (2, 7, 255, "l"), (4, 9, 256, "u"), (2, 3, 1028, "ul")])
@pytest.mark.parametrize("pair", [True, False])
def test_a_second_bias_is_summed_apart(D, S, K, sides, pair):
    """The sums of another bias beside the pass's own, with and without a second coefficient: the other
    outputs keep the bits of the pass without it, its sums those of float64 to their rounding."""
    dev = device()
    M = D * S
    announce(f"relaxation with a second bias D={D} S={S} K={K} sides={sides} pair={pair}")
    g = torch.Generator().manual_seed(D + 3 * S + 7 * K + pair)
    r = lambda *shape: torch.randn(*shape, generator=g).to(dev)   # noqa: E731
    A, b = {q: r(M, K) for q in sides}, {q: r(M) for q in sides}
    A2, b2 = ({q: r(M, K) for q in sides}, {q: r(M) for q in sides}) if pair else ({}, {})
    lo, kbias, kbias2 = r(D, K), r(K), r(K)
    hi = lo + torch.rand(D, K, generator=g).to(dev) * 2
    out, want = ({q: torch.empty(M, K, device=dev) for q in sides} for _ in range(2))
    bo, bw, k2 = ({q: torch.empty(M, device=dev) for q in sides} for _ in range(3))
    p = lambda m, q: _lib.ptr(m.get(q))   # noqa: E731
    box = (_lib.ptr(lo), _lib.ptr(hi), None, 0, None, 0, _lib.ptr(kbias))
    _lib.call("bf_crown_relu_relax_biases_lu", p(A, "u"), p(A, "l"), p(A2, "u"), p(A2, "l"), D, S, K, *box,
              _lib.ptr(kbias2), p(b, "u"), p(b, "l"), p(b2, "u"), p(b2, "l"), p(out, "u"), p(out, "l"), p(bo, "u"),
              p(bo, "l"), p(k2, "u"), p(k2, "l"), _lib.stream_handle())
    rows = (p(want, "u"), p(want, "l"), p(bw, "u"), p(bw, "l"))
    if pair:
        _lib.call("bf_crown_relu_relax_sum_lu", p(A, "u"), p(A, "l"), p(A2, "u"), p(A2, "l"), D, S, K, *box, p(b, "u"),
                  p(b, "l"), p(b2, "u"), p(b2, "l"), *rows, _lib.stream_handle())
    else:
        _lib.call("bf_crown_relu_relax_lu", p(A, "u"), p(A, "l"), S * K, D, S, K, *box, None, p(b, "u"), p(b, "l"),
                  *rows, None, None, _lib.stream_handle())
    torch.cuda.synchronize()
    for q in sides:
        assert torch.equal(out[q], want[q]) and torch.equal(bo[q], bw[q])
        ref = out[q].double() @ kbias2.double()
        size = out[q].double().abs() @ kbias2.double().abs()
        assert bool(((k2[q].double() - ref).abs() <= (K + 8) * 2.0 ** -24 * size).all())
