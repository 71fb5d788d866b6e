"""The contractions on packed weight parts (three bf16 parts per value on the bf16 matrix
cores): every epilogue against float64 at the fp32 contraction's tolerance, on row, column
and K tails of the 128 x 128 tile; the error against float64 beside the fp32 tiles'; operands
that are not finite; and the host-side rule for the shapes they take."""

import os

import pytest
import torch

from boundflow_amd import _lib
from tests.gpu_util import announce, contraction_tol, device

gpu = pytest.mark.gpu


def config(*a):
    return int(_lib.load().bf_gemm_parts_config(*a))


def test_shapes_taken():
    if not _lib.LIB_PATH.exists():
        pytest.skip("library not built (run python -m boundflow_amd.build)")
    if os.environ.get("BOUNDFLOW_GEMM_TILE"):
        pytest.skip("tile forced by the environment")
    tile = lambda *a: chr(config(*a)) if config(*a) else ""   # noqa: E731
    for form in (0, 1, 2):
        assert tile(128000, 500, 500, 500, 2, form) == "P" and tile(36864, 256, 256, 9, 1, form) == "P"
        assert tile(36864, 256, 16, 9, 1, form) == "P" and not tile(36864, 256, 15, 9, 1, form)   # a whole stage
        assert not tile(10 ** 7, 256, 256, 10 ** 6, 1, form)                        # rows past 32-bit offsets
        assert not tile(0, 256, 256, 9, 1, form) and not tile(36864, 256, 256, 9, 3, form)
        assert not tile(36864, 256, 256, 0, 1, form) and not tile(255, 256, 256, 9, 1, form)
    # stores: 64 x 64 below 1536 such tiles, past K = 512 only with one per CU
    assert tile(64 * 1536, 64, 256, 9, 1, 0) == "P" and tile(64 * 1535, 64, 256, 9, 1, 0) == "S"
    assert tile(256, 64, 512, 9, 1, 0) == "S" and not tile(256, 64, 516, 9, 1, 0) and tile(64 * 128, 64, 516, 9, 2, 0) == "S"
    # the norm epilogue's tile is its partial norms' width (64 columns on short grids); the others 128 tiles
    assert tile(576, 784, 256, 9, 2, 1) == "S" and not tile(576, 784, 256, 9, 2, 2)
    assert tile(64 * 128, 128, 256, 9, 2, 1) == "P" and not tile(64 * 128, 128, 256, 9, 1, 1)
    assert tile(128 * 127 + 1, 128, 64, 9, 1, 2) == "P" and not tile(128 * 127, 128, 64, 9, 1, 2)
    assert not config(36864, 256, 256, 9, 1, 3)


@pytest.mark.parametrize("gains,M,N,K,nz,form", [
    # stores: fewer 64 x 64 tiles than CUs, one or two a CU, 128 x 128 tiles
    (True, 2304, 256, 128, 1, 0), (False, 2304, 256, 256, 1, 0), (True, 2304, 256, 500, 1, 0), (False, 2304, 256, 250, 1, 0),
    (True, 4096, 256, 256, 1, 0), (False, 4096, 256, 512, 1, 0), (True, 4096, 256, 500, 1, 0), (True, 8192, 256, 512, 1, 0),
    (False, 2304, 256, 128, 1, 3), (True, 2304, 256, 100, 1, 3), (True, 4096, 256, 256, 1, 3),
    (False, 36864, 256, 64, 1, 0), (True, 36864, 256, 50, 1, 0), (True, 49152, 256, 64, 1, 0), (True, 128000, 500, 500, 2, 0),
    # norms: the 64-column tile, the 128-column one over a few columns
    (True, 288, 784, 64, 2, 1), (False, 288, 784, 96, 2, 1), (True, 288, 784, 100, 2, 1), (True, 100000, 65, 50, 2, 1),
    (False, 100000, 5, 50, 2, 1),
    # relaxation: a second round of workgroups that fills, one that does not
    (False, 9216, 256, 60, 1, 2), (True, 9216, 256, 64, 1, 2), (False, 36864, 256, 256, 1, 2),
    (True, 18432, 500, 500, 1, 2), (False, 36864, 256, 64, 2, 2), (True, 36864, 256, 128, 2, 2),
    (True, 50000, 50, 50, 2, 2), (False, 8192, 256, 50, 1, 2),
    (False, 255, 256, 64, 1, 0), (False, 36864, 256, 256, 3, 0)])
def test_shapes_that_gain(gains, M, N, K, nz, form):
    if not _lib.LIB_PATH.exists():
        pytest.skip("library not built (run python -m boundflow_amd.build)")
    if os.environ.get("BOUNDFLOW_GEMM_TILE"):
        pytest.skip("tile forced by the environment")
    assert bool(_lib.load().bf_gemm_parts_pays(M, N, K, 9, nz, form)) == gains
    assert not gains or config(M, N, K, 9, nz, form % 3)


def pack(W, trans_b):
    n, p = W.shape
    N, K = (n, p) if trans_b else (p, n)
    out = torch.empty(int(_lib.load().bf_gemm_parts_floats(N, K)), device=W.device)
    _lib.call("bf_gemm_pack_parts", 1, _lib.ptr_array([W]), _lib.i64_array([p]), _lib.i32_array([int(trans_b)]),
              _lib.i64_array([N]), _lib.i64_array([K]), _lib.ptr_array([out]), _lib.stream_handle())
    return out


def gen(*key):
    return torch.Generator().manual_seed(sum((i + 1) * int(k) for i, k in enumerate(key)))


# tiles of 128 x 128 and 64 x 64, stages of 16 k: one row past a tile and one short of it, one column
# past a 32-column block and past a tile, K of one to three whole float4s past a stage
@gpu
@pytest.mark.parametrize("M,N,K,S", [(49153, 128, 64, 9), (98303, 127, 68, 16384), (32897, 161, 76, 1),
                                     (32769, 129, 252, 9), (12800, 500, 500, 512), (256, 1, 64, 9), (257, 65, 68, 300),
                                     (575, 97, 508, 9), (2304, 256, 512, 9), (8191, 127, 1028, 1),
                                     # K no multiple of four: rows copied float by float
                                     (49153, 129, 17, 9), (98303, 63, 50, 16384), (257, 65, 31, 300), (2303, 50, 333, 1)])
@pytest.mark.parametrize("trans_b", [True, False])
def test_store_matches_fp64(M, N, K, S, trans_b):
    dev = device()
    announce(f"parts store M={M} N={N} K={K} S={S} trans_b={trans_b}")
    assert config(M, N, K, S, 1, 0)
    g = gen(M, N, K, trans_b)
    A = torch.randn(M, K, generator=g)
    B = torch.randn(N, K, generator=g)
    r, v = torch.randn(M, generator=g), torch.randn(-(-M // S), N, generator=g)
    rv = r.double()[:, None] * v.double()[torch.arange(M) // S]
    W = (B if trans_b else B.t().contiguous()).to(dev)
    Ad, rd, vd = A.to(dev), r.to(dev), v.to(dev)
    ref = A.double() @ B.double().t()
    for rank1 in (False, True):
        C = torch.full((M, N), float("nan"), device=dev)
        _lib.call("bf_gemm_rank1_parts", _lib.ptr(Ad), K, _lib.ptr(pack(W, trans_b)), _lib.ptr(C), N, M, N, K, S,
                  _lib.ptr(rd if rank1 else None), _lib.ptr(vd if rank1 else None), N, _lib.stream_handle())
        torch.cuda.synchronize()
        want = ref + rv if rank1 else ref
        tol = contraction_tol(A, B.t(), K) + (rv.abs() * 2.0 ** -22 if rank1 else 0.0) + 1e-30
        err = (C.cpu().double() - want).abs()
        assert bool((err <= tol).all()), float((err / tol).max())


@gpu
@pytest.mark.parametrize("M,N,K", [(36864, 256, 256), (16384, 129, 500), (2304, 256, 512)])
@pytest.mark.parametrize("positive", [False, True])
def test_error_is_not_above_the_fp32_tiles(M, N, K, positive):
    """Root mean square error against float64, beside that of the fp32 MFMA contraction."""
    dev = device()
    g = torch.Generator(device=dev).manual_seed(M + N + K + positive)
    A, B = torch.randn(M, K, generator=g, device=dev), torch.randn(N, K, generator=g, device=dev)
    if positive:
        A, B = A.abs(), B.abs()
    ref = A.double() @ B.double().t()
    C, C32 = torch.empty(M, N, device=dev), torch.empty(M, N, device=dev)
    _lib.call("bf_gemm_rank1_parts", _lib.ptr(A), K, _lib.ptr(pack(B, True)), _lib.ptr(C), N, M, N, K, 9, None, None,
              0, _lib.stream_handle())
    _lib.call("bf_gemm", _lib.ptr(A), K, _lib.ptr(B), K, 1, 0, _lib.ptr(C32), N, M, N, K, _lib.stream_handle())
    torch.cuda.synchronize()
    err, err32 = (float((c.double() - ref).norm() / ref.norm()) for c in (C, C32))
    announce(f"parts error {err:.3e}, fp32 tiles {err32:.3e} (M={M} N={N} K={K} positive={positive})")
    assert err <= err32


@gpu
@pytest.mark.parametrize("M,N,K", [(36864, 256, 256), (2304, 256, 64), (9216, 97, 50), (2304, 500, 100), (36864, 129, 500)])
@pytest.mark.parametrize("nonzeros", [1, 2, 4, 16])
def test_sparse_rows_are_no_further_off_than_the_fp32_tiles(M, N, K, nonzeros):
    """Rows of few nonzero coefficients (stable-off ReLUs leave such): the fp32 contraction rounds a sum
    once per nonzero.  One product alone is within fp32's own rounding: what is left out of it and the
    rounding of its low sum are below 9 x 2^-33 of it, 2^-6 of half a unit in the last place."""
    dev = device()
    announce(f"parts sparse rows M={M} N={N} K={K} nonzeros={nonzeros}")
    assert config(M, N, K, 9, 1, 0)
    g = torch.Generator(device=dev).manual_seed(M + N + K + nonzeros)
    A, B = torch.randn(M, K, generator=g, device=dev), torch.randn(N, K, generator=g, device=dev)
    at = torch.rand(M, K, generator=g, device=dev).topk(nonzeros, dim=1).indices
    A = A * torch.zeros_like(A).scatter_(1, at, 1.0)
    C, C32 = torch.empty(M, N, device=dev), torch.empty(M, N, device=dev)
    _lib.call("bf_gemm_rank1_parts", _lib.ptr(A), K, _lib.ptr(pack(B, True)), _lib.ptr(C), N, M, N, K, 9, None, None,
              0, _lib.stream_handle())
    _lib.call("bf_gemm", _lib.ptr(A), K, _lib.ptr(B), K, 1, 0, _lib.ptr(C32), N, M, N, K, _lib.stream_handle())
    torch.cuda.synchronize()
    ref = A.double() @ B.double().t()
    err, err32 = (float((c.double() - ref).norm() / ref.norm()) for c in (C, C32))
    announce(f"parts error {err:.4e}, fp32 tiles {err32:.4e}")
    assert err <= err32 * (1 + 2.0 ** -6)
    if nonzeros == 1:
        assert bool(((C.double() - ref).abs() <= 2.0 ** -24 * (1 + 2.0 ** -6) * ref.abs()).all())


@gpu
@pytest.mark.parametrize("D,S,N,P,cvec,extra,bounds", [(1600, 9, 64, 129, True, True, 1), (300, 33, 100, 500, False, False, 2),
                                                       (6000, 3, 128, 160, True, False, 2), (40, 500, 252, 96, True, True, 1),
                                                                  (1000, 50, 50, 50, True, True, 1), (2000, 9, 77, 130, False, False, 2)])
def test_relaxation_epilogue_matches_fp64(D, S, N, P, cvec, extra, bounds):
    """9 and 3 rows per domain: a tile spans 16 domains (entries in LDS) and 44 (read from memory)."""
    dev = device()
    M = D * S
    announce(f"parts relaxation epilogue D={D} S={S} N={N} P={P} cvec={cvec} extra={extra} bounds={bounds}")
    assert config(M, P, N, S, bounds, 2)
    g = gen(D, S, N, P)
    W = torch.randn(N, P, generator=g) / N ** 0.5
    lo = torch.randn(D, P, generator=g)
    hi = lo + torch.rand(D, P, generator=g) * 2
    table = torch.empty(D, P, 4, device=dev)
    lo_d, hi_d = lo.to(dev), hi.to(dev)
    _lib.call("bf_relu_relax_table", _lib.ptr(lo_d), _lib.ptr(hi_d), None, 0, D, P, _lib.ptr(table),
              _lib.stream_handle())
    tab = table.cpu().double()[torch.arange(M) // S]
    bias, cen, add = torch.randn(P, generator=g), torch.randn(D, P, generator=g), torch.randn(D, P, generator=g)
    sides = ("l",) if bounds == 1 else ("u", "l")
    A = {q: torch.randn(M, N, generator=g) for q in sides}
    b0 = {q: torch.randn(M, generator=g) for q in sides}
    d = lambda t: t.to(dev)   # noqa: E731
    Ad, bd = {q: d(t) for q, t in A.items()}, {q: d(t) for q, t in b0.items()}
    out = {q: torch.empty(M, P, device=dev) for q in sides}
    pre = torch.empty(M, P, device=dev) if extra else None
    bo = {q: torch.empty(M, device=dev) for q in sides}
    co = {q: torch.empty(M, device=dev) for q in sides} if cvec else {}
    ws = torch.empty(int(_lib.load().bf_crown_relu_linear_relu_fwd_workspace(D, S, P)), device=dev)
    bias_d, cen_d, add_d, Wd = d(bias), d(cen) if cvec else None, d(add) if extra else None, pack(d(W), False)
    p = lambda m, q: _lib.ptr(m.get(q))   # noqa: E731
    _lib.call("bf_crown_linear_relu_fwd_parts", p(Ad, "u"), p(Ad, "l"), S * N, D, S, N, _lib.ptr(Wd), P, p(bd, "u"),
              p(bd, "l"), _lib.ptr(table), _lib.ptr(add_d), P, _lib.ptr(bias_d), _lib.ptr(cen_d), P, _lib.ptr(ws),
              p(out, "u"), p(out, "l"), None, _lib.ptr(pre), p(bo, "u"), p(bo, "l"), p(co, "u"), p(co, "l"),
              _lib.stream_handle())
    torch.cuda.synchronize()
    dom = torch.arange(M) // S
    for q in sides:
        C = A[q].double() @ W.double()
        tolC = contraction_tol(A[q], W, N) + 1e-30
        take_u = C < 0 if q == "l" else C >= 0
        nxt = C * torch.where(take_u, tab[..., 0], tab[..., 2])
        beta = C * torch.where(take_u, tab[..., 1], tab[..., 3])
        # a product within rounding of zero may take the other slope: off by its own size
        big = torch.maximum(tab[..., 0], tab[..., 2])
        tol = tolC * 2 * big + 2.0 ** -22 * nxt.abs()
        if q == "l" and extra:
            nxt = nxt + add.double()[dom]
            tol = tol + 2.0 ** -22 * nxt.abs()
            err = (pre.cpu().double() - C).abs()
            assert bool((err <= tolC).all()), float((err / tolC).max())
        err = (out[q].cpu().double() - nxt).abs()
        assert bool((err <= tol).all()), f"{q}: {float((err / tol).max())}"
        tol_b = tolC * 2 * torch.maximum(tab[..., 1], tab[..., 3])
        for got, want, size, room in (
                (bo[q], b0[q].double() + (beta + nxt * bias.double()).sum(1),
                 b0[q].double().abs() + (beta.abs() + (nxt * bias.double()).abs()).sum(1),
                 (tol_b + tol * bias.double().abs()).sum(1)),
                (co.get(q), (nxt * cen.double()[dom]).sum(1), (nxt * cen.double()[dom]).abs().sum(1),
                 (tol * cen.double()[dom].abs()).sum(1))):
            if got is None:
                continue
            err = (got.cpu().double() - want).abs()
            lim = room + (P + 8) * 2.0 ** -24 * size
            assert bool((err <= lim).all()), f"{q} sums: {float((err / lim).max())}"


@gpu
@pytest.mark.parametrize("D,S,N,I,box,norm_p", [(1600, 9, 64, 129, False, 0), (900, 9, 100, 784, True, 0),
                                                (1025, 9, 256, 65, False, 1), (700, 13, 68, 161, False, 2),
                                                (64, 9, 256, 784, True, 0), (29, 9, 64, 65, False, 2),
                                                (400, 50, 50, 5, True, 0), (64, 9, 77, 784, False, 1)])
def test_concretize_matches_fp64(D, S, N, I, box, norm_p):
    dev = device()
    M = D * S
    announce(f"parts concretize D={D} S={S} N={N} I={I} box={box} norm_p={norm_p}")
    assert config(M, I, N, S, 2, 1)
    g = gen(D, S, N, I)
    A = {q: torch.randn(M, N, generator=g) for q in "ul"}
    W = torch.randn(N, I, generator=g) * 0.1
    rad = torch.rand(D, I, generator=g) if box else None
    w64 = rad.double()[torch.arange(M) // S] if box else torch.ones(M, I, dtype=torch.float64)
    cen, b = {q: torch.randn(M, generator=g) for q in "ul"}, {q: torch.randn(M, generator=g) for q in "ul"}
    hs = torch.randn(M, generator=g)
    eps = 1.0 if box else 0.05
    d = lambda t: None if t is None else t.to(dev)   # noqa: E731
    dA, dc, db, drad, dhs = {q: d(A[q]) for q in "ul"}, {q: d(cen[q]) for q in "ul"}, {q: d(b[q]) for q in "ul"}, d(rad), d(hs)
    ws = torch.empty(int(_lib.load().bf_crown_linear_concretize_workspace(D, S, I)), device=dev)
    got = {q: torch.empty(M, device=dev) for q in "ul"}
    h = torch.empty(M, I, device=dev)
    Wd = pack(d(W), False)
    _lib.call("bf_crown_linear_concretize_parts", _lib.ptr(dA["u"]), _lib.ptr(dA["l"]), S * N, D, S, N, _lib.ptr(Wd), I,
              _lib.ptr(drad), eps, norm_p, _lib.ptr(dc["u"]), _lib.ptr(dc["l"]), _lib.ptr(db["u"]), _lib.ptr(db["l"]),
              _lib.ptr(dhs), _lib.ptr(h), _lib.ptr(ws), _lib.ptr(got["l"]), _lib.ptr(got["u"]), _lib.stream_handle())
    torch.cuda.synchronize()
    for q, sign in (("u", 1.0), ("l", -1.0)):
        C = A[q].double() @ W.double()
        tolC = contraction_tol(A[q], W, N)
        norm = {0: (C.abs() * w64).sum(1), 1: C.abs().max(1).values, 2: C.norm(dim=1)}[norm_p]
        room = {0: (tolC * w64).sum(1), 1: tolC.max(1).values, 2: tolC.norm(dim=1)}[norm_p]
        want = cen[q].double() + sign * eps * norm + b[q].double()
        tol = eps * (room + I * 2.0 ** -23 * norm) + 2.0 ** -22 * (cen[q].double().abs() + b[q].double().abs() + eps * norm)
        err = (got[q].cpu().double() - want).abs()
        assert bool((err <= tol).all()), f"{q}: {float((err / tol).max())}"
        if q == "l" and norm_p == 0:
            sure = C.abs() > tolC
            seed = hs.double()[:, None] * torch.sign(C) * w64
            assert torch.equal(h.cpu().double()[sure], seed[sure].float().double())


@gpu
@pytest.mark.parametrize("M,N,K", [(65536, 128, 68), (9100, 128, 68), (9100, 128, 69)])   # both tiles, both copies
def test_operands_that_are_not_finite(M, N, K):
    """Infinities, NaN and values between the largest bf16 and the largest fp32 give what the fp32
    contraction gives, and leave every other row and column alone."""
    dev = device()
    g = gen(M, N, K)
    A = torch.randn(M, K, generator=g)
    B = torch.randn(N, K, generator=g)
    A[5, 3], A[300, 66], A[5000, 0], A[9000, K - 1] = float("inf"), float("nan"), 3.4e38, -float("inf")
    B[7, 2], B[40, K - 1], B[100, 1] = float("inf"), float("nan"), -3.4e38
    Ad, Bd = A.to(dev), B.to(dev)
    C, C32 = torch.empty(M, N, device=dev), torch.empty(M, N, device=dev)
    _lib.call("bf_gemm_rank1_parts", _lib.ptr(Ad), K, _lib.ptr(pack(Bd, True)), _lib.ptr(C), N, M, N, K, 9, None, None,
              0, _lib.stream_handle())
    _lib.call("bf_gemm", _lib.ptr(Ad), K, _lib.ptr(Bd), K, 1, 0, _lib.ptr(C32), N, M, N, K, _lib.stream_handle())
    torch.cuda.synchronize()
    got, want = C.cpu(), C32.cpu()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(torch.isinf(got), torch.isinf(want)) and torch.equal(got[torch.isinf(got)], want[torch.isinf(want)])
    fine = torch.isfinite(want)
    room = 2 * contraction_tol(A, B.t(), K)
    room = torch.where(torch.isfinite(room), room, torch.zeros_like(room))
    plain = fine & (room > 0) & (want.abs() < 1e30)
    err = (got.double() - want.double()).abs()
    assert bool((err[plain] <= room[plain]).all())
    rest = fine & ~plain
    assert bool((err[rest] <= 1e-4 * want.double().abs()[rest]).all())


# powers of two on A and on B: subnormal values and those whose third bf16 part would be, on either side;
# values past 2^103 and sums past 2^79, which the tiles compute again
@gpu
@pytest.mark.parametrize("a_exp,b_exp", [(-118, 100), (-140, 120), (100, -118), (120, -140), (-60, -80), (-110, -16),
                                         (104, -90), (-90, 104), (50, 40), (-126, 102), (123, -146)])
@pytest.mark.parametrize("M,N,K", [(36864, 256, 64), (2304, 97, 50)])   # both tiles, both copies
def test_operands_of_any_size_keep_their_bits(a_exp, b_exp, M, N, K):
    dev = device()
    announce(f"parts operands of 2^{a_exp} and 2^{b_exp} M={M} N={N} K={K}")
    g = gen(M, N, K, abs(a_exp), abs(b_exp))
    scale = lambda t, e: (t.double() * 2.0 ** e).float()   # noqa: E731
    A, B = scale(torch.randn(M, K, generator=g), a_exp), scale(torch.randn(N, K, generator=g), b_exp)
    Ad, Bd = A.to(dev), B.to(dev)
    C, C32 = torch.empty(M, N, device=dev), torch.empty(M, N, device=dev)
    _lib.call("bf_gemm_rank1_parts", _lib.ptr(Ad), K, _lib.ptr(pack(Bd, True)), _lib.ptr(C), N, M, N, K, 9, None, None,
              0, _lib.stream_handle())
    _lib.call("bf_gemm", _lib.ptr(Ad), K, _lib.ptr(Bd), K, 1, 0, _lib.ptr(C32), N, M, N, K, _lib.stream_handle())
    torch.cuda.synchronize()
    # (float64 of the scaled products: past float32's range at either end they would be neither's)
    ref = (A.double() * 2.0 ** -a_exp) @ (B.double() * 2.0 ** -b_exp).t()
    err, err32 = (float((c.cpu().double() * 2.0 ** -(a_exp + b_exp) - ref).norm() / ref.norm()) for c in (C, C32))
    announce(f"parts error {err:.4e}, fp32 tiles {err32:.4e}")
    assert err <= err32 * (1 + 2.0 ** -6)


@gpu
def test_unaligned_rows_and_refused_shapes():
    dev = device()
    g = torch.Generator(device=dev).manual_seed(3)
    A, B = torch.randn(2304 * 64 + 1, generator=g, device=dev), torch.randn(128, 64, generator=g, device=dev)
    W = pack(B, True)

    def run(a, M, K):
        C = torch.empty(M, 128, device=dev)
        _lib.call("bf_gemm_rank1_parts", _lib.ptr(a), K, _lib.ptr(W), _lib.ptr(C), 128, M, 128, K, 9, None, None, 0,
                  _lib.stream_handle())
        return C

    off = A[1:].reshape(2304, 64)                       # one float off 16-byte alignment: the same bits
    assert torch.equal(run(off, 2304, 64), run(off.clone(), 2304, 64))
    with pytest.raises(_lib.HipError):
        run(off, 64, 64)                                # too few rows
