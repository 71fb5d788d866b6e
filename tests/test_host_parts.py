"""Which weights a query packs, on the CPU: what its backward and its reverse pass read, and no more."""

import os

import pytest
import torch

from boundflow_amd import _lib, crown

pytestmark = [
    pytest.mark.skipif(not _lib.LIB_PATH.exists(), reason="library not built (run python -m boundflow_amd.build)"),
    pytest.mark.skipif(bool(os.environ.get("BOUNDFLOW_GEMM_TILE")), reason="tile forced by the environment")]


def _layers(*dims):
    g = torch.Generator().manual_seed(len(dims))
    return [crown.AffineLayer(kind="linear", op_index=i, in_name=f"a{i}", out_name=f"h{i}", in_shape=(a,),
                              out_shape=(b,), bias=None, weight=torch.randn(b, a, generator=g)) for i, (a, b) in enumerate(zip(dims, dims[1:]))]


# rows, rows per domain, widths.  64800 rows: every contraction on packed parts, the relaxation in the
# epilogue.  2304 of 500 values: the backward's stores are packed, the reverse pass's are split over K.
# 73728 of 128: the relaxation epilogue stays on the fp32 tiles, the reverse pass's store does not.
@pytest.mark.parametrize("M,S,dims,below,reverse", [
    (64800, 9, (784, 256, 256, 256, 10), {0, 1}, {0, 1, 2}), (2304, 9, (784, 500, 500, 500, 10), {1}, set()),
    (73728, 9, (784, 128, 128, 128, 10), {0}, {0, 1, 2})])
@pytest.mark.parametrize("gradient", [False, True])
def test_a_query_packs_what_it_reads(monkeypatch, M, S, dims, below, reverse, gradient):
    asked = []
    monkeypatch.setattr(crown, "weight_parts", lambda w, t, also=(): asked.extend([(w, t), *also]))
    layers = _layers(*dims)
    k = len(layers) - 2   # the last layer is the specs' head
    crown.chain_parts(layers, k, M, S, 1, {"grad_rows": torch.ones(1)} if gradient else {})
    at = {id(layer.weight): i for i, layer in enumerate(layers)}
    got = [{at[id(w)] for w, t in asked if t == side} for side in (False, True)]
    assert got == [below | {k}, reverse if gradient else set()]
