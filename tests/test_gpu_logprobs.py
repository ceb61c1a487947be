"""GPU: the split log-probability rows against the one-workgroup form of the same entry, at the
edges of its slices (4096 elements per workgroup, 1024 per wave) and on rows with ties, infinities
and NaN. Picks are equal; log-probabilities differ by the order of float32 sums: each form's sum of
up to 2^19 terms in [0, 1] is a tree of at most 2 * 9 + 148 additions, so within 2^-16 relative."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _one_workgroup(x, tokens, k):
    from mlx_dspark._hip import call, ptr, stream_ptr
    R, V = x.shape
    chosen = torch.empty(R, device=x.device)
    ids = torch.empty((R, max(k, 1)), dtype=torch.int32, device=x.device)
    vals = torch.empty((R, max(k, 1)), device=x.device)
    call("dsk_row_logprobs", ptr(x), x.stride(0), R, V, ptr(tokens), k, ptr(chosen), ptr(ids), ptr(vals),
         stream_ptr())
    return chosen, ids[:, :k], vals[:, :k]


def _split(x, tokens, k):
    from mlx_dspark._hip import call, lib, ptr, stream_ptr
    R, V = x.shape
    chosen = torch.empty(R, device=x.device)
    ids = torch.empty((R, max(k, 1)), dtype=torch.int32, device=x.device)
    vals = torch.empty((R, max(k, 1)), device=x.device)
    need = lib.dsk_row_logprobs_ws_bytes(R, V, k)
    if need == 0:
        return None
    ws = torch.empty(need, dtype=torch.uint8, device=x.device)
    call("dsk_row_logprobs_ws", ptr(x), x.stride(0), R, V, ptr(tokens), k, ptr(chosen), ptr(ids), ptr(vals), ptr(ws),
         need, stream_ptr())
    return chosen, ids[:, :k], vals[:, :k]


@pytest.mark.parametrize("V,k,split", [(1000, 5, False), (1000, 64, False), (4095, 64, False), (32000, 0, False),
                                       (24000, 1, False), (4096, 20, True), (13000, 5, True), (24000, 2, False), (151936, 0, True)])
def test_short_rows_take_one_workgroup(dev, monkeypatch, V, k, split):
    """Rows whose split costs more than it saves keep the single kernel."""
    from mlx_dspark import ops
    names, real = [], ops.call
    monkeypatch.setattr(ops, "call", lambda name, *a: (names.append(name), real(name, *a))[1])
    x = torch.randn(3, V, generator=torch.Generator().manual_seed(V)).to(dev)
    ops.row_logprobs(x, torch.zeros(3, dtype=torch.int32, device=dev), k)
    assert names == ["dsk_row_logprobs_ws" if split else "dsk_row_logprobs"]


@pytest.mark.parametrize("V,k", [(1, 1), (63, 64), (1024, 3), (1025, 64), (4096, 20), (4097, 20), (9000, 0),
                                 (151937, 5), (1 << 19, 2), ((1 << 19) + 1, 2)])
def test_split_rows_equal_one_workgroup(dev, V, k):
    from mlx_dspark import ops
    print(f"logprobs V={V} k={k}", flush=True)
    g = torch.Generator().manual_seed(V + k)
    x = torch.randn(6, V + 3, generator=g) * 4
    x[1] = x[1].round()                     # many ties, across slices
    x[2] = -float("inf")                    # no distribution
    x[3, : V // 2] = -float("inf")          # whole slices masked
    x[4, V // 3] = float("nan")
    x[5, V // 2] = float("inf")
    x = x.to(dev)[:, 1:V + 1]               # rows at odd addresses and strides
    tokens = torch.tensor([0, V - 1, 0, V - 1, 0, V + 9], dtype=torch.int32, device=dev)
    ref, split = _one_workgroup(x, tokens, k), _split(x, tokens, k)
    assert (split is None) == (V > 1 << 19)
    for got in (ops.row_logprobs(x, tokens, k), split or ref):
        for a, b, name in zip(got, ref, ("chosen", "ids", "vals")):
            a, b = a.cpu().numpy(), b.cpu().numpy()
            if name == "ids":
                assert np.array_equal(a, b)
            else:
                np.testing.assert_allclose(a, b, rtol=2.0 ** -16, atol=2.0 ** -16)
