"""GPU parity of row sampling on both sides of the few-rows rule (up to four rows the gather pass
finds the threshold buckets itself and rows are cut into up to 64 slices) and of 16 slices per row
(their maxima read a lane each beyond, in turn up to it): tokens and probabilities
bit-identical to the oracle for every truncation, at vocabularies of one slice, of slices that do
not divide, and unaligned ones, with heavy ties and an all-equal row."""

import numpy as np
import pytest
import torch

from oracle import accept as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,V", [(1, 511), (1, 151936), (3, 33001), (4, 40960), (4, 32771), (5, 40960), (17, 9001),
                                 (70, 9001)])
@pytest.mark.parametrize("T,tp,tk", [(1.0, 0.9, 0), (0.7, 1.0, 20), (0.8, 0.95, 50), (1.0, 0.0, 0), (0.5, 1.0, 0)])
def test_sample_rows_few(dev, R, V, T, tp, tk):
    from mlx_dspark.ops import sample_rows
    rng = np.random.default_rng(R * 7 + V)
    logits = (rng.standard_normal((R, V)) * 2).astype(np.float32)
    logits[0] = np.round(logits[0])          # heavy ties
    if R > 1:
        logits[1] = 1.5                      # one bucket holds the whole row
    ref_tok, ref_p = A.sample_rows(logits, T, tp, tk, False, seed=7, offset=3, row0=1)
    pr = torch.full((R, V), -1.0, dtype=torch.float32, device=dev)
    tok, _ = sample_rows(torch.from_numpy(logits).to(dev), T, tp, tk, seed=7, offset=3, row0=1, probs_out=pr)
    torch.cuda.synchronize()
    assert np.array_equal(tok.cpu().numpy(), ref_tok)
    assert np.array_equal(pr.cpu().numpy(), ref_p)
