"""softmax_topk_cumsum on rows whose groups are too few to bound the candidates:
both sides of the rule, ties, misaligned rows, special values."""
import numpy as np
import pytest
import torch

from oracle import tallax_oracle as O

pytestmark = pytest.mark.gpu


def _rows(rng, cols):
    x = (rng.standard_normal((6, cols)) * 3).astype(np.float32)
    x[1] = np.round(x[1])                                  # heavy ties
    x[2] = 0.5                                             # one value
    x[3, rng.random(cols) < 0.7] = -np.inf                 # masked
    x[4] = np.sort(x[4])
    x[5, ::2] = -0.0
    x[5, 1::4] = 0.0
    return x


# groups of 16 elements below, at and above 1.25 k (40941 columns: 2559 groups, the
# last short row at k = 2048; 40942: 2560), rows whose ties overflow the candidate
# pool on both sides; k = cols; short odd rows
@pytest.mark.parametrize("cols,k", [(10926, 1616), (8193, 2048), (16384, 2048), (40959, 2048), (40961, 2048),
                                    (40941, 2048), (40942, 2048), (20461, 1024), (20462, 1024),
                                    (2048, 2048), (517, 300), (1, 1), (33, 2), (5000, 256)])
def test_short_rows(gpu, cols, k):
    from tallax_amd import prefill
    print(f"prefill short cols={cols} k={k}", flush=True)
    rng = np.random.default_rng(cols + k)
    x = _rows(rng, cols)
    probs, idx, cum, cut = prefill.softmax_topk_cumsum(torch.from_numpy(x).to(gpu), k, 0.9)
    # the k largest logits, ties to the lowest index (-0 == +0)
    order = np.argsort(-(x + 0.0), axis=1, kind="stable")[:, :k]
    assert np.array_equal(idx.cpu().numpy(), order)
    e = np.exp(x.astype(np.float64) - x.max(axis=1, keepdims=True))
    want = np.take_along_axis(e / e.sum(axis=1, keepdims=True), order, 1)
    # float32 softmax: the documented 1e-5 relative of float64
    np.testing.assert_allclose(probs.cpu().numpy(), want, rtol=1e-5, atol=1e-38)
    assert np.array_equal(cum.cpu().numpy().view(np.uint32), O.cumsum(probs.cpu().numpy(), 1).view(np.uint32))
    assert np.array_equal(cut.cpu().numpy(), (cum.cpu().numpy() < np.float32(0.9)).sum(axis=1))
