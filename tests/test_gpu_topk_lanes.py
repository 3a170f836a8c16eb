"""topk_lanes_kernel at the edges of its list lengths, lanes per row, passes and
of its dispatch, against the oracle bit for bit."""
import numpy as np
import pytest
import torch

from gpu_util import bits, from_dev_vals, host_values, to_dev
from oracle import tallax_oracle as O

pytestmark = pytest.mark.gpu

# every count of lanes per row, full and one past it; one pass and several;
# rows of whole 16-byte vectors and not; the largest k of each list and the
# smallest of the next; row counts on both sides of the dispatch's lines
CASES = [
    (4097, 16, 16), (1000, 17, 9), (300, 32, 32), (257, 31, 17), (70, 64, 8), (70, 65, 8), (8192, 64, 9),
    (8191, 64, 9), (33, 128, 8), (4096, 128, 16), (4095, 128, 16), (16384, 128, 32), (16383, 128, 17), (65, 129, 8),
    (9, 256, 16), (8192, 256, 17), (5, 512, 8), (5, 513, 9), (4096, 512, 32), (3, 1024, 8), (3, 1025, 8),
    (2048, 1024, 32), (256, 2048, 16), (257, 2048, 16), (1024, 2048, 32), (1, 2047, 1), (1024, 2049, 8),
    (1023, 2049, 8), (1024, 4096, 32), (1025, 4097, 17), (1024, 8192, 8), (1024, 8191, 16), (1024, 8193, 8),
    (3072, 64, 8), (3071, 64, 8), (3072, 33, 1), (3071, 33, 1), (512, 65, 8), (511, 65, 8), (512, 128, 8), (511, 128, 1),
]


@pytest.mark.parametrize("rows,cols,k", CASES)
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_topk_lanes(gpu, rows, cols, k, dtype):
    from tallax_amd import tax
    print(f"top_k lanes rows={rows} cols={cols} k={k} {dtype}", flush=True)
    rng = np.random.default_rng(rows * 7 + cols + k)
    x = np.round(rng.standard_normal((rows, cols)) * 8).astype(np.float32) / 4  # ties
    fmin = np.float32(-3.3895314e38) if dtype == "bf16" else np.finfo(np.float32).min
    special = np.array([np.nan, -0.0, 0.0, np.inf, -np.inf, fmin, -np.nan], np.float32)
    mask = rng.random((rows, cols)) < 0.1
    x[mask] = rng.choice(special, int(mask.sum()))
    x[::13] = -np.inf                     # rows with nothing admissible
    xv = host_values(x, dtype)
    vals, idx = tax.top_k(to_dev(x, dtype, gpu), k)
    ov, oi = O.top_k(xv, k, dtype)
    assert np.array_equal(idx.cpu().numpy(), oi)
    assert np.array_equal(bits(from_dev_vals(vals)), bits(ov))


def test_topk_lanes_unaligned(gpu):
    """A base that is not 16-byte aligned takes element loads."""
    from tallax_amd import tax
    rng = np.random.default_rng(2)
    buf = torch.from_numpy(rng.standard_normal(500 * 128 + 1).astype(np.float32)).to(gpu)
    x = buf[1:].view(500, 128)
    vals, idx = tax.top_k(x, 8)
    ov, oi = O.top_k(x.cpu().numpy(), 8)
    assert np.array_equal(idx.cpu().numpy(), oi) and np.array_equal(bits(vals.cpu().numpy()), bits(ov))
