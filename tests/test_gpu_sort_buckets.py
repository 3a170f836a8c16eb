"""The splitter merge of wide rows: the bins of a bucket and their fallback to
the radix sort, at the edges of the row lengths that choose chunks, samples and
bucket sizes, against the oracle bit for bit."""
import numpy as np
import pytest
import torch

from gpu_util import bits, to_dev
from oracle import tallax_oracle as O

pytestmark = pytest.mark.gpu


def _row(rng, cols, kind):
    if kind == "probs":
        z = np.exp(rng.standard_normal(cols) * 2)
        return (z / z.sum()).astype(np.float32)
    if kind == "normal":       # both signs: the bucket around zero spans many exponents
        return rng.standard_normal(cols).astype(np.float32)
    if kind == "bunched":      # most keys in a small part of every bucket's range: radix sort
        x = rng.standard_normal(cols) * 1e-3
        x[::97] = rng.standard_normal(x[::97].size) * 1e30
        x[::7] = 0.0
        return (1.0 + x).astype(np.float32)
    if kind == "ties":         # few values: no bins
        return rng.integers(0, 5, cols).astype(np.float32)
    if kind == "sorted":       # every bucket lies in one run
        return np.sort(rng.standard_normal(cols)).astype(np.float32)
    x = rng.standard_normal(cols).astype(np.float32)   # special
    u = rng.random(cols)
    x[u < 0.2] = np.nan
    x[(u >= 0.2) & (u < 0.3)] = np.inf
    x[(u >= 0.3) & (u < 0.5)] = -0.0
    return x


KINDS = ["probs", "normal", "bunched", "ties", "sorted", "special"]


# the first row past two whole chunks, a run of one record, the longest row of
# fine samples and the first of coarse ones, the first of 25 whole chunks
@pytest.mark.parametrize("cols", [32769, 40961, 65536, 131071, 262144, 262145, 393217])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("descending,stable", [(False, True), (True, True), (True, False)])
def test_bucket_sort(gpu, cols, dtype, descending, stable):
    from tallax_amd import tax
    print(f"bucket sort {dtype} cols={cols} desc={descending} stable={stable}", flush=True)
    rng = np.random.default_rng(cols + descending)
    x = np.stack([_row(rng, cols, k) for k in KINDS])
    got = tax.sort(to_dev(x, dtype, gpu), num_keys=1, is_stable=stable, return_argsort=True, descending=descending)
    want, _ = O.sort([O.round_to_dtype(x, dtype)], 1, is_stable=stable, return_argsort=True, descending=descending,
                     dtypes=[dtype])
    assert np.array_equal(got[1].cpu().numpy(), want[1])
    assert np.array_equal(bits(got[0].float().cpu().numpy()), bits(want[0]))


@pytest.mark.parametrize("rows", [1, 40])   # smaller buckets for few rows
@pytest.mark.parametrize("descending", [False, True])
def test_bucket_sort_int_and_second_key(gpu, rows, descending):
    from tallax_amd import tax
    rng = np.random.default_rng(rows)
    cols = 50257
    a = rng.integers(0, 64, (rows, cols)).astype(np.int32)
    b = rng.integers(-2**31, 2**31, (rows, cols), dtype=np.int64).astype(np.int32)
    da, db = torch.from_numpy(a).to(gpu), torch.from_numpy(b).to(gpu)
    got = tax.sort([da, db], num_keys=2, return_argsort=True, descending=descending)
    want, _ = O.sort([a, b], 2, return_argsort=True, descending=descending, dtypes=["i32", "i32"])
    for g, w in zip(got, want):
        assert np.array_equal(g.cpu().numpy(), w)
    got = tax.sort(db, num_keys=1, return_argsort=True, descending=descending)
    want, _ = O.sort([b], 1, return_argsort=True, descending=descending, dtypes=["i32"])
    for g, w in zip(got, want):
        assert np.array_equal(g.cpu().numpy(), w)
