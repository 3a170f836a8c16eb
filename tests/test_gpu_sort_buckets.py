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


# every instance of the bucket kernel (4096 records, 8192, 16384) and the first
# row past the longest sorted in half chunks, with a second key and a permutation
# to compose; keys that spread over the bins, keys that tie, and bf16 values held
# in f32 (low digits that no key varies in)
@pytest.mark.parametrize("cols", [50257, 229377, 262145, 393217])
@pytest.mark.parametrize("first", ["i32", "ties", "bf16"])
@pytest.mark.parametrize("second", ["f32", "bf16"])
@pytest.mark.parametrize("descending", [False, True])
def test_bucket_sort_two_keys(gpu, cols, first, second, descending):
    from tallax_amd import tax
    print(f"bucket sort two keys cols={cols} {first} {second} desc={descending}", flush=True)
    rng = np.random.default_rng(cols)
    rows = 3
    b = np.round(rng.standard_normal((rows, cols)) * 64).astype(np.float32) / 8
    db, bt = to_dev(b, second, gpu), O.round_to_dtype(b, second)
    if first == "bf16":   # not a packed key: it comes back as float32
        a = rng.standard_normal((rows, cols)).astype(np.float32)
        da, a, dt = to_dev(a, "bf16", gpu), O.round_to_dtype(a, "bf16"), "bf16"
    else:
        lim = 4 if first == "ties" else 2**31 - 1
        a = rng.integers(-lim, lim, (rows, cols), dtype=np.int64).astype(np.int32)
        da, dt = torch.from_numpy(a).to(gpu), "i32"
    got = tax.sort([da, db], num_keys=2, return_argsort=True, descending=descending)
    want, _ = O.sort([a, bt], 2, return_argsort=True, descending=descending, dtypes=[dt, second])
    for g, w in zip(got, want):
        g = g.cpu().numpy() if g.dtype != torch.bfloat16 else g.float().cpu().numpy()
        assert np.array_equal(g if g.dtype == np.int32 else bits(g), w if w.dtype == np.int32 else bits(w))


@pytest.mark.parametrize("cols", [32769, 229376, 229377, 262144, 300001, 393217])
@pytest.mark.parametrize("descending", [False, True])
def test_bucket_sort_coarse_floats(gpu, cols, descending):
    """bf16 values held in float32, of both signs: the low digits are all zeros or
    all ones, and the radix sort skips what no key of a bucket varies in."""
    from tallax_amd import tax
    print(f"bucket sort coarse floats cols={cols} desc={descending}", flush=True)
    x = O.round_to_dtype(np.random.default_rng(cols).standard_normal((3, cols)).astype(np.float32) * 3, "bf16")
    got = tax.sort(torch.from_numpy(x).to(gpu), num_keys=1, is_stable=True, return_argsort=True, descending=descending)
    want, _ = O.sort([x], 1, is_stable=True, return_argsort=True, descending=descending, dtypes=["f32"])
    assert np.array_equal(got[1].cpu().numpy(), want[1])
    assert np.array_equal(bits(got[0].cpu().numpy()), bits(want[0]))
