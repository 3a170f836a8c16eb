"""Rows too long for one workgroup: segments with fewer than 128 eligible
values, and parts of rows that do not divide, against the oracle bit for bit."""
import numpy as np
import pytest
import torch

from gpu_util import bits, from_dev_vals, host_values, to_dev
from oracle import tallax_oracle as O
from test_gpu_select import _make

pytestmark = pytest.mark.gpu


def _check(gpu, rows, cols, k, dtype, kind, threads, segments=None):
    from tallax_amd import _lib, sampling, tax
    print(f"split rows={rows} cols={cols} k={k} {dtype} {kind}", flush=True)
    x = _make(rows, cols, kind, seed=rows * 31 + cols)
    xd, xv = to_dev(x, dtype, gpu), host_values(x, dtype)
    plan = _lib.select_plan(rows, cols, _lib.dtype_code(xd))
    assert plan["threads"] == threads and (segments is None or plan["segments"] == segments), plan
    vals, idx = tax.top_k(xd, k)
    ov, oi = O.top_k(xv, k, dtype)
    assert np.array_equal(idx.cpu().numpy(), oi)
    assert np.array_equal(bits(from_dev_vals(vals)), bits(ov))
    rng = np.random.default_rng(cols)
    temp = rng.uniform(0.5, 1.5, rows).astype(np.float32)
    topk = rng.integers(1, 200, rows).astype(np.int32)
    topp = rng.uniform(0.7, 1.0, rows).astype(np.float32)
    meta = sampling.SamplingMetadata(*(torch.from_numpy(a).to(gpu) for a in (topk, topp, temp)))
    tok = sampling.sample((3, 77), xd, meta).cpu().numpy()
    assert np.array_equal(tok, O.sample((3, 77), xv, topk, topp, temp, dtype=dtype))


# rows of segments: every class of ineligible value fills the list's end, in
# rows whose masked stretches span several segments, aligned or not, and in
# the row's short last segment
@pytest.mark.parametrize("rows,cols,k,dtype,kind", [
    (8, 200003, 128, "f32", "masked_mix"),
    (8, 200003, 64, "f32", "masked_mix"),
    (16, 311299, 128, "bf16", "masked_mix"),
    (9, 155653, 100, "bf16", "masked_mix"),
    (4, 81931, 128, "f32", "nan_heavy"),
    (5, 200003, 128, "f32", "masked5"),
    (6, 155653, 128, "bf16", "special"),
])
def test_segments_with_few_eligible(gpu, rows, cols, k, dtype, kind):
    _check(gpu, rows, cols, k, dtype, kind, 256)


# rows that do not divide: parts of whole vectors with a shorter last one, at
# both ends of the 128..256 part workgroups, misaligned rows among them
@pytest.mark.parametrize("rows,cols,k,dtype,kind,parts", [
    (64, 77827, 128, "f32", "masked_mix", 2),    # the shortest such row
    (64, 151937, 50, "f32", "normal", 2),
    (128, 155623, 128, "f32", "masked_mix", 2),  # parts of 19 vectors per thread
    (44, 220001, 64, "f32", "masked_mix", 3),
    (32, 311233, 100, "f32", "special", 4),
    (64, 155653, 64, "bf16", "masked_mix", 2),
    (70, 200003, 128, "bf16", "tieblock", 2),
    (43, 400003, 50, "bf16", "normal", 3),
])
def test_uneven_parts(gpu, rows, cols, k, dtype, kind, parts):
    _check(gpu, rows, cols, k, dtype, kind, 1024, parts)


# rows whose vectors do not fill the waves that give the bound: their shares of
# the places at a few vectors per wave, a partial wave, and the last short row
@pytest.mark.parametrize("cols,dtype", [(1025, "f32"), (1031, "f32"), (1300, "f32"), (2044, "f32"), (2049, "f32"),
                                        (1025, "bf16"), (1100, "bf16"), (1528, "bf16"), (2050, "bf16"),
                                        (4090, "bf16"), (4097, "bf16")])
@pytest.mark.parametrize("k,kind", [(64, "normal"), (128, "normal"), (128, "masked_mix"), (100, "ints"),
                                    (64, "sorted_desc"), (128, "special")])
def test_bound_of_short_rows(gpu, cols, dtype, k, kind):
    _check(gpu, 40, cols, k, dtype, kind, 1024, 1)


# a last segment of a handful of elements, fewer than a list holds: nothing
# ineligible in it, or all of it
@pytest.mark.parametrize("rows,cols,dtype", [(4, 77827, "f32"), (2, 155653, "f32"), (5, 311299, "f32"),
                                             (3, 155653, "bf16"), (2, 163841, "bf16")])
@pytest.mark.parametrize("kind", ["normal", "masked_mix", "special"])
@pytest.mark.parametrize("tail", [None, np.nan, -np.inf])
def test_short_last_segment(gpu, rows, cols, dtype, kind, tail):
    from tallax_amd import _lib, tax
    print(f"short last segment rows={rows} cols={cols} {dtype} {kind} {tail}", flush=True)
    x = _make(rows, cols, kind, seed=cols)
    if tail is not None:
        x[:, -8:] = tail
    xd, xv = to_dev(x, dtype, gpu), host_values(x, dtype)
    assert _lib.select_plan(rows, cols, _lib.dtype_code(xd))["threads"] == 256
    vals, idx = tax.top_k(xd, 128)
    ov, oi = O.top_k(xv, 128, dtype)
    assert np.array_equal(idx.cpu().numpy(), oi)
    assert np.array_equal(bits(from_dev_vals(vals)), bits(ov))


# whole rows and parts with too many candidates: many elements equal to the
# k-th largest, in the first vectors of the row, in its last ones, everywhere;
# few and many distinct values; candidates staged and not; both zeros; NaNs
def _tied(rows, cols, kind, seed):
    rng = np.random.default_rng(seed)
    if kind == "rounded":
        return np.round(rng.standard_normal((rows, cols)) * 1.5).astype(np.float32)
    if kind == "dense":       # a tenth of the row at the top value
        return (rng.random((rows, cols)) < 0.1).astype(np.float32) + 3
    if kind == "late":        # the ties in the row's last vectors, a few larger ones anywhere
        x = rng.standard_normal((rows, cols)).astype(np.float32)
        x[:, -min(cols, 2500):] = 7.0
        for r in range(rows):
            x[r, rng.choice(cols, min(cols, 40), replace=False)] = 8.0 + rng.integers(0, 3)
        return x
    if kind == "zeros":       # the k-th largest is a zero of either sign, NaNs and infinities about
        x = -np.abs(rng.standard_normal((rows, cols))).astype(np.float32)
        x[rng.random((rows, cols)) < 0.2] = 0.0
        x[rng.random((rows, cols)) < 0.2] = -0.0
        x[rng.random((rows, cols)) < 0.1] = np.nan
        x[:, ::997] = np.inf
        return x
    if kind == "nans":        # vectors of positive NaNs, few or no eligible values
        x = np.full((rows, cols), np.nan, np.float32)
        for r in range(rows - 1):
            x[r, rng.choice(cols, 60, replace=False)] = rng.integers(-2, 3, 60)
            x[r, rng.choice(cols, 10, replace=False)] = -np.inf
        return x
    if kind == "ramp":        # no ties, yet one thread's vectors hold the largest
        x = rng.standard_normal((rows, cols)).astype(np.float32)
        x[:, :min(cols, 4000)] += 50 + np.arange(min(cols, 4000), dtype=np.float32) / 64
        return x
    x = np.full((rows, cols), -5.0, np.float32)   # negative constant
    x[:, cols // 2] = np.finfo(np.float32).min
    return x


@pytest.mark.parametrize("kind", ["rounded", "dense", "late", "zeros", "nans", "ramp", "negconst"])
@pytest.mark.parametrize("cols,dtype", [(1100, "f32"), (8193, "f32"), (40000, "f32"), (77820, "f32"), (151936, "f32"),
                                        (4097, "bf16"), (25000, "bf16"), (65537, "bf16"), (128256, "bf16"),
                                        (155641, "bf16"), (262144, "bf16")])
@pytest.mark.parametrize("k", [50, 128])
def test_raised_threshold(gpu, cols, dtype, kind, k):
    from tallax_amd import _lib, tax
    print(f"raised threshold cols={cols} k={k} {dtype} {kind}", flush=True)
    x = _tied(4, cols, kind, seed=cols + k)
    xd, xv = to_dev(x, dtype, gpu), host_values(x, dtype)
    assert _lib.select_plan(4, cols, _lib.dtype_code(xd))["threads"] == 1024
    vals, idx = tax.top_k(xd, k)
    ov, oi = O.top_k(xv, k, dtype)
    assert np.array_equal(idx.cpu().numpy(), oi)
    assert np.array_equal(bits(from_dev_vals(vals)), bits(ov))
