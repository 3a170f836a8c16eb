"""The wide sampler's single-read path on rows that are not whole aligned
16-byte vectors: both edges of the row, their vectors in one thread, the longest
rows, against the oracle bit for bit."""
import numpy as np
import pytest
import torch

from gpu_util import bits, host_values, to_dev
from oracle import tallax_oracle as O
from test_gpu_select import _make, _sampler_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cols,dtype", [(8193, "bf16"), (16385, "bf16"), (50257, "bf16"), (110978, "bf16"),
                                        (155641, "bf16"), (155649, "bf16"), (4097, "f32"), (47070, "f32"),
                                        (77821, "f32"), (77825, "f32")])
@pytest.mark.parametrize("k,kind", [(1024, "normal"), (300, "special"), (512, "ints"), (1024, "negative")])
def test_wide_edges(gpu, cols, dtype, k, kind):
    from tallax_amd import sampling
    print(f"wide edges cols={cols} {dtype} k={k} {kind}", flush=True)
    x = _make(9, cols, kind, seed=cols + k)   # nine rows: every misalignment
    x[:, 0] = 50.0                            # candidates at both edges
    x[:, -1] = 60.0
    vals, idx = sampling.wide_top_k(to_dev(x, dtype, gpu), k)
    wv, wi = O.top_k(host_values(x, dtype), k, dtype)
    assert np.array_equal(idx.cpu().numpy(), wi)
    assert np.array_equal(bits(vals.cpu().numpy()), bits(wv))


def test_wide_edges_tokens(gpu):
    from tallax_amd import sampling
    x, temp, topk, topp = _sampler_inputs(33, 50257, seed=9)
    meta = sampling.SamplingMetadata(*(torch.from_numpy(a).to(gpu) for a in (topk, topp, temp)))
    key = torch.tensor([5, 6], dtype=torch.int32, device=gpu)
    got = sampling.sample(key, to_dev(x, "bf16", gpu), meta, max_k=1024)
    want = O.sample((5, 6), host_values(x, "bf16"), topk, topp, temp, dtype="bf16", max_k=1024)
    assert np.array_equal(got.cpu().numpy(), want)


# rows that end in the radix select, read as whole aligned vectors: row lengths
# about a workgroup step of 8192 slots, ties at both edges of the row, the row
# before and after full of larger values
@pytest.mark.parametrize("cols,dtype", [(1031, "bf16"), (8185, "bf16"), (8191, "bf16"), (16386, "bf16"),
                                        (200003, "bf16"), (1025, "f32"), (8190, "f32"), (8195, "f32"), (16387, "f32"),
                                        (100001, "f32")])
@pytest.mark.parametrize("k,kind", [(1024, "negative"), (512, "edges"), (700, "const"), (300, "masked5"),
                                    (1000, "nan_heavy")])
def test_wide_edges_radix(gpu, cols, dtype, k, kind):
    from tallax_amd import sampling
    print(f"wide edges radix cols={cols} {dtype} k={k} {kind}", flush=True)
    if kind == "edges":   # more than 2048 ties, the first and last columns among them
        x = -np.abs(np.random.default_rng(cols).standard_normal((9, cols))).astype(np.float32) - 1
        x[:, :min(cols, 1500)] = -0.5
        x[:, -min(cols, 1500):] = -0.5
    else:
        x = _make(9, cols, kind, seed=cols + k)
    x[::2] += 100.0       # every second row lies above its neighbours
    vals, idx = sampling.wide_top_k(to_dev(x, dtype, gpu), k)
    wv, wi = O.top_k(host_values(x, dtype), k, dtype)
    assert np.array_equal(idx.cpu().numpy(), wi)
    assert np.array_equal(bits(vals.cpu().numpy()), bits(wv))
