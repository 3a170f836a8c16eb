"""cumsum's tile scans at the edges of a tile, of a lane's eight elements, of a
wave's groups and of the dispatch, against the oracle bit for bit."""
import numpy as np
import pytest
import torch

from gpu_util import bits
from oracle import tallax_oracle as O

pytestmark = pytest.mark.gpu

# one workgroup per row: the first lengths past one tile, an eighth more or
# less, a chunk of 64 tiles and one element past it; three launches: rows that
# end inside a lane's eight elements, fewer tiles per row than a wave takes,
# below and above 65536 tiles (one and four groups of tiles per wave)
SHAPES = [(1, 129), (5, 135), (7, 136), (3, 137), (2, 8192), (2, 8193), (40, 16385), (260, 8191),
          (2000, 131), (900, 1030), (2100, 1999), (34000, 250), (129, 65537)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("reverse", [False, True])
def test_cumsum_tiles(gpu, shape, reverse):
    from tallax_amd import tax
    print(f"cumsum tiles {shape} reverse={reverse}", flush=True)
    rng = np.random.default_rng(shape[0] + shape[1])
    x = rng.standard_normal(shape).astype(np.float32)
    x.flat[::53] = -0.0
    got = tax.cumsum(torch.from_numpy(x).to(gpu), 1, reverse=reverse).cpu().numpy()
    assert np.array_equal(bits(got), bits(O.cumsum(x, 1, reverse)))
    xi = rng.integers(-2**31, 2**31, shape, dtype=np.int64).astype(np.int32)   # wraps
    got = tax.cumsum(torch.from_numpy(xi).to(gpu), 1, reverse=reverse).cpu().numpy()
    a = np.flip(xi, 1) if reverse else xi
    r = np.cumsum(a.astype(np.int64), axis=1)
    r = np.flip(r, 1) if reverse else r
    assert np.array_equal(got, (r & 0xFFFFFFFF).astype(np.uint32).view(np.int32))


def test_cumsum_unaligned_view(gpu):
    """A row start that is only 4-byte aligned (a view into a larger buffer)."""
    from tallax_amd import tax
    rng = np.random.default_rng(5)
    buf = torch.from_numpy(rng.standard_normal(3 * 9001 + 1).astype(np.float32)).to(gpu)
    x = buf[1:].view(3, 9001)
    got = tax.cumsum(x, 1).cpu().numpy()
    assert np.array_equal(bits(got), bits(O.cumsum(x.cpu().numpy(), 1)))


# the chain's stretches of 32 totals: one, a partial second, both of a pair of
# stretches and one more, several lines per workgroup, more than one staged block
@pytest.mark.parametrize("shape,axis", [((33 * 8 + 3, 5), 0), ((34 * 8, 5), 0), ((65 * 8 + 1, 700), 0),
                                        ((97 * 8, 1100), 0), ((1, 128 * 4200), 1), ((20000, 129 * 8), 0),
                                        ((1, 128 * 16400), 1)])
@pytest.mark.parametrize("reverse", [False, True])
def test_cumsum_chain_stretches(gpu, shape, axis, reverse):
    from tallax_amd import tax
    print(f"cumsum chain {shape} axis={axis} reverse={reverse}", flush=True)
    rng = np.random.default_rng(shape[0] + shape[1])
    x = rng.standard_normal(shape).astype(np.float32)
    got = tax.cumsum(torch.from_numpy(x).to(gpu), axis, reverse=reverse).cpu().numpy()
    assert np.array_equal(bits(got), bits(O.cumsum(x, axis, reverse)))
