"""The batched pair sums of launches with many tiles (GPU): a tile's four runs
on four wavefronts of one workgroup, where fewer tiles take a run per
workgroup.  Same terms, same order: a problem has the same bits in a small
batch and beside a problem of thousands of tiles, at the sizes where runs,
chunks of 64 records, pairs and groups of four end."""
import numpy as np
import pytest

from test_gpu_batch_sums import SIZES, _system

pytestmark = pytest.mark.gpu
MORE = [(64, 255), (65, 256), (66, 257), (259, 260), (515, 96), (1025, 70), (3, 1), (4, 2), (6, 4)]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("transpose,large", [(False, (262200, 9)), (True, (30, 41000))])
def test_bits_do_not_depend_on_the_batch(nnk, precision, transpose, large):
    rng = np.random.default_rng(8)
    sizes = SIZES + MORE
    systems = [_system(nnk, rng, n, q) for n, q in sizes + [large]]
    eps = rng.uniform(0.01, 0.1, len(systems))
    few = nnk.BatchedMobility(systems[:-1], eps[:-1], precision=precision, hipGraph=False)
    many = nnk.BatchedMobility(systems, eps, precision=precision, hipGraph=True)
    for _ in range(2):
        x = rng.standard_normal(many.n)
        y = many.apply(x, transpose=transpose)
        np.testing.assert_array_equal(y[:few.n], few.apply(x[:few.n], transpose=transpose))
        assert np.isfinite(y).all() and (np.abs(y[few.n:]) > 0).any()
