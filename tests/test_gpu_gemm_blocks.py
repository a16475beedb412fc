"""The direct FP64 gather GEMM with as many operator blocks as a job may have
(GPU): the list of a tile's active blocks holds them all, in each launch
shape and in the ordered one.  Bound as in test_gpu_gemm_direct."""
import ctypes
import os

import numpy as np
import pytest

from test_gpu_gemm_direct import EPS, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,nb,widths,ordered", [
    (24, 24, 17, (37,), 0), (24, 20, 512, (5, 40), 0),    # 32 x 16 tiles, eight wavefronts
    (24, 6, 100, (8200,), 0),                             # 48 x 32, four wavefronts
    (24, 6, 33, (65500,), 0),                             # 48 x 128, one
    (24, 24, 17, (37,), 1), (24, 20, 512, (5, 40), 1)])
def test_many_blocks(nnk, M, K, nb, widths, ordered):
    nnk.lib()
    st = ctypes.CDLL(os.path.join(os.path.dirname(nnk.library_path()), "libnnk_selftest.so"))
    c, ref, mod = _run(st, M, K, nb, widths, 1, ordered)
    assert (np.abs(c - ref) <= (nb * K + 8) * EPS * mod).all()
