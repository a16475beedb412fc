"""One step of the GMRES orthogonalisation (GPU): slices that end within the
vectors, groups of four vectors per wavefront, and more vectors than one chunk
of coefficients (1,024) holds, against numpy.  Per slice and pass a dot product
has at most n terms, so the coefficients are within n eps |V_j| |w|; a pass
changes an entry by at most (k + n) eps of its terms; two passes leave y
orthogonal to (k + n) eps."""
import ctypes
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


@pytest.mark.parametrize("n,k", [(1, 1), (63, 5), (130, 31), (129, 128), (1500, 33), (20000, 7), (16384, 96),
                                 (16385, 65), (1300, 1023), (1300, 1024), (1300, 1025), (2600, 2100)])
def test_two_passes(nnk, n, k):
    nnk.lib()
    st = ctypes.CDLL(os.path.join(os.path.dirname(nnk.library_path()), "libnnk_selftest.so"))
    d = ctypes.POINTER(ctypes.c_double)
    rng = np.random.default_rng(n + k)
    V = np.linalg.qr(rng.standard_normal((n, k)))[0].T.copy()
    w0 = V.T @ rng.standard_normal(k) + (1e-3 * rng.standard_normal(n) if n > k else 0.0)
    m1 = k + 3
    w, y, hc = w0.copy(), np.full(n, 7.0), np.full(2 * m1 + 1, 7.0)
    assert st.nnk_selftest_cgs2(ctypes.c_int64(n), k, m1, V.ctypes.data_as(d), w.ctypes.data_as(d),
                                y.ctypes.data_as(d), hc.ctypes.data_as(d)) == 0
    scale = np.linalg.norm(w0)
    assert (np.abs(hc[:k] - V @ w0) <= n * EPS * scale).all()
    assert (hc[k:m1] == 7).all() and (hc[m1 + k:2 * m1] == 7).all()      # only the k coefficients of each pass
    ref = w0 - V.T @ hc[:k]
    bound = (k + n) * EPS * (np.abs(w0) + np.abs(V).T @ np.abs(hc[:k]))
    assert (np.abs(hc[m1:m1 + k] - V @ ref) <= n * EPS * np.linalg.norm(ref) + np.abs(V) @ bound).all()
    ref = ref - V.T @ hc[m1:m1 + k]
    assert (np.abs(w - ref) <= 2 * bound).all()
    assert abs(hc[-1] - np.linalg.norm(w)) <= n * EPS * hc[-1]
    if n > k:
        np.testing.assert_allclose(y * hc[-1], w, rtol=4 * EPS, atol=0)
        assert np.abs(V @ y).max() <= (k + n) * EPS
