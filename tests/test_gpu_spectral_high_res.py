"""Whole matvecs in frequency space at the larger surface resolutions (GPU),
where the check-to-equivalent inverses amplify rounding most: the comparison
with the dense class tiles of test_gpu_spectral, at the same bound."""
import pytest

import test_gpu_spectral

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("res", [7, 8, 9, 10])
def test_high_resolutions(nnk, res):
    test_gpu_spectral.test_matvec_matches_dense_translations(nnk, res)
