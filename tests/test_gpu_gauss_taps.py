"""GPU: the one-launch Gaussian taps against the float64 formula, for tap counts
from one to several per thread and float32 / float64 sigmas."""
import numpy as np
import pytest
import torch

from rubix_amd import ops
from rubix_amd.autograd import _norm_gauss

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n,sigma", [(1, 2.0), (2, 0.5), (25, 1.2), (26, 4.0), (256, 30.0), (1001, 90.0)])
def test_gauss_taps_match_float64(n, sigma, dtype):
    x = np.arange(n) - (n - 1) / 2
    s = torch.tensor(sigma, dtype=dtype, device="cuda")
    taps, rev, dtaps = ops.gauss_taps(torch.as_tensor(x, device="cuda"), s)
    g, dg = _norm_gauss(x, float(s))
    # one rounding to float32; the float64 sums differ by their order only
    np.testing.assert_allclose(taps.cpu().numpy(), g, rtol=1.2e-7)
    np.testing.assert_array_equal(rev.cpu().numpy(), taps.cpu().numpy()[::-1])
    np.testing.assert_allclose(dtaps.cpu().numpy(), dg, rtol=1e-11, atol=1e-13 * np.abs(dg).max())
