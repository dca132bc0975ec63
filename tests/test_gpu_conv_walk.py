"""GPU: the convolutions along an axis and their dots at the edges of their
splits: tap counts with and without a register walk, axes shorter than the
kernel, one past a segment or a row item, inner sizes around a wavefront;
against the float64 definition out[x] = sum_t taps[t] in[x + start - t]."""
import numpy as np
import pytest
import torch

from rubix_amd import ops

pytestmark = pytest.mark.gpu


def _ref(x, taps, start):
    n = x.shape[1]
    out = np.zeros(x.shape, np.float64)
    for t, tap in enumerate(taps):
        for o in range(n):
            s = o + start - t
            if 0 <= s < n:
                out[:, o] += tap * x[:, s]
    return out


@pytest.mark.parametrize("m,start", [(1, 0), (3, 1), (8, 3), (11, 5), (15, 7), (15, 0), (15, 14), (25, 12),
                                     (26, 12), (31, 15)])
@pytest.mark.parametrize("n_outer,n_axis,n_inner", [(2, 1, 63), (1, 2, 65), (3, 16, 64), (2, 33, 1),
                                                    (1, 49, 130), (2, 241, 3), (1, 1024, 1),
                                                    (2, 1027, 1), (5, 2051, 1)])
def test_conv_and_dot_match_float64(m, start, n_outer, n_axis, n_inner):
    rng = np.random.default_rng(m * 1000 + n_axis)
    x = rng.normal(size=(n_outer, n_axis, n_inner)).astype(np.float32)
    a = rng.normal(size=x.shape).astype(np.float32)
    taps = rng.normal(size=m)
    dev = "cuda"
    tx, ta = torch.as_tensor(x, device=dev), torch.as_tensor(a, device=dev)
    t32 = torch.as_tensor(taps.astype(np.float32), device=dev)
    got = ops.conv_axis(tx, t32, n_outer, n_axis, n_inner, start).cpu().numpy()
    ref = _ref(x.astype(np.float64), taps.astype(np.float32).astype(np.float64), start)
    # a sum of m float32 products: m rounding errors of the largest partial sum
    bound = 6e-8 * m * (np.abs(taps).sum() * np.abs(x).max() + 1e-30)
    assert np.abs(got - ref).max() <= bound
    dot = float(ops.conv_axis_dot(ta, tx, torch.as_tensor(taps, device=dev), n_outer, n_axis, n_inner,
                                  start))
    terms = a.astype(np.float64) * _ref(x.astype(np.float64), taps, start)
    assert abs(dot - terms.sum()) <= 1e-12 * (np.abs(terms).sum() + 1e-30)


def test_infinities_stay_within_the_kernel():
    """A value outside the kernel's reach does not touch an output, even where
    it is not finite (no product with a padded tap or a value outside)."""
    for m, start in ((15, 7), (25, 12), (26, 12)):
        for n_inner in (1, 64):
            x = torch.zeros(1, 200, n_inner, device="cuda")
            x[:, 100] = float("inf")
            out = ops.conv_axis(x, torch.ones(m, device="cuda"), 1, 200, n_inner, start)[0, :, 0].cpu()
            hit = np.zeros(200, bool)
            lo = 100 - start
            hit[lo:lo + m] = True
            assert bool((torch.isinf(out).numpy() == hit).all()), (m, n_inner)
            assert not bool(torch.isnan(out).any())
