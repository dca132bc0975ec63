"""GPU: the fused forward where knots are denser than bins: 2, 3 or 4 strided
bins per lane at the edges of their axis lengths, windows that just fit and that
do not; cube and gradients against the float64 oracle."""
import pytest

import tests.test_gpu_fused_runs as runs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nt,n_wave,knots", [
    (2, 3000, "linear"), (63, 400, "linear"), (300, 700, "linear"), (512, 1900, "linear"),
    (512, 2600, "log"), (513, 1900, "linear"), (768, 2500, "irregular"), (769, 2500, "linear"),
    (1024, 2600, "linear"), (1025, 2600, "linear"), (1536, 2500, "log"), (1537, 5400, "linear"),
    (2048, 6000, "linear"), (2049, 6000, "linear"), (3072, 5200, "linear"), (3073, 5200, "linear")])
def test_dense_knots_match_oracle(nt, n_wave, knots):
    runs.test_shapes_and_layouts_match_oracle(nt, n_wave, knots, 4700, 8800)
