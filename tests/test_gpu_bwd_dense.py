"""GPU: the adjoint where knots are denser than bins (groups of 64 bins searched
among staged records) at the edges of its range: one group, a partial one, an
empty second slab, windows at and past the record space, targets past both grid
ends, uneven knots; cube and gradients against the float64 oracle."""
import pytest

import tests.test_gpu_fused_runs as runs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nt,n_wave,knots,t0,t1", [
    (2, 12, "linear", 4000, 4800), (64, 160, "linear", 4000, 7000), (65, 200, "linear", 4000, 7000),
    (129, 500, "log", 4000, 7000), (300, 560, "linear", 4700, 8800), (400, 590, "irregular", 4700, 8800),
    (700, 2600, "linear", 4700, 8800), (900, 3600, "linear", 4700, 8800),
    (640, 1500, "linear", 2500, 9800), (1921, 2700, "log", 4700, 8800), (3000, 4400, "linear", 4700, 8800)])
def test_dense_adjoint_matches_oracle(nt, n_wave, knots, t0, t1):
    runs.test_shapes_and_layouts_match_oracle(nt, n_wave, knots, t0, t1)
