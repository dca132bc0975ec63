"""GPU: the chunk plan of one workgroup at the edges of its key count (the
segment cube sums every star once whatever plan it takes), the sort of no
stars, and a column spread over its rows."""
import numpy as np
import pytest
import torch

from rubix_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,n_keys", [(1, 1), (5, 1023), (3000, 1024), (3000, 1025), (100_001, 3),
                                      (20_000, 8191), (20_000, 8192), (20_000, 8193)])
def test_segment_sums_count_every_star(n, n_keys):
    rng = np.random.default_rng(n + n_keys)
    ids = rng.integers(0, n_keys, n).astype(np.int32)
    ids[: n // 3] = n_keys - 1  # several chunks of one key
    rows = rng.integers(0, 16, (n, 5)).astype(np.float32)  # exact in float32
    cube = ops.segment_cube(torch.as_tensor(rows, device="cuda"), torch.as_tensor(ids, device="cuda"),
                            n_keys, n_keys)
    ref = np.zeros((n_keys, 5))
    np.add.at(ref, ids, rows.astype(np.float64))
    np.testing.assert_array_equal(cube.cpu().numpy().reshape(n_keys, 5), ref)


def test_sort_of_no_stars():
    perm, srt, off = ops.spaxel_sort(torch.empty(0, dtype=torch.int32, device="cuda"), 7)
    assert perm.numel() == 0 and off.cpu().tolist() == [0] * 8


@pytest.mark.parametrize("n,cols,col", [(0, 3, 2), (1, 1, 0), (257, 3, 0), (1000, 3, 2), (70_001, 4, 1)])
def test_column_rows(n, cols, col):
    v = torch.randn(n, device="cuda")
    want = torch.zeros(n, cols)
    want[:, col] = v.cpu()
    assert torch.equal(ops.column_rows(v, (n, cols), col).cpu(), want)
