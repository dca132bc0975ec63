"""GPU: the stable spaxel sort at the edges of the workgroup plan (16 wavefronts
down to 2 as the key counters fill LDS, one wavefront a tile past that; 1 to 16
rounds; stars around a workgroup's tile; radix digits), against numpy's stable
argsort."""
import numpy as np
import pytest
import torch

from rubix_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,n_keys", [
    (1023, 10), (1024, 10), (1025, 10),                     # one workgroup's tile and one past it
    (5000, 2046), (5000, 2047), (5000, 2048),               # 16 and 12 wavefronts, odd and even counters
    (3000, 8191), (3000, 10_922), (3000, 16_382), (3000, 16_383), (3000, 16_384),  # 4, 2 and one wavefront
    (524_288, 100), (524_289, 100), (1_048_577, 100), (5_000_011, 3),  # 1, 2, 4 and 16 rounds
    (20_000_003, 2500), (2_000_003, 120_000),               # many tiles a bucket; radix passes
])
def test_sort_matches_stable_argsort(n, n_keys):
    rng = np.random.default_rng(n + n_keys)
    ids = rng.integers(-1, n_keys + 1, n).astype(np.int32)
    ids[rng.random(n) < 0.3] = n_keys - 1
    perm, srt, off = ops.spaxel_sort(torch.as_tensor(ids, device="cuda"), n_keys)
    bucket = np.where((ids >= 0) & (ids < n_keys), ids, n_keys)
    ref = np.argsort(bucket, kind="stable")
    np.testing.assert_array_equal(perm.cpu().numpy(), ref)
    np.testing.assert_array_equal(srt.cpu().numpy(), ids[ref])
    np.testing.assert_array_equal(off.cpu().numpy(), np.searchsorted(bucket[ref], np.arange(n_keys + 1)))
