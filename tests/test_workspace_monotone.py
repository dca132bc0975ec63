"""A workspace sized for a program's most stars and bins takes every smaller
call: the sizes never shrink as the counts grow (host arithmetic only)."""
import pytest

from rubix_amd import _lib

# around the steps of the tile and chunk rules: rounds of a sort tile double
# past 512 workgroups, chunks lengthen by one star at multiples of 8 slots
STARS = sorted({0, 1, 63, 64, 65, 1000, 10 ** 6, 10 ** 7}
               | {c * w * k + d for c in (512, 4096, 8192, 14336) for w in (8, 9, 64, 256, 768, 1024)
                  for k in (1, 2) for d in (-1, 0, 1)})


@pytest.mark.parametrize("keys", [1, 49, 2500, 16383, 16384, 40000, 310000])
def test_sort_workspace_never_shrinks(keys):
    L = _lib.load()
    sizes = [L.rbx_spaxel_sort_workspace_size(n, keys) for n in STARS]
    assert all(a <= b for a, b in zip(sizes, sizes[1:]))


@pytest.mark.parametrize("keys", [1, 625, 10000])
def test_cube_workspace_never_shrinks(keys):
    L = _lib.load()
    bins = (1, 50, 1000, 1024, 1025, 2048, 2049, 3721, 4096, 4097, 8192, 9000)
    size = {(n, b): L.rbx_cube_workspace_size(n, keys, b) for n in STARS for b in bins}
    for b in bins:
        row = [size[n, b] for n in STARS]
        assert all(x <= y for x, y in zip(row, row[1:])), b
    for n in STARS:
        row = [size[n, b] for b in bins]
        assert all(x <= y for x, y in zip(row, row[1:])), n
