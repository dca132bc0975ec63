"""GPU: the adjoint pass that gives the transposed convolution and the dot with
the derivative taps together, at the edges of its split (tap counts with and
without a joint pass, kernels off centre, axes shorter than the kernel, one past
a segment or a row item, inner sizes around a wavefront), against the float64
definition conv(x)[o] = sum_t taps[t] x[o + start - t]."""
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from rubix_amd import _lib, ops

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


def _check(got, dot, dot32, a, x, rev, dtaps, start, add):
    m = len(rev)
    ref = _ref(a.astype(np.float64), rev.astype(np.float64), m - 1 - start)
    # a sum of m float32 products: m rounding errors of the largest partial sum
    assert np.abs(got - ref).max() <= 6e-8 * m * np.abs(rev).sum() * np.abs(a).max()
    terms = a.astype(np.float64) * _ref(x.astype(np.float64), dtaps, start)
    size = np.abs(terms).sum() + abs(add)
    assert abs(float(dot) - (terms.sum() + add)) <= 1e-12 * size
    assert abs(float(dot32) - float(dot)) <= 6e-8 * abs(float(dot))


@pytest.mark.parametrize("m,start", [(1, 0), (3, 1), (8, 3), (13, 6), (15, 7), (15, 0), (15, 14), (17, 8),
                                     (25, 12), (31, 15)])
@pytest.mark.parametrize("n_outer,n_axis,n_inner", [(2, 1, 63), (1, 2, 65), (3, 16, 64), (2, 33, 1),
                                                    (1, 49, 130), (2, 241, 3), (1, 1025, 1), (5, 2051, 1)])
def test_axis(m, start, n_outer, n_axis, n_inner):
    rng = np.random.default_rng(m * 1000 + n_axis)
    x = rng.normal(size=(n_outer, n_axis, n_inner)).astype(np.float32)
    a = rng.normal(size=x.shape).astype(np.float32)
    rev, dtaps = rng.normal(size=m).astype(np.float32), rng.normal(size=m)
    t = [torch.as_tensor(v, device="cuda") for v in (a, x, rev, dtaps)]
    for add in (None, 3.25):
        tadd = None if add is None else torch.tensor(add, dtype=torch.float64, device="cuda")
        din, dot, dot32 = ops.conv_axis_bwd(*t, n_outer, n_axis, n_inner, start, add=tadd)
        _check(din.cpu().numpy(), dot, dot32, a, x, rev, dtaps, start, add or 0.0)


@pytest.mark.parametrize("m,start", [(3, 1), (15, 7), (15, 6), (8, 3), (21, 10)])
@pytest.mark.parametrize("axis", [0, 1])
@pytest.mark.parametrize("packed", [True, False])
def test_batch(m, start, axis, packed):
    rng = np.random.default_rng(m + axis)
    nbs, nt = (1, 5, 17), 70
    gap = 0 if packed else 1  # rows of no galaxy in between take the general path
    begin = np.cumsum([0] + [nb * nb + gap for nb in nbs])
    n_rows = int(begin[-1])
    a = rng.normal(size=(n_rows, nt)).astype(np.float32)
    x = rng.normal(size=a.shape).astype(np.float32)
    rev, dtaps = rng.normal(size=m).astype(np.float32), rng.normal(size=m)
    t = [torch.as_tensor(v, device="cuda") for v in (a, x, rev, dtaps)]
    arr = (_lib.RbxGalaxy * len(nbs))()
    for g, nb in enumerate(nbs):
        arr[g].star_begin, arr[g].spaxel_begin, arr[g].nb = g, int(begin[g]), nb
    table = torch.from_numpy(np.frombuffer(bytes(arr), dtype=np.uint8).copy()).to("cuda")
    layout = SimpleNamespace(table=table, n_gal=len(nbs), n_rows=n_rows)
    din, dot, dot32 = ops.conv_batch_bwd(t[0], t[1], layout, axis, t[2], t[3], start)
    got, ref_dot, size = din.cpu().numpy(), 0.0, 0.0
    for g in range(len(nbs)):
        nb = nbs[g]
        sl = slice(begin[g], begin[g] + nb * nb)
        ag, xg = (v[sl].astype(np.float64).reshape(nb, nb, nt) for v in (a, x))
        if axis == 1:
            r = _ref(ag, rev.astype(np.float64), m - 1 - start)
            d = ag * _ref(xg, dtaps, start)
        else:
            r = _ref(ag.swapaxes(0, 1), rev.astype(np.float64), m - 1 - start).swapaxes(0, 1)
            d = ag * _ref(xg.swapaxes(0, 1), dtaps, start).swapaxes(0, 1)
        assert np.abs(got[sl].reshape(nb, nb, nt) - r).max() <= 6e-8 * m * np.abs(rev).sum() * np.abs(a).max()
        ref_dot += d.sum()
        size += np.abs(d).sum()
    assert abs(float(dot) - ref_dot) <= 1e-12 * size
    assert abs(float(dot32) - float(dot)) <= 6e-8 * abs(float(dot))
