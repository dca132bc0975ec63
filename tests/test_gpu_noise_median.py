"""GPU: the median of the flux image and the spaxels that hold it around the
sizes where the selection changes its loads, with ties, one odd value and
values over the whole exponent range; against numpy's stable order."""
import numpy as np
import pytest
import torch

from rubix_amd import _lib

pytestmark = pytest.mark.gpu


def _stats(flux):
    n = len(flux)
    cube = torch.as_tensor(flux.reshape(n, 1), device="cuda")
    sn = torch.full((n,), 2.0, device="cuda")
    f, s2n, out = torch.empty(n, device="cuda"), torch.empty(n, device="cuda"), torch.empty_like(cube)
    st = torch.zeros(16, dtype=torch.uint8, device="cuda")
    _lib.call("rbx_apply_noise", _lib.ptr(cube), n, 1, _lib.ptr(sn), 7, 1, _lib.ptr(f), _lib.ptr(s2n),
              _lib.ptr(st), _lib.ptr(out), _lib.stream_handle(cube.device))
    raw = st.cpu().numpy()
    return raw[:4].view(np.float32)[0], raw[4:16].view(np.int32), s2n.cpu().numpy()


@pytest.mark.parametrize("n", [1, 2, 3, 1023, 1024, 1025, 8193, 16383, 16384, 16385, 90001, 98304])
@pytest.mark.parametrize("kind", ["spread", "close", "ties", "equal"])
def test_median_and_its_spaxels(n, kind):
    rng = np.random.default_rng(n)
    flux = {"spread": lambda: 10.0 ** rng.uniform(-30, 30, n),
            "close": lambda: 1.0 + rng.uniform(0, 1e-3, n),
            "ties": lambda: rng.integers(1, 5, n).astype(float),
            "equal": lambda: np.full(n, 3.5)}[kind]().astype(np.float32)
    order = np.argsort(flux, kind="stable")
    lo, hi = int(order[(n - 1) // 2]), int(order[n // 2])
    median, idx, s2n = _stats(flux)
    want = np.float32((flux[lo] + flux[hi]) * np.float32(0.5))
    assert median == want
    assert list(idx) == [lo, hi, 0]
    np.testing.assert_array_equal(s2n, (np.sqrt(want) / np.float32(2.0)) / np.sqrt(flux))


@pytest.mark.parametrize("n,at", [(5, 4), (16384, 16383), (16385, 16384), (40000, 17)])
@pytest.mark.parametrize("value", [0.0, -1.0, float("nan")])
def test_a_spaxel_without_flux_makes_the_median_zero(n, at, value):
    flux = np.full(n, 2.0, np.float32)
    flux[at] = value
    median, idx, s2n = _stats(flux)
    assert median == 0.0 and list(idx) == [-1, -1, 1] and not s2n.any()


@pytest.mark.parametrize("n_spaxel,nt", [(3, 1), (5, 5), (1, 2049), (2, 4099), (8191, 3), (8192, 6),
                                         (8193, 257)])
def test_rows_of_any_length_and_count(n_spaxel, nt):
    """Noise and adjoint at the edges of the row splits, from the library's own draws."""
    rng = np.random.default_rng(n_spaxel + nt)
    cube = rng.uniform(0.5, 1.5, (n_spaxel, nt)).astype(np.float32)
    g = rng.normal(size=cube.shape).astype(np.float32)
    dev = "cuda"
    tc, tg = torch.as_tensor(cube, device=dev), torch.as_tensor(g, device=dev)
    sn = torch.as_tensor(rng.uniform(1, 9, n_spaxel).astype(np.float32), device=dev)
    z = torch.empty_like(tc)
    h = _lib.stream_handle(tc.device)
    _lib.call("rbx_noise_sample", z.numel(), 11, 0, _lib.ptr(z), h)
    f, s2n = torch.empty(n_spaxel, device=dev), torch.empty(n_spaxel, device=dev)
    out, din = torch.empty_like(tc), torch.empty_like(tc)
    st = torch.zeros(16, dtype=torch.uint8, device=dev)
    ws = torch.empty(8 * n_spaxel, dtype=torch.uint8, device=dev)
    _lib.call("rbx_apply_noise", _lib.ptr(tc), n_spaxel, nt, _lib.ptr(sn), 11, 0, _lib.ptr(f),
              _lib.ptr(s2n), _lib.ptr(st), _lib.ptr(out), h)
    _lib.call("rbx_apply_noise_bwd", _lib.ptr(tc), _lib.ptr(tg), n_spaxel, nt, _lib.ptr(f), _lib.ptr(s2n),
              _lib.ptr(st), 11, 0, _lib.ptr(ws), ws.numel(), _lib.ptr(din), h)
    zz, s = z.cpu().numpy(), s2n.cpu().numpy()
    np.testing.assert_array_equal(out.cpu().numpy(), cube + cube * (zz * s[:, None]))
    F, S, Z, G = (v.astype(np.float64) for v in (f.cpu().numpy(), s, zz, g))
    A = (G * cube.astype(np.float64) * Z).sum(1)
    order = np.argsort(f.cpu().numpy(), kind="stable")
    M = (F[order[(n_spaxel - 1) // 2]] + F[order[n_spaxel // 2]]) * 0.5
    dF = -A * S / (2 * F)
    for k in ((n_spaxel - 1) // 2, n_spaxel // 2):
        dF[order[k]] += 0.5 * (A * S).sum() / (2 * M)
    direct = G * Z * S[:, None]
    ref = G + direct + dF[:, None]
    # float32 roundings of the product, the direct sum, dL/dF and the last sum
    bound = 6e-8 * (2 * np.abs(direct) + np.abs(G + direct) + np.abs(dF)[:, None] + np.abs(ref)) + 1e-30
    # M is stored in float32, and the medians' term is a sum over all rows
    bound += 1e-7 * np.abs(dF)[:, None]
    assert (np.abs(din.cpu().numpy() - ref) <= bound).all()
