"""GPU: the fused forward's workgroup shapes and its two bin layouts (runs of
four consecutive bins where knots are sparse, strided bins elsewhere) at the
edges of their ranges: one bin, one past a wavefront's or workgroup class's
bins, targets reaching past both ends of the template grid, bins crossing 2 or
3 segments, irregular knots and bins; cube and gradients against the float64
oracle on the reference's float32 knots."""
import numpy as np
import pytest
import torch

from oracle import ref_torch as RT
from rubix_amd import ops, synthetic as S
from rubix_amd.autograd import FusedDatacube
from tests.helpers import rel_err

pytestmark = pytest.mark.gpu
TOL = 1e-5  # the parity bound of the cube and its gradients


def _wave(kind, n_wave):
    if kind == "linear":
        return np.linspace(3000.0, 9000.0, n_wave)
    if kind == "log":
        return np.geomspace(3000.0, 9000.0, n_wave)
    rng = np.random.default_rng(4)  # irregular spacing, up to a factor 4
    d = rng.uniform(0.5, 2.0, n_wave - 1)
    return 3000.0 + 6000.0 * np.concatenate([[0.0], np.cumsum(d) / d.sum()])


def _target(kind, n, t0, t1):
    if n == 1:
        return np.array([5000.0])
    if kind == "irregular":
        rng = np.random.default_rng(5)
        d = rng.uniform(0.4, 1.6, n - 1)
        return t0 + (t1 - t0) * np.concatenate([[0.0], np.cumsum(d) / d.sum()])
    return np.linspace(t0, t1, n)


@pytest.mark.parametrize("nt,n_wave,knots,t0,t1", [
    (1, 300, "linear", 0, 0), (255, 120, "linear", 4000, 7000), (257, 100, "log", 4000, 7000),
    (513, 200, "linear", 4000, 7000), (1000, 700, "linear", 3400, 8395),
    (1025, 300, "irregular", 3400, 8395), (1483, 2111, "log", 4750, 8751),
    (2049, 500, "linear", 2500, 9800), (3721, 1000, "linear", 4700, 9350),
    (4096, 1800, "linear", 4700, 8800), (4097, 900, "linear", 4700, 8800),
    (8192, 1500, "linear", 4000, 8800), (700, 60, "linear", 2000, 12000)])
def test_shapes_and_layouts_match_oracle(nt, n_wave, knots, t0, t1):
    n, nb = 150, 3
    st = S.make_stars(n, seed=nt)
    st["velocity"][:5, 2] = [2000.0, -2000.0, 0.0, 700.0, -700.0]
    grid = S.make_ssp_grid(4, 6, n_wave, (3000.0, 9000.0), seed=1)
    grid["wave"] = _wave(knots, n_wave).astype(np.float32)
    geom = dict(wave_target=_target(knots, nt, t0, t1).astype(np.float32), z=0.05, edges=np.arange(nb + 1))
    ids = np.random.default_rng(nt).integers(0, nb * nb, n)
    ids[n // 2:] = 4  # one long chunk
    cot = np.random.default_rng(1).normal(size=(nb * nb, nt))
    t = {k: torch.tensor(st[k], dtype=torch.float64, requires_grad=True)
         for k in ("mass", "age", "metallicity")}
    v = torch.tensor(st["velocity"][:, 2], dtype=torch.float64, requires_grad=True)
    ref = RT.star_cube(t["mass"], t["age"], t["metallicity"], v, torch.tensor(ids), grid, geom,
                       torch.float64).reshape(nb * nb, nt)
    rg = torch.autograd.grad(ref, [t["mass"], t["age"], t["metallicity"], v], torch.tensor(cot))
    dev = "cuda"
    ssp = ops.PreparedSSP(grid["flux"], grid["ax_met"], grid["ax_age"], grid["wave"], geom["z"],
                          True, dev)
    tg = ops.TargetGrid(geom["wave_target"], dev)
    g = {k: torch.tensor(st[k], device=dev, requires_grad=True)
         for k in ("mass", "age", "metallicity", "velocity")}
    cube = FusedDatacube.apply(g["mass"], g["age"], g["metallicity"], g["velocity"],
                               torch.tensor(ids, dtype=torch.int32, device=dev), ssp, tg, nb * nb,
                               nb * nb, 2, ops.SPEED_OF_LIGHT)
    got = torch.autograd.grad(cube, list(g.values()),
                              torch.tensor(cot, dtype=torch.float32, device=dev))
    assert rel_err(cube.detach().cpu().numpy(), ref.detach().numpy()) <= TOL
    if nt > 1:  # one bin: Nn = 0, sf = 0
        for a, b in zip(got[:3], rg[:3]):
            assert rel_err(a.cpu().numpy(), b.numpy()) <= TOL
        assert rel_err(got[3][:, 2].cpu().numpy(), rg[3].numpy()) <= TOL
