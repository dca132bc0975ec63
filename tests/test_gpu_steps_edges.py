"""GPU: the per-step kernels at the edges of their splits: row lengths off a
multiple of four, targets of one bin, past a group of bins in flight, past the
LDS-held forward, starting below, inside and past the template grid, knots
denser and sparser than the bins; against the float64 oracle on the
reference's float32 knots."""
import numpy as np
import pytest
import torch

from oracle import ref_torch as RT
from rubix_amd import ops
from rubix_amd.autograd import Resample, ScaleByMass, SegmentCube
from tests.helpers import rel_err

pytestmark = pytest.mark.gpu
TOL = 1e-5  # the parity bound of the steps and their gradients
DEV = "cuda"


@pytest.mark.parametrize("nt,ns,t0,t1", [(1, 7, 5000, 5000), (255, 61, 4000, 7000), (257, 1003, 4000, 7000),
                                         (1025, 998, 2500, 9800), (2047, 502, 4700, 8000),
                                         (3721, 5001, 4700, 9350), (1000, 6000, 6000, 6400),
                                         (5300, 301, 3500, 9000)])
def test_resample_and_adjoint(nt, ns, t0, t1):
    n, z = 20, 0.05
    rng = np.random.default_rng(nt + ns)
    wave = np.linspace(3000, 9000, ns).astype(np.float32)
    tw = np.linspace(t0, t1, nt).astype(np.float32)
    spec = rng.uniform(0.5, 1.5, (n, ns)).astype(np.float32)
    vel = rng.normal(0, 200, (n, 3)).astype(np.float32)
    g = rng.normal(size=(n, nt)).astype(np.float32)
    grid = rng.uniform(0.5, 1.5, (2, 2, ns))
    ssp = ops.PreparedSSP(grid, [0.0, 1.0], [0.0, 1.0], wave, z, False, DEV)
    tg = ops.TargetGrid(tw, DEV)
    s, v = torch.tensor(spec, device=DEV, requires_grad=True), torch.tensor(vel, device=DEV, requires_grad=True)
    out = Resample.apply(s, v, ssp, tg, 2, ops.SPEED_OF_LIGHT)
    gs, gv = torch.autograd.grad(out, [s, v], torch.tensor(g, device=DEV))
    s64 = torch.tensor(spec, dtype=torch.float64, requires_grad=True)
    v64 = torch.tensor(vel[:, 2], dtype=torch.float64, requires_grad=True)
    w32 = torch.tensor(1 + z, dtype=torch.float32) * torch.tensor(wave)
    knots = RT.reference_knots(w32, v64, torch.exp(v64 / RT.SPEED_OF_LIGHT))
    ref = RT.resample(s64, knots, torch.tensor(tw, dtype=torch.float64))
    if nt == 1:  # one bin has no width: the total is 0, the factor 0
        assert not bool(out.any()) and not bool(gs.any())
        return
    rs, rv = torch.autograd.grad(ref, [s64, v64], torch.tensor(g, dtype=torch.float64))
    assert rel_err(out.detach().cpu().numpy(), ref.detach().numpy()) <= TOL
    assert rel_err(gs.cpu().numpy(), rs.numpy()) <= TOL
    assert rel_err(gv[:, 2].cpu().numpy(), rv.numpy()) <= TOL


def test_resample_past_the_lds_forward():
    n, nt = 3, 17_001  # more bins than the forward holds in LDS
    rng = np.random.default_rng(3)
    wave = np.linspace(3000, 9000, 2003).astype(np.float32)
    tw = np.linspace(4000, 8000, nt).astype(np.float32)
    spec = rng.uniform(0.5, 1.5, (n, 2003)).astype(np.float32)
    vel = rng.normal(0, 200, (n, 3)).astype(np.float32)
    ssp = ops.PreparedSSP(rng.uniform(0.5, 1.5, (2, 2, 2003)), [0.0, 1.0], [0.0, 1.0], wave, 0.0, False, DEV)
    out = ops.resample(ssp, ops.TargetGrid(tw, DEV), torch.tensor(spec, device=DEV), torch.tensor(vel, device=DEV))
    v64 = torch.tensor(vel[:, 2], dtype=torch.float64)
    knots = RT.reference_knots(torch.tensor(wave), v64, torch.exp(v64 / RT.SPEED_OF_LIGHT))
    ref = RT.resample(torch.tensor(spec, dtype=torch.float64), knots, torch.tensor(tw, dtype=torch.float64))
    assert rel_err(out.cpu().numpy(), ref.numpy()) <= TOL


@pytest.mark.parametrize("n,nw", [(1, 1), (5, 3), (300, 255), (700, 257), (2000, 1030)])
def test_rows_by_quads(n, nw):
    rng = np.random.default_rng(n)
    x = torch.tensor(rng.normal(size=(n, nw)).astype(np.float32), device=DEV, requires_grad=True)
    m = torch.tensor(rng.normal(size=n).astype(np.float32), device=DEV, requires_grad=True)
    ids = torch.tensor(rng.integers(-1, 5, n).astype(np.int32), device=DEV)
    g = torch.tensor(rng.normal(size=(4, nw)).astype(np.float32), device=DEV)
    out = ScaleByMass.apply(x, m)
    cube = SegmentCube.apply(out, ids, 4, 5)
    gx, gm = torch.autograd.grad(cube, [x, m], g)
    xd, md, gd, k = (t.detach().double().cpu().numpy() for t in (x, m, g, ids))
    ok = (k >= 0) & (k < 4)
    ref = np.zeros((4, nw))
    np.add.at(ref, k[ok].astype(int), (xd * md[:, None])[ok])
    up = np.where(ok[:, None], gd[np.where(ok, k, 0).astype(int)], 0.0)
    assert rel_err(cube.detach().cpu().numpy(), ref) <= TOL
    assert rel_err(gx.cpu().numpy(), up * md[:, None]) <= TOL
    assert rel_err(gm.cpu().numpy(), (up * xd).sum(1)) <= TOL
