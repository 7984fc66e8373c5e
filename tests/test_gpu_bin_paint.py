"""The paint and the readout's adjoint of particles in any order (sorted by
mesh tiles of 8 x 16 x 16 cells), against the oracle summing in float64.

Every deposit is a float32 product: a weight's three factors take one rounding
each, their product two and that with the particle's weight one; the sums are
float64, rounded once (the scatter of the sizes below the rule rounds once per
deposit).  So a cell is within 8 2^-24 of the sum of its |deposits|, plus, on
the scatter, one 2^-24 of it per deposit.
"""
import numpy as np
import pytest
import torch

import flowpm_amd as fa
from flowpm_amd import _lib
from oracle import pm as opm

pytestmark = pytest.mark.gpu


def _positions(kind, n, batch, npart, gen):
  side = torch.tensor(n, dtype=torch.float32)
  if kind == "uniform":
    return torch.rand(batch, npart, 3, generator=gen) * side
  if kind == "far":  # many box lengths away, both sides
    return (torch.rand(batch, npart, 3, generator=gen) * 8 - 4) * side
  if kind == "cell":  # all in one cell across the mesh's edge
    return torch.rand(batch, npart, 3, generator=gen) * 0.9 - 0.95
  q = torch.as_tensor(np.indices(n).reshape(3, -1).T.astype(np.float32))
  return q + 0.8 * torch.randn(batch, *q.shape, generator=gen)


def _check(out, pos, w, n):
  B = pos.shape[0]
  zero = torch.zeros(B, *n, dtype=torch.float64)
  # (float32 factors, which near a cell's far face have absolute errors,
  # summed in float64)
  ref = opm.cic_paint(zero, pos, w)
  mag = opm.cic_paint(zero, pos, w.abs())
  cnt = opm.cic_paint(zero, pos, torch.ones_like(w))
  err = (out.double().cpu() - ref).abs()
  # (cnt: the weighted number of deposits; small ones' roundings are small)
  tol = (8 + 8 * (pos.shape[1] < 40000) * (1 + cnt)) * 2.0**-24 * mag
  assert bool((err <= tol).all()), float((err - tol).max())


# sides below, at and above a tile's, one-cell sides, ragged ones; a chunk of
# 2048 particles less one, one more; more chunks than a tile's workgroup has
# threads (256); more than one member
CASES = [("uniform", (5, 7, 9), 1, 70000), ("uniform", (1, 40, 3), 2, 36863),
         ("uniform", (8, 16, 16), 1, 69633), ("uniform", (9, 17, 33), 3, 24577),
         ("uniform", (64, 50, 70), 1, 530000), ("far", (24, 33, 18), 2, 36000),
         ("cell", (12, 20, 40), 1, 70000), ("grid", (64, 40, 48), 2, 122880),
         ("uniform", (16, 16, 16), 1, 3), ("uniform", (30, 30, 30), 1, 2049)]


@pytest.mark.parametrize("kind,n,batch,npart", CASES)
def test_paint_in_any_order(gpu, kind, n, batch, npart):
  gen = torch.Generator().manual_seed(4)
  pos = _positions(kind, n, batch, npart, gen)
  w = torch.randn(batch, pos.shape[1], generator=gen)
  base = torch.zeros(batch, *n)
  if pos.shape[1] != n[0] * n[1] * n[2]:  # (the grid's paint has its own test)
    out = fa.cic_paint(base.to(gpu), pos.to(gpu), weight=w.to(gpu))
    _check(out, pos, w, n)
    # onto a mesh that holds something already
    more = fa.cic_paint(out, pos.to(gpu), weight=-w.to(gpu))
    assert (more.abs() <= 2.0**-17 * (1 + out.abs())).all() or \
        pos.shape[1] < 40000 or kind == "cell"
  mesh = torch.randn(batch, *n, generator=gen).to(gpu).requires_grad_()
  dpos = pos.to(gpu).requires_grad_()
  gm, gp = torch.autograd.grad(fa.cic_readout(mesh, dpos), [mesh, dpos],
                               w.to(gpu))
  _check(gm, pos, w, n)
  # the same position gradient as without the mesh's
  (alone,) = torch.autograd.grad(fa.cic_readout(mesh, dpos), dpos, w.to(gpu))
  assert torch.equal(gp, alone)


def test_weights_without_a_value(gpu):
  """inf and nan weights reach their own corner cells only, and particles
  without a position none."""
  n, npart = (20, 24, 28), 70000
  gen = torch.Generator().manual_seed(9)
  pos = torch.rand(1, npart, 3, generator=gen) * torch.tensor(n)
  pos[0, :2] = torch.tensor([[3.5, 15.5, 15.5], [7.5, 2.5, 27.5]])
  pos[0, 2, 1] = float("nan")
  pos[0, 3, 0] = float("inf")
  w = torch.ones(1, npart)
  w[0, 0], w[0, 1] = float("inf"), float("nan")
  out = fa.cic_paint(torch.zeros(1, *n, device=gpu), pos.to(gpu),
                     weight=w.to(gpu)).cpu()
  bad = torch.zeros(1, *n, dtype=torch.bool)
  bad[0, 3:5, 15:17, 15:17] = True
  bad[0, 7:9, 2:4, [27, 0]] = True
  assert torch.equal(~torch.isfinite(out), bad)
  keep = torch.ones(npart, dtype=torch.bool)
  keep[:4] = False
  ref = opm.cic_paint(torch.zeros(1, *n).double(), pos[:, keep])
  assert ((out.double() - ref).abs()[~bad] <= 1e-5 * (1 + ref[~bad])).all()
