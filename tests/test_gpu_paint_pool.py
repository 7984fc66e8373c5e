"""Bricks whose boxes are beyond their own piece of the arena: some in the
pool, and the rest, with the pool full, through float atomics.  Density and
three-channel paint, against the float64 oracle.

The accumulation is 32-bit fixed point per brick of at most 2048 particles: a
deposit is rounded by at most 2^-30 of the sum of the brick's |weights|, so a
cell of the density that takes k deposits is off by at most k 2^-19, plus a
few float32 roundings of its value (as on every path).  The gradient of the
force goes through the three-channel paint and five float32 transforms: 1e-4
of its norm covers some hundred roundings of 2^-24 amplified tenfold by the
differences across a cell, and a box that lies elsewhere moves it by 1e-2 and
more.
"""
import numpy as np
import pytest
import torch

import flowpm_amd as fa
from flowpm_amd import tfpm
from oracle import pm as opm
from oracle.background import GrowthTable, planck15

pytestmark = pytest.mark.gpu


def _positions(n, batch, amp, far, f=1, seed=11):
  """A grid moved by amp spacings rms, and by 2.2 mesh cells (boxes of some 24000 cells:
  between a piece and the largest box) in the bricks of far."""
  gen = torch.Generator().manual_seed(seed)
  q = torch.as_tensor(np.indices(n).reshape(3, -1).T.astype(np.float32))
  a = torch.full((q.shape[0], 1), amp)
  if far == "few":
    a[(q[:, 0] < 8 / f) & (q[:, 1] < 32 / f) & (q[:, 2] < 16 / f)] = 2.2 / f
  elif far == "all":
    a[:] = 2.2 / f
  return q + a * torch.randn(batch, *q.shape, generator=gen) - 1.75


CASES = [((64, 64, 64), 1, 0.4, "few"), ((64, 64, 64), 1, 0.4, "all"),
         ((60, 40, 54), 2, 1.0, "few"), ((44, 50, 37), 1, 1.0, "all")]


@pytest.mark.parametrize("n,batch,amp,far", CASES)
def test_density_through_the_pool(gpu, n, batch, amp, far):
  pos = _positions(n, batch, amp, far)
  out = fa.cic_paint(torch.zeros(batch, *n, device=gpu), pos.to(gpu))
  out = out.double().cpu()
  ref = opm.cic_paint(torch.zeros(batch, *n).double(), pos.double())
  nb, _ = opm._cic_corners(pos.double(), list(n))
  cnt = torch.stack([torch.bincount(
      ((i[..., 0] * n[1] + i[..., 1]) * n[2] + i[..., 2]).reshape(-1),
      minlength=ref[0].numel()) for i in nb]).reshape(ref.shape)
  tol = cnt * 2.0**-19 + (8 + cnt) * 2.0**-23 * ref.abs()
  assert bool(((out - ref).abs() <= tol).all())


@pytest.mark.parametrize("n,batch,amp,far,f", [
    c + (1,) for c in (CASES[0], CASES[1], ((60, 40, 48), 2, 1.0, "few"))
] + [((16, 24, 32), 1, 0.3, "few", 2), ((20, 24, 30), 1, 0.5, "all", 2)])
def test_three_channels_through_the_pool(gpu, n, batch, amp, far, f):
  pos = _positions(n, batch, amp, far, f)
  gen = torch.Generator().manual_seed(5)
  g = torch.randn(batch, pos.shape[1], 3, generator=gen)
  zero = torch.zeros_like(pos)

  def grad(dev, dt, run):
    st = torch.stack([pos, zero, zero]).to(dev, dt).requires_grad_()
    (run(st)[2] * g.to(dev, dt)).sum().backward()
    return st.grad[0].double().cpu()

  growth = GrowthTable(planck15())
  ref = grad("cpu", torch.float64,
             lambda st: opm.force(growth, st, list(n), f))
  cosmo = fa.cosmology.Planck15()
  got = [grad(gpu, torch.float32,
              lambda st: tfpm.force(cosmo, st, list(n), f)) for _ in range(2)]
  for o in got:  # (the second paint of a process reuses the first's memory)
    assert (o - ref).norm() <= 1e-4 * ref.norm(), float(
        (o - ref).norm() / ref.norm())
