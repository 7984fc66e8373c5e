"""Boxes of bricks of few particles (a finer force mesh), around the largest one
they get: the force and its gradient against the float64 oracle.

Five float32 transforms and the two paints: 1e-4 in norm covers some hundred
roundings of 2^-24 amplified tenfold by the differences across a cell; a brick
that is lost, or painted twice, moves it by 1e-2 and more.
"""
import numpy as np
import pytest
import torch

import flowpm_amd as fa
from flowpm_amd import tfpm
from oracle import pm as opm
from oracle.background import GrowthTable, planck15

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f,n,amp,most", [(2, (24, 32, 32), 1.6, 20480),
                                          (4, (12, 16, 16), 1.1, 16384)])
def test_boxes_around_the_largest(gpu, f, n, amp, most):
  gen = torch.Generator().manual_seed(31)
  q = torch.as_tensor(np.indices(n).reshape(3, -1).T.astype(np.float32))
  x = (q + amp * torch.randn(q.shape, generator=gen) - 1.75)[None]
  e = (8 // f, 16 // f, 16 // f)
  m = (x[0] * f).floor().reshape(*n, 3)
  b = m.unfold(0, e[0], e[0]).unfold(1, e[1], e[1]).unfold(2, e[2], e[2])
  b = b.flatten(4)
  vol = (b.amax(-1) - b.amin(-1) + 2).prod(-1)
  # (a fifth of the bricks or more on either side)
  assert 0.2 < float((vol > most).float().mean()) < 0.8
  g = torch.randn(1, x.shape[1], 3, generator=gen)

  def both(dev, dt, run):
    st = torch.stack([x, 0 * x, 0 * x]).to(dev, dt).requires_grad_()
    out = run(st)[2]
    (out * g.to(dev, dt)).sum().backward()
    return out.detach().double().cpu(), st.grad[0].double().cpu()

  growth, cosmo = GrowthTable(planck15()), fa.cosmology.Planck15()
  ref = both("cpu", torch.float64, lambda s: opm.force(growth, s, list(n), f))
  got = both(gpu, torch.float32, lambda s: tfpm.force(cosmo, s, list(n), f))
  for r, o in zip(ref, got):
    assert (o - r).norm() <= 1e-4 * r.norm(), float((o - r).norm() / r.norm())
