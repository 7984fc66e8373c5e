"""The tape of a differentiable run is of the kind that it is filled as: with one
particle per cell it holds potentials whatever set_compact_tape says, and takes
their size; with a finer force mesh both kinds exist, and give the same states
and gradients bit for bit.
"""
import numpy as np
import pytest
import torch

import flowpm_amd as fa
from flowpm_amd import _lib, _plans, tfpm
from oracle import pm as opm
from oracle.background import GrowthTable, planck15

pytestmark = pytest.mark.gpu

STAGES = [0.1, 0.3, 0.6, 1.0]


def _state(n, batch, amp, gpu):
  gen = torch.Generator().manual_seed(3)
  q = torch.as_tensor(np.indices(n).reshape(3, -1).T.astype(np.float32))
  x = q + amp * torch.randn(batch, *q.shape, generator=gen)
  p = 0.05 * torch.randn(batch, *q.shape, generator=gen)
  g = torch.randn(3, batch, *q.shape, generator=gen)
  return torch.stack([x, p, 0 * x]).to(gpu), g.to(gpu)


@pytest.fixture(params=[False, None, True])
def compact(request):
  tfpm.set_compact_tape(request.param)
  yield request.param
  tfpm.set_compact_tape(None)


@pytest.mark.parametrize("f", [1, 2])
def test_tape_takes_the_size_of_its_kind(gpu, compact, f):
  n = (16, 24, 32)
  st, _ = _state(n, 2, 0.2, gpu)
  out = fa.nbody(fa.cosmology.Planck15(), st.requires_grad_(), STAGES, list(n),
                 pm_nc_factor=f, checkpoint_every=0)
  plan = _plans.get(gpu, 2, *[f * m for m in n])
  kind = "" if compact is False and f == 2 else "compact_"
  want = getattr(_lib.lib(), "pmx_nbody_%stape_floats" % kind)(
      plan.handle, int(np.prod(n)), len(STAGES) - 1)
  assert out.grad_fn.saved_tensors[0].numel() == want


def test_the_policy_asks_for_the_size_that_is_used(gpu, compact, monkeypatch):
  asked = []
  monkeypatch.setattr(tfpm, "_tape_fits",
                      lambda plan, N, k, dev, name: asked.append(name) or True)
  n = (16, 24, 32)
  st, _ = _state(n, 1, 0.2, gpu)
  for f in (1, 2):
    fa.nbody(fa.cosmology.Planck15(), st.clone().requires_grad_(), STAGES,
             list(n), pm_nc_factor=f)
  full = "pmx_nbody_tape_floats"
  small = "pmx_nbody_compact_tape_floats"
  assert asked == [small, full if compact is False else small]


@pytest.mark.parametrize("batch", [1, 2])
def test_both_tapes_of_a_finer_mesh_agree(gpu, batch):
  n = (16, 20, 24)
  st, g = _state(n, batch, 0.3, gpu)
  res = []
  for kind in (False, True):
    tfpm.set_compact_tape(kind)
    try:
      oc = torch.tensor(0.2589, dtype=torch.float64, requires_grad=True)
      x = st.clone().requires_grad_()
      out = fa.nbody(fa.cosmology.Planck15(Omega_c=oc), x, STAGES, list(n),
                     pm_nc_factor=2, checkpoint_every=0)
      for keep in (True, False):  # a second pass reads an intact tape
        res.append((out.detach(),) + torch.autograd.grad(
            out, (x, oc), g, retain_graph=keep))
    finally:
      tfpm.set_compact_tape(None)
  for r in res[1:]:
    assert all(torch.equal(a, b) for a, b in zip(res[0], r))


def test_finer_mesh_gradient_against_oracle(gpu, compact):
  """Of a single force: five float32 transforms, 1e-4 in norm (some hundred
  roundings of 2^-24 amplified tenfold by the differences across a cell)."""
  n = (16, 20, 24)
  st, g = _state(n, 1, 0.3, gpu)
  ref = st.double().cpu().requires_grad_()
  (opm.force(GrowthTable(planck15()), ref, list(n), 2) *
   g.double().cpu()).sum().backward()
  x = st.clone().requires_grad_()
  (fa.tfpm.force(fa.cosmology.Planck15(), x, list(n), 2) * g).sum().backward()
  err = (x.grad.double().cpu() - ref.grad)[0].norm() / ref.grad[0].norm()
  assert err <= 1e-4, float(err)
