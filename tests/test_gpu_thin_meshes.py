"""Runs on meshes with a side too short for the bricks' boxes: large batches form
force meshes, small ones read the potential.  With displacements so small that
every brick has its box the paint repeats bit for bit, and a batch agrees with
its two halves bit for bit, as the two ways form the same sums in the same
order: states, gradients, with either tape, checkpoints, and a single force.
"""
import numpy as np
import pytest
import torch

import flowpm_amd as fa

pytestmark = pytest.mark.gpu

# (the halves are below the 200000 particles the rule asks for)
CASES = [((12, 40, 32), 14), ((40, 20, 24), 12), ((24, 32, 20), 14)]


def _state(n, batch, gpu):
  gen = torch.Generator().manual_seed(7)
  q = torch.as_tensor(np.indices(n).reshape(3, -1).T.astype(np.float32))
  x = q + 0.5 + 0.02 * torch.randn(batch, *q.shape, generator=gen)
  p = 0.01 * torch.randn(batch, *q.shape, generator=gen)
  c = torch.randn(3, batch, *q.shape, generator=gen)
  return torch.stack([x, p, torch.zeros_like(x)]).to(gpu), c.to(gpu)


def _grad(fn, st, c):
  st = st.clone().requires_grad_()
  out = fn(st)
  (g,) = torch.autograd.grad(out, st, c)
  return out.detach(), g


@pytest.mark.parametrize("n,batch", CASES)
@pytest.mark.parametrize("how", ["run", "force", "taped", "full tape", "kept",
                                 "recomputed"])
def test_batch_equals_its_halves(gpu, n, batch, how):
  cosmo = fa.cosmology.Planck15()
  st, c = _state(n, batch, gpu)
  assert batch * np.prod(n) >= 200000 > batch // 2 * np.prod(n)
  every = {"kept": 1, "recomputed": 2}.get(how, 0)

  def run(s):
    if how == "force":
      return fa.tfpm.force(cosmo, s, list(n))
    return fa.nbody(cosmo, s, [0.1, 0.12, 0.14, 0.16], list(n),
                    checkpoint_every=every)

  fa.tfpm.set_compact_tape(False if how == "full tape" else None)
  fa.tfpm.set_keep_potentials(how == "kept")
  try:
    if how == "run":
      go = lambda s, g: (run(s),)
    else:
      go = lambda s, g: _grad(run, s, g)
    whole = go(st, c)
    h = batch // 2
    halves = [go(s.contiguous(), g.contiguous())
              for s, g in ((st[:, :h], c[:, :h]), (st[:, h:], c[:, h:]))]
  finally:
    fa.tfpm.set_compact_tape(None)
    fa.tfpm.set_keep_potentials(None)
  for k, w in enumerate(whole):
    assert torch.equal(w, torch.cat([x[k] for x in halves], 1)), k
