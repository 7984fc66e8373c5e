"""Forces of particles whose bricks have no box, on a mesh large enough that they
may read a force mesh formed for them: from the potential (few such bricks) and
from that mesh (many), against float64 differences and sums of the potential
that the run itself kept.

A difference and its share of the 8 corners' sum are some 12 float32 roundings
of the potential's values: 16 2^-24 of the sum of the absolute terms.
"""
import numpy as np
import pytest
import torch

import flowpm_amd as fa  # noqa: F401
from flowpm_amd import _lib, _plans

pytestmark = pytest.mark.gpu
FAC = 0.46


def _readout(field, x, n, absolute):
  """sum over corners of w times the fourth-order differences (float64)."""
  lo = x.floor()
  out = torch.zeros_like(x)
  size = torch.tensor(n, device=x.device)
  d1, d2 = 2.0 / 3.0, 1.0 / 12.0

  def at(i):
    i = torch.remainder(i, size)
    return field[(i[:, 0] * n[1] + i[:, 1]) * n[2] + i[:, 2]]

  for k in range(8):
    off = torch.tensor([k & 1, k >> 1 & 1, k >> 2], device=x.device)
    cell = lo.long() + off
    w = (1.0 - (x - (lo + off)).abs()).prod(-1)
    for e in range(3):
      s = torch.zeros(3, dtype=torch.long, device=x.device)
      s[e] = 1
      p1, m1, p2, m2 = at(cell + s), at(cell - s), at(cell + 2 * s), at(
          cell - 2 * s)
      out[:, e] += w * (d1 * (p1 + m1) + d2 * (p2 + m2) if absolute else d1 *
                        (p1 - m1) - d2 * (p2 - m2))
  return out


# share of the bricks whose particles lie anywhere: below and above an eighth
@pytest.mark.parametrize("share", [0.06, 0.5, 1.0])
def test_forces_without_a_box(gpu, share):
  n = (256, 256, 64)
  N = n[0] * n[1] * n[2]
  gen = torch.Generator(device=gpu).manual_seed(17)
  q = torch.stack(torch.meshgrid(*[torch.arange(m, device=gpu) for m in n],
                                 indexing="ij"), -1).reshape(N, 3)
  size = torch.tensor(n, device=gpu, dtype=torch.float32)
  brick = (q[:, 0] // 8 * 16 + q[:, 1] // 16) * 4 + q[:, 2] // 16
  far = torch.rand(2048, generator=gen, device=gpu)[brick] < share
  x = torch.where(
      far[:, None],
      torch.rand(N, 3, generator=gen, device=gpu) * 3 * size - size,
      q + 0.3 * torch.randn(N, 3, generator=gen, device=gpu))
  state = torch.zeros(3, 1, N, 3, device=gpu)
  state[0, 0] = x
  plan = _plans.get(gpu, 1, *n)
  L = _lib.lib()
  work = torch.empty(L.pmx_nbody_work_floats(plan.handle), device=gpu)
  tape = torch.empty(L.pmx_nbody_compact_tape_floats(plan.handle, N, 0),
                     device=gpu)
  _lib.call("pmx_nbody_run_compact_taped", plan.handle, _lib.ptr(state), N,
            1.0, FAC, None, 0, _lib.ptr(tape), _lib.ptr(work),
            _lib.stream_of(state))
  phi = tape[3 * N:].double()
  pick = torch.randperm(N, generator=gen, device=gpu)[:400000]
  xs = x[pick].double()
  ref = FAC * _readout(phi, xs, n, False)
  tol = 16 * 2.0**-24 * FAC * _readout(phi.abs(), xs, n, True)
  err = (state[2, 0, pick].double() - ref).abs()
  assert bool((err <= tol).all()), float((err - tol).max())
