"""The time loop's readout from the potential (one particle per cell) against
the general path: the float4 force mesh and the separate readout + kick +
drift, from the same density.  Both form the same differences and sums in the
same order, so the states agree bit for bit wherever the paint is
deterministic (no brick spills to float atomics); where bricks spill the two
densities differ by their rounding, a few 2^-23 of a cell's value per deposit.
"""
import numpy as np
import pytest
import torch

import flowpm_amd as fa
from flowpm_amd import _lib, _plans

pytestmark = pytest.mark.gpu


def _general(st, n, fac, coef):
  """Jump-start force and KDK steps by the separate entry points."""
  B, N = st.shape[1], st.shape[2]
  plan = _plans.get(st.device, B, *n)
  s = _lib.stream_of(st)

  def force(flags, k2, k1, d):
    rho = fa.cic_paint(torch.zeros(B, *n, device=st.device), st[0])
    f4 = torch.empty(B, *n, 4, device=st.device)
    phi = torch.empty_like(rho)
    _lib.call("pmx_force_mesh_f4", plan.handle, _lib.ptr(rho),
              _lib.ptr(plan.spec()), _lib.ptr(phi), _lib.ptr(f4), 1.0 / N, s)
    m = [f4[..., i].contiguous() for i in range(3)]
    _lib.call("pmx_readout_kick_drift", _lib.ptr(st[0]), _lib.ptr(st[1]),
              _lib.ptr(st[2]), *[_lib.ptr(q) for q in m], B, N, *n, 1.0, fac,
              k2, k1, d, flags, s)

  steps = len(coef) // 3
  force(2 if steps else 0, 0.0, coef[0] if steps else 0.0,
        coef[1] if steps else 0.0)
  for i in range(steps):
    last = i + 1 == steps
    force(1 if last else 3, coef[3 * i + 2], 0.0 if last else coef[3 * i + 3],
          0.0 if last else coef[3 * i + 4])
  return st


# amp: rms displacement in cells.  Small sides: boxes longer than the mesh;
# 4 cells: boxes of several LDS windows and, on the small meshes, bricks
# beyond their slot (read from the mesh); partial bricks and ragged sides
@pytest.mark.parametrize("n,batch,amp", [
    ((8, 8, 8), 1, 0.2), ((12, 16, 8), 2, 0.3), ((20, 24, 12), 1, 1.0),
    ((32, 32, 32), 2, 0.5), ((40, 24, 60), 1, 1.5), ((64, 96, 48), 1, 0.5),
    ((48, 64, 80), 1, 4.0), ((128, 64, 64), 1, 3.0)])
def test_box_readout_equals_force_mesh(gpu, n, batch, amp):
  gen = torch.Generator().manual_seed(3)
  N = n[0] * n[1] * n[2]
  q = torch.as_tensor(np.indices(n).reshape(3, -1).T.astype(np.float32))
  st = torch.stack([q + amp * torch.randn(batch, N, 3, generator=gen) - 1.75,
                    0.1 * torch.randn(batch, N, 3, generator=gen),
                    torch.zeros(batch, N, 3)]).to(gpu)
  # a particle without a position takes no force and paints nothing
  st[0, 0, N // 2, 1] = float("nan")
  coef = [0.3, 0.5, 0.2, 0.1, 0.4, 0.25]
  plan = _plans.get(gpu, batch, *n)
  work = torch.empty(_lib.lib().pmx_nbody_work_floats(plan.handle),
                     dtype=torch.float32, device=gpu)
  for steps in (0, 2):
    c = coef[:3 * steps]
    ref = _general(st.clone(), n, 0.46, c)
    out = st.clone()
    _lib.call("pmx_nbody_run", plan.handle, _lib.ptr(out), N, 1.0, 0.46,
              _lib.dbl(c), 0, steps, 1, _lib.ptr(work), _lib.stream_of(out))
    again = _general(st.clone(), n, 0.46, c)
    own = torch.nan_to_num(ref - again).abs().max()
    diff = torch.nan_to_num(ref - out).abs().max()
    assert torch.equal(torch.isnan(ref), torch.isnan(out))
    # deterministic: bit for bit; else the rounding of the density, which
    # moves the forces (order 1) by far less than 1e-4
    assert diff == 0 if own == 0 else diff < 1e-4, (steps, diff, own)
