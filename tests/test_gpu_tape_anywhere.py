"""A caller's tape may begin at any float: the taped run and its reverse sweep
give the same bits as with one that begins at 16 bytes.
"""
import numpy as np
import pytest
import torch

from flowpm_amd import _lib, _plans

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps", [0, 2])
@pytest.mark.parametrize("skip", [1, 2])
def test_tape_at_any_float(gpu, steps, skip):
  n, B = (24, 32, 40), 2
  N = int(np.prod(n))
  gen = torch.Generator().manual_seed(6)
  q = torch.as_tensor(np.indices(n).reshape(3, -1).T.astype(np.float32))
  x = q + 0.3 * torch.randn(B, N, 3, generator=gen)
  st = torch.stack([x, 0.1 * torch.randn(B, N, 3, generator=gen), 0 * x])
  g = torch.randn(3, B, N, 3, generator=gen).to(gpu)
  plan = _plans.get(gpu, B, *n)
  L, p = _lib.lib(), _lib.ptr
  coef = _lib.dbl([0.3, 0.5, 0.2, 0.1, 0.4, 0.25][:3 * steps])
  work = torch.empty(L.pmx_nbody_adj_work_floats(plan.handle, N, 0),
                     device=gpu)
  size = L.pmx_nbody_compact_tape_floats(plan.handle, N, steps)
  res = []
  for at in (0, skip):
    tape = torch.empty(size + at, device=gpu)[at:]
    assert tape.data_ptr() % 16 == 4 * at
    out, gs = st.to(gpu), g.clone()
    s = _lib.stream_of(out)
    _lib.call("pmx_nbody_run_compact_taped", plan.handle, p(out), N, 1.0, 0.46,
              coef, steps, p(tape), p(work), s)
    _lib.call("pmx_nbody_adjoint_compact_taped", plan.handle, p(tape), steps, N,
              1.0, 0.46, coef, p(gs), p(work), None, s)
    res.append((out, gs))
  for a, b in zip(*res):
    assert torch.equal(a, b)
