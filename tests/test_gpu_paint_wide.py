"""The accuracy of bricks whose boxes are beyond 64 KB.

Only the particles of two such bricks have a weight, so that no other brick's
32-bit accumulation is in the mesh.  Their deposits are float32 products (a
weight's three factors are off by at most 2^-25 each, the products by 2^-24 of
themselves), summed in 64-bit fixed point whose unit is far below that, and
rounded once per box and once where boxes overlap: in the root mean square the
mesh is off by less than 8 2^-24 of itself.
"""
import numpy as np
import pytest
import torch

import flowpm_amd as fa
from oracle import pm as opm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("weights", ["ones", "wide"])
@pytest.mark.parametrize("n", [(64, 64, 64), (60, 54, 70)])
def test_large_boxes_are_summed_like_floats(gpu, n, weights):
  gen = torch.Generator().manual_seed(21)
  q = torch.as_tensor(np.indices(n).reshape(3, -1).T.astype(np.float32))
  far = (q[:, 0] < 8) & (q[:, 1] < 32) & (q[:, 2] < 16)
  a = torch.where(far, 2.2, 0.4)[:, None]
  # (away from the mesh's edge, where weights round by themselves)
  pos = (q + a * torch.randn(q.shape, generator=gen) + 20.0)[None]
  w = far.float()
  if weights == "wide":  # of either sign, over several orders of magnitude
    w = w * torch.exp(2.0 * torch.randn(w.shape, generator=gen)) * \
        torch.sign(torch.randn(w.shape, generator=gen))
  for k in range(2):  # boxes beyond 64 KB, up to 128 KB
    b = pos[0, far & (q[:, 1] // 16 == k)]
    e = b.floor().amax(0) - b.floor().amin(0) + 2
    assert 16384 < float(e.prod()) <= 32768, e
  out = fa.cic_paint(torch.zeros(1, *n, device=gpu), pos.to(gpu),
                     weight=w[None].to(gpu)).double().cpu()
  ref = opm.cic_paint(torch.zeros(1, *n).double(), pos.double(),
                      w[None].double())
  err = float((out - ref).norm() / ref.norm())
  print("%s %s: %.3g" % (n, weights, err))
  assert err <= 8 * 2.0**-24
