"""Batches of small meshes, around the number of planes from which the z and y
passes are two launches again: up to 64 cells a side both ways do the same
operations in the same order, so a batch and its two halves agree bit for bit.
"""
import pytest
import torch

import flowpm_amd as fa

pytestmark = pytest.mark.gpu


# planes of the batch: over the limit (2048, 4096 at 32), its halves below it
@pytest.mark.parametrize("n,nx,batch", [(8, 8, 258), (12, 12, 172),
                                        (20, 8, 260), (24, 24, 86),
                                        (32, 32, 130), (40, 8, 514)])
def test_batch_equals_its_halves(gpu, n, nx, batch):
  field = torch.randn(batch, nx, n, n,
                      generator=torch.Generator().manual_seed(n)).to(gpu)
  h = batch // 2
  spec = fa.r2c3d(field)
  assert torch.equal(spec, torch.cat([fa.r2c3d(field[:h]),
                                      fa.r2c3d(field[h:])]))
  back = fa.c2r3d(spec)
  assert torch.equal(back, torch.cat([fa.c2r3d(spec[:h]),
                                      fa.c2r3d(spec[h:])]))
  assert (back - field).norm() <= 128 * 2.0**-24 * field.norm()
