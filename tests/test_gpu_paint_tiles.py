"""The paint of one particle per cell at the edges of its mesh tiles and of
its boxes, against the float64 oracle.

The accumulation is 32-bit fixed point per brick of at most 2048 particles of
weight 1: one deposit is rounded by at most 2^-31 2^12 (the bricks' unit is
2^(ex - 30), ex <= 12), so a cell that takes k deposits is off by at most
k 2^-19, plus a few float32 roundings of its value.  Bricks that spill to
float atomics are within the same bound.
"""
import numpy as np
import pytest
import torch

import flowpm_amd as fa
from oracle import pm as opm

pytestmark = pytest.mark.gpu


def _check(gpu, n, batch, amp, seed, shift=0.0):
  gen = torch.Generator().manual_seed(seed)
  q = torch.as_tensor(np.indices(n).reshape(3, -1).T.astype(np.float32))
  pos = q + shift + amp * torch.randn(batch, *q.shape, generator=gen)
  mesh = torch.zeros(batch, *n)
  out = fa.cic_paint(mesh.to(gpu), pos.to(gpu)).double().cpu()
  ref = opm.cic_paint(mesh.double(), pos.double())
  # deposits per cell: every particle's 8 corners with weight 1
  nb, _ = opm._cic_corners(pos.double(), list(n))
  cnt = torch.stack([torch.bincount(
      ((i[..., 0] * n[1] + i[..., 1]) * n[2] + i[..., 2]).reshape(-1),
      minlength=ref[0].numel()) for i in nb]).reshape(ref.shape)
  tol = cnt * 2.0**-19 + (8 + cnt) * 2.0**-23 * ref.abs()
  assert bool(((out - ref).abs() <= tol).all()), float(
      ((out - ref).abs() - tol).max())


# sides below, at and above the tiles' 16 cells and 4, 8 or 16 planes; z
# sides that are no multiple of 4 (no 16-byte stores); boxes that nearly span
# a short z side (their cells are read one by one); more than one member
@pytest.mark.parametrize("n,batch,amp", [
    ((5, 7, 9), 1, 0.3), ((16, 16, 16), 2, 0.1), ((17, 15, 20), 1, 0.3),
    ((24, 33, 18), 2, 0.5), ((8, 40, 10), 3, 1.0), ((36, 20, 31), 1, 2.0),
    ((9, 64, 48), 1, 3.0)])
def test_paint_tile_edges(gpu, n, batch, amp):
  _check(gpu, n, batch, amp, 7)


# both sides of the rule that picks the tile: fewer than 256 tiles of 16
# planes, from 256, from 1024
@pytest.mark.parametrize("n,batch", [
    ((64, 64, 60), 3), ((64, 64, 60), 4), ((64, 64, 64), 15),
    ((64, 64, 64), 16), ((20, 128, 256), 4)])
def test_paint_tile_rule(gpu, n, batch):
  _check(gpu, n, batch, 1.5, 8, shift=-3.25)
