"""Catalogues of more chunks than a tile's workgroup takes at a time (512 of 2048
particles): the second round of its loop over the chunks, and the further
shares of tiles with more than 8192 entries, some of which begin or end in
that round.

A deposit is a float32 product, off by 8 2^-24 of itself at most; a tile's sums
are float64, rounded once, and each further share is rounded once and added with
one rounding of the cell: with s shares a cell is within (8 + 2 s) 2^-24 of the
sum of its |deposits|.  A chunk that is left out or taken twice moves the sum of
all cells by 2048 deposits, which is asked for to 2^-24 of each deposit.
"""
import pytest
import torch

import flowpm_amd as fa
from flowpm_amd import _lib
from oracle import pm as opm

pytestmark = pytest.mark.gpu

CHUNK, ROUND, SHARE = 2048, 512, 8192


@pytest.mark.parametrize("kind,n,batch,npart", [
    ("uniform", (40, 36, 50), 1, 1100003), ("uniform", (40, 36, 50), 2, 1050001),
    ("cells", (24, 40, 33), 1, 1300003), ("late", (24, 40, 33), 1, 1080001)])
def test_more_chunks_than_a_round(gpu, kind, n, batch, npart):
  assert -(-npart // CHUNK) > ROUND
  assert _lib.lib().pmx_cic_readout_adj_work_floats(batch, npart, *n) > 0
  gen = torch.Generator().manual_seed(12)
  pos = torch.rand(batch, npart, 3, generator=gen) * torch.tensor(
      n, dtype=torch.float32)
  if kind == "cells":  # half of them in three cells of two tiles
    spot = torch.tensor([[3.0, 4.0, 5.0], [6.0, 15.0, 7.0], [20.0, 30.0, 20.0]])
    pos[:, ::2] = spot[torch.randint(3, pos[:, ::2].shape[:2], generator=gen)] \
        + 0.9 * torch.rand(pos[:, ::2].shape, generator=gen)
  elif kind == "late":  # a tile's particles in the last chunks only
    pos[:, -40000:] = 17.0 + 5.0 * torch.rand(batch, 40000, 3, generator=gen)
  w = torch.randn(batch, npart, generator=gen)
  out = fa.cic_paint(torch.zeros(batch, *n, device=gpu), pos.to(gpu),
                     weight=w.to(gpu)).double().cpu()
  mesh = torch.zeros(batch, *n, device=gpu, requires_grad=True)
  (adj,) = torch.autograd.grad(fa.cic_readout(mesh, pos.to(gpu)), mesh,
                               w.to(gpu))
  zero = torch.zeros(batch, *n, dtype=torch.float64)
  # (float32 factors, as the kernels', summed in float64)
  ref, mag = opm.cic_paint(zero, pos, w), opm.cic_paint(zero, pos, w.abs())
  tol = (8 + 2 * _most_shares(pos, n)) * 2.0**-24 * mag
  for got in (out, adj.double().cpu()):
    err = (got - ref).abs()
    assert bool((err <= tol).all()), float((err - tol).max())
    assert abs(float((got - ref).sum())) <= 8 * 2.0**-24 * float(mag.sum())


def _most_shares(pos, n):
  """The shares of the fullest tile (8 x 16 x 16 cells), counting a particle in
  each tile that a corner of its lies in."""
  most = 0
  for p in pos:
    i = p.floor().long()
    tiles = []
    for k in range(8):
      off = torch.tensor([k & 1, k >> 1 & 1, k >> 2])
      t = torch.remainder(i + off, torch.tensor(n)) // torch.tensor([8, 16, 16])
      tiles.append((t[:, 0] * 64 + t[:, 1]) * 64 + t[:, 2])
    tiles = torch.stack(tiles, 1).sort(1).values
    new = torch.ones_like(tiles, dtype=torch.bool)
    new[:, 1:] = tiles[:, 1:] != tiles[:, :-1]
    most = max(most, int(torch.bincount(tiles[new]).max()))
  return -(-most // SHARE)
