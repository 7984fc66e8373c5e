"""Bricks with boxes of nearly 64 KB, all of them at once: each has its own
piece of the arena, so none is added with float atomics and the paint repeats
bit for bit.
"""
import numpy as np
import pytest
import torch

import flowpm_amd as fa

pytestmark = pytest.mark.gpu


def test_boxes_up_to_64_kb_all_fit(gpu):
  n = (64, 64, 64)
  gen = torch.Generator().manual_seed(8)
  q = torch.as_tensor(np.indices(n).reshape(3, -1).T.astype(np.float32))
  pos = q + 0.4 * torch.randn(q.shape, generator=gen)
  # bricks of 8 x 16 x 16 particles: the first two of each span a box of
  # 24 x 26 x 26 cells, 63.4 of its 64 KB
  for x in range(0, 64, 8):
    for y in range(0, 64, 16):
      for z in range(0, 64, 16):
        i = (x * 64 + y) * 64 + z
        o = torch.tensor([x, y, z], dtype=torch.float32)
        pos[i] = o + torch.tensor([-7.5, -4.5, -4.5])
        pos[i + 1] = o + torch.tensor([14.5, 19.5, 19.5])
  zero = torch.zeros(1, *n, device=gpu)
  pos = pos[None].to(gpu)
  first = fa.cic_paint(zero, pos)
  for _ in range(7):
    assert torch.equal(fa.cic_paint(zero, pos), first)
