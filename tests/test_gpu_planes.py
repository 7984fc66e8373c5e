"""Transforms whose z and y passes run as one launch (square y-z planes of up
to 128 x 128) against torch's float64 transform, on both sides of the limit and
for sides of every radix.

An axis takes at most 4 stages of some 5 roundings each, three axes 60: in
norm the float32 result is off by less than 64 2^-24 of it.
"""
import pytest
import torch

import flowpm_amd as fa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [8, 12, 16, 20, 24, 32, 40, 48, 60, 64, 80, 96, 100,
                               120, 128, 160])
@pytest.mark.parametrize("nx,batch", [(8, 1), (20, 3)])
def test_square_planes(gpu, n, nx, batch):
  gen = torch.Generator().manual_seed(n)
  field = torch.randn(batch, nx, n, n, generator=gen)
  norm = nx * n * n
  spec = fa.r2c3d(field.to(gpu))
  ref = torch.fft.fftn(field.double(), dim=(1, 2, 3)) / norm
  got = spec.cpu().to(torch.complex128)
  assert (got - ref).norm() <= 64 * 2.0**-24 * ref.norm()
  back = fa.c2r3d(spec).double().cpu()
  assert (back - field).norm() <= 128 * 2.0**-24 * field.double().norm()
