"""The full spectrum of r2c3d and the projection of c2r3d at every number of
lanes a row takes (rows of 8 to 1024 elements, 5 to 513 of the half spectrum),
with a number of rows that is no multiple of a workgroup's.

The full spectrum's upper half is the conjugate of the lower one bit for bit
(it is the same half spectrum), and c2r3d sees only the Hermitian part of what
it is given: adding an anti-Hermitian field, here i times the spectrum of
another real field, leaves the projection where it was but for the rounding of
the sums, 2^-24 of each, and the transform's own, 64 2^-24 in norm.
"""
import pytest
import torch

import flowpm_amd as fa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,batch", [((12, 20, 8), 1), ((8, 12, 12), 3),
                                     ((8, 20, 16), 1), ((12, 8, 20), 5),
                                     ((8, 12, 32), 1), ((20, 8, 60), 1),
                                     ((8, 12, 64), 3), ((8, 8, 128), 1),
                                     ((8, 12, 1024), 1)])
def test_rows_of_every_length(gpu, n, batch):
  gen = torch.Generator().manual_seed(n[2])
  a = torch.randn(batch, *n, generator=gen).to(gpu)
  b = torch.randn(batch, *n, generator=gen).to(gpu)
  ka, kb = fa.r2c3d(a), fa.r2c3d(b)
  ref = torch.fft.fftn(a.double().cpu(), dim=(1, 2, 3)) / (n[0] * n[1] * n[2])
  got = ka.cpu().to(torch.complex128)
  assert (got - ref).norm() <= 64 * 2.0**-24 * ref.norm()
  mirror = torch.roll(torch.flip(ka, (1, 2, 3)), (1, 1, 1), (1, 2, 3)).conj()
  z = torch.arange(n[2], device=gpu)
  own = (z != 0) & (z != n[2] // 2)  # (those two planes mirror in themselves)
  assert torch.equal(ka[..., own], mirror[..., own].resolve_conj())
  back = fa.c2r3d(ka + 1j * kb)
  tol = 128 * 2.0**-24 * (a.double().norm() + b.double().norm())
  assert (back - a).double().norm() <= tol
