"""Full-box transforms by register lines and planes, and the potential stage
fused into them, at every length they cover, against numpy."""
import numpy as np
import pytest
import torch

from jrystal_amd import _ops
from jrystal_amd.objective import EnergyPlan

pytestmark = pytest.mark.gpu

PLANES = (32, 35, 36, 40, 42, 45, 48, 49, 50, 54, 56, 60, 63, 64, 70, 72, 75,
          80)
LINES = PLANES + (81, 84, 90, 96, 98, 100, 105, 108, 112, 120, 126, 128)


@pytest.mark.parametrize("n", LINES)
def test_transforms_of_every_length(n):
  # each axis in turn, the square inner planes, odd batches, an LDS-staged
  # neighbour length (12) and a non-square plane
  shapes = [(3, n, 12, 12), (n, 12, 5), (2, 5, n, 12), (1, 7, 12, n),
            (n, 35, n)]
  if n in PLANES:
    shapes += [(1, 3, n, n), (5, n, n)]
  rng = np.random.default_rng(n)
  for shape in shapes:
    x = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    t = torch.tensor(x, device="cuda")
    print(shape, flush=True)
    for fn, ref in ((_ops.FFT3, np.fft.fftn(x, axes=(-3, -2, -1))),
                    (_ops.IFFT3, np.fft.ifftn(x, axes=(-3, -2, -1)) *
                     np.prod(shape[-3:]))):
      y = fn.apply(t, 0.5).cpu().numpy()
      # three FP64 transforms of about log2(n) butterfly levels each
      err = np.linalg.norm(y - 0.5 * ref) / np.linalg.norm(0.5 * ref)
      assert err < 2e-15 * np.log2(np.prod(shape[-3:]))


def _potential(rho, G, vol, pos, chg, ks_spin=False):
  """(E_H, E_ext, E_x, v_s) of rho (ns, ...) in numpy (LDA exchange; v_s in
  the band driver's form, vxc_lda, for two channels)."""
  N = rho[0].size
  g2 = (G**2).sum(-1)
  inv = np.where(g2 > 0, 1 / np.where(g2 > 0, g2, 1), 0)
  f = np.fft.fftn(rho.sum(0))
  ph = sum(z * np.exp(-1j * (G @ r)) for z, r in zip(chg, pos))
  ve = -4 * np.pi * N / vol * ph / (g2 + 1e-10)
  ve[0, 0, 0] = 0
  eh = 2 * np.pi * vol / N**2 * np.sum(np.abs(f)**2 * inv)
  ee = vol / N**2 * np.sum(np.conj(ve) * f).real
  v = np.fft.ifftn(4 * np.pi * f * inv + ve).real
  cx = 0.75 * (3 / np.pi)**(1 / 3)
  if len(rho) == 1:
    ex = -cx * np.cbrt(rho[0])
    return eh, ee, vol / N * np.sum(ex * rho[0]), (v + 4 / 3 * ex)[None]
  e = 0.5 * (-cx * np.cbrt(2 * rho[0]) - cx * np.cbrt(2 * rho[1]))
  vs = [v + e + r * -cx / (3 * np.cbrt(2 * r)**2) for r in rho]
  return eh, ee, vol / N * np.sum(e * rho.sum(0)), np.stack(vs)


@pytest.mark.parametrize("n,nz", [(n, n) for n in PLANES] +
                         [(36, z) for z in LINES[-12:]] + [(64, 45)])
def test_fused_potential_stage(n, nz):
  """Energies of the evaluation's own density, and band mode's potential
  energy sum f <psi|v|psi> = (vol / N) sum_r v rho at a given density."""
  cell = np.array([[7.1, 0.3, 0.0], [0.0, 6.7, -0.4], [0.2, 0.0, 6.6 * nz / n]])
  vol = float(np.linalg.det(cell))
  B = 2 * np.pi * np.linalg.inv(cell).T
  fr = [np.fft.fftfreq(m, 1 / m) for m in (n, n, nz)]
  M = np.stack(np.meshgrid(*fr, indexing="ij"), -1)
  G = M @ B
  mask = (np.abs(M / np.array([n, n, nz]))**2).sum(-1) <= 0.16**2
  pos, chg = np.array([[0.1, 0.2, 0.3], [2.5, 2.9, 3.1]]), np.array([4.0, 3.0])
  for ns in (1, 2):
    occ = np.full((ns, 1, 2), 2.0 / ns)
    kpts = np.zeros((1, 3))
    plan = EnergyPlan(pos, chg, cell, mask, kpts, occ)
    gen = torch.Generator(device="cuda").manual_seed(n)
    w = [torch.randn(plan.param_shape, generator=gen, device="cuda",
                     dtype=torch.float64) for _ in range(2)]
    r = plan.evaluate(*w, grad=False, density=True)
    rho = r["density"].cpu().numpy()
    e = r["energies"].cpu().numpy()
    eh, ee, ex, _ = _potential(rho, G, vol, pos, chg)
    np.testing.assert_allclose(e[1:4], [eh, ee, ex], rtol=1e-12)
    fixed = 0.02 + 0.01 * np.cos(np.arange(ns * n * n * nz)).reshape(rho.shape)
    plan.set_fixed_density(fixed)
    e = plan.evaluate(*w, grad=False)["energies"].cpu().numpy()
    v = _potential(fixed, G, vol, pos, chg)[3]
    # sums over N points with cancellation between the signs of v
    np.testing.assert_allclose(e[1], vol / rho[0].size * np.sum(v * rho),
                               rtol=1e-11)
    plan.close()
