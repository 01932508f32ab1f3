"""Cholesky inverse and adjoint factors on 16 x 16 tiles, through jrx_qr and
jrx_qr_backward: band counts around the tile edges, against LAPACK."""
import numpy as np
import pytest
import torch

from jrystal_amd import _lib, _ops
from jrystal_amd.objective import EnergyPlan

pytestmark = pytest.mark.gpu


def _householder(w):
  """Q, R of w (g, b) with a real positive diagonal of R."""
  q, r = np.linalg.qr(w)
  ph = np.diag(r) / np.abs(np.diag(r))
  return q * ph, r / ph[:, None]


@pytest.mark.parametrize("nb", (1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63,
                                64, 65, 80, 81, 96, 97, 112, 113, 127, 128))
def test_qr_and_adjoint_of_every_tile_count(nb):
  L, P, ng = _lib.lib(), 2, 300
  rng = np.random.default_rng(nb)
  w = rng.standard_normal((P, ng, nb)) + 1j * rng.standard_normal((P, ng, nb))
  # the second problem needs the second pass: columns of unequal size that
  # share a common part
  w[1] = w[1] * np.logspace(0, 2, nb) + 3 * w[1, :, :1]
  qb = rng.standard_normal((P, nb, ng)) + 1j * rng.standard_normal((P, nb, ng))
  dev = lambda x: torch.tensor(x, device="cuda")  # noqa: E731
  wr, wi = dev(w.real.copy()), dev(w.imag.copy())
  q = torch.empty((P, nb, ng), dtype=torch.complex128, device="cuda")
  ri = torch.empty((P, nb, nb), dtype=torch.complex128, device="cuda")
  ws, wp = _ops.workspace(L.jrx_qr_workspace_bytes(P, ng, nb))
  s = _lib.stream_ptr()
  _lib.check(L.jrx_qr(wr.data_ptr(), wi.data_ptr(), P, ng, nb, q.data_ptr(),
                      ri.data_ptr(), wp, ws.numel() - 256, s))
  gr, gi = torch.empty_like(wr), torch.empty_like(wi)
  qbd = dev(qb)
  _lib.check(L.jrx_qr_backward(q.data_ptr(), qbd.data_ptr(), ri.data_ptr(), P,
                               ng, nb, gr.data_ptr(), gi.data_ptr(), wp,
                               ws.numel() - 256, s))
  Q, Ri = q.cpu().numpy(), ri.cpu().numpy()
  G = gr.cpu().numpy() + 1j * gi.cpu().numpy()
  for p in range(P):
    ref, r = _householder(w[p])
    inv = np.linalg.inv(r)
    # forward errors scale with the condition number of W
    tol = 1e-14 * np.linalg.cond(w[p])
    assert np.allclose(Q[p].conj() @ Q[p].T, np.eye(nb), atol=1e-13)
    assert np.linalg.norm(Q[p].T - ref) <= tol * np.sqrt(nb)
    assert np.linalg.norm(Ri[p] - inv) <= tol * nb * np.linalg.norm(inv)
    assert np.all(np.tril(Ri[p], -1) == 0)
    M = -(qb[p].conj() @ ref)  # -Qbar^H Q
    low = np.tril(M, -1)
    C = low + low.conj().T + np.diag(np.diag(M).real)
    want = (qb[p].T + ref @ C) @ inv.conj().T
    assert np.linalg.norm(G[p] - want) <= 10 * tol * nb * \
        np.linalg.norm(want)


@pytest.mark.parametrize("nb", (3, 20, 40, 70, 128))
def test_dependent_columns_give_nan(nb):
  """A Gram matrix with a non-positive pivot poisons the result."""
  L, ng = _lib.lib(), 200
  w = np.random.default_rng(0).standard_normal((1, ng, nb))
  w[0, :, nb // 2] = 0.0
  wr = torch.tensor(w, device="cuda")
  wi = torch.zeros_like(wr)
  q = torch.empty((1, nb, ng), dtype=torch.complex128, device="cuda")
  ri = torch.empty((1, nb, nb), dtype=torch.complex128, device="cuda")
  ws, wp = _ops.workspace(L.jrx_qr_workspace_bytes(1, ng, nb))
  _lib.check(L.jrx_qr(wr.data_ptr(), wi.data_ptr(), 1, ng, nb, q.data_ptr(),
                      ri.data_ptr(), wp, ws.numel() - 256, _lib.stream_ptr()))
  assert torch.isnan(torch.view_as_real(q)).any()


@pytest.mark.parametrize("nb", (1, 16, 17, 32, 33, 48, 64, 65, 100, 128))
def test_one_pass_columns_have_unit_norm(nb):
  """Rounding of the pivots' inverse square roots alone: columns with one
  nonzero entry c each have an exactly diagonal Gram matrix, so that the
  adaptive QR takes one pass and |Q| = |c| / sqrt(fl(c^2)).  With u = 2^-53:
  half of the square's u, 1.25 u of the root (1.4e-16) and u of the product
  make less than 3 u."""
  f = np.arange(16)
  f = np.where(f < 8, f, f - 16)
  mask = f[:, None, None]**2 + f[:, None]**2 + f**2 <= 21
  ng, nk = int(mask.sum()), 8
  plan = EnergyPlan(np.zeros((1, 3)), np.array([4.0]), 8.0 * np.eye(3), mask,
                    np.zeros((nk, 3)), np.ones((1, nk, nb)))
  rng = np.random.default_rng(nb)
  c = np.exp(rng.uniform(-20.0, 20.0, (nk, nb)))
  rows = np.stack([rng.permutation(ng)[:nb] for _ in range(nk)])
  w = np.zeros((1, nk, ng, nb))
  np.put_along_axis(w[0], rows[:, None], c[:, None], axis=1)
  w = torch.tensor(w, device="cuda")
  plan.evaluate(w, torch.zeros_like(w), grad=False)
  q = plan.orthonormal_params()[0].cpu().numpy()[0]
  got = np.take_along_axis(q, rows[:, None], axis=1)[:, 0]
  assert np.count_nonzero(q) == nk * nb
  assert np.max(np.abs(got - 1)) <= 3 * 2.0**-53
