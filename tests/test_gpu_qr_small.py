"""Cholesky inverse and adjoint factors on 16 x 16 tiles, through jrx_qr and
jrx_qr_backward: band counts around the tile edges, against LAPACK."""
import numpy as np
import pytest
import torch

from jrystal_amd import _lib, _ops

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
