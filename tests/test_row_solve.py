"""The register Cholesky solve (32-lane teams) where a 16-lane row or a padded
group of four columns begins or ends: residuals against the backward error
bound of a float32 Cholesky solve, |M x - b| <= g |L| |L'| |x| with
g = 4 (3 n + 4) eps: gamma_{3 n + 1} of the textbook bound, with 4 for the
hardware's square root and reciprocal in place of correctly rounded ones."""
import numpy as np
import pytest
import torch

import helpers
import mjx_warp_amd as mjw
from mjx_warp_amd import models

pytestmark = pytest.mark.gpu


def _within(M, x, b):
  n = M.shape[-1]
  g = 4 * (3 * n + 4) * np.finfo(np.float32).eps
  for w in range(len(M)):
    A, y = M[w].astype(np.float64), x[w].astype(np.float64)
    L = np.abs(np.linalg.cholesky(A))
    assert np.all(np.abs(A @ y - b[w]) <= g * (L @ (L.T @ np.abs(y)))), w


@pytest.mark.parametrize("nv", [1, 4, 5, 15, 16, 17, 20, 28, 29, 31, 32])
def test_row_solve(nv):
  nworld = 3  # an odd world: half a wavefront without one
  mjm = models.chain(nv)
  m = mjw.put_model(mjm)
  d = mjw.make_data(mjm, nworld=nworld, nconmax=16 * nworld, njmax=64 * nworld)
  rng = np.random.default_rng(nv)
  A = rng.normal(size=(nworld, nv, nv))
  M = (A @ A.transpose(0, 2, 1) + nv * np.eye(nv)).astype(np.float32)
  b = rng.normal(size=(nworld, nv)).astype(np.float32)
  helpers.set_field(d, "qM", M)
  mjw.factor_m(m, d)
  x, y = torch.zeros(nworld, nv, device="cuda"), torch.as_tensor(b, device="cuda")
  mjw.solve_m(m, d, x, y)
  torch.cuda.synchronize()
  _within(M, x.cpu().numpy(), b)
  # the fused step's factor and solve stay in registers
  helpers.set_field(d, "qpos", rng.uniform(-0.3, 0.3, (nworld, nv)))
  helpers.set_field(d, "qvel", rng.uniform(-0.3, 0.3, (nworld, nv)))
  mjw.step_fused(m, d)
  torch.cuda.synchronize()
  f = {k: helpers.data_numpy(d, k) for k in ("qM", "qacc_smooth", "qfrc_smooth")}
  _within(f["qM"].reshape(nworld, nv, nv), f["qacc_smooth"].reshape(nworld, nv), f["qfrc_smooth"].reshape(nworld, nv))
