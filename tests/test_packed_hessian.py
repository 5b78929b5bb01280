"""The 64-lane solver's packed Newton Hessian (two rows per lane) against the
square one in LDS (MJH_SOLVER_WIDE=0): the same bits."""

import numpy as np
import pytest
import torch

import mjx_warp_amd as mjw
from mjx_warp_amd import models

import helpers

pytestmark = pytest.mark.gpu


def _state(links, balls, nworld):
  """A hanging chain and spheres lying a little in the floor on a lattice."""
  rng = np.random.default_rng(links + balls)
  q = np.zeros((nworld, links + 7 * balls))
  q[:, :links] = rng.uniform(-0.1, 0.1, (nworld, links))
  for k in range(balls):
    a = links + 7 * k
    q[:, a:a + 2] = [0.15 * (k % 5) - 0.3, 0.15 * (k // 5) - 0.3]
    q[:, a:a + 2] += rng.uniform(-0.01, 0.01, (nworld, 2))
    q[:, a + 2] = rng.uniform(0.047, 0.051, nworld)
    q[:, a + 3] = 1.0
  return q, rng.normal(0.0, 0.3, (nworld, links + 6 * balls))


# nv 33, 63, 64, 65, 80, 81, 128, 129: one row set with a remainder, a lane
# less than full, full, one row in the second set, a whole panel there, one
# more, the largest, and the first that is not packed
@pytest.mark.parametrize("links,balls", [(3, 5), (3, 10), (4, 10), (5, 10), (2, 13), (3, 13), (2, 21), (3, 21)])
def test_packed_equals_square(links, balls, monkeypatch):
  mjm = models.box_world(links, (0.05,) * balls)
  m = mjw.put_model(mjm)
  nv = int(mjm.nv)
  q, v = _state(links, balls, 3)
  out = []
  for square in (False, True):
    if square:
      monkeypatch.setenv("MJH_SOLVER_WIDE", "0")
    d = mjw.make_data(mjm, nworld=3, nconmax=3 * 4 * nv, njmax=3 * 20 * nv)
    helpers.set_field(d, "qpos", q)
    helpers.set_field(d, "qvel", v)
    mjw.step_fused(m, d)
    torch.cuda.synchronize()
    assert int(helpers.data_numpy(d, "nefc")[0]) > 0
    out.append({f: helpers.data_numpy(d, f) for f in ("qacc", "qfrc_constraint", "qvel", "efc_cost")})
  for f, a in out[0].items():
    assert np.isfinite(a).all() and np.array_equal(a, out[1][f]), f
