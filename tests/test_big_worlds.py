"""Worlds with 65 to 256 constraint rows (the big-world launch): found by the
bit map in Data.step_desc and, without one, in place -- the same bits."""

import numpy as np
import pytest
import torch

import mjx_warp_amd as mjw
from mjx_warp_amd import models

import helpers

pytestmark = pytest.mark.gpu


def _lying(mjm, nworld, every):
  """Humanoids in the air, every `every`-th one lying in the floor."""
  rng = np.random.default_rng(nworld)
  q = np.tile(np.asarray(mjm.key_qpos[2]), (nworld, 1))  # "no_efc"
  low = np.arange(nworld) % every == every - 1
  q[low, 2] = rng.uniform(0.02, 0.05, int(low.sum()))
  q[low, 3:7] = [np.sqrt(0.5), 0.0, np.sqrt(0.5), 0.0]
  q[low, 7:] = rng.normal(0.0, 0.1, (int(low.sum()), mjm.nq - 7))
  return q


# one world; the map's first word full and a second begun; more words than
# lanes; the last world count the map holds and the first it does not
@pytest.mark.parametrize("nworld,every", [(1, 1), (33, 1), (2081, 3), (32768, 4096), (32769, 4096)])
@pytest.mark.parametrize("fused", [True, False])
def test_big_world_map_equals_in_place(nworld, every, fused):
  mjm = models.humanoid(iterations=10, ls_iterations=20)
  m = mjw.put_model(mjm)
  out = []
  for desc in (True, False):
    # each lying world reaches about 30 contacts and 140 rows, the others none
    k = nworld // every + 1
    d = mjw.make_data(mjm, nworld=nworld, nconmax=40 * nworld, njmax=200 * k)
    if not desc:
      d.ndesc = 0
      d.step_desc = torch.zeros(0, dtype=torch.int32, device=d.qpos.device)
    helpers.set_field(d, "qpos", _lying(mjm, nworld, every))
    (mjw.step_fused if fused else mjw.step)(m, d)
    torch.cuda.synchronize()
    rows = helpers.data_numpy(d, "world_efc").reshape(-1, 2)[:nworld, 1]
    assert np.sum(rows > 64) >= 1 and rows.max() <= 256, rows.max()
    assert not np.any(helpers.data_numpy(d, "overflow")) and not np.any(helpers.data_numpy(d, "world_flags"))
    out.append({f: getattr(d, f).cpu() for f in ("qpos", "qvel", "qacc", "qfrc_constraint")})
  for f, a in out[0].items():
    assert torch.isfinite(a).all()
    assert torch.equal(a, out[1][f]), f
