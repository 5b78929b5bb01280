"""Sweep-and-prune collision by several wavefronts a world, and by one inside
the fused step: the pairs and their order against the oracle, at the sizes
where the path changes (the smallest, one geom past a team's or workgroup's
multiple, the last sorted by counting and the first by radix, the last with
staged filter ints) and where a wavefront has more pairs than it has bits for."""
import numpy as np
import pytest
import torch

import helpers
import mjx_warp_amd as mjw
from oracle import oracle
from mjx_warp_amd import mjcf
from test_gpu_parity import _gpu_and_oracle

pytestmark = pytest.mark.gpu


def _scene(ngeom, movers, spread):
  """movers free spheres and capsules among static ones over a floor, in a
  box of `spread` m whose projections on the sweep direction overlap the more
  the smaller it is."""
  rng = np.random.default_rng(ngeom)
  n = ngeom - 1
  pos = rng.uniform(-spread, spread, (n, 3)) + [0, 0, spread]
  rad = rng.uniform(0.05, 0.12, n)
  at = lambda i: f'pos="{pos[i, 0]:.3f} {pos[i, 1]:.3f} {pos[i, 2]:.3f}"'
  geom = lambda i, p: f'<geom {p} type="{"sphere" if i % 2 else "capsule"}" size="{rad[i]:.3f} 0.1"/>'
  bodies = "".join(f'<body {at(i)}><freejoint/>{geom(i, "")}</body>' for i in range(movers))
  static = "".join(geom(i, at(i)) for i in range(movers, n))
  return mjcf.from_xml_string('<mujoco><option jacobian="dense"/><worldbody><geom type="plane" size="5 5 .1"/>'
                              f'{static}{bodies}</worldbody></mujoco>')


def _same_pairs(d, hd, nworld):
  gp = helpers.world_blocks(helpers.data_numpy(d, "world_pair"), nworld)
  op = helpers.world_blocks(hd["world_pair"], nworld)
  assert [n for _, n in gp] == [n for _, n in op]
  assert min(n for _, n in gp) > 0
  assert np.array_equal(helpers.gather_world_rows(helpers.data_numpy(d, "collision_pair"), gp),
                        helpers.gather_world_rows(hd["collision_pair"], op))
  gc = helpers.world_blocks(helpers.data_numpy(d, "world_con"), nworld)
  oc = helpers.world_blocks(hd["world_con"], nworld)
  assert [n for _, n in gc] == [n for _, n in oc]


def _inputs(mjm, nworld, nconmax_w):
  q = np.tile(mjm.qpos0, (nworld, 1))
  rng = np.random.default_rng(3)
  for k in range(0, mjm.nq, 7):
    q[1:, k:k + 3] += rng.normal(0, 0.05, (nworld - 1, 3))
  return _gpu_and_oracle(mjm, nworld, q, nconmax_w=nconmax_w, njmax_w=4)


@pytest.mark.parametrize("ngeom,spread", [(101, 1.0), (129, 1.0), (513, 1.0), (1024, 2.0), (1025, 0.8)])
def test_pair_waves_match_oracle(ngeom, spread):
  mjm = _scene(ngeom, 40, spread)
  assert mjm.nv > 32
  m, d, hm, hd = _inputs(mjm, 3, 8192)
  mjw.kinematics(m, d)
  mjw.collision(m, d)
  torch.cuda.synchronize()
  oracle.run("kinematics", hm, hd)
  oracle.run("collision", hm, hd)
  _same_pairs(d, hd, 3)


@pytest.mark.parametrize("ngeom,movers", [(101, 5), (400, 5), (101, 8), (400, 8)])
def test_fused_step_pairs_match_oracle(ngeom, movers):
  """nv 30 (32-lane teams) and 48 (64-lane teams)."""
  mjm = _scene(ngeom, movers, 0.5)
  mjm.opt.disableflags |= int(mjw.DisableBit.CONSTRAINT)
  m, d, hm, hd = _inputs(mjm, 3, 8192)
  mjw.step(m, d)
  torch.cuda.synchronize()
  oracle.run("kinematics", hm, hd)
  oracle.run("collision", hm, hd)
  _same_pairs(d, hd, 3)


# one wavefront a world, two worlds (nv 30) or one (nv 48) in it: the smallest
# model, more candidates than a lane has bits for (64 chunks of 32 or 64), the
# last with staged filter ints and the first without
@pytest.mark.parametrize("ngeom,spread", [(101, 0.5), (400, 0.3), (1024, 1.0), (1025, 1.0)])
@pytest.mark.parametrize("movers", [5, 8])
def test_one_wavefront_pairs_match_oracle(ngeom, spread, movers):
  mjm = _scene(ngeom, movers, spread)
  assert mjm.nv == 6 * movers
  mjm.opt.disableflags |= int(mjw.DisableBit.CONSTRAINT)
  m, d, hm, hd = _inputs(mjm, 3, 32768)
  mjw.step_fused(m, d)
  torch.cuda.synchronize()
  oracle.run("kinematics", hm, hd)
  oracle.run("collision", hm, hd)
  assert not np.any(hd["overflow"])
  _same_pairs(d, hd, 3)
  if ngeom == 400:
    assert helpers.data_numpy(d, "sap_cumulative_sum").reshape(3, -1)[:, ngeom - 1].min() > 64 * 64
