"""The fused step's LDS-resident forward stages against the per-stage entry
points: every field the stages write, and the pools per world."""

from pathlib import Path

import numpy as np
import pytest
import torch

import mjx_warp_amd as mjw
from mjx_warp_amd import mjcf, models

import helpers

pytestmark = pytest.mark.gpu

GOLDEN = Path(__file__).parent / "golden"
# the suite's tolerance for kinematics, inertias and smooth forces
TOL = 2e-4
WORLD = ("xpos", "xquat", "xmat", "xipos", "ximat", "xanchor", "xaxis", "geom_xpos", "geom_xmat", "site_xpos",
         "site_xmat", "subtree_com", "cdof", "cinert", "crb", "qM", "actuator_length", "actuator_moment",
         "actuator_velocity", "actuator_force", "cvel", "cdof_dot", "qfrc_bias", "qfrc_spring", "qfrc_damper",
         "qfrc_passive", "qfrc_actuator", "qfrc_smooth", "rne_cacc", "rne_cfrc")
CONTACT = ("dist", "pos", "frame", "includemargin", "friction", "solref", "solimp", "dim", "geom")
ROW = ("J", "D", "aref", "pos", "margin")


def _scene(name):
  if name.endswith(".xml"):
    return mjcf.from_xml_path(str(GOLDEN / name))
  if name == "humanoid":
    return models.humanoid(iterations=2, ls_iterations=4)
  if name == "three":  # 64-lane teams, sparse mass matrix
    return mjcf.from_xml_path(str(models.ASSETS / "n_humanoids.xml"))
  if name == "chain1":  # one dof
    return models.chain(1)
  if name == "crowd":  # 35 pairs and contacts: more than a team's lanes, three chunks of rows
    return models.box_world(2, (0.6,) * 5)
  return models.box_world(8, (0.05,) * 4)  # nv 32


@pytest.mark.parametrize("name", ["humanoid", "three", "chain1", "crowd", "box", "pendula.xml", "constraints.xml",
                                  "collision.xml"])
@pytest.mark.parametrize("nworld", [1, 5])
def test_resident_forward_equals_stages(name, nworld):
  mjm = _scene(name)
  m = mjw.put_model(mjm)
  rng = np.random.default_rng(nworld)
  q = np.tile(np.asarray(mjm.qpos0, np.float64), (nworld, 1)) + rng.normal(0.0, 0.05, (nworld, mjm.nq))
  v = rng.normal(0.0, 0.3, (nworld, mjm.nv))
  u = rng.uniform(-1.0, 1.0, (nworld, mjm.nu))
  x = rng.normal(0.0, 1.0, (nworld, mjm.nbody, 6))
  out = []
  for step in (mjw.step_fused, mjw.step):
    d = mjw.make_data(mjm, nworld=nworld, nconmax=256 * nworld, njmax=1024 * nworld)
    helpers.set_field(d, "qpos", q)
    helpers.set_field(d, "qvel", v)
    helpers.set_field(d, "ctrl", u)
    helpers.set_field(d, "xfrc_applied", x)
    step(m, d)
    torch.cuda.synchronize()
    out.append(d)
  get = lambda k, f: helpers.data_numpy(out[k], f)
  for f in ("ncollision", "ncon", "nefc", "overflow"):
    assert np.array_equal(get(0, f), get(1, f)), (f, get(0, f), get(1, f))
  close = lambda a, b, f: np.testing.assert_allclose(a, b, atol=TOL * (1.0 + np.nanmax(np.abs(b), initial=0.0)), err_msg=f)
  for f in WORLD:
    close(get(0, f), get(1, f), f)
  for fields, prefix, world in ((CONTACT, "contact_", "world_con"), (ROW, "efc_", "world_efc")):
    blocks = [helpers.world_blocks(get(k, world), nworld) for k in range(2)]
    assert [n for _, n in blocks[0]] == [n for _, n in blocks[1]]
    for f in fields:
      a, b = (helpers.gather_world_rows(get(k, prefix + f), blocks[k]) for k in range(2))
      close(a, b, prefix + f)


def _more_bodies_than_lanes(n):
  """n bodies under the world, all but three fixed, joints of three kinds."""
  joint = {0: '<joint axis="0 1 0" stiffness="2" damping=".1"/>', 15: '<joint type="ball"/>',
           31: '<joint type="slide" axis="0 0 1"/>'}
  body = lambda i: (f'<body pos=".02 0 -.05" euler="0 {3 * i} 5"><inertial pos="0 0 .01" mass=".1" diaginertia="1e-4 2e-4 3e-4"/>'
                    + joint.get(i, "") + ('<geom size=".02"/>' if i % 15 == 0 else ""))
  return mjcf.from_xml_string('<mujoco><option jacobian="dense"/><worldbody><geom type="plane" size="5 5 .1"/>'
                              + "".join(body(i) for i in range(n)) + "</body>" * n + "</worldbody></mujoco>")


def _heap():
  """64-lane teams, 90 and more pairs: the pair list is emptied and begun again."""
  ball = lambda i: f'<body pos="{.02 * (i % 4)} {.02 * (i // 4)} .05"><freejoint/><geom size=".1"/></body>'
  return mjcf.from_xml_string('<mujoco><option jacobian="dense"/><worldbody><geom type="plane" size="5 5 .1"/>'
                              + "".join(ball(i) for i in range(14)) + "</worldbody></mujoco>")


@pytest.mark.parametrize("name", ["humanoid", "three", "crowd", "box", "pendula.xml", "constraints.xml", "collision.xml",
                                  "bodies33", "bodies63", "bodies64", "chain32", "heap"])
def test_resident_forward_is_the_stages_bit_for_bit(name):
  nworld = 5
  # (63 bodies: with the world's the most that the resident form takes)
  mjm = (_more_bodies_than_lanes(int(name[6:])) if name.startswith("bodies") else _heap() if name == "heap"
         else models.chain(32) if name == "chain32" else _scene(name))
  m = mjw.put_model(mjm)
  rng = np.random.default_rng(nworld)
  q = np.tile(np.asarray(mjm.qpos0, np.float64), (nworld, 1)) + rng.normal(0.0, 0.05, (nworld, mjm.nq))
  state = {"qpos": q, "qvel": rng.normal(0.0, 0.3, (nworld, mjm.nv)), "ctrl": rng.uniform(-1.0, 1.0, (nworld, mjm.nu)),
           "xfrc_applied": rng.normal(0.0, 1.0, (nworld, mjm.nbody, 6)), "qfrc_applied": rng.normal(0.0, 1.0, (nworld, mjm.nv))}
  out = []
  for step in (mjw.step_fused, mjw.step):
    d = mjw.make_data(mjm, nworld=nworld, nconmax=256 * nworld, njmax=1024 * nworld)
    for f, v in state.items():
      helpers.set_field(d, f, v)
    step(m, d)
    torch.cuda.synchronize()
    out.append(d)
  get = lambda k, f: helpers.data_numpy(out[k], f)
  assert not np.any(get(0, "overflow"))
  if name == "heap":
    assert min(n for _, n in helpers.world_blocks(get(0, "world_pair"), nworld)) > 64
  for f in WORLD:
    assert np.array_equal(get(0, f), get(1, f), equal_nan=True), f
  for fields, prefix, world in ((CONTACT, "contact_", "world_con"), (ROW, "efc_", "world_efc")):
    blocks = [helpers.world_blocks(get(k, world), nworld) for k in range(2)]
    assert [n for _, n in blocks[0]] == [n for _, n in blocks[1]]
    for f in fields:
      a, b = (helpers.gather_world_rows(get(k, prefix + f), blocks[k]) for k in range(2))
      assert np.array_equal(a, b, equal_nan=True), prefix + f
