"""The work that programs have this framework do, as measurable cases.

Every case goes through the public entry points of `mjx_warp_amd`: whole
steps (fused, per stage, replayed from a HIP graph, heterogeneous batches),
the differentiable rollout, and the single stages that planners, samplers and
inverse-dynamics programs call on their own (kinematics to bias forces and
the mass-matrix solve, collision, the constraint solver).  Models are the
repository's: the 27-dof humanoid (Newton 10 / 20, implicitfast), three
attached humanoids (nv 81, sparse mass matrix, Euler), hinge chains (CG,
Euler), chains and spheres in a walled box, and 256 free bodies in a box.

Step cases start every pass from the case's own state (positions, velocities,
controls and the solver's warm start are copied in, as a sampler that
evaluates controls from one state does).
"""

from __future__ import annotations

import functools
import math

import numpy as np
import torch

import mjx_warp_amd as mjw
from mjx_warp_amd import derivative, mjcf, models

DEV = "cuda"


def listed():
  return [
    # one simulated robot in a control loop: latency of the functional step
    {"name": "step_single", "kind": "functional", "model": "humanoid", "nworld": 1},
    # a small batch of hinge chains with the CG solver, one call per step
    {"name": "step_chain_small", "kind": "step", "model": "chain", "links": 5, "nworld": 37, "nstep": 1, "fused": False},
    # the batched fused step, the usual reinforcement-learning batch
    {"name": "step_fused_8192", "kind": "step", "model": "humanoid", "nworld": 8192, "nstep": 2, "fused": True, "pose": "squat"},
    # a large batch in which many robots lie on the floor (many constraint rows)
    {"name": "step_fallen_24576", "kind": "step", "model": "humanoid", "nworld": 24576, "nstep": 2, "fused": True, "pose": "fallen"},
    # the reference-shaped step, one launch per stage, on a ragged batch
    {"name": "step_plain_1000", "kind": "step", "model": "humanoid", "nworld": 1000, "nstep": 1, "fused": False, "pose": "squat"},
    # a captured rollout replayed as one graph
    {"name": "graph_chain_4096", "kind": "graph", "model": "chain", "links": 3, "nworld": 4096, "nstep": 10},
    # wide models: three humanoids in one world, nv 81, 64-lane path
    {"name": "step_wide_1024", "kind": "step", "model": "n_humanoids", "nworld": 1024, "nstep": 1, "fused": True, "pose": "squat"},
    # many models in one batch, domain randomisation over morphologies
    {"name": "multi_16384", "kind": "multi", "nworld": 16384, "max_links": 8, "max_spheres": 4, "nstep": 2},
    # trajectory optimisation: forward rollout and its adjoint
    {"name": "rollout_grad_1024", "kind": "grad", "nworld": 1024, "nstep": 8},
    # kinematics to bias forces and the mass-matrix solve, stage by stage
    {"name": "smooth_4096", "kind": "smooth", "model": "humanoid", "nworld": 4096},
    # sweep-and-prune collision of piles of free bodies
    {"name": "collide_pile_256", "kind": "collide", "nbody": 256, "nworld": 256},
    # the constraint solver on rows that the caller laid out
    {"name": "solve_4096", "kind": "solve", "nworld": 4096, "rows": 24},
  ]


def _log(rng, lo, hi):
  return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
  kind = rng.choice(["functional", "step", "step", "step", "graph", "multi", "grad", "smooth", "collide", "solve"])
  if kind == "functional":
    return {"kind": kind, "model": "humanoid", "nworld": _log(rng, 1, 300)}
  if kind == "step":
    model = rng.choice(["humanoid", "humanoid", "chain", "n_humanoids"])
    if model == "chain":
      return {"kind": kind, "model": model, "links": rng.randint(2, 20), "nworld": _log(rng, 1, 20000),
              "nstep": rng.randint(1, 2), "fused": rng.random() < 0.5}
    top = 20000 if model == "humanoid" else 700
    return {"kind": kind, "model": model, "nworld": _log(rng, 16, top), "nstep": rng.randint(1, 2),
            "fused": rng.random() < 0.7, "pose": rng.choice(["squat", "fallen"]) if model == "humanoid" else "squat"}
  if kind == "graph":
    return {"kind": kind, "model": "chain", "links": rng.randint(2, 12), "nworld": _log(rng, 16, 4000),
            "nstep": rng.randint(2, 10)}
  if kind == "multi":
    return {"kind": kind, "nworld": _log(rng, 200, 12000), "max_links": rng.randint(3, 8),
            "max_spheres": rng.randint(1, 4), "nstep": 1}
  if kind == "grad":
    return {"kind": kind, "nworld": _log(rng, 32, 1000), "nstep": rng.randint(2, 6)}
  if kind == "smooth":
    model = rng.choice(["humanoid", "n_humanoids"])
    return {"kind": kind, "model": model, "nworld": _log(rng, 64, 4000 if model == "humanoid" else 500)}
  if kind == "collide":
    return {"kind": kind, "nbody": rng.randint(100, 250), "nworld": _log(rng, 8, 250)}
  return {"kind": kind, "nworld": _log(rng, 64, 4000), "rows": rng.randint(4, 40)}


# ---------------------------------------------------------------- models

@functools.lru_cache(maxsize=None)
def _compiled(kind, *args):
  if kind == "humanoid":
    return models.humanoid(iterations=10, ls_iterations=20)
  if kind == "chain":  # hung so that the straight chain's tip grazes the floor
    return mjcf.from_xml_string(models.chain_xml(args[0], anchor_z=0.5 * args[0]))
  if kind == "n_humanoids":
    return mjcf.from_xml_path(str(models.ASSETS / "n_humanoids.xml"))
  if kind == "box":
    return models.box_world(args[0], args[1])
  return models.contact_heavy(args[0])


def _model(case):
  return _compiled("chain", case["links"]) if case["model"] == "chain" else _compiled(case["model"])


def _dev(a):
  return torch.tensor(np.asarray(a), dtype=torch.float32, device=DEV)


def _capacity(case, mjm):
  """(contacts, rows) per world: the benchmark's for the humanoid."""
  if case["model"] == "humanoid":
    return 64, 4 * 64 + 21
  if case["model"] == "chain":
    return 8 * mjm.nbody, 32 * mjm.nbody + mjm.njnt
  return 192, 4 * 192 + 63


def _humanoid_state(rng, key_qpos, n, pose):
  """[n, 28] positions and [n, 27] velocities: the squat keyframe with its
  feet from a little in the floor to above it, or ("fallen") every third
  robot lying near the floor in any orientation, limbs spread."""
  q = np.tile(np.asarray(key_qpos, np.float64), (n, 1))
  q[:, 0:2] += rng.normal(0.0, 0.05, (n, 2))
  q[:, 2] += rng.uniform(-0.005, 0.12, n)
  q[:, 7:] += rng.normal(0.0, 0.05, (n, 21))
  rot = rng.normal(0.0, 0.05, (n, 3))
  v = rng.normal(0.0, 0.3, (n, 27))
  if pose == "fallen":
    low = np.arange(n) % 3 == 0
    k = int(low.sum())
    q[low, 2] = rng.uniform(0.1, 0.2, k)
    q[low, 7:] = rng.normal(0.0, 0.15, (k, 21))
    q[low, 3:7] = [math.sqrt(0.5), 0.0, math.sqrt(0.5), 0.0]  # on the back or the belly
    rot[low] = rng.normal(0.0, 0.1, (k, 3))
  ang = np.linalg.norm(rot, axis=1, keepdims=True)
  dq = np.concatenate([np.cos(0.5 * ang), rot * (np.sin(0.5 * ang) / ang)], 1)
  q[:, 3:7] = _qmul(q[:, 3:7], dq)
  q[:, 3:7] /= np.linalg.norm(q[:, 3:7], axis=1, keepdims=True)
  return q, v


def _states(case, mjm, rng):
  n = case["nworld"]
  if case["model"] == "chain":
    return rng.uniform(-0.5, 0.5, (n, mjm.nq)), rng.normal(0.0, 0.1, (n, mjm.nv))
  key = _compiled("humanoid").key_qpos[0]
  pose = case.get("pose", "squat")
  if case["model"] == "humanoid":
    return _humanoid_state(rng, key, n, pose)
  qs, vs = [], []
  for k in range(mjm.nq // 28):
    q, v = _humanoid_state(rng, key, n, pose)
    q[:, 0:2] += np.asarray(mjm.qpos0)[28 * k:28 * k + 2]
    qs.append(q)
    vs.append(v)
  return np.concatenate(qs, 1), np.concatenate(vs, 1)


_GRAPHS = []  # captured rollouts live as long as the program, as a server's do


def _reset(s):
  torch._foreach_copy_(s["dst"], s["src"])


# ---------------------------------------------------------------- prepare / run

def prepare(case, seed):
  rng = np.random.default_rng(seed)
  return _PREPARE[case["kind"]](case, rng)


def run(state):
  return _RUN[state["kind"]](state)


def _prepare_step(case, rng):
  mjm = _model(case)
  n = case["nworld"]
  m = mjw.put_model(mjm)
  ncon, nrow = _capacity(case, mjm)
  d = mjw.make_data(mjm, nworld=n, nconmax=ncon * n, njmax=nrow * n)
  q, v = _states(case, mjm, rng)
  src = [_dev(q), _dev(v), torch.zeros((n, mjm.nv), device=DEV), _dev(rng.uniform(-1.0, 1.0, (n, mjm.nu)))]
  s = {"kind": case["kind"], "m": m, "d": d, "nstep": case.get("nstep", 1), "fused": case.get("fused", True),
       "src": src, "dst": [d.qpos, d.qvel, d.qacc_warmstart, d.ctrl]}
  if mjm.nu == 0:
    s["src"], s["dst"] = s["src"][:3], s["dst"][:3]
  _reset(s)
  if case["kind"] == "graph":
    s["graph"] = mjw.StepGraph(m, d, nstep=case["nstep"])
    _GRAPHS.append(s["graph"])
  if case["kind"] == "functional":
    s["f"] = mjw.FunctionalStep(m, d)
  return s


def _run_step(s):
  _reset(s)
  m, d = s["m"], s["d"]
  if s["nstep"] > 1:
    mjw.rollout(m, d, s["nstep"], s["fused"])
  elif s["fused"]:
    mjw.step_fused(m, d)
  else:
    mjw.step(m, d)
  return d.qpos, d.qvel


def _run_functional(s):
  return s["f"](s["src"][0], s["src"][1], s["src"][3])


def _run_graph(s):
  _reset(s)
  s["graph"].replay()
  return s["d"].qpos, s["d"].qvel


def _prepare_multi(case, rng):
  spec = models.heterogeneous_groups(case["nworld"], max_links=case["max_links"], max_spheres=case["max_spheres"])
  groups, src, dst = [], [], []
  for links, radii, n in spec:
    mjm = _compiled("box", links, radii)
    m = mjw.put_model(mjm)
    ncon = 8 * (links + len(radii))
    d = mjw.make_data(mjm, nworld=n, nconmax=ncon * n, njmax=(4 * ncon + mjm.njnt) * n)
    q, v = np.zeros((n, mjm.nq)), rng.normal(0.0, 0.3, (n, mjm.nv))
    q[:, :links] = rng.normal(0.0, 0.1, (n, links))
    for k, r in enumerate(radii):  # a quarter of the box each, resting on the floor, against a wall or falling
      a = links + 7 * k
      side = np.array([1.0 if k & 1 else -1.0, 1.0 if k & 2 else -1.0])
      q[:, a:a + 2] = 0.3 * side + rng.uniform(-0.1, 0.1, (n, 2))
      q[:, a + 2] = r + rng.uniform(-0.001, 0.1, n)
      q[:, a + 3] = 1.0
    groups.append((m, d))
    src += [_dev(q), _dev(v), torch.zeros((n, mjm.nv), device=DEV)]
    dst += [d.qpos, d.qvel, d.qacc_warmstart]
  s = {"kind": "multi", "groups": groups, "src": src, "dst": dst, "nstep": case["nstep"],
       "multi": mjw.MultiStep(groups)}
  _reset(s)
  return s


def _run_multi(s):
  _reset(s)
  for _ in range(s["nstep"]):
    s["multi"].step()
  return [(torch.cat([d.qpos.reshape(-1) for _, d in s["groups"]]),
           torch.cat([d.qvel.reshape(-1) for _, d in s["groups"]]))]


def _prepare_grad(case, rng):
  mjm = _compiled("humanoid")
  m = mjw.put_model(mjm)
  n, t = case["nworld"], case["nstep"]
  r = derivative.Rollout(mjm, m, n, t, nconmax=64 * n, njmax=277 * n)
  q, v = _humanoid_state(rng, mjm.key_qpos[0], n, "squat")
  q[:, 2] += 0.1  # landing during the rollout or just before it
  return {"kind": "grad", "r": r, "q": _dev(q), "v": _dev(v), "u": _dev(rng.uniform(-1.0, 1.0, (t, n, mjm.nu)))}


def _run_grad(s):
  v = s["v"].detach().requires_grad_(True)
  u = s["u"].detach().requires_grad_(True)
  qpos, qvel = s["r"](s["q"], v, u)
  loss = ((qpos[..., 2] - 1.3) ** 2).sum() + 1e-3 * (u**2).sum()
  gv, gu = torch.autograd.grad(loss, (v, u))
  return qpos.detach(), qvel.detach(), gv, gu


def _prepare_smooth(case, rng):
  mjm = _model(case)
  n = case["nworld"]
  m = mjw.put_model(mjm)
  d = mjw.make_data(mjm, nworld=n, nconmax=n, njmax=n)
  q, v = _states(case, mjm, rng)
  d.qpos.copy_(_dev(q))
  d.qvel.copy_(_dev(v))
  return {"kind": "smooth", "m": m, "d": d, "tau": _dev(rng.normal(0.0, 10.0, (n, mjm.nv))),
          "acc": torch.zeros((n, mjm.nv), device=DEV)}


def _run_smooth(s):
  m, d = s["m"], s["d"]
  mjw.kinematics(m, d)
  mjw.com_pos(m, d)
  mjw.crb(m, d)
  mjw.factor_m(m, d)
  mjw.com_vel(m, d)
  mjw.passive(m, d)
  mjw.rne(m, d)
  mjw.solve_m(m, d, s["acc"], s["tau"])
  return {"xpos": d.xpos, "xquat": d.xquat, "geom_xpos": d.geom_xpos, "subtree_com": d.subtree_com, "cdof": d.cdof,
          "cinert": d.cinert, "cvel": d.cvel, "qM": d.qM, "qfrc_bias": d.qfrc_bias, "qfrc_passive": d.qfrc_passive,
          "acc": s["acc"]}


def _pile(case, rng):
  """Positions [n, nbody, 3] and rotations [n, nbody, 3, 3]: bodies on a
  jittered lattice that neighbours overlap on, as in a settled pile."""
  n, nb = case["nworld"], case["nbody"]
  cell = np.arange(nb)
  at = np.stack([cell % 8, (cell // 8) % 8, cell // 64], 1) * [0.24, 0.24, 0.2] + [-0.84, -0.84, 0.1]
  p = at[None] + rng.uniform(-0.06, 0.06, (n, nb, 3))
  q = rng.normal(size=(n, nb, 4))
  q /= np.linalg.norm(q, axis=2, keepdims=True)
  return p, _qmat(q)


def _prepare_collide(case, rng):
  mjm = _compiled("pile", case["nbody"])
  n, nb = case["nworld"], case["nbody"]
  m = mjw.put_model(mjm)
  d = mjw.make_data(mjm, nworld=n, nconmax=24 * nb * n, njmax=n)
  p, r = _pile(case, rng)
  # geoms 0-4 are the floor and the walls; each body holds one geom at its origin
  gp = np.tile(np.asarray(mjm.geom_pos)[None], (n, 1, 1))
  gr = np.tile(_qmat(np.asarray(mjm.geom_quat))[None], (n, 1, 1, 1))
  gp[:, 5:], gr[:, 5:] = p, r
  d.geom_xpos.copy_(_dev(gp))
  d.geom_xmat.copy_(_dev(gr))
  return {"kind": "collide", "m": m, "d": d}


def _run_collide(s):
  d = s["d"]
  mjw.collision(s["m"], d)
  # the contact pool's order over worlds is not fixed; these are
  return {"ncollision": d.ncollision, "ncon": d.ncon, "order": d.sap_sort_index, "lower": d.sap_projection_lower,
          "upper": d.sap_projection_upper, "range": d.sap_range}


def _solve_inputs(case, rng):
  """Rows of contacts (a normal and two tangents as four pyramid edges) and
  limits of each world, back to back: (M, qfrc_smooth, warm, counts, J, D, aref)."""
  n, nv = case["nworld"], 27
  a = rng.normal(size=(n, nv, nv)) * 0.2
  scale = np.exp(rng.uniform(math.log(0.2), math.log(3.0), (n, nv)))
  M = (a @ a.transpose(0, 2, 1) + np.eye(nv)) * scale[:, :, None] * scale[:, None, :]
  counts = 4 * rng.integers(0, case["rows"] // 2 + 1, n)
  counts[::16] = 4 * 20  # a few worlds with many
  total = int(counts.sum())
  basis = rng.normal(size=(total // 4, 3, nv)) * (rng.random((total // 4, 1, nv)) < 0.6)
  J = np.stack([basis[:, 0] + s * basis[:, t] for t in (1, 2) for s in (1.0, -1.0)], 1).reshape(total, nv)
  # impedances of 0.8 to 0.95 on the rows' own inverse inertia, as the row builder sets D
  smooth = rng.normal(0.0, 20.0, (n, nv))
  world = np.repeat(np.arange(n), counts)
  Minv = np.linalg.inv(M)
  own = np.einsum("ri,rij,rj->r", J, Minv[world], J).reshape(-1, 4).mean(1)
  imp = rng.uniform(0.8, 0.95, total // 4)
  D = (imp / ((1.0 - imp) * np.maximum(own, 1e-3))).repeat(4)
  free = np.einsum("nij,nj->ni", Minv, smooth)
  aref = np.einsum("ri,ri->r", J, free[world]).reshape(-1, 4).mean(1)
  aref = (aref + np.sqrt(own) * rng.normal(0.0, 5.0, total // 4)).repeat(4)
  warm = free + rng.normal(0.0, 1.0, (n, nv))
  f32 = lambda x: np.asarray(x, np.float32)
  M = f32(M)
  return M, f32(smooth), f32(warm), counts, f32(J), f32(D), f32(aref)


def _prepare_solve(case, rng):
  mjm = _compiled("humanoid")
  n = case["nworld"]
  M, qs, warm, counts, J, D, aref = _solve_inputs(case, rng)
  total = int(counts.sum())
  m = mjw.put_model(mjm)
  d = mjw.make_data(mjm, nworld=n, nconmax=n, njmax=total + 64)
  d.qM.copy_(_dev(M))
  d.qfrc_smooth.copy_(_dev(qs))
  d.qacc_smooth.copy_(torch.linalg.solve(_dev(M).double(), _dev(qs).double()).float())
  d.efc.J[:total].copy_(_dev(J))
  d.efc.D[:total].copy_(_dev(D))
  d.efc.aref[:total].copy_(_dev(aref))
  d.efc.worldid.fill_(-1)
  d.efc.worldid[:total].copy_(torch.tensor(np.repeat(np.arange(n), counts), dtype=torch.int32))
  d.nefc.fill_(total)
  return {"kind": "solve", "m": m, "d": d, "src": [_dev(warm)], "dst": [d.qacc_warmstart]}


def _run_solve(s):
  _reset(s)
  mjw.solve(s["m"], s["d"])
  return s["d"].qacc, s["d"].qfrc_constraint


_PREPARE = {"step": _prepare_step, "functional": _prepare_step, "graph": _prepare_step, "multi": _prepare_multi,
            "grad": _prepare_grad, "smooth": _prepare_smooth, "collide": _prepare_collide, "solve": _prepare_solve}
_RUN = {"step": _run_step, "functional": _run_functional, "graph": _run_graph, "multi": _run_multi,
        "grad": _run_grad, "smooth": _run_smooth, "collide": _run_collide, "solve": _run_solve}


# ---------------------------------------------------------------- work

def _step_words(mjm):
  """Words of a world's fields with a counterpart in mjData that a step
  reads or writes, each once."""
  nv, nb, nu = mjm.nv, mjm.nbody, mjm.nu
  r = mjm.nq + 3 * nv + nu + 6 * nb
  w = (mjm.nq + 23 * nv + 57 * nb + 6 * mjm.njnt + 12 * mjm.ngeom + 12 * mjm.nsite + 3 * nu + nu * nv)
  return r + w + 2 * (mjm.nM if nv >= 60 else nv * nv)


def _step_flops(mjm, newton=4):
  nv = mjm.nv
  return 600.0 * mjm.nbody + (2 + newton) * nv**3 / 3 + newton * 30.0 * 4 * nv


def work(case):
  k, n = case["kind"], case["nworld"]
  if k in ("step", "functional", "graph"):
    mjm, t = _model(case), case.get("nstep", 1)
    return {"bytes": 4.0 * n * t * _step_words(mjm), "flops": n * t * _step_flops(mjm)}
  if k == "multi":
    b = f = 0.0
    for links, radii, c in models.heterogeneous_groups(n, max_links=case["max_links"], max_spheres=case["max_spheres"]):
      mjm = _compiled("box", links, radii)
      b += 4.0 * c * case["nstep"] * _step_words(mjm)
      f += c * case["nstep"] * _step_flops(mjm)
    return {"bytes": b, "flops": f}
  if k == "grad":
    mjm = _compiled("humanoid")
    t = case["nstep"]
    # each step forward, its fields read once more by the reverse pass
    return {"bytes": 2 * 4.0 * n * t * _step_words(mjm), "flops": 3.0 * n * t * _step_flops(mjm)}
  if k == "smooth":
    mjm = _model(case)
    words = (mjm.nq + 3 * mjm.nv + 72 * mjm.nbody + 6 * mjm.njnt + 12 * mjm.ngeom + 12 * mjm.nv
             + 2 * (mjm.nM if mjm.nv >= 60 else mjm.nv**2))
    return {"bytes": 4.0 * n * words, "flops": n * (900.0 * mjm.nbody + mjm.nv**3 / 3)}
  if k == "collide":
    ng = case["nbody"] + 5
    # poses in, the sweep's arrays and about two contacts per body (30 words each) out
    return {"bytes": 4.0 * n * (12 * ng + 9 * ng + 2 * 30 * case["nbody"]), "flops": 300.0 * n * ng}
  rows = n * case["rows"]
  return {"bytes": 4.0 * (n * (27 * 27 + 8 * 27) + rows * (27 + 4)),
          "flops": n * 4 * 27**3 / 3 + 5.0 * rows * 27 * 27}


# ---------------------------------------------------------------- exact values

def exact(case, seed):
  """64-bit values for the stages that have a closed one; whole steps go
  through a truncated iterative solve and have none."""
  rng = np.random.default_rng(seed)
  if case["kind"] == "smooth":
    return _exact_smooth(case, rng)
  if case["kind"] == "collide":
    return _exact_collide(case, rng)
  if case["kind"] == "solve":
    return _exact_solve(case, rng)
  return None


def _qmul(a, b):
  aw, ax, ay, az = np.moveaxis(a, -1, 0)
  bw, bx, by, bz = np.moveaxis(b, -1, 0)
  return np.stack([aw * bw - ax * bx - ay * by - az * bz, aw * bx + ax * bw + ay * bz - az * by,
                   aw * by - ax * bz + ay * bw + az * bx, aw * bz + ax * by - ay * bx + az * bw], -1)


def _qmat(q):
  w, x, y, z = np.moveaxis(np.asarray(q, np.float64), -1, 0)
  return np.stack([w * w + x * x - y * y - z * z, 2 * (x * y - w * z), 2 * (x * z + w * y),
                   2 * (x * y + w * z), w * w - x * x + y * y - z * z, 2 * (y * z - w * x),
                   2 * (x * z - w * y), 2 * (y * z + w * x), w * w - x * x - y * y + z * z], -1).reshape(q.shape[:-1] + (3, 3))


def _spatial(inert, v):
  """A 10-word inertia times a motion vector (rotation first)."""
  i, v = np.moveaxis(inert, -1, 0), np.moveaxis(v, -1, 0)
  return np.stack([i[0] * v[0] + i[3] * v[1] + i[4] * v[2] - i[8] * v[4] + i[7] * v[5],
                   i[3] * v[0] + i[1] * v[1] + i[5] * v[2] + i[8] * v[3] - i[6] * v[5],
                   i[4] * v[0] + i[5] * v[1] + i[2] * v[2] - i[7] * v[3] + i[6] * v[4],
                   i[8] * v[1] - i[7] * v[2] + i[9] * v[3], i[6] * v[2] - i[8] * v[0] + i[9] * v[4],
                   i[7] * v[0] - i[6] * v[1] + i[9] * v[5]], -1)


def _cross_motion(u, v):
  return np.concatenate([np.cross(u[..., :3], v[..., :3]),
                         np.cross(u[..., 3:], v[..., :3]) + np.cross(u[..., :3], v[..., 3:])], -1)


def _cross_force(v, f):
  return np.concatenate([np.cross(v[..., :3], f[..., :3]) + np.cross(v[..., 3:], f[..., 3:]),
                         np.cross(v[..., :3], f[..., 3:])], -1)


def _exact_smooth(case, rng):
  """Rigid-body kinematics, mass matrix, bias and passive forces of trees of
  free and hinge joints, and M x = tau, vectorised over the worlds."""
  mjm = _model(case)
  n, nb, nv = case["nworld"], mjm.nbody, mjm.nv
  q, v = _states(case, mjm, rng)
  f = lambda x: np.asarray(x, np.float32).astype(np.float64)
  q, v, tau = f(q), f(v), f(rng.normal(0.0, 10.0, (n, nv)))
  par, root = np.asarray(mjm.body_parentid), np.asarray(mjm.body_rootid)
  pos, quat = np.zeros((n, nb, 3)), np.zeros((n, nb, 4))
  quat[:, 0, 0] = 1.0
  anchor, axis = np.zeros((n, mjm.njnt, 3)), np.zeros((n, mjm.njnt, 3))
  for b in range(1, nb):
    j0, jn = int(mjm.body_jntadr[b]), int(mjm.body_jntnum[b])
    if jn == 1 and mjm.jnt_type[j0] == 0:
      a = int(mjm.jnt_qposadr[j0])
      p, qq = q[:, a:a + 3], q[:, a + 3:a + 7]
      anchor[:, j0], axis[:, j0] = p, f(mjm.jnt_axis[j0])
    else:
      pq = quat[:, par[b]]
      p = np.einsum("nij,j->ni", _qmat(pq), f(mjm.body_pos[b])) + pos[:, par[b]]
      qq = _qmul(pq, np.tile(f(mjm.body_quat[b]), (n, 1)))
      for j in range(j0, j0 + jn):
        a = int(mjm.jnt_qposadr[j])
        jx, jp = f(mjm.jnt_axis[j]), f(mjm.jnt_pos[j])
        R = _qmat(qq)
        anchor[:, j], axis[:, j] = R @ jp + p, R @ jx
        h = 0.5 * (q[:, a] - f(mjm.qpos0)[a])
        qq = _qmul(qq, np.concatenate([np.cos(h)[:, None], np.sin(h)[:, None] * jx], 1))
        p = anchor[:, j] - _qmat(qq) @ jp
    pos[:, b], quat[:, b] = p, qq / np.linalg.norm(qq, axis=1, keepdims=True)
  xmat = _qmat(quat)
  xipos = pos + np.einsum("nbij,bj->nbi", xmat, f(mjm.body_ipos))
  ximat = _qmat(_qmul(quat, np.broadcast_to(f(mjm.body_iquat), quat.shape)))
  gb = np.asarray(mjm.geom_bodyid)
  geom = pos[:, gb] + np.einsum("ngij,gj->ngi", xmat[:, gb], f(mjm.geom_pos))
  mass = f(mjm.body_mass)
  mom, tot = xipos * mass[:, None], mass.copy()
  for b in range(nb - 1, 0, -1):
    mom[:, par[b]] += mom[:, b]
    tot[par[b]] += tot[b]
  com = mom / np.where(tot > 0, tot, 1.0)[:, None]
  dif = xipos - com[:, root]
  I = np.einsum("nbij,bj,nbkj->nbik", ximat, f(mjm.body_inertia), ximat)
  I += mass[:, None, None] * (np.sum(dif**2, -1)[..., None, None] * np.eye(3) - dif[..., :, None] * dif[..., None, :])
  cin = np.stack([I[..., 0, 0], I[..., 1, 1], I[..., 2, 2], I[..., 0, 1], I[..., 0, 2], I[..., 1, 2],
                  *np.moveaxis(mass[:, None] * dif, -1, 0), np.broadcast_to(mass, (n, nb))], -1)
  cdof, cvel, dofs = np.zeros((n, nv, 6)), np.zeros((n, nb, 6)), [[] for _ in range(nb)]
  acc, pas = np.zeros((n, nb, 6)), np.zeros((n, nv))
  acc[:, 0, 3:] = -f(mjm.opt.gravity)
  damp = f(mjm.dof_damping)
  for b in range(1, nb):
    vb, ab = cvel[:, par[b]].copy(), acc[:, par[b]].copy()
    for j in range(int(mjm.body_jntadr[b]), int(mjm.body_jntadr[b]) + int(mjm.body_jntnum[b])):
      a = int(mjm.jnt_dofadr[j])
      off = com[:, root[b]] - anchor[:, j]
      if mjm.jnt_type[j] == 0:
        cdof[:, a:a + 3, 3:] = np.eye(3)
        ax = xmat[:, b].transpose(0, 2, 1)
        cdof[:, a + 3:a + 6, :3], cdof[:, a + 3:a + 6, 3:] = ax, np.cross(ax, off[:, None])
        ids = range(a, a + 6)
        vb += np.einsum("nk,nkc->nc", v[:, a:a + 3], cdof[:, a:a + 3])
        for k in ids[3:]:
          ab += _cross_motion(vb, cdof[:, k]) * v[:, k, None]
        vb += np.einsum("nk,nkc->nc", v[:, a + 3:a + 6], cdof[:, a + 3:a + 6])
      else:
        cdof[:, a, :3], cdof[:, a, 3:] = axis[:, j], np.cross(axis[:, j], off)
        ids = [a]
        ab += _cross_motion(vb, cdof[:, a]) * v[:, a, None]
        vb += cdof[:, a] * v[:, a, None]
        qa = int(mjm.jnt_qposadr[j])
        pas[:, a] -= f(mjm.jnt_stiffness)[j] * (q[:, qa] - f(mjm.qpos_spring)[qa])
      for k in ids:
        pas[:, k] -= damp[k] * v[:, k]
        dofs[b].append(k)
    cvel[:, b], acc[:, b] = vb, ab
  force = _spatial(cin, acc) + _cross_force(cvel, _spatial(cin, cvel))
  crb = cin.copy()
  for b in range(nb - 1, 0, -1):
    force[:, par[b]] += force[:, b]
    if par[b]:
      crb[:, par[b]] += crb[:, b]
  bias, M = np.zeros((n, nv)), np.zeros((n, nv, nv))
  dp, db = np.asarray(mjm.dof_parentid), np.asarray(mjm.dof_bodyid)
  for i in range(nv):
    bias[:, i] = np.sum(cdof[:, i] * force[:, db[i]], -1)
    buf = _spatial(crb[:, db[i]], cdof[:, i])
    j = i
    while j >= 0:
      M[:, i, j] = M[:, j, i] = np.sum(cdof[:, j] * buf, -1)
      j = int(dp[j])
    M[:, i, i] += f(mjm.dof_armature)[i]
  x = np.linalg.solve(M, tau[..., None])[..., 0]
  if nv >= 60:  # rows i, parent(i), ... as MuJoCo's sparse layout
    at = []
    for i in range(nv):
      j = i
      while j >= 0:
        at.append(i * nv + j)
        j = int(dp[j])
    M = M.reshape(n, nv * nv)[:, at]
  return {"xpos": pos, "xquat": quat, "geom_xpos": geom, "subtree_com": None if tot[1:].min() <= 0 else com,
          "cdof": cdof, "cinert": cin, "cvel": cvel, "qM": M, "qfrc_bias": bias, "qfrc_passive": pas, "acc": x}


def _exact_collide(case, rng):
  mjm = _compiled("pile", case["nbody"])
  n = case["nworld"]
  f = lambda x: np.asarray(x, np.float32).astype(np.float64)
  gp = np.tile(f(mjm.geom_pos)[None], (n, 1, 1))
  gp[:, 5:] = f(_pile(case, rng)[0])
  way = f([0.5935, 0.7790, 0.1235])
  c = gp @ (way / np.linalg.norm(way))
  rb = f(mjm.geom_rbound)
  rad = np.where(rb == 0.0, 1e9, rb) + f(mjm.geom_margin)
  return {"ncollision": None, "ncon": None, "order": None, "lower": np.sort(c - rad, 1), "upper": c + rad, "range": None}


def _exact_solve(case, rng):
  """The minimum of 1/2 (x - a)' M (x - a) + 1/2 sum D min(0, J x - aref)^2
  by Newton steps with a bisected line search."""
  M, qs, warm, counts, J, D, aref = _solve_inputs(case, rng)
  t = lambda x: torch.tensor(x, dtype=torch.float64, device=DEV if torch.cuda.is_available() else "cpu")
  n, nv, top = case["nworld"], 27, int(counts.max()) if len(counts) else 0
  row = np.concatenate([np.arange(c) for c in counts]) if counts.sum() else np.zeros(0, int)
  w = np.repeat(np.arange(n), counts)
  Jp, Dp, Ap = np.zeros((n, top, nv)), np.zeros((n, top)), np.zeros((n, top))
  Jp[w, row], Dp[w, row], Ap[w, row] = J, D, aref
  M, J, D, aref, qs = t(M), t(Jp), t(Dp), t(Ap), t(qs)
  x = torch.linalg.solve(M, qs)

  def slope(x):
    r = (J @ x[..., None])[..., 0] - aref
    a = (r < 0) * D
    return (M @ x[..., None])[..., 0] - qs + (J.transpose(1, 2) @ (a * r)[..., None])[..., 0], a

  for _ in range(40):
    g, a = slope(x)
    p = -torch.linalg.solve(M + J.transpose(1, 2) @ (a[..., None] * J), g)
    lo, hi = torch.zeros(n, 1, dtype=x.dtype, device=x.device), torch.ones(n, 1, dtype=x.dtype, device=x.device) * 2
    for _ in range(50):
      mid = 0.5 * (lo + hi)
      down = ((slope(x + mid * p)[0] * p).sum(1, keepdim=True)) < 0
      lo, hi = torch.where(down, mid, lo), torch.where(down, hi, mid)
    x = x + 0.5 * (lo + hi) * p
  g, a = slope(x)
  r = (J @ x[..., None])[..., 0] - aref
  return x, -(J.transpose(1, 2) @ (a * r)[..., None])[..., 0]
