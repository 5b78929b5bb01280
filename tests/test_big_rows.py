"""The big-world solve at the row counts where its work changes hands: the last
rows staged in LDS and the first read from global memory, for the launches of
few, some and many worlds, and the most rows it takes -- the same bits wherever a
row is read from, against the optimum in 64 bits; in a captured graph; and on
rows that the caller laid out, again and again on the same Data."""
import numpy as np
import pytest
import torch

import helpers
import mjx_warp_amd as mjw
from mjx_warp_amd import mjcf, models
from test_big_worlds import _lying

pytestmark = pytest.mark.gpu


def _solved(nv, rows, nworld):
  """One world's rows, in every world: the constraint cost's minimiser."""
  mjm = mjcf.from_xml_string(models.chain_xml(nv).replace('solver="CG"', 'solver="Newton"').replace(
      "<option ", '<option jacobian="dense" '))
  m = mjw.put_model(mjm)
  rng = np.random.default_rng(1000 * nv + rows)
  A = rng.normal(size=(nv, nv))
  M = (A @ A.T / nv + np.eye(nv)).astype(np.float32)
  J = rng.normal(size=(rows, nv)).astype(np.float32)
  D = rng.uniform(0.5, 1.5, rows).astype(np.float32)
  aref = rng.normal(0.0, 10.0, rows).astype(np.float32)
  qs = rng.normal(0.0, 10.0, nv).astype(np.float32)
  total = nworld * rows
  d = mjw.make_data(mjm, nworld=nworld, nconmax=nworld, njmax=total)
  dev = lambda a: torch.as_tensor(a, device="cuda")
  d.qM.copy_(dev(M).expand(nworld, nv, nv).reshape(d.qM.shape))
  d.qfrc_smooth.copy_(dev(qs).expand(nworld, nv))
  mjw.factor_m(m, d)
  mjw.solve_m(m, d, d.qacc_smooth, d.qfrc_smooth)
  d.efc.J.copy_(dev(J).repeat(nworld, 1))
  d.efc.D.copy_(dev(D).repeat(nworld))
  d.efc.aref.copy_(dev(aref).repeat(nworld))
  d.efc.worldid.copy_(torch.arange(nworld, device="cuda", dtype=torch.int32).repeat_interleave(rows))
  d.nefc.fill_(total)
  mjw.solve(m, d)
  torch.cuda.synchronize()
  return M, J, D, aref, qs, d


@pytest.mark.parametrize("nv,rows", [(32, 101), (32, 102), (32, 145), (32, 146), (32, 243), (32, 244), (32, 256),
                                     (28, 164), (28, 165), (28, 253), (28, 254), (27, 256), (8, 65), (8, 256)])
def test_rows_past_the_staged_ones(nv, rows):
  xs = []
  for nworld in (2, 1100, 2100):
    M, J, D, aref, qs, d = _solved(nv, rows, nworld)
    q = d.qacc.cpu().numpy()
    assert np.array_equal(q, np.broadcast_to(q[:1], q.shape))
    xs.append(q[0])
  assert np.array_equal(xs[0], xs[1]) and np.array_equal(xs[0], xs[2])
  M, J, D, aref, qs, x = (a.astype(np.float64) for a in (M, J, D, aref, qs, xs[0]))
  smooth = np.linalg.solve(M, qs)
  best = smooth.copy()
  for _ in range(200):  # Newton with halving
    act = J @ best < aref
    grad = M @ best - qs + J[act].T @ (D[act] * (J[act] @ best - aref[act]))
    step = -np.linalg.solve(M + J[act].T @ (D[act, None] * J[act]), grad)
    cost = lambda v: 0.5 * (v - smooth) @ M @ (v - smooth) + 0.5 * np.sum(D * np.minimum(J @ v - aref, 0.0) ** 2)
    t = 1.0
    while cost(best + t * step) > cost(best) and t > 1e-12:
      t *= 0.5
    best = best + t * step
  # the solver stops where the cost, in 32 bits, falls no more: a sum of rows
  # squares, each of a sum of nv products, and M's form (textbook constants
  # times 4); and a gap g above the optimum is within sqrt(2 g / lowest
  # eigenvalue of M) of it
  jar, size = np.minimum(J @ x - aref, 0.0), np.abs(J) @ np.abs(x) + np.abs(aref)
  e = np.abs(x - smooth)
  gap = 4 * np.finfo(np.float32).eps * (np.sum(D * (rows / 2 * jar**2 + nv * np.abs(jar) * size)) + nv * e @ np.abs(M) @ e)
  assert np.sum((x - best) ** 2) <= 2 * gap / np.linalg.eigvalsh(M)[0]
  assert np.sum(jar < 0) > rows // 8


@pytest.mark.parametrize("links", [16, 32])  # the launch's LDS as it comes, and asked for
def test_captured(links):
  mjm = models.chain(links)
  m = mjw.put_model(mjm)
  out = []
  for graph in (True, False):
    d = mjw.make_data(mjm, nworld=3, nconmax=24 * links, njmax=64 * links)
    q = np.random.default_rng(links).uniform(-0.3, 0.3, (3, links))
    helpers.set_field(d, "qpos", q)
    g = mjw.StepGraph(m, d, nstep=1) if graph else None
    for _ in range(3):
      if graph:
        g.replay()
      else:
        mjw.step_fused(m, d)
      torch.cuda.synchronize()
    assert helpers.data_numpy(d, "world_efc").reshape(-1, 2)[:3, 1].min() > 64
    out.append((d.qpos.clone(), d.qvel.clone()))
  assert all(torch.equal(a, b) for a, b in zip(*out))


def _lay_out(d2, d, layout, rng):
  """d's smooth quantities and rows into d2's pool, its blocks left stale."""
  for f in ("qM", "qLD", "qacc_smooth", "qfrc_smooth"):
    getattr(d2, f).copy_(getattr(d, f))
  d2.qacc_warmstart.zero_()
  blocks = helpers.world_blocks(helpers.data_numpy(d, "world_efc"), d.nworld)
  tag = np.concatenate([np.full(n, w) for w, (_, n) in enumerate(blocks)])
  src = np.concatenate([np.arange(b, b + n) for b, n in blocks])
  if layout == "interleaved":  # a random merge that keeps each world's order
    seq = rng.permutation(tag)
    take = np.empty(len(seq), int)
    for w in range(d.nworld):
      take[seq == w] = np.flatnonzero(tag == w)
    src, tag = src[take], seq
  n, njmax = len(src), d2.njmax
  for f in ("J", "D", "aref", "pos", "margin"):
    full = helpers.data_numpy(d, "efc_" + f)[src]
    helpers.set_field(d2, "efc_" + f, np.concatenate([full, np.zeros((njmax - n,) + full.shape[1:], full.dtype)]))
  helpers.set_field(d2, "efc_worldid", np.concatenate([tag, np.full(njmax - n, -1)]).astype(np.int32))
  helpers.set_field(d2, "nefc", np.array([n], np.int32))


@pytest.mark.parametrize("desc", [True, False])
@pytest.mark.parametrize("layouts", [("blocks", "interleaved"), ("interleaved", "blocks")])
def test_caller_laid_big_worlds(layouts, desc):
  nworld = 5
  mjm = models.humanoid(iterations=10, ls_iterations=20)
  m = mjw.put_model(mjm)
  d2 = mjw.make_data(mjm, nworld=nworld, nconmax=8, njmax=2500)
  if not desc:
    d2.ndesc = 0
    d2.step_desc = torch.zeros(0, dtype=torch.int32, device="cuda")
  rng = np.random.default_rng(len(layouts[0]))
  for turn, layout in enumerate(layouts):  # the second turn's big worlds are others
    d = mjw.make_data(mjm, nworld=nworld, nconmax=64 * nworld, njmax=277 * nworld)
    helpers.set_field(d, "qpos", np.roll(_lying(mjm, nworld, 2), turn, 0))
    mjw.forward(m, d)
    torch.cuda.synchronize()
    rows = helpers.data_numpy(d, "world_efc").reshape(-1, 2)[:nworld, 1]
    assert [i for i in range(nworld) if rows[i] > 64] == ([1, 3] if turn == 0 else [2, 4]) and rows.max() <= 256
    _lay_out(d2, d, layout, rng)
    mjw.solve(m, d2)
    torch.cuda.synchronize()
    assert not np.any(helpers.data_numpy(d2, "world_flags"))
    for f in ("qacc", "qfrc_constraint"):
      assert torch.equal(getattr(d2, f), getattr(d, f)), (turn, f)
