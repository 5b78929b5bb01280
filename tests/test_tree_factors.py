"""Mass-matrix factors on 64-lane teams: the packed blocks (one row a lane, two
rows, the largest packed and the first that is not), small blocks, and the
sparse L'DL factor (its look-up table in LDS, also on 32-lane teams, more
ancestors than a pass takes, and a matrix too large for the table), against
float32 backward error bounds: |M x - b| <= g |L| |L'| |x| and |M - L' D L| <= g |L'| |D| |L|, with
g = 4 (3 n + 4) eps and 4 (n + 4) eps (the textbook constants times 4)."""
import numpy as np
import pytest
import torch

import helpers
import mjx_warp_amd as mjw
from mjx_warp_amd import mjcf, models

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float32).eps


@pytest.mark.parametrize("nv", [33, 64, 65, 81, 128, 129])
def test_packed_blocks(nv):
  mjm = models.chain(nv)
  m = mjw.put_model(mjm)
  d = mjw.make_data(mjm, nworld=2, nconmax=16, njmax=4 * nv)
  rng = np.random.default_rng(nv)
  A = rng.normal(size=(2, nv, nv))
  M = (A @ A.transpose(0, 2, 1) + nv * np.eye(nv)).astype(np.float32)
  b = rng.normal(size=(2, nv)).astype(np.float32)
  field = "qMd" if m.opt.is_sparse else "qM"
  helpers.set_field(d, field, M)
  mjw.factor_m(m, d)
  x = torch.zeros(2, nv, device="cuda")
  mjw.solve_m(m, d, x, torch.as_tensor(b, device="cuda"))
  torch.cuda.synchronize()
  for w in range(2):
    H, y = M[w].astype(np.float64), x[w].cpu().numpy().astype(np.float64)
    L = np.abs(np.linalg.cholesky(H))
    assert np.all(np.abs(H @ y - b[w]) <= 4 * (3 * nv + 4) * EPS * (L @ (L.T @ np.abs(y))))


def _chains(n, trees):
  link = lambda k: ('<body><joint axis="0 1 0"/><geom type="capsule" fromto="0 0 0 0 0 -0.1" size="0.02"/>'
                    + (link(k - 1) if k > 1 else "") + "</body>")
  return mjcf.from_xml_string('<mujoco><option jacobian="dense"/><worldbody>' + trees * link(n) + "</worldbody></mujoco>")


# a tree per lane from one dof to the most it takes (more trees than lanes
# too), then packed: both sides of each change of panel width, several panels
@pytest.mark.parametrize("n,trees", [(1, 65), (2, 17), (5, 7), (6, 70), (7, 5), (8, 5), (9, 4), (12, 3), (13, 3), (17, 2)])
def test_small_blocks(n, trees):
  nv = n * trees
  mjm = _chains(n, trees)
  assert mjm.nv == nv > 32
  m = mjw.put_model(mjm)
  d = mjw.make_data(mjm, nworld=2, nconmax=16, njmax=16)
  rng = np.random.default_rng(n)
  M = np.zeros((2, nv, nv), np.float32)
  for k in range(0, nv, n):
    A = rng.normal(size=(2, n, n))
    M[:, k:k + n, k:k + n] = A @ A.transpose(0, 2, 1) + n * np.eye(n)
  b = rng.normal(size=(2, nv)).astype(np.float32)
  helpers.set_field(d, "qM", M)
  mjw.factor_m(m, d)
  x = torch.zeros(2, nv, device="cuda")
  mjw.solve_m(m, d, x, torch.as_tensor(b, device="cuda"))
  torch.cuda.synchronize()
  F = helpers.data_numpy(d, "qLD").astype(np.float64)
  for w in range(2):
    H, y = M[w].astype(np.float64), x[w].cpu().numpy().astype(np.float64)
    L = np.abs(np.linalg.cholesky(H))
    assert np.all(np.abs(H - F[w] @ F[w].T) <= 4 * (n + 4) * EPS * (L @ L.T))
    assert np.all(np.abs(H @ y - b[w]) <= 4 * (3 * n + 4) * EPS * (L @ (L.T @ np.abs(y))))


@pytest.mark.parametrize("nv", [40, 100])
def test_solve_divides_at_the_ends_of_the_range(nv):
  """A diagonal factor: every entry is two divisions, to the bit, for divisors
  and dividends down to subnormal and up to the largest, and a quotient that
  overflows (which the zeros off the diagonal then carry on as NaN)."""
  mjm = models.chain(nv)
  m = mjw.put_model(mjm)
  rng = np.random.default_rng(nv)
  f32 = np.float32
  mant = lambda: rng.uniform(1, 2, nv).astype(f32)
  ones = np.ones(nv, f32)
  scale = lambda e: (mant() * f32(2.0) ** np.asarray(e, f32)).astype(f32)
  sub = rng.integers(1, 1 << 23, nv).astype(np.uint32).view(f32)
  cases = [(mant(), scale(-rng.integers(100, 126, nv))), (mant(), sub), (scale(-rng.integers(100, 126, nv)), scale(rng.integers(-126, -100, nv))),
           (sub, sub), (scale(rng.integers(100, 127, nv)), scale(rng.integers(60, 127, nv))), (mant(), np.where(np.arange(nv) % 3 == 0, f32(0), mant())),
           (scale(rng.integers(-20, 20, nv)), scale(rng.integers(-60, 60, nv))), (ones * f32(0.01), np.where(np.arange(nv) == nv - 2, f32(3e38), mant()))]
  d = mjw.make_data(mjm, nworld=len(cases), nconmax=16, njmax=16)
  L = np.stack([np.diag(l) for l, _ in cases])
  helpers.set_field(d, "qLDd" if m.opt.is_sparse else "qLD", L)
  y = torch.as_tensor(np.stack([y for _, y in cases]), device="cuda")
  x = torch.zeros(len(cases), nv, device="cuda")
  mjw.solve_m(m, d, x, y)
  torch.cuda.synchronize()
  with np.errstate(all="ignore"):
    for w, (l, b) in enumerate(cases):
      q = (b / l).astype(f32)
      bad = np.flatnonzero(~np.isfinite(q))
      if bad.size:
        q[bad[0] + 1:] = np.nan
      want = (q / l).astype(f32)
      if np.any(~np.isfinite(want)):
        want[: np.flatnonzero(~np.isfinite(want))[-1]] = np.nan
      assert np.array_equal(x[w].cpu().numpy(), want, equal_nan=True), w


@pytest.mark.parametrize("nv", [2, 17, 32, 33, 60, 126, 128])
def test_sparse_factor(nv):
  mjm = models.chain(nv)
  mjm.opt.jacobian = 1
  m = mjw.put_model(mjm)
  assert m.opt.is_sparse
  d = mjw.make_data(mjm, nworld=3, nconmax=48, njmax=12 * nv)
  rng = np.random.default_rng(nv)
  helpers.set_field(d, "qpos", rng.uniform(-0.3, 0.3, (3, nv)))
  mjw.kinematics(m, d)
  mjw.com_pos(m, d)
  mjw.crb(m, d)
  mjw.factor_m(m, d)
  torch.cuda.synchronize()
  # a chain: row i of the sparse layout is M(i, i), M(i, i - 1), ...
  rows = lambda a: [np.pad(r[::-1], (0, nv - len(r))) for r in np.split(a, np.cumsum(np.arange(1, nv)))]
  S, F = (helpers.data_numpy(d, k).reshape(3, -1).astype(np.float64) for k in ("qM", "qLD"))
  inv = helpers.data_numpy(d, "qLDiagInv").reshape(3, nv)
  for w in range(3):
    T, U = np.array(rows(S[w])), np.array(rows(F[w]))
    M = T + np.tril(T, -1).T
    D, L = np.diag(U).copy(), np.tril(U, -1) + np.eye(nv)
    assert np.all(np.abs(M - L.T @ (D[:, None] * L)) <= 4 * (nv + 4) * EPS * (np.abs(L.T) @ (np.abs(D)[:, None] * np.abs(L))))
    assert np.allclose(inv[w] * D, 1, rtol=0, atol=2 * EPS)
