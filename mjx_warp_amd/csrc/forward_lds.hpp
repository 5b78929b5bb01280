// The forward stages of one world (kinematics to qfrc_smooth and the
// constraint rows) with the world's state resident in LDS, for the fused
// launches.
//
// The stage functions of smooth.hpp, forward.hpp and constraint.hpp pass a
// world's fields on through global memory: each stage waits for the stores
// of the one before it, walks chains of dependent model loads level by level
// and writes [n, k] fields a lane per row, a cache request per word.  Here
// the fields that later stages read stay in LDS, the model's per-body and
// per-joint constants are loaded once before the level loops, what does not
// depend on the tree (joint angles, actuator moments) is computed before
// them, and the fields go to global memory with lanes over consecutive
// words.  The arithmetic of every field, and its order, is the stage
// functions'; they remain for the per-stage entry points and for models that
// fwd_resident refuses.
//
// What bounds it: with 8192 worlds, four wavefronts per SIMD, the latency of
// the dependent steps (LDS and L2) of each world; so the layout is kept to
// 1280 floats per world at humanoid size (16 workgroups of two worlds per
// CU; larger models, see fwd_resident).
#pragma once

#include "constraint.hpp"
#include "forward.hpp"

namespace mjh {

// Contacts per chunk of the constraint rows here (see make_constraint_rows).
constexpr int kFwdRowChunk = 16;

// LDS layout, offsets in floats.  Kept to the end: qpos, qvel, cdof, cinert,
// sc.  From B on by phase: kinematics (jloc, anchor, axis, lmat, ipos and,
// behind everything that comes before the geoms are placed, lpos / lquat);
// composite inertias and the packed mass matrix; the geom table and the list
// of pairs, which stay while the velocity phase (cdot, vel) runs behind
// them; the constraint rows' workspace.
struct FwdLds {
  int qpos, qvel, cdof, cinert, sc;
  int jloc, anchor, axis, lmat, ipos, lpos, lquat;
  int crb, par, tri;
  int geom, list, cdot, vel;
  int rows, total;
};
constexpr int kGeomRec = 15;  // position, rotation, bounding radius, margin, type
__host__ __device__ inline int fwd_max(int a, int b) { return a > b ? a : b; }
__host__ __device__ inline FwdLds fwd_lds(int nq, int nv, int nb, int nj, int ng, int nu, int team) {
  FwdLds l;
  l.qpos = 0;
  l.qvel = l.qpos + nq;
  l.cdof = l.qvel + nv;
  l.cinert = l.cdof + 6 * nv;
  l.sc = l.cinert + 10 * nb;
  const int B = (l.sc + 3 * nb + 3) & ~3;  // jloc is read as float4s
  l.jloc = B;
  l.anchor = B + 8 * nj;
  l.axis = l.anchor + 3 * nj;
  l.lmat = l.axis + 3 * nj;
  l.ipos = l.lmat + 9 * nb;
  l.crb = B;
  l.par = B + 10 * nb;
  l.tri = l.par + nv;
  l.geom = B;
  l.list = B + kGeomRec * ng;
  const int kin = l.ipos + 3 * nb, crb_end = l.tri + (team == 64 ? 0 : nv * (nv + 1) / 2), geom_end = l.list + 2 * team;
  l.lpos = fwd_max(kin, fwd_max(crb_end, geom_end));
  l.lquat = l.lpos + 3 * nb;
  l.cdot = geom_end;
  l.vel = l.cdot + 6 * nv;
  l.rows = B;
  const int vel_end = l.vel + fwd_max(18 * nb, 6 * nb + fwd_max(nv, 2 * nu));
  l.total = (fwd_max(l.lquat + 4 * nb, fwd_max(vel_end, B + 29 * kFwdRowChunk)) + 3) & ~3;
  return l;
}
__host__ __device__ inline FwdLds fwd_lds(const mjhModel& m, int team) {
  return fwd_lds(m.nq, m.nv, m.nbody, m.njnt, m.ngeom, m.nu, team);
}
// Whether the layout serves the model on teams of this size: pairs from the
// nxn table, at most 64 bodies (a dof's subtree as one 64-bit mask), two dofs
// per lane and at most `limit` floats.  The limit is eight workgroups a CU (2560
// floats on 32-lane teams, 5120 on 64-lane ones; two wavefronts a SIMD), and
// sixteen on 32-lane teams where groups of other models share the launch and its
// LDS.  Fused steps in us, stage functions / resident, at 1024, 8192 and 32768
// worlds: a 20-link chain (1316 floats) 162 / 138, 289 / 299, 1021 / 759; the
// humanoid with four more bodies (1396) 313 / 294, 534 / 532, 1746 / 1494; a
// 32-link chain (2036) 217 / 177, 563 / 436, 1814 / 1387.
__host__ __device__ inline bool fwd_resident(const mjhModel& m, int team, int limit) {
  return m.ngeom <= MJH_NXN_TABLE_MAX && m.nbody <= 64 && m.nv <= 2 * team && fwd_lds(m, team).total <= limit;
}

// n consecutive words from LDS to global memory, lanes over words
template <int TEAM>
MJH_DEV void flush_words(float* dst, const float* src, int n, const Team<TEAM>& t) {
#pragma unroll 4
  for (int i = t.lane; i < n; i += TEAM) dst[i] = src[i];
}

// What a lane keeps of the body it places: entry `lane` of body_tree.
struct BodyConst {
  int b, pid, ja, jn, da, dn;
  unsigned types;  // joint types, two bits each, of the first 16
};
MJH_DEV BodyConst body_const(const mjhModel& m, int k) {
  BodyConst c;
  c.b = m.body_tree[k];
  c.pid = m.body_parentid[c.b];
  c.ja = m.body_jntadr[c.b];
  c.jn = m.body_jntnum[c.b];
  c.da = m.body_dofadr[c.b];
  c.dn = m.body_dofnum[c.b];
  c.types = 0;
  for (int j = 0; j < c.jn && j < 16; j++) c.types |= (unsigned)m.jnt_type[c.ja + j] << (2 * j);
  return c;
}
MJH_DEV int body_joint_type(const mjhModel& m, const BodyConst& c, int j) {
  return j < 16 ? (int)((c.types >> (2 * j)) & 3u) : m.jnt_type[c.ja + j];
}
// f(constants) for the bodies of body_tree[beg, end), a lane per body; c0:
// the constants of the lane's own entry
template <int TEAM, class F>
MJH_DEV void level_bodies(const mjhModel& m, int beg, int end, const BodyConst& c0, const Team<TEAM>& t, F f) {
  if (t.lane >= beg && t.lane < end) f(c0);
  for (int k = t.lane + TEAM; k < end; k += TEAM)
    if (k >= beg) f(body_const(m, k));
}

// collision_driver.py:480-508 on the geom table's records
MJH_DEV bool bounds_hit(const float* f1, const float* f2) {
  const float s1 = f1[12], s2 = f2[12];
  const float bound = s1 + s2 + fmaxf(f1[13], f2[13]);
  const V3 dif = V3{f2[0], f2[1], f2[2]} - V3{f1[0], f1[1], f1[2]};
  if (s1 != 0.0f && s2 != 0.0f) return dot(dif, dif) <= bound * bound;
  if (s1 == 0.0f) return dot(dif, V3{f1[5], f1[8], f1[11]}) <= bound;
  return dot(-dif, V3{f2[5], f2[8], f2[11]}) <= bound;
}

template <int TEAM>
MJH_DEV void forward_resident(const mjhModel& m, const mjhData& d, float* lds, const Team<TEAM>& t) {
  const int w = t.valid ? t.world : 0, lane = t.lane;
  const bool ok = t.valid;
  const int nq = m.nq, nv = m.nv, nb = m.nbody, nj = m.njnt, ng = m.ngeom, nu = m.nu;
  const FwdLds L = fwd_lds(m, TEAM);
  float* const qpos = lds + L.qpos;
  float* const qvel = lds + L.qvel;
  float* const cdof = lds + L.cdof;
  float* const cinert = lds + L.cinert;
  float* const sc = lds + L.sc;
  float* const lpos = lds + L.lpos;
  float* const lquat = lds + L.lquat;
  const bool act_on = nu > 0 && !(m.opt.disableflags & mjhDSBL_ACTUATION);

  // smooth.py:469-536 first: the moments are in memory by the time the
  // actuators read them
  transmission(m, d, t);
  BodyConst c0{};
  unsigned long long below0 = 0, below1 = 0;  // bodies that dof `lane` (+ TEAM) moves
  if (ok) {
    const float* gq = WPTR(d.qpos, w, nq);
    const float* gv = WPTR(d.qvel, w, nv);
    for (int i = lane; i < nq; i += TEAM) qpos[i] = gq[i];
    for (int i = lane; i < nv; i += TEAM) qvel[i] = gv[i];
    if (lane < nb) c0 = body_const(m, lane);
    if (lane < nv)
      for (int b = 0; b < nb; b++) below0 |= (unsigned long long)(m.body_dof_tree[b * nv + lane] ? 1 : 0) << b;
    if (lane + TEAM < nv)
      for (int b = 0; b < nb; b++) below1 |= (unsigned long long)(m.body_dof_tree[b * nv + lane + TEAM] ? 1 : 0) << b;
  }
  wave_fence();

  // ---- smooth.py:32-145 kinematics: the joints' constants and angles
  // (lanes over joints) ...
  float4* const jloc = reinterpret_cast<float4*>(lds + L.jloc);
  float* const anchor = lds + L.anchor;
  float* const axis = lds + L.axis;
  float* const lmat = lds + L.lmat;
  float* const ipos = lds + L.ipos;
  float* const gximat = WPTR(d.ximat, w, nb * 9);
  if (ok) {
    for (int j = lane; j < nj; j += TEAM) {
      const int jt = m.jnt_type[j], qa = m.jnt_qposadr[j];
      const V3 ax = ld3(m.jnt_axis + 3 * j), jp = ld3(m.jnt_pos + 3 * j);
      jloc[2 * j] = make_float4(ax.x, ax.y, ax.z, jt < mjhJNT_SLIDE ? __int_as_float(qa) : qpos[qa] - m.qpos0[qa]);
      jloc[2 * j + 1] = make_float4(jp.x, jp.y, jp.z, 0.0f);
    }
    if (lane == 0) {
      st3(lpos, V3{0.f, 0.f, 0.f});
      st4(lquat, Q4{1.f, 0.f, 0.f, 0.f});
      const M33 I = {{1.f, 0.f, 0.f, 0.f, 1.f, 0.f, 0.f, 0.f, 1.f}};
      st9(lmat, I);
      st3(ipos, V3{0.f, 0.f, 0.f});
      st9(gximat, I);
    }
  }
  wave_fence();
  // ... and the poses level by level
  for (int l = 1; l < m.nlevel; l++) {
    if (ok)
      level_bodies(m, m.body_treeadr[l], level_end(m, l), c0, t, [&](const BodyConst& c) {
        V3 pos;
        Q4 quat;
        if (c.jn == 1 && body_joint_type(m, c, 0) == mjhJNT_FREE) {
          const float4 a4 = jloc[2 * c.ja];
          const int qa = __float_as_int(a4.w);
          pos = ld3(qpos + qa);
          quat = ld4(qpos + qa + 3);
          st3(anchor + 3 * c.ja, pos);
          st3(axis + 3 * c.ja, V3{a4.x, a4.y, a4.z});
        } else {
          pos = mulmv(ld9(lmat + 9 * c.pid), ld3(m.body_pos + 3 * c.b)) + ld3(lpos + 3 * c.pid);
          quat = mul_quat(ld4(lquat + 4 * c.pid), ld4(m.body_quat + 4 * c.b));
          for (int j = 0; j < c.jn; j++) {
            const int jj = c.ja + j, jt = body_joint_type(m, c, j);
            const float4 a4 = jloc[2 * jj], p4 = jloc[2 * jj + 1];
            const V3 jaxis = V3{a4.x, a4.y, a4.z}, jpos = V3{p4.x, p4.y, p4.z};
            const V3 anch = rot_vec_quat(jpos, quat) + pos;
            const V3 ax = rot_vec_quat(jaxis, quat);
            if (jt == mjhJNT_BALL) {
              quat = mul_quat(quat, ld4(qpos + __float_as_int(a4.w)));
              pos = anch - rot_vec_quat(jpos, quat);
            } else if (jt == mjhJNT_SLIDE) {
              pos = pos + ax * a4.w;
            } else if (jt == mjhJNT_HINGE) {
              quat = mul_quat(quat, axis_angle_to_quat(jaxis, a4.w));
              pos = anch - rot_vec_quat(jpos, quat);
            }
            st3(anchor + 3 * jj, anch);
            st3(axis + 3 * jj, ax);
          }
        }
        quat = qnormalize(quat);
        st3(lpos + 3 * c.b, pos);
        st4(lquat + 4 * c.b, quat);
        st9(lmat + 9 * c.b, quat_to_mat(quat));
        st3(ipos + 3 * c.b, pos + rot_vec_quat(ld3(m.body_ipos + 3 * c.b), quat));
        st9(gximat + 9 * c.b, quat_to_mat(mul_quat(quat, ld4(m.body_iquat + 4 * c.b))));
      });
    wave_fence();
  }

  // ---- smooth.py:148-245 com_pos
  if (ok)
    for (int b = lane; b < nb; b += TEAM) st3(sc + 3 * b, ld3(ipos + 3 * b) * m.body_mass[b]);
  wave_fence();
  if (ok && lane < 3)
    for (int b = nb - 1; b >= 0; b--) sc[3 * m.body_parentid[b] + lane] += sc[3 * b + lane];
  wave_fence();
  if (ok)
    for (int b = lane; b < nb; b += TEAM) st3(sc + 3 * b, ld3(sc + 3 * b) * (1.0f / m.subtree_mass[b]));
  wave_fence();
  if (ok) {
    sync();  // the inertia frames' stores
    for (int b = lane; b < nb; b += TEAM) {
      body_cinert(cinert + 10 * b, ld9(gximat + 9 * b), ld3(m.body_inertia + 3 * b), m.body_mass[b],
                  ld3(ipos + 3 * b) - ld3(sc + 3 * m.body_rootid[b]));
    }
    for (int j = lane; j < nj; j += TEAM) {
      const int b = m.jnt_bodyid[j];
      joint_cdof(cdof + 6 * m.jnt_dofadr[j], m.jnt_type[j], ld3(axis + 3 * j), lmat + 9 * b,
                 ld3(sc + 3 * m.body_rootid[b]) - ld3(anchor + 3 * j));
    }
  }
  wave_fence();
  if (ok) {
    flush_words(WPTR(d.xpos, w, nb * 3), lpos, 3 * nb, t);
    flush_words(WPTR(d.xquat, w, nb * 4), lquat, 4 * nb, t);
    flush_words(WPTR(d.xmat, w, nb * 9), lmat, 9 * nb, t);
    flush_words(WPTR(d.xipos, w, nb * 3), ipos, 3 * nb, t);
    flush_words(WPTR(d.xanchor, w, nj * 3), anchor, 3 * nj, t);
    flush_words(WPTR(d.xaxis, w, nj * 3), axis, 3 * nj, t);
    flush_words(WPTR(d.subtree_com, w, nb * 3), sc, 3 * nb, t);
    flush_words(WPTR(d.cinert, w, nb * 10), cinert, 10 * nb, t);
    flush_words(WPTR(d.cdof, w, nv * 6), cdof, 6 * nv, t);
    float* sxpos = WPTR(d.site_xpos, w, m.nsite * 3);
    float* sxmat = WPTR(d.site_xmat, w, m.nsite * 9);
    for (int s = lane; s < m.nsite; s += TEAM) {
      const int b = m.site_bodyid[s];
      const Q4 q = ld4(lquat + 4 * b);
      st3(sxpos + 3 * s, ld3(lpos + 3 * b) + rot_vec_quat(ld3(m.site_pos + 3 * s), q));
      st9(sxmat + 9 * s, quat_to_mat(mul_quat(q, ld4(m.site_quat + 4 * s))));
    }
  }
  wave_fence();

  // ---- smooth.py:248-314 crb
  {
    float* const lcrb = lds + L.crb;
    int* const lpar = reinterpret_cast<int*>(lds + L.par);
    float* const tri = lds + L.tri;
    float* const qMg = WPTR(d.qMd, w, nv * nv);
    if (ok) {
      for (int i = lane; i < nb * 10; i += TEAM) lcrb[i] = cinert[i];
      for (int i = lane; i < nv; i += TEAM) lpar[i] = m.dof_parentid[i];
      if (TEAM != 64) {
        for (int i = lane; i < nv * (nv + 1) / 2; i += TEAM) tri[i] = 0.0f;
      } else {
        for_each_tree_block(m, [&](int dof, int n) {
          for (int p = lane; p < n * n; p += TEAM) qMg[(dof + p / n) * nv + dof + p % n] = 0.0f;
        });
      }
    }
    if (TEAM == 64) sync();
    wave_fence();
    if (ok && lane < 10)
      for (int b = nb - 1; b >= 1; b--) {
        const int p = m.body_parentid[b];
        if (p != 0) lcrb[10 * p + lane] += lcrb[10 * b + lane];
      }
    wave_fence();
    if (ok) {
      for (int i = lane; i < nv; i += TEAM) {
        const S6 ci = ld6(cdof + 6 * i);
        const S6 buf = inert_vec(lcrb + 10 * m.dof_bodyid[i], ci);
        const float diag = m.dof_armature[i] + dot6(ci, buf);
        if (TEAM != 64) tri[i * (i + 1) / 2 + i] = diag;
        else qMg[i * nv + i] = diag;
        for (int j = lpar[i]; j >= 0; j = lpar[j]) {
          const float v = dot6(ld6(cdof + 6 * j), buf);
          if (TEAM != 64) {
            tri[i * (i + 1) / 2 + j] = v;
          } else {
            qMg[i * nv + j] = v;
            qMg[j * nv + i] = v;
          }
        }
      }
      flush_words(WPTR(d.crb, w, nb * 10), lcrb, 10 * nb, t);
    }
    wave_fence();
    if (TEAM == 64) sync();
    if (ok) {
      if (TEAM != 64) {
#pragma unroll 4
        for (int r = 0; r < nv; r++)
          if (lane < nv) qMg[r * nv + lane] = lane <= r ? tri[r * (r + 1) / 2 + lane] : tri[lane * (lane + 1) / 2 + r];
      }
      if (m.opt.is_sparse) {
        float* S = WPTR(d.qM, w, m.nM);
        if (TEAM == 64) {
          dense_to_sparse(m, qMg, S, t);
        } else {
          for (int i = lane; i < nv; i += TEAM) {
            int a = m.dof_Madr[i];
            for (int j = i; j >= 0; j = lpar[j]) S[a++] = tri[i * (i + 1) / 2 + j];
          }
        }
      }
    }
    wave_fence();
  }

  // ---- the geoms' poses, kept as records with the bounding test's numbers
  float* const geom = lds + L.geom;
  int* const list = reinterpret_cast<int*>(lds + L.list);
  if (ok) {
    for (int g = lane; g < ng; g += TEAM) {
      const int b = m.geom_bodyid[g];
      const Q4 q = ld4(lquat + 4 * b);
      float* r = geom + kGeomRec * g;
      st3(r, ld3(lpos + 3 * b) + rot_vec_quat(ld3(m.geom_pos + 3 * g), q));
      st9(r + 3, quat_to_mat(mul_quat(q, ld4(m.geom_quat + 4 * g))));
      r[12] = m.geom_rbound[g];
      r[13] = m.geom_margin[g];
      r[14] = __int_as_float(m.geom_type[g]);
    }
  }
  wave_fence();
  if (ok) {
    float* gxpos = WPTR(d.geom_xpos, w, ng * 3);
    float* gxmat = WPTR(d.geom_xmat, w, ng * 9);
    for (int i = lane; i < 3 * ng; i += TEAM) gxpos[i] = geom[kGeomRec * (i / 3) + i % 3];
#pragma unroll 2
    for (int i = lane; i < 9 * ng; i += TEAM) gxmat[i] = geom[kGeomRec * (i / 9) + 3 + i % 9];
  }

  // ---- collision: the candidate pairs that pass the bounding test go to a
  // list (type-ordered, in candidate order), on which the narrowphase runs
  // with a lane per pair; run in place, each round of candidates with a hit
  // ran it for the few lanes that had one.  A list that fills up is worked
  // off and begun again; the pairs are then enumerated once more for the
  // write pass.
  const bool fp = !(m.opt.disableflags & mjhDSBL_FILTERPARENT);
  const bool build_rows = !(m.opt.disableflags & mjhDSBL_CONSTRAINT);
  const bool do_limit = build_rows && !(m.opt.disableflags & mjhDSBL_LIMIT) && m.nlimited > 0;
  const bool do_crow = build_rows && !(m.opt.disableflags & mjhDSBL_CONTACT) && m.opt.cone == mjhCONE_PYRAMIDAL;
  const int ncand = m.nnxn;
  const GeomRecords poses{geom};
  auto for_hits = [&](auto f) {  // f(pairs on the list); returns how often the list was emptied before the last
    int n = 0, emptied = 0;
    for (int p0 = 0; p0 < ncand; p0 += TEAM) {
      const int p = p0 + lane;
      bool hit = false;
      int g1 = 0, g2 = 0;
      if (ok && p < ncand) {
        const int e = m.nxn_pair[p];
        g1 = e & 0x7fff;
        g2 = (e >> 15) & 0x7fff;
        hit = !(fp && ((e >> 30) & 1)) && bounds_hit(geom + kGeomRec * g1, geom + kGeomRec * g2);
      }
      int tot;
      const int off = team_exscan_bits<TEAM, 1>(hit ? 1 : 0, &tot);
      if (hit) {
        const int t1 = __float_as_int(geom[kGeomRec * g1 + 14]), t2 = __float_as_int(geom[kGeomRec * g2 + 14]);
        list[n + off] = t1 > t2 ? g2 | g1 << 7 : g1 | g2 << 7;
      }
      n += tot;
      if (n > TEAM) {  // the next round might not fit
        wave_fence();
        f(n);
        wave_fence();
        n = 0;
        emptied++;
      }
    }
    wave_fence();
    f(n);
    wave_fence();
    return make_int2(n, emptied);
  };
  int npair = 0, ncon = 0, ncact = 0, nlim = 0;
  const int2 left = for_hits([&](int n) {
    npair += n;
    for (int h = lane; h < n; h += TEAM) {
      const int e = list[h], g1 = e & 127, g2 = (e >> 7) & 127;
      ContactSink s{&d, 0, 0, 0, w, false, 0, 0};
      if (do_crow) {
        s.dim = pair_condim(m, g1, g2);
        s.incl = pair_includemargin(m, g1, g2);
      }
      narrowphase_pair(m, poses, g1, g2, s);
      ncon += s.k;
      ncact += s.nact;
      list[h] = e | s.k << 14;
    }
  });
  if (ok && do_limit)
    for (int k = lane; k < m.nlimited; k += TEAM) {
      float pos, J;
      nlim += limit_active(m, qpos, m.jnt_limited_slide_hinge_adr[k], &pos, &J) ? 1 : 0;
    }
  ncon = team_sum_int<TEAM>(ncon);
  ncact = team_sum_int<TEAM>(ncact);
  nlim = team_sum_int<TEAM>(nlim);
  const int nrow = build_rows ? nlim + 4 * ncact : 0;
  int pbase, cbase, ebase;
  team_reserve3<TEAM>(d.ncollision, ok ? npair : 0, d.ncon, ok ? ncon : 0, d.nefc, ok ? nrow : 0, &pbase, &cbase,
                      &ebase);
  if (ok) {
    const int cap = d.nconmax;
    const int npw = npair <= 0 ? 0 : max(0, min(npair, cap - pbase));
    const int ncw = ncon <= 0 ? 0 : max(0, min(ncon, cap - cbase));
    if (lane == 0) {
      d.world_pair[2 * w] = pbase;
      d.world_pair[2 * w + 1] = npw;
      if (pbase + npair > cap) atomicAdd(d.overflow + 0, min(npair, pbase + npair - cap));
      d.world_con[2 * w] = cbase;
      d.world_con[2 * w + 1] = ncw;
      if (cbase + ncon > cap) atomicAdd(d.overflow + 1, min(ncon, cbase + ncon - cap));
    }
    int kp = 0, kc = 0;
    auto write = [&](int n, bool counted) {
      for (int h0 = 0; h0 < n; h0 += TEAM) {
        const int h = h0 + lane;
        int c = 0, g1 = 0, g2 = 0;
        if (h < n) {
          const int e = list[h];
          g1 = e & 127;
          g2 = (e >> 7) & 127;
          const int i = kp + h;
          if (pbase + i < cap) {
            d.collision_pair[2 * (pbase + i)] = g1;
            d.collision_pair[2 * (pbase + i) + 1] = g2;
            d.collision_worldid[pbase + i] = w;
          }
          if (i < npw) {  // contacts only of pairs inside the pair pool
            c = (e >> 14) & 7;
            if (!counted) {
              ContactSink s{&d, 0, 0, 0, w, false, 0, 0};
              narrowphase_pair(m, poses, g1, g2, s);
              c = s.k;
            }
          }
        }
        int ctot;
        const int coff = team_exscan_bits<TEAM, 3>(c, &ctot);
        if (c > 0) {
          ContactSink s{&d, cbase, cap, kc + coff, w, true, 0, 0};
          narrowphase_pair(m, poses, g1, g2, s);
          const int fit = min(cbase + kc + coff + c, cap) - (cbase + kc + coff);
          if (fit > 0) contact_params(m, d, g1, g2, cbase + kc + coff, fit);
        }
        kc += ctot;
      }
      kp += n;
    };
    if (left.y == 0) write(left.x, true);
    else for_hits([&](int n) { write(n, false); });
  }

  // ---- smooth.py:539-606 com_vel
  float* const cdot = lds + L.cdot;
  float* const cvel = lds + L.vel;
  if (ok) {
    const float* gdot = WPTR(d.cdof_dot, w, nv * 6);
    for (int j = lane; j < nj; j += TEAM)
      if (m.jnt_type[j] == mjhJNT_FREE) {  // not com_vel's to write: zero, or the caller's
        const int da = m.jnt_dofadr[j];
        for (int i = 0; i < 18; i++) cdot[6 * da + i] = gdot[6 * da + i];
      }
    if (lane < 6) cvel[lane] = 0.0f;
  }
  wave_fence();
  for (int l = 1; l < m.nlevel; l++) {
    if (ok)
      level_bodies(m, m.body_treeadr[l], level_end(m, l), c0, t, [&](const BodyConst& c) {
        int da = c.da;
        S6 v = ld6(cvel + 6 * c.pid);
        for (int j = 0; j < c.jn; j++) da = joint_velocity(v, body_joint_type(m, c, j), da, cdof, cdot, qvel);
        st6(cvel + 6 * c.b, v);
      });
    wave_fence();
  }
  if (ok) {
    flush_words(WPTR(d.cvel, w, nb * 6), cvel, 6 * nb, t);
    flush_words(WPTR(d.cdof_dot, w, nv * 6), cdot, 6 * nv, t);
  }

  // ---- passive.py:27-108; spring in the room of rne's accelerations
  float* const spring = cvel + 6 * nb;
  float pas[2] = {0.0f, 0.0f};
  {
    const bool off = m.opt.disableflags & mjhDSBL_PASSIVE;
    float* qfrc_passive = WPTR(d.qfrc_passive, w, nv);
    if (ok && !off) {
      for (int i = lane; i < nv; i += TEAM) spring[i] = 0.0f;
    }
    wave_fence();
    if (ok && !off)
      for (int j = lane; j < nj; j += TEAM) joint_spring(m, j, qpos, spring);
    wave_fence();
    if (ok) {
      float* gspring = WPTR(d.qfrc_spring, w, nv);
      float* gdamper = WPTR(d.qfrc_damper, w, nv);
#pragma unroll
      for (int k = 0; k < 2; k++) {
        const int i = lane + k * TEAM;
        if (i >= nv) break;
        if (!off) {
          const float f = -m.dof_damping[i] * qvel[i];
          gspring[i] = spring[i];
          gdamper[i] = f;
          pas[k] = settle(f + spring[i]);
        }
        qfrc_passive[i] = pas[k];
      }
    }
    wave_fence();
  }

  // ---- smooth.py:398-466 rne
  float bias[2] = {0.0f, 0.0f};
  {
    float* const cacc = cvel + 6 * nb;
    float* const cfrc = cvel + 12 * nb;
    if (ok && lane < 6) {
      const bool nograv = m.opt.disableflags & mjhDSBL_GRAVITY;
      const float gl = lane == 3 ? m.opt.gravity[0] : (lane == 4 ? m.opt.gravity[1] : m.opt.gravity[2]);
      cacc[lane] = (lane < 3 || nograv) ? 0.0f : -gl;
    }
    wave_fence();
    for (int l = 0; l < m.nlevel; l++) {
      if (ok)
        level_bodies(m, m.body_treeadr[l], level_end(m, l), c0, t, [&](const BodyConst& c) {
          S6 a = ld6(cacc + 6 * c.pid);
          for (int i = 0; i < c.dn; i++) {
            const float qv = qvel[c.da + i];
#pragma unroll
            for (int k = 0; k < 6; k++) a.v[k] += cdot[6 * (c.da + i) + k] * qv;
          }
          st6(cacc + 6 * c.b, a);
        });
      wave_fence();
    }
    if (ok)
      for (int b = lane; b < nb; b += TEAM)
        st6(cfrc + 6 * b, body_force(cinert + 10 * b, ld6(cacc + 6 * b), ld6(cvel + 6 * b)));
    wave_fence();
    if (ok && lane < 6)
      for (int b = nb - 1; b >= 0; b--) cfrc[6 * m.body_parentid[b] + lane] += cfrc[6 * b + lane];
    wave_fence();
    if (ok) {
      flush_words(WPTR(d.rne_cacc, w, nb * 6), cacc, 6 * nb, t);
      flush_words(WPTR(d.rne_cfrc, w, nb * 6), cfrc, 6 * nb, t);
      float* gbias = WPTR(d.qfrc_bias, w, nv);
#pragma unroll
      for (int k = 0; k < 2; k++) {
        const int i = lane + k * TEAM;
        if (i >= nv) break;
        bias[k] = settle(dot6(ld6(cdof + 6 * i), ld6(cfrc + 6 * m.dof_bodyid[i])));
        gbias[i] = bias[k];
      }
    }
    wave_fence();
  }

  // ---- forward.py:423-496, 503-641: the actuators, velocities and forces in
  // LDS (entries that the tile loop does not reach keep what memory holds)
  float act[2] = {0.0f, 0.0f};
  {
    float* const avel = cvel;
    float* const aforce = cvel + nu;
    float* const gact = WPTR(d.qfrc_actuator, w, nv);
    float* const gvel = WPTR(d.actuator_velocity, w, nu);
    const float* moment = WPTR(d.actuator_moment, w, nu * nv);
    sync();  // the moments' stores
    if (ok) {
      for (int a = lane; a < nu; a += TEAM) avel[a] = gvel[a];
      if (m.opt.is_sparse) {
        for (int a = lane; a < nu; a += TEAM) {
          float s = 0.0f;
#pragma unroll 8
          for (int j = 0; j < nv; j++) s += moment[(size_t)a * nv + j] * qvel[j];
          avel[a] = s;
        }
      } else {
        for_each_act_tile(m, m.nact_group, [&](int onv, int onu, int tnv, int tnu) {
          if (tnu == 0 || tnv == 0) return;
          for (int a = lane; a < tnu; a += TEAM) {
            float s = 0.0f;
            const float* row = moment + (onu + a) * nv + onv;
#pragma unroll 8
            for (int j = 0; j < tnv; j++) s += row[j] * qvel[onv + j];
            avel[onu + a] = s;
          }
        });
      }
    }
    wave_fence();
    if (ok) {
      for (int a = lane; a < nu; a += TEAM) gvel[a] = avel[a];
      if (!act_on) {
        float* act_dot = WPTR(d.act_dot, w, m.na);
        for (int i = lane; i < m.na; i += TEAM) act_dot[i] = 0.0f;
      } else {
        float* gforce = WPTR(d.actuator_force, w, nu);
        for (int a = lane; a < nu; a += TEAM) {
          const float f = actuator_force(m, a, d.actuator_length[(size_t)w * nu + a], avel[a], d.ctrl[(size_t)w * nu + a]);
          aforce[a] = f;
          gforce[a] = f;
        }
      }
    }
    wave_fence();
    if (ok) {
#pragma unroll
      for (int k = 0; k < 2; k++) {
        const int i = lane + k * TEAM;
        if (i >= nv) break;
        float q = 0.0f;
        if (act_on) {
          q = gact[i];
          if (m.opt.is_sparse) {
            float s = 0.0f;
#pragma unroll 8
            for (int a = 0; a < nu; a++) s += moment[(size_t)a * nv + i] * aforce[a];
            q = s;
          } else {
            for_each_act_tile(m, m.nact_group, [&](int onv, int onu, int tnv, int tnu) {
              if (tnu == 0 || i < onv || i >= onv + tnv) return;
              float s = 0.0f;
#pragma unroll 8
              for (int a = 0; a < tnu; a++) s += moment[(onu + a) * nv + i] * aforce[onu + a];
              q = s;
            });
          }
          const int j = m.dof_jntid[i];
          if (m.jnt_actfrclimited[j]) q = fminf(fmaxf(q, m.jnt_actfrcrange[2 * j]), m.jnt_actfrcrange[2 * j + 1]);
        }
        act[k] = settle(q);
        gact[i] = act[k];
      }
    }
    wave_fence();
  }

  // ---- forward.py:644-661 and support.py:140-172: qfrc_smooth; the bodies'
  // applied forces and their offsets staged, a dof's bodies taken off its mask
  {
    float* const body = cvel;  // offset, force, torque
    const float* xfrc = WPTR(d.xfrc_applied, w, nb * 6);
    const float* xipos = WPTR(d.xipos, w, nb * 3);
    if (ok)
      for (int b = lane; b < nb; b += TEAM) {
        st3(body + 9 * b, ld3(xipos + 3 * b) - ld3(sc + 3 * m.body_rootid[b]));
        st6(body + 9 * b + 3, ld6(xfrc + 6 * b));
      }
    wave_fence();
    if (ok) {
      const float* app = WPTR(d.qfrc_applied, w, nv);
      float* qs = WPTR(d.qfrc_smooth, w, nv);
#pragma unroll
      for (int k = 0; k < 2; k++) {
        const int i = lane + k * TEAM;
        if (i >= nv) break;
        const S6 c = ld6(cdof + 6 * i);
        const V3 rot = V3{c.v[0], c.v[1], c.v[2]}, lin = V3{c.v[3], c.v[4], c.v[5]};
        float acc = 0.0f;
        for (unsigned long long left_b = k == 0 ? below0 : below1; left_b; left_b &= left_b - 1) {
          const int b = __ffsll(left_b) - 1;
          if (b < m.dof_bodyid[i]) continue;
          const V3 off = ld3(body + 9 * b), f = ld3(body + 9 * b + 3), tq = ld3(body + 9 * b + 6);
          acc += dot(lin, f) + dot(rot, tq) + dot(cross(rot, off), f);
        }
        const float q = settle(pas[k] - bias[k] + act[k] + app[i]);
        qs[i] = q + acc;
      }
    }
    wave_fence();
  }

  // ---- constraint.py:213-240 (the contacts' stores are long done)
  if (build_rows) {
    sync();
    make_constraint_rows<TEAM, kFwdRowChunk>(m, d, lds + L.rows, t, ebase, nrow, nlim, qpos, qvel, cdof, sc,
                                             [&](int b, int i) { return ((i < TEAM ? below0 : below1) >> b) & 1ull; });
  }
}

}  // namespace mjh
