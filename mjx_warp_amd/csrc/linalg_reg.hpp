// Register-resident dense linear algebra for 32-lane teams (nv <= 32).
//
// A world's nv x nv symmetric positive definite matrix is held one row per
// lane (lane i owns row i in VGPRs), padded to NVC (a multiple of 4) with
// identity rows so that every loop has a compile-time trip count.  Block-
// diagonal matrices (one block per kinematic tree, as the reference's dense
// tiles, io.py:150-162) are factored as a whole: entries outside a lane's
// block are zero, so the factor's blocks equal the per-block factors.
//
// Team primitives used here and by the register solver: DPP sums, lane
// broadcasts and LDS broadcast buffers.  LDS instructions of one wavefront
// execute in issue order, so a write followed by reads of the same wavefront
// needs no barrier, only a compiler fence.
#pragma once

#include <type_traits>

#include "common.hpp"

namespace mjh {

constexpr int kRegTeam = 32;
constexpr int kRegNvMax = 32;
// LDS floats a 32-lane team needs at least: RegChol's column broadcast
// buffer (one float per lane)
constexpr int kRegLdsMin = 32;

// Row stride of nvc-column rows staged in LDS (matrix rows, Jacobian rows):
// an odd number of float4s (nvc or nvc + 4), so that a row is read as float4s
// -- by every lane at once (the Hessian's rank-1 updates) or a row per lane
// without bank conflicts -- and a column entry per lane stays conflict free.
__host__ __device__ constexpr int reg_row_stride(int nvc) { return (nvc / 4) % 2 ? nvc : nvc + 4; }
// LDS floats of the broadcast buffer and one staged matrix
__host__ __device__ constexpr int lds_reg_matrix(int nvc) { return kRegLdsMin + nvc * reg_row_stride(nvc); }

MJH_DEV void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  asm volatile("" ::: "memory");
}

// `yes` in the lanes of a constant mask (over the 32 lanes of a team), `no` in
// the others.  The mask is two scalar moves at its use, where a comparison
// with the lane number is a vector instruction for each column, and masks that
// the compiler knows of leave a loop for scalar registers that it then spills.
// kDpp: the result is a DPP operand, read two wait states after the write at the
// earliest (the compiler keeps that distance for its own instructions only).
template <unsigned MASK, bool kDpp = false>
MJH_DEV float pick(float yes, float no) {
  float r;
  if constexpr (kDpp)
    asm("s_mov_b32 vcc_lo, %3\n\ts_mov_b32 vcc_hi, vcc_lo\n\tv_cndmask_b32_e32 %0, %1, %2, vcc\n\ts_nop 1"
        : "=v"(r) : "v"(no), "v"(yes), "i"(MASK) : "vcc");
  else
    asm("s_mov_b32 vcc_lo, %3\n\ts_mov_b32 vcc_hi, vcc_lo\n\tv_cndmask_b32_e32 %0, %1, %2, vcc"
        : "=v"(r) : "v"(no), "v"(yes), "i"(MASK) : "vcc");
  return r;
}
// lane k, and the lanes past k
constexpr unsigned lane_mask(int k) { return 1u << k; }
constexpr unsigned past_mask(int k) { return k < 31 ? ~0u << (k + 1) : 0u; }
// y - z[k] h in one 16-lane row of each team (HIGH: the upper), z[k] from lane
// k of that row.  The wait is for a z written just before.
template <int K, bool HIGH>
MJH_DEV void sub_row(float* y, float z, float h) {
  if constexpr (HIGH)
    asm("s_nop 1\n\tv_fmac_f32_dpp %0, -%1, %2 row_newbcast:%3 row_mask:0xa bank_mask:0xf"
        : "+v"(*y) : "v"(z), "v"(h), "i"(K));
  else
    asm("s_nop 1\n\tv_fmac_f32_dpp %0, -%1, %2 row_newbcast:%3 row_mask:0x5 bank_mask:0xf"
        : "+v"(*y) : "v"(z), "v"(h), "i"(K));
}
// Calls f(std::integral_constant<int, k>) for k = B .. E - 1.
template <int B, int E, class F>
MJH_DEV void unrolled(F f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    unrolled<B + 1, E>(f);
  }
}

// p, opaque to the optimiser: address arithmetic on it is redone at each use
// instead of being hoisted out of a loop into live VGPRs.
typedef __attribute__((address_space(1))) const float gfloat;
MJH_DEV gfloat* opaque(const float* p) {
  gfloat* q = (gfloat*)p;
  asm volatile("" : "+v"(q));
  return q;
}
MJH_DEV int opaque(int i) {
  asm volatile("" : "+v"(i));
  return i;
}

// v, computed before any memory access that follows: keeps the compiler from
// issuing the loads of several dot products together, whose operands then
// hold the registers of another wavefront per SIMD (200 VGPRs against 150).
MJH_DEV float settle(float v) {
  asm volatile("" : "+v"(v) : : "memory");
  return v;
}

// Calls f(std::integral_constant<int, NVC>) with NVC = nv rounded up to 4.
template <class F>
MJH_DEV auto with_nvc(int nv, F f) {
  switch ((nv + 3) / 4) {
    case 1: return f(std::integral_constant<int, 4>{});
    case 2: return f(std::integral_constant<int, 8>{});
    case 3: return f(std::integral_constant<int, 12>{});
    case 4: return f(std::integral_constant<int, 16>{});
    case 5: return f(std::integral_constant<int, 20>{});
    case 6: return f(std::integral_constant<int, 24>{});
    case 7: return f(std::integral_constant<int, 28>{});
    default: return f(std::integral_constant<int, 32>{});
  }
}

// The tree block [beg, end) holding `dof` (padding lanes: [dof, dof + 1)).
MJH_DEV void tree_block(const mjhModel& m, int dof, int* beg, int* end) {
  *beg = dof;
  *end = dof + 1;
  for_each_tree_block(m, [&](int d0, int n) {
    if (dof >= d0 && dof < d0 + n) {
      *beg = d0;
      *end = d0 + n;
    }
  });
}

// Staged rows (stride reg_row_stride(NVC)) into the blocks [beg, end) of A
// (global, [nv, nv]), a row at a time with lanes over columns (a column's
// block holds the rows [beg, end) too); lower: zeros above the diagonal.
template <int NVC>
MJH_DEV void store_blocks(float* A, int nv, int beg, int end, int lane, const float* rows, bool lower) {
  if (lane < nv) {
#pragma unroll 4
    for (int r = 0; r < nv; r++)
      if (r >= beg && r < end) A[r * nv + lane] = (lower && lane > r) ? 0.0f : rows[r * reg_row_stride(NVC) + lane];
  }
  wave_fence();
}

template <int NVC>
struct RegChol {
  static_assert(NVC % 4 == 0 && NVC <= kRegNvMax, "padded dof count");
  int lane;     // 0..31: the row this lane owns
  float* cbuf;  // [kRegLdsMin] LDS column broadcast buffer of the team
  float h[NVC];  // matrix row, then factor row (lower part)
  float rdiag;   // 1 / L[lane][lane]

  // Row `lane` of a symmetric matrix read column-wise from global memory
  // (A[j * nv + lane], coalesced across the team), restricted to the lane's
  // tree block [beg, end); padding rows are identity rows.
  // `diag` is added to the lane's diagonal entry.
  MJH_DEV void load_sym(const float* A, int nv, int beg, int end, float diag = 0.0f) {
    const int ln = opaque(lane);
    gfloat* Ac = opaque(A) + (ln < nv ? ln : 0);
#pragma unroll
    for (int j = 0; j < NVC; j++) {
      const float v = Ac[(j < nv ? j : 0) * nv] + (j == ln ? diag : 0.0f);
      h[j] = (ln < nv && j >= beg && j < end) ? v : (j == ln ? 1.0f : 0.0f);
    }
    rdiag = 1.0f;
  }

  static constexpr int JS = reg_row_stride(NVC);
  // the staged row this lane reads: its own (lanes past the padding read the
  // last row; nothing they derive from it reaches another lane)
  MJH_DEV const float4* row4(const float* rows) const {
    return reinterpret_cast<const float4*>(rows + (lane < NVC ? lane : NVC - 1) * JS);
  }

  // Row `lane` of a matrix staged by stage_sym, of a mass matrix that crb
  // wrote: entries of dofs in different trees are zero, so no block to select.
  MJH_DEV void load_rows(const float* rows) {
    const float4* r = row4(rows);
#pragma unroll
    for (int q = 0; q < NVC / 4; q++) {
      const float4 v = r[q];
      h[4 * q] = v.x;
      h[4 * q + 1] = v.y;
      h[4 * q + 2] = v.z;
      h[4 * q + 3] = v.w;
    }
    rdiag = 1.0f;
  }

  // The lower factor's row `lane` from global memory, restricted to the
  // lane's block (from column beg to before the diagonal), by way of the staging
  // buffer `rows` (NVC rows): a row per lane read in place touches a cache
  // line per lane with every load.
  MJH_DEV void load_lower(const float* L, int nv, int beg, float* rows) {
    gfloat* Lc = opaque(L) + (lane < nv ? lane : 0);
    wave_fence();
    if (lane < NVC) {
#pragma unroll 7  // seven or eight: the same within 1 % at 27 dofs
      for (int r = 0; r < nv; r++) rows[r * JS + lane] = Lc[r * nv];
    }
    wave_fence();
    const float4* r4 = row4(rows);
    const int ln = opaque(lane);
    const bool dof = ln < nv;
#pragma unroll
    for (int q = 0; q < NVC / 4; q++) {
      const float4 v = r4[q];
      const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int j = 4 * q + u;
        h[j] = (dof && j >= beg && j < ln) ? e[u] : 0.0f;
      }
    }
    rdiag = dof ? 1.0f / rows[ln * JS + ln] : 1.0f;
    wave_fence();
  }
  // rdiag as load_lower sets it, from a factor that store_rows staged
  MJH_DEV void divide_diag(const float* rows, int nv) { rdiag = lane < nv ? 1.0f / rows[lane * JS + lane] : 1.0f; }

  // Cholesky H = L L' of the lane-owned rows (right-looking, one column
  // broadcast through LDS per step).  Lane i keeps L[i][0..i-1] in h[0..i-1],
  // zeros from there on and 1 / L[i][i] in rdiag: what solve() reads.
  // kDiag: the diagonal of L is in h[i] too, to be stored (drop_diag() then
  // makes it a factor for solve()).  rsq: 1 / L[i][i] from one reciprocal square root, which
  // differs from square root and reciprocal in the last bit (callers keep the
  // form they have, so that their results stay as they are).
  template <bool kDiag = true>
  MJH_DEV void factor(bool rsq = false) {
    const int ln = lane;
    wave_fence();
    cbuf[ln] = h[0];
    unrolled<0, NVC>([&](auto col) {
      constexpr int k = col;
      wave_fence();
      float c[NVC];
#pragma unroll
      for (int q = k / 4; q < NVC / 4; q++) {
        const float4 v = reinterpret_cast<const float4*>(cbuf)[q];
        c[4 * q] = v.x;
        c[4 * q + 1] = v.y;
        c[4 * q + 2] = v.z;
        c[4 * q + 3] = v.w;
      }
      const float dkk = c[k];
      float lkk = __builtin_amdgcn_sqrtf(dkk);
      asm("" : "+v"(lkk));  // else the compiler may make a rsq of the two
      const float inv = rsq ? __builtin_amdgcn_rsqf(dkk) : __builtin_amdgcn_rcpf(lkk);
      // L[i][k] L[j][k] = H[i][k] H[j][k] / dkk
      const float hk = pick<past_mask(k)>(h[k], 0.0f);
      const float g = hk * (inv * inv);
      // the next column first, and on its way to the other lanes while the rest
      // is worked
      if constexpr (k + 1 < NVC) {
        h[k + 1] = fmaf(-g, c[k + 1], h[k + 1]);
        wave_fence();
        cbuf[ln] = h[k + 1];
      }
#pragma unroll
      for (int j = k + 2; j < NVC; j++) h[j] = fmaf(-g, c[j], h[j]);
      rdiag = pick<lane_mask(k)>(inv, rdiag);
      h[k] = hk * inv;
      if (kDiag) h[k] = pick<lane_mask(k)>(lkk, h[k]);
    });
  }
  MJH_DEV void drop_diag() {
    unrolled<0, NVC>([&](auto k) { h[k] = pick<lane_mask(k)>(0.0f, h[k]); });
  }

  // x = inv(L L') b with L from factor() / load_lower() (h zero from the
  // diagonal on); b, x one entry per lane (padding lanes carry 0).
  // The two substitutions are a serial chain of NVC steps each, and where
  // wavefronts are many their instructions are what the solver issues, so a
  // step is kept inside the 16-lane row that owns it: its value comes by the
  // row's own broadcast within the multiply-add, and what one row owes the
  // other passes at once, when the row is done.  (A value for both rows at every
  // step, masks compared with the lane number and five-level sums were 680
  // vector instructions at 28 columns; these are 362.  8192 humanoids 908 to 880 us
  // for two steps, 24576 lying ones 3773 to 3682.)
  MJH_DEV float solve(float b) const {
    constexpr int N0 = NVC < 16 ? NVC : 16;
    // forward: y = inv(L) b, column by column
    float y = b;
    unrolled<0, N0>([&](auto k) { sub_row<k, false>(&y, y * rdiag, h[k]); });
    if constexpr (NVC > 16) {
      const float z = __int_as_float(swap_rows(__float_as_int(y * rdiag)).even);
      unrolled<0, 16>([&](auto k) { sub_row<k, true>(&y, z, h[k]); });
      unrolled<16, NVC>([&](auto k) { sub_row<k - 16, true>(&y, y * rdiag, h[k]); });
    }
    y *= rdiag;
    asm("" : "+v"(y));  // rounded here, not within the differences below
    // backward: x = inv(L') y, x[k] = (y[k] - sum_{j>k} L[j][k] x[j]) / L[k][k],
    // the sums in the order of sum32.  The lanes j <= k have a zero L or a
    // zero x, so the levels that would add only those are left out.
    float x = 0.0f;
    auto row_sum = [&](int k) {
      float p = h[k] * x;
      asm("" : "+v"(p));
      p += dpp_f<0xB1>(p);
      p += dpp_f<0x4E>(p);
      if ((k & 15) < 12) p += dpp_f<0x141>(p);
      if ((k & 15) < 8) p += dpp_f<0x140>(p);
      return p;
    };
    unrolled<0, NVC - N0>([&](auto i) {
      constexpr int k = NVC - 1 - i;
      x = pick<lane_mask(k)>((y - row_sum(k)) * rdiag, x);
    });
    float upper = 0.0f;
    if constexpr (NVC > 16) upper = __int_as_float(swap_rows(__float_as_int(upper_sums(x))).odd);
    unrolled<0, N0>([&](auto i) {
      constexpr int k = N0 - 1 - i;
      float s = row_sum(k);
      if (NVC > 16) s += upper;
      x = pick<lane_mask(k)>((y - s) * rdiag, x);
    });
    return x;
  }

  // In lane l the sum over l's row of L[j][l % 16] x[j], added as sum32 adds a
  // row: of the 16 columns' sums each level hands the half that the partner
  // lane keeps to it (15 adds for 16 sums of four levels).  Lane l keeps the
  // column c = l % 16 through all levels: level 1 decides bit 0 ^ bit 2 of c,
  // level 2 bit 1 ^ bit 2, level 3 bit 2 ^ bit 3 and level 4 bit 3, each of
  // which differs between that level's partners and is the same between those
  // of all later ones (l ^ 1, l ^ 2, l ^ 7, l ^ 15).
  MJH_DEV float upper_sums(float x) const {
    float a[16], b[8], c[4], e[2];
#pragma unroll
    for (int k = 0; k < 16; k++) {
      a[k] = h[k] * x;
      asm("" : "+v"(a[k]));
    }
    // lanes with bit 0 ^ bit 2, bit 1 ^ bit 2, bit 2 ^ bit 3, bit 3
    constexpr unsigned m1 = 0x5a5a5a5au, m2 = 0x3c3c3c3cu, m3 = 0x0ff00ff0u, m4 = 0xff00ff00u;
    // pairs of columns that differ in the level's bit and agree in the later
    // levels': c and c ^ 1, then c ^ 2, c ^ 7 and c ^ 15
#pragma unroll
    for (int i = 0; i < 8; i++) {  // columns 2 i, 2 i + 1; the first has bit 0 ^ bit 2 = (i >> 1) & 1
      const int f = (i >> 1) & 1;
      const float lo = a[2 * i + f], hi = a[2 * i + 1 - f];
      b[i] = pick<m1>(hi, lo) + dpp_f<0xB1>(pick<m1, true>(lo, hi));
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {  // b[2 i], b[2 i + 1] are columns 4 i.. and 4 i + 2..
      const int f = i & 1;
      const float lo = b[2 * i + f], hi = b[2 * i + 1 - f];
      c[i] = pick<m2>(hi, lo) + dpp_f<0x4E>(pick<m2, true>(lo, hi));
    }
#pragma unroll
    for (int i = 0; i < 2; i++) {  // c[2 i], c[2 i + 1] are columns 8 i.. and 8 i + 4..
      const int f = i;
      const float lo = c[2 * i + f], hi = c[2 * i + 1 - f];
      e[i] = pick<m3>(hi, lo) + dpp_f<0x141>(pick<m3, true>(lo, hi));
    }
    return pick<m4>(e[1], e[0]) + dpp_f<0x140>(pick<m4, true>(e[0], e[1]));
  }

  // Writes the rows into the blocks [beg, end) of A (global, [nv, nv]) by
  // way of the staging buffer `rows` (NVC rows): stored a row at a time with
  // lanes over columns, where a row per lane sent every word to the cache as
  // a request of its own.  lower: the factor's lower triangle and zeros above
  // the diagonal inside a block, as the reference's tile factor
  // (smooth.py:353-379).
  MJH_DEV void store_rows(float* A, int nv, int beg, int end, float* rows, bool lower) const {
    wave_fence();
    if (lane < NVC) {
      float4* r4 = reinterpret_cast<float4*>(rows + lane * JS);
#pragma unroll
      for (int q = 0; q < NVC / 4; q++) r4[q] = make_float4(h[4 * q], h[4 * q + 1], h[4 * q + 2], h[4 * q + 3]);
    }
    wave_fence();
    store_blocks<NVC>(A, nv, beg, end, lane, rows, lower);
  }
};

// Stages the symmetric matrix A (global, [nv, nv]) into LDS rows (NVC rows
// of stride reg_row_stride(NVC)), padded with identity rows: lane i loads
// column i, coalesced across the team, as row i.
template <int NVC>
MJH_DEV void stage_sym(const float* A, int nv, int lane, float* rows) {
  const int ln = opaque(lane);
  gfloat* Ac = opaque(A) + (ln < nv ? ln : 0);
  float4 v[NVC / 4];
#pragma unroll
  for (int q = 0; q < NVC / 4; q++) {
    float e[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int j = 4 * q + u;
      const float a = Ac[(j < nv ? j : 0) * nv];
      e[u] = (ln < nv && j < nv) ? a : (j == ln ? 1.0f : 0.0f);
    }
    v[q] = make_float4(e[0], e[1], e[2], e[3]);
  }
  wave_fence();
  if (ln < NVC) {
    float4* r4 = reinterpret_cast<float4*>(rows + ln * reg_row_stride(NVC));
#pragma unroll
    for (int q = 0; q < NVC / 4; q++) r4[q] = v[q];
  }
  wave_fence();
}

// qLD = tree-block Cholesky factors of qM, in registers (32-lane teams);
// lds: lds_reg_matrix
MJH_DEV void reg_factor_blocks(const mjhModel& m, const float* M, float* L, float* lds, const Team<kRegTeam>& t) {
  const int nv = m.nv;
  int beg, end;
  tree_block(m, t.lane, &beg, &end);
  with_nvc(nv, [&](auto nvc) {
    RegChol<decltype(nvc)::value> c{t.lane, lds};
    c.load_sym(M, nv, beg, end);
    c.factor();
    c.store_rows(L, nv, beg, end, lds + kRegLdsMin, true);
    return 0;
  });
}

// x = inv(M) y from the tree-block factor L (qLD), in registers; x may
// alias y; lds: lds_reg_matrix
MJH_DEV void reg_solve_blocks(const mjhModel& m, const float* L, float* x, const float* y, float* lds,
                              const Team<kRegTeam>& t) {
  const int nv = m.nv;
  int beg, end;
  tree_block(m, t.lane, &beg, &end);
  const float b = t.lane < nv ? y[t.lane] : 0.0f;
  const float r = with_nvc(nv, [&](auto nvc) {
    RegChol<decltype(nvc)::value> c{t.lane, lds};
    c.load_lower(L, nv, beg, lds + kRegLdsMin);
    return c.solve(b);
  });
  if (t.lane < nv) x[t.lane] = r;
}

}  // namespace mjh
