// Per-reactor variable-order BDF (CVODE v5.8.0 algorithm) on one wavefront.
//
// Layout: lane j < nsp holds species j, lane nsp holds y_T = T/Tref (the
// reference state order), lanes above are padding (identically zero, zero
// error weight).  Every CVODE vector (Nordsieck history zn[0..5], ewt,
// acor, ...) is one register per lane; CVODE's scalars are wave-uniform.
//
// Linear algebra: the analytic Jacobian
// (applications/cfd_plugin/reactor_nvector_serial.cpp:610-771) is assembled
// column by column into the wave's LDS and saved to HBM for reuse; the Newton
// matrix M = I - gamma*J is inverted in registers by Gauss-Jordan elimination
// without pivoting (row per lane, columns rotated one register per step so
// every register index is a compile-time constant), and each Newton solve is
// then an LDS matrix-vector product.  This is the explicit-inverse scheme of
// the reference GPU path (interfaces/cublas_manager/cublas_manager.cu:73-91,
// getrf/getri without pivoting + block-diagonal matvec); a zero pivot is a
// recoverable setup failure, like a singular dense factorisation in CVODE.
//
// CVODE structure restated (names kept): cvStep, cvPredict, cvSet/cvSetBDF,
// cvSetTqBDF, cvNls + SUNNonlinSol_Newton, cvLsSetup/cvLsLinSys, cvLsSolve
// (with the 2/(1+gamrat) BDF correction), cvHandleNFlag, cvDoErrorTest,
// cvCompleteStep, cvPrepareNextStep, cvChooseEta, cvSetEta, cvAdjustOrder,
// cvRescale, cvRestore, cvHin, CVodeGetDky; the plugin's driver loop is
// applications/cfd_plugin/solver_cvode.cpp:220-299.
#pragma once

#include <cfloat>
#include <utility>

#include "bdf_launch.h"
#include "chem_device.h"

namespace zrk {

constexpr int kQmax = 5;

// ---------------------------------------------------------------------------
// Reference analytic Jacobian into LDS, column-major J[c*kNP + row], and a
// copy to HBM (savedJ).  inv_rho_prev is the inverse density of the last RHS
// call (at y), which the reference reuses for the 1/C factors
// (reactor_nvector_serial.cpp:625-637).  Returns the inverse density of the
// last RHS evaluated here (the reference's carried value).  t2l: kNP doubles
// of LDS scratch.  Jl is column-major with column stride ld >= nsp + 1 and
// only rows <= nsp are written (the term table holds no terms for lanes at
// or beyond nsp); saved is column-major with stride kNP.
//
// Species block: lane i walks row i's term list (sorted by column), so each
// entry has one writer and the loads of the list are coalesced across lanes;
// the temperature row and the MW_i/MW_j scaling follow column by column.
// Every entry is accumulated in FP64; MT = float stores the finished entries
// in FP32 (the FP32 preconditioner keeps its Jacobian in FP32).
// ---------------------------------------------------------------------------
//
// solveT = false (temperature held, not a state variable): the temperature
// row and column are zero and the finite-difference evaluation is skipped,
// as the reference's Jacobian without temperature has neither
// (reactor_nvector_serial.cpp:641-643, 691-750).
template <typename MT, class Team>
__device__ __forceinline__ double jacobian_lds(const Team& team, const DevMech& m, const RhsLds& s, double P,
                                               double v0, const BdfOpts& o, double y, double fy,
                                               double inv_rho_prev, MT* __restrict__ Jl, int ld,
                                               MT* __restrict__ saved,
                                               double* __restrict__ t2l, RhsSrc src = {},
                                               bool solveT = true) {
  const int lane = lane_id();
  const int nsp = m.nsp;
  const bool sp = lane < nsp;
  const bool act = lane <= nsp;
  const double mmf = o.min_mass_fraction;
  double t1 = y;
  if (sp && fabs(t1) < mmf) t1 = (t1 < 0.0) ? -mmf : mmf;
  const double t2 = sp ? m.mw[lane] / t1 * inv_rho_prev : 0.0;
  t2l[lane] = t2;
  // d(ydot)/dT by forward difference at the unfloored state.  Evaluated
  // first: it does not depend on the floored evaluation, and its inverse
  // density is the one carried on (it is the reference's last call).
  const double yT = bcast(y, nsp);
  double dT = yT * sqrt(DBL_EPSILON);
  const double Tp = yT + dT;
  dT = Tp - yT;
  const double t4in = (lane == nsp) ? Tp : (sp ? y : 0.0);
  double colT = 0.0;
  RhsAux aux2;
  if (solveT) {
    double t4;
    rhs_team(team, m, s, P, v0, o.Tref, o.step_limiter, t4in, t4, aux2, src);
    colT = act ? (t4 - fy) * (1.0 / dT) : 0.0;
  }
  // floored evaluation: rates of progress for every species term
  double t3;
  RhsAux aux;
  rhs_team(team, m, s, P, v0, o.Tref, o.step_limiter, t1, t3, aux, src);
  if (!solveT) aux2.inv_rho = aux.inv_rho;  // the last evaluation's
  const double Tdot = bcast(t3, nsp);
  const double RuTemp = kRu * yT;
  const double mult = -1.0 / aux.cp_mix;
  const double mwi = sp ? m.mw[lane] : 0.0;
  if (act)
    for (int c = 0; c < nsp; ++c) Jl[c * ld + lane] = MT(0);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  {
    // each product ROP*invC is rounded once, then added or subtracted as the
    // reference's J -= ROP*invC / J += ROP*invC, so balanced terms cancel exactly
    const uint4* __restrict__ jr = m.jr + lane;
    const int nb = m.jr_blocks;
    int cur = -1;
    double v = 0.0;
    auto term = [&](unsigned t) {
      const int col = (int)((t >> 16) & 0xFFu);
      if (col != 0xFF) {
        if (col != cur) {
          cur = col;
          v = 0.0;
        }
        if (Team::kExt && (t & kJtNonInt)) {
          // (multiplier * ROP) / C_col (non_integer_reaction_network.cpp:493-506)
          const double2 e = m.ni_jt[t & 0xFFFFu];
          v = __dadd_rn(v, __dmul_rn(__dmul_rn(e.x, s.rop[(int)e.y]), t2l[col]));
        } else {
          const double p = __dmul_rn(s.rop[t & 0xFFFFu], t2l[col]);
          v = (t & 0x80000000u) ? __dsub_rn(v, p) : __dadd_rn(v, p);
        }
        Jl[col * ld + lane] = (MT)v;
      }
    };
    uint4 w = nb > 0 ? jr[0] : make_uint4(0, 0, 0, 0);
    for (int b = 0; b < nb; ++b) {
      const uint4 x = w;
      if (b + 1 < nb) w = jr[(b + 1) * kWave];
      term(x.x);
      term(x.y);
      term(x.z);
      term(x.w);
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  for (int c = 0; c < nsp; ++c) {
    const double v = sp ? (double)Jl[c * ld + lane] : 0.0;
    // d(Tdot)/dy_c from the concentration-space column
    double val = 0.0;
    if (solveT) {
      const double sc = wave_sum(v * aux.h);
      val = sc * RuTemp;
      val += Tdot * bcast(aux.cpm, c) * m.mw[c];
      val *= m.inv_mw[c] * mult;
    }
    const double out = sp ? v * (mwi * m.inv_mw[c]) : (lane == nsp ? val : 0.0);
    if (act) Jl[c * ld + lane] = (MT)out;
    saved[c * kNP + lane] = (MT)out;
  }
  if (act) Jl[nsp * ld + lane] = (MT)colT;
  saved[nsp * kNP + lane] = (MT)colT;
  return aux2.inv_rho;
}

// ---------------------------------------------------------------------------
// The same Jacobian for a team of several wavefronts (nsp < 64W): thread i
// owns row i; J and saved are column-major with column stride js; t2l and hl
// are kState and nsp doubles of LDS scratch (hl may be s.C).  js >= nsp + 1.  The temperature row is a
// matrix-vector product read from LDS (column c by thread c) instead of one reduction per column.
// ---------------------------------------------------------------------------
template <typename MT, class Team>
__device__ __forceinline__ double jacobian_team(const Team& team, const DevMech& m,
                                                const RhsLds& s, double P, double v0,
                                                const BdfOpts& o, double y, double fy,
                                                double inv_rho_prev, MT* __restrict__ J,
                                                MT* __restrict__ saved, int js,
                                                double* __restrict__ t2l,
                                                double* __restrict__ hl, RhsSrc src = {},
                                                bool solveT = true) {
  const int tid = team.tid();
  const int nsp = m.nsp;
  const bool sp = tid < nsp;
  const bool act = tid <= nsp;
  const double mmf = o.min_mass_fraction;
  double t1 = y;
  if (sp && fabs(t1) < mmf) t1 = (t1 < 0.0) ? -mmf : mmf;
  if (tid < Team::kState) t2l[tid] = sp ? m.mw[tid] / t1 * inv_rho_prev : 0.0;
  const double yT = team.from(y, nsp);
  double dT = yT * sqrt(DBL_EPSILON);
  const double Tp = yT + dT;
  dT = Tp - yT;
  double colT = 0.0;
  RhsAux aux2;
  if (solveT) {
    double t4;
    rhs_team(team, m, s, P, v0, o.Tref, o.step_limiter, (tid == nsp) ? Tp : (sp ? y : 0.0), t4,
             aux2, src);
    colT = act ? (t4 - fy) * (1.0 / dT) : 0.0;
  }
  double t3;
  RhsAux aux;
  rhs_team(team, m, s, P, v0, o.Tref, o.step_limiter, t1, t3, aux, src);
  if (!solveT) aux2.inv_rho = aux.inv_rho;  // the last evaluation's
  const double Tdot = team.from(t3, nsp);
  if (sp) hl[tid] = aux.h;
  for (int k = tid; k < nsp * js; k += Team::kThreads) J[k] = MT(0);
  team.sync();
  if (tid < m.jr_stride) {
    // rows beyond the table's stride have no terms (team larger than needed)
    const uint4* __restrict__ jr = m.jr + tid;
    const int nb = m.jr_blocks;
    const int js_tab = m.jr_stride;
    int cur = -1;
    double v = 0.0;
    auto term = [&](unsigned t) {
      const int col = (int)((t >> 16) & 0xFFu);
      if (col != 0xFF) {
        if (col != cur) {
          cur = col;
          v = 0.0;
        }
        if (Team::kExt && (t & kJtNonInt)) {
          const double2 e = m.ni_jt[t & 0xFFFFu];
          v = __dadd_rn(v, __dmul_rn(__dmul_rn(e.x, s.rop[(int)e.y]), t2l[col]));
        } else {
          const double p = __dmul_rn(s.rop[t & 0xFFFFu], t2l[col]);
          v = (t & 0x80000000u) ? __dsub_rn(v, p) : __dadd_rn(v, p);
        }
        J[col * js + tid] = (MT)v;
      }
    };
    uint4 w = nb > 0 ? jr[0] : make_uint4(0, 0, 0, 0);
    for (int b = 0; b < nb; ++b) {
      const uint4 x = w;
      if (b + 1 < nb) w = jr[(b + 1) * js_tab];
      term(x.x);
      term(x.y);
      term(x.z);
      term(x.w);
    }
  }
  team.sync();
  // temperature row: thread c forms d(Tdot)/dy_c from column c
  double trow = 0.0;
  if (sp && solveT) {
    double acc = 0.0;
    for (int i = 0; i < nsp; ++i) acc += (double)J[tid * js + i] * hl[i];
    trow = acc * (kRu * yT);
    trow += Tdot * aux.cpm * m.mw[tid];
    trow *= m.inv_mw[tid] * (-1.0 / aux.cp_mix);
  }
  team.sync();
  // row i of the species block: J_ic *= MW_i / MW_c; then the temperature row
  // (column c's entry at row nsp) and the finite-difference column
  if (sp) {
    const double mwi = m.mw[tid];
    for (int c = 0; c < nsp; ++c) {
      const MT out = (MT)((double)J[c * js + tid] * (mwi * m.inv_mw[c]));
      J[c * js + tid] = out;
      saved[c * js + tid] = out;
    }
    J[tid * js + nsp] = (MT)trow;
    saved[tid * js + nsp] = (MT)trow;
  }
  if (act) {
    J[nsp * js + tid] = (MT)colT;
    saved[nsp * js + tid] = (MT)colT;
  }
  team.sync();
  return aux2.inv_rho;
}

// Gauss-Jordan inverse (no pivoting) of the N x N leading block of a matrix
// held one row per lane in R[0..kC-1]; padding rows/columns must be identity.
// MT is the working precision (double, or float for the FP32 preconditioner).
// Returns false on a zero pivot.
//
// The pivot row is broadcast from its lane with readlane (no LDS round trip)
// and is not normalised when it is used: row k is kept unscaled with a
// per-row factor s_k = 1/a_kk set at its pivot step, and every other row i
// subtracts g_i * (row k) with g_i = a_ik / a_kk, which does not depend on
// how row k is scaled.  The pivot column becomes -g_i (1 on the pivot row,
// whose factor carries 1/a_kk), and every row is multiplied by its factor at
// the end.  Per column and pivot that is one broadcast and one fma.
// Register indices must be compile-time constants, so pivots are taken in
// blocks of kGjBlock whose pivot columns sit in registers 0..kGjBlock-1, and
// the registers are rotated by kGjBlock after each block: on return register
// c holds logical column (c + gj_rotation<kC>(N)) mod kC of the inverse.
constexpr int kGjBlock = 8;
template <int kC = kNP>
__host__ __device__ constexpr int gj_rotation(int N) {
  return (((N + kGjBlock - 1) / kGjBlock) * kGjBlock) % kC;
}

// kC >= N: the columns held (a multiple of kGjBlock).
template <typename MT, int kC>
__device__ __forceinline__ bool gj_invert(MT (&R)[kC], int N) {
  const int lane = lane_id();
  bool ok = true;
  MT s = MT(1);
  for (int k0 = 0; k0 < N; k0 += kGjBlock) {
#pragma unroll
    for (int kk = 0; kk < kGjBlock; ++kk) {
      const int k = k0 + kk;
      if (k < N) {
        const MT f = R[kk];
        const MT piv = bcast(f, k);
        if (piv == MT(0)) ok = false;
        const MT rp = MT(1) / piv;
        const bool me = (lane == k);
        const MT g = me ? MT(0) : f * rp;
        if (me) s = rp;
#pragma unroll
        for (int c = 0; c < kC; ++c)
          if (c != kk) R[c] = fma(-g, bcast(R[c], k), R[c]);
        R[kk] = me ? MT(1) : -g;
      }
    }
    MT t[kGjBlock];
#pragma unroll
    for (int c = 0; c < kGjBlock; ++c) t[c] = R[c];
#pragma unroll
    for (int c = 0; c < kC - kGjBlock; ++c) R[c] = R[c + kGjBlock];
#pragma unroll
    for (int c = 0; c < kGjBlock; ++c) R[kC - kGjBlock + c] = t[c];
  }
#pragma unroll
  for (int c = 0; c < kC; ++c) R[c] *= s;
  return ok;
}

// ---------------------------------------------------------------------------
// Blocked Gauss-Jordan inverse (no pivoting) on MFMA by a team of wavefronts
// (FP32 tiles for the FP32 Newton matrix, FP64 tiles for the FP64 one).  The
// N x N matrix is padded with the identity to 16 x 16 tiles that stay in the
// wavefronts' registers from the first load to the last store (GjGrid: tile
// (ib, jb) on wavefront (ib mod GR, jb mod GC)); only the row and the column of
// the current block step pass through LDS, laid out as MFMA operands.  Block
// step K with the diagonal tile D = A[K,K]:
//   row tiles      A[K,J] <- D^-1 A[K,J]                 (J != K)
//   column tiles   A[I,K] <- -A[I,K] D^-1                (I != K)
//   -- barrier --
//   other tiles    A[I,J] <- A[I,J] - A[I,K] A[K,J]      (I != K, J != K; old A[I,K])
//   the wavefront with tile (K+1, K+1) forms it first and inverts it
//   the tiles of row and column K+1 are published
//   -- barrier --
// What bounds it: with the tiles in LDS (each read and written once a block
// step) the LDS pipe and the wait for it took 224,000 cycles at 161 rows and
// 8 wavefronts, against 42,000 for its MFMAs; from registers the operands are
// one 16-byte read a tile row and a tile column.
// v_mfma_f32_16x16x4f32 / v_mfma_f64_16x16x4f64 operand layouts (one 16 x 16
// block):
//   A[i][k] (16 x 4): lane l holds i = l % 16, k = l / 16
//   B[k][j] (4 x 16): lane l holds k = l / 16, j = l % 16
//   C[i][j] (16 x 16): register v of lane l holds j = l % 16 and i = 4 (l / 16) + v
//                      (FP32) or i = l / 16 + 4 v (FP64)
// ---------------------------------------------------------------------------
// 16 x 16 x 4 MFMA by element type: v_mfma_f32_16x16x4f32 for the FP32
// Newton matrices, v_mfma_f64_16x16x4f64 for the FP64 ones.  Both take one A
// element (row lane % 16, k lane / 16) and one B element (k lane / 16, column
// lane % 16) per lane and accumulate the 16 x 16 tile as 4 elements per lane
// in column lane % 16, but in different rows (row(lk, v), lk = lane / 16):
// the FP32 instruction holds rows 4 lk + v, the FP64 one rows lk + 4 v
// (checked on gfx950 against a host product).
template <typename T>
struct Mfma16;
template <>
struct Mfma16<float> {
  typedef float v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 mac(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lk, int v) { return 4 * lk + v; }
};
template <>
struct Mfma16<double> {
  typedef double v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 mac(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lk, int v) { return lk + 4 * v; }
};

// reciprocal of a pivot: the FP32 inverse only preconditions the Newton
// iteration (its residual and convergence test stay in FP64), so the
// hardware reciprocal (1 ulp) serves; the FP64 inverse divides exactly
__device__ __forceinline__ float pivot_recip(float p) { return __builtin_amdgcn_rcpf(p); }
__device__ __forceinline__ double pivot_recip(double p) { return 1.0 / p; }

// x of lane K of this lane's row of 16 lanes (DPP row_newbcast).
template <int K>
__device__ __forceinline__ float row16_bcast(float x) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x150 + K, 0xF, 0xF, true));
}
template <int K>
__device__ __forceinline__ double row16_bcast(double x) {
  return dpp_move<0x150 + K>(x);
}
// x of the lane at the same place in row G of 16 lanes.
template <int G>
__device__ __forceinline__ unsigned group16_bcast(unsigned u) {
  const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const unsigned v = (G & 1) ? r[1] : r[0];
  const auto q = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return (G & 2) ? q[1] : q[0];
}
template <int G>
__device__ __forceinline__ float group16_bcast(float x) {
  return __uint_as_float(group16_bcast<G>(__float_as_uint(x)));
}
template <int G>
__device__ __forceinline__ double group16_bcast(double x) {
  return __hiloint2double((int)group16_bcast<G>((unsigned)__double2hiint(x)),
                          (int)group16_bcast<G>((unsigned)__double2loint(x)));
}

// Gauss-Jordan inverse of a 16 x 16 matrix by one wavefront, with the deferred
// row scaling of gj_invert: lane 16 g + i holds row i's columns 4 g .. 4 g + 3.
// A pivot step is one cross-row broadcast of the pivot column's entries and one
// DPP broadcast and one fma per column held (4), where a whole row per lane
// would take 15 readlanes and 15 fmas on a quarter of the lanes.
template <int K, typename T>
__device__ __forceinline__ void gj_pivot16(T (&d)[4], T& s, bool& ok, int i, int g) {
  constexpr int G = K >> 2, CK = K & 3;
  const T f = group16_bcast<G>(d[CK]);  // this row's entry of column K
  const T piv = bcast(d[CK], 16 * G + K);
  if (piv == T(0)) ok = false;
  const T rp = pivot_recip(piv);
  const bool me = (i == K);
  const T gi = me ? T(0) : f * rp;
  if (me) s = rp;
  const bool own = (g == G);
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const T u = fma(-gi, row16_bcast<K>(d[c]), d[c]);
    d[c] = (c == CK && own) ? (me ? T(1) : -gi) : u;
  }
}

template <typename T, int... K>
__device__ __forceinline__ bool gj_invert16(T (&d)[4], std::integer_sequence<int, K...>) {
  const int lane = lane_id();
  bool ok = true;
  T s = T(1);
  (gj_pivot16<K>(d, s, ok, lane & 15, lane >> 4), ...);
#pragma unroll
  for (int c = 0; c < 4; ++c) d[c] *= s;
  return ok;
}

// One operand tile in LDS (kGjTile elements): lane l's four elements (k = l / 16 + 4 s, s = 0..3, of row
// or column l % 16) in 16 (FP32) or 32 bytes, the four groups of 16 lanes 68
// elements apart so that the scattered writes below are free of bank conflicts.
__device__ __forceinline__ constexpr int gj_place(int rc, int k) {
  return (k & 3) * 68 + rc * 4 + (k >> 2);
}


// Wavefront grid and tiles per wavefront of a team whose state takes W wavefronts,
// with gj_buffers(W) buffers of the published row and column (two save the 8
// wavefronts a barrier a block step, 10 % of the inverse at 161 rows).
template <int W>
struct GjGrid;
template <>
struct GjGrid<1> {  // one wavefront: up to 64 rows
  static constexpr int GR = 1, GC = 1, TR = 4, TC = 4, kBuf = gj_buffers(1);
};
// One wavefront, up to 32 rows: the larger grid's updates of absent tile rows are left out
// (24 species, 4,096 reactors: 18.5 to 18.0 ms).
struct GjGridSmall {
  static constexpr int GR = 1, GC = 1, TR = 2, TC = 2, kBuf = gj_buffers(1);
};
template <>
struct GjGrid<2> {  // 4 wavefronts: up to 128 rows
  static constexpr int GR = 2, GC = 2, TR = 4, TC = 4, kBuf = gj_buffers(2);
};
template <>
struct GjGrid<3> {  // 8 wavefronts: up to 192 rows
  static constexpr int GR = 4, GC = 2, TR = 3, TC = 6, kBuf = gj_buffers(3);
};

// The tiles: lane's elements of tile (a, b) of this wavefront are in rows
// 16 (wr + GR a) + Mfma16<T>::row(lk, v) of column 16 (wc + GC b) + li.
template <class G, typename T>
struct GjTiles {
  using v4 = typename Mfma16<T>::v4;
  v4 x[G::TR][G::TC];
  int wr, wc, li, lk;
  __device__ __forceinline__ explicit GjTiles(int wave)
      : wr(wave / G::GC), wc(wave % G::GC), li(lane_id() & 15), lk(lane_id() >> 4) {}
  __device__ __forceinline__ int row(int a, int v) const {
    return 16 * (wr + G::GR * a) + Mfma16<T>::row(lk, v);
  }
  __device__ __forceinline__ int col(int b) const { return 16 * (wc + G::GC * b) + li; }
};

// Four elements of a lane's operand.
template <typename T>
__device__ __forceinline__ typename Mfma16<T>::v4 gj_operand(const T* __restrict__ tile, int li,
                                                             int lk) {
  return *reinterpret_cast<const typename Mfma16<T>::v4*>(tile + lk * 68 + li * 4);
}

// Inverts the padded matrix in t; L: gj_lds_elems(nb, W) elements of LDS (16-byte
// aligned), free on entry.  Returns false on a zero pivot of a diagonal tile
// (every thread gets the same answer through *flag, one element of LDS).
template <class G, class Team, typename T>
__device__ __forceinline__ bool gj_invert_tiles(const Team& team, GjTiles<G, T>& t, int nb,
                                                T* __restrict__ L, T* __restrict__ flag) {
  using M = Mfma16<T>;
  using v4 = typename M::v4;
  const int li = t.li, lk = t.lk;
  const int panel = nb * kGjTile;
  T* const dA = L + 2 * G::kBuf * panel;  // D^-1 as left operand
  T* const dB = dA + kGjTile;             // and as right operand
  T* const dt = dB + kGjTile;             // the tile to invert
  const auto wave_fence = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  // the diagonal tile's inverse by the wavefront that holds it (tile d)
  const auto invert = [&](const v4& d) {
#pragma unroll
    for (int v = 0; v < 4; ++v) dt[li * 20 + M::row(lk, v)] = d[v];
    wave_fence();
    T r[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) r[c] = dt[(4 * lk + c) * 20 + li];
    const bool ok = gj_invert16(r, std::make_integer_sequence<int, 16>{});
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      dA[gj_place(li, 4 * lk + c)] = r[c];
      dB[gj_place(4 * lk + c, li)] = r[c];
    }
    if (!ok && lane_id() == 0) *flag = T(0);
  };
  // this wavefront's tile row of block row K, and its tile column of block
  // column K (-1: none); register arrays are indexed at compile time only
  const auto row_of = [&](int K) { return K % G::GR == t.wr ? K / G::GR : -1; };
  const auto col_of = [&](int K) { return K % G::GC == t.wc ? K / G::GC : -1; };
  // the old column and the row of step K
  const auto col_panel = [&](int K) { return L + 2 * (K % G::kBuf) * panel; };
  // publish the tiles of row and column K
  const auto publish = [&](int K) {
    T* const cp = col_panel(K);
    T* const rowp = cp + panel;
    const int aK = row_of(K), bK = col_of(K);
#pragma unroll
    for (int b = 0; b < G::TC; ++b)
      if (b == bK) {
#pragma unroll
        for (int a = 0; a < G::TR; ++a) {
          const int ib = t.wr + G::GR * a;
          if (ib >= nb) continue;
#pragma unroll
          for (int v = 0; v < 4; ++v)
            cp[ib * kGjTile + gj_place(M::row(lk, v), li)] = t.x[a][b][v];
        }
      }
#pragma unroll
    for (int a = 0; a < G::TR; ++a)
      if (a == aK) {
#pragma unroll
        for (int b = 0; b < G::TC; ++b) {
          const int jb = t.wc + G::GC * b;
          if (jb >= nb) continue;
#pragma unroll
          for (int v = 0; v < 4; ++v)
            rowp[jb * kGjTile + gj_place(li, M::row(lk, v))] = t.x[a][b][v];
        }
      }
  };
  if (team.tid() == 0) *flag = T(1);
  team.sync();
  if (t.wr == 0 && t.wc == 0) invert(t.x[0][0]);
  if (nb == 1) {  // the diagonal tile is all of it
    team.sync();
#pragma unroll
    for (int v = 0; v < 4; ++v)
      if (t.wr == 0 && t.wc == 0) t.x[0][0][v] = dB[gj_place(li, M::row(lk, v))];
    team.sync();
    return *flag != T(0);
  }
  publish(0);
  team.sync();
  for (int K = 0; K < nb; ++K) {
    const int next = K + 1;
    const int aK = row_of(K), bK = col_of(K);
    T* const cp = col_panel(K);
    T* const rowp = cp + panel;
    // row tiles D^-1 A[K,J], column tiles -A[I,K] D^-1 and the diagonal tile; a
    // wavefront's tiles of either kind are independent chains
    if (aK >= 0) {
      v4 r[G::TC], acc[G::TC];
      const v4 l = gj_operand(dA, li, lk);
#pragma unroll
      for (int b = 0; b < G::TC; ++b) {
        r[b] = gj_operand(rowp + min(t.wc + G::GC * b, nb - 1) * kGjTile, li, lk);
        acc[b] = v4{T(0), T(0), T(0), T(0)};
      }
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int b = 0; b < G::TC; ++b) acc[b] = M::mac(l[s], r[b][s], acc[b]);
      wave_fence();
#pragma unroll
      for (int b = 0; b < G::TC; ++b) {
        const int jb = t.wc + G::GC * b;
        if (jb >= nb || jb == K) continue;
#pragma unroll
        for (int v = 0; v < 4; ++v)
          rowp[jb * kGjTile + gj_place(li, M::row(lk, v))] = acc[b][v];
      }
#pragma unroll
      for (int a = 0; a < G::TR; ++a)
        if (a == aK)
#pragma unroll
          for (int b = 0; b < G::TC; ++b) t.x[a][b] = acc[b];
    }
    if (bK >= 0) {
      v4 l[G::TR], acc[G::TR];
      const v4 r = gj_operand(dB, li, lk);
#pragma unroll
      for (int a = 0; a < G::TR; ++a) {
        l[a] = gj_operand(cp + min(t.wr + G::GR * a, nb - 1) * kGjTile, li, lk);
        acc[a] = v4{T(0), T(0), T(0), T(0)};
      }
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int a = 0; a < G::TR; ++a) acc[a] = M::mac(-l[a][s], r[s], acc[a]);
      if (aK >= 0) {  // the diagonal tile
        v4 d;
#pragma unroll
        for (int v = 0; v < 4; ++v) d[v] = dB[gj_place(li, M::row(lk, v))];
#pragma unroll
        for (int a = 0; a < G::TR; ++a)
          if (a == aK) acc[a] = d;
      }
#pragma unroll
      for (int b = 0; b < G::TC; ++b)
        if (b == bK)
#pragma unroll
          for (int a = 0; a < G::TR; ++a) t.x[a][b] = acc[a];
    }
    team.sync();
    // the operands of the step's updates (with one buffer, before anyone publishes
    // the next step's)
    const int aN = row_of(next), bN = col_of(next);
    v4 l[G::TR], r[G::TC], d = t.x[0][0];
#pragma unroll
    for (int a = 0; a < G::TR; ++a) {
      l[a] = gj_operand(cp + min(t.wr + G::GR * a, nb - 1) * kGjTile, li, lk);
#pragma unroll
      for (int s = 0; s < 4; ++s) l[a][s] = -l[a][s];
    }
#pragma unroll
    for (int b = 0; b < G::TC; ++b)
      r[b] = gj_operand(rowp + min(t.wc + G::GC * b, nb - 1) * kGjTile, li, lk);
    if (G::kBuf == 1) team.sync();
    // tile (next, next) and its inverse first (the update below forms it again)
    if (next < nb && aN >= 0 && bN >= 0) {
      v4 dl = l[0], dr = r[0];
#pragma unroll
      for (int a = 0; a < G::TR; ++a)
        if (a == aN) dl = l[a];
#pragma unroll
      for (int b = 0; b < G::TC; ++b)
        if (b == bN) dr = r[b];
#pragma unroll
      for (int a = 0; a < G::TR; ++a)
#pragma unroll
        for (int b = 0; b < G::TC; ++b)
          if (a == aN && b == bN) d = t.x[a][b];
#pragma unroll
      for (int s = 0; s < 4; ++s) d = M::mac(dl[s], dr[s], d);
      invert(d);
    }
    // the other tiles, a tile column at a time (a zero left operand leaves the
    // tiles of row K as they are)
#pragma unroll
    for (int a = 0; a < G::TR; ++a)
#pragma unroll
      for (int s = 0; s < 4; ++s) l[a][s] = a == aK ? T(0) : l[a][s];
#pragma unroll
    for (int b = 0; b < G::TC; ++b) {
      if (b == bK || t.wc + G::GC * b >= nb) continue;
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int a = 0; a < G::TR; ++a) t.x[a][b] = M::mac(l[a][s], r[b][s], t.x[a][b]);
    }
    if (next < nb) publish(next);
    team.sync();
  }
  return *flag != T(0);
}

// Loads the padded matrix: entry(v, r, c) is its element for r, c < N from the
// element v of J (column-major, column stride js).  Tiles beyond the matrix are
// skipped (nothing reads them); a partial tile loads clamped places and selects,
// so no load waits behind a branch of its own.  All loads first, then the
// entries a tile at a time: formed all at once they take 250 registers, which
// the caller then has to save.
template <class G, typename T, class F>
__device__ __forceinline__ void gj_load_tiles(GjTiles<G, T>& t, const T* __restrict__ J, int js,
                                              int N, F&& entry) {
#pragma unroll
  for (int a = 0; a < G::TR; ++a)
#pragma unroll
    for (int b = 0; b < G::TC; ++b) {
      t.x[a][b] = typename Mfma16<T>::v4{T(0), T(0), T(0), T(0)};
      if (16 * (t.wr + G::GR * a) < N && 16 * (t.wc + G::GC * b) < N) {
        const T* __restrict__ col = J + min(t.col(b), N - 1) * js;
#pragma unroll
        for (int v = 0; v < 4; ++v) t.x[a][b][v] = col[min(t.row(a, v), N - 1)];
      }
    }
#pragma unroll
  for (int a = 0; a < G::TR; ++a)
#pragma unroll
    for (int b = 0; b < G::TC; ++b) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int r = t.row(a, v), c = t.col(b);
        const T e = entry(t.x[a][b][v], min(r, N - 1), min(c, N - 1));
        t.x[a][b][v] = (r < N && c < N) ? e : (r == c ? T(1) : T(0));
      }
    }
}

// Stores the tiles into the N x N matrix A, column-major with column stride js.
template <class G, typename T>
__device__ __forceinline__ void gj_store_tiles(const GjTiles<G, T>& t, int N, int js,
                                               T* __restrict__ A) {
#pragma unroll
  for (int a = 0; a < G::TR; ++a)
#pragma unroll
    for (int b = 0; b < G::TC; ++b) {
      const int r0 = 16 * (t.wr + G::GR * a), c0 = 16 * (t.wc + G::GC * b), c = t.col(b);
      if (r0 + 16 <= N && c0 + 16 <= N) {
#pragma unroll
        for (int v = 0; v < 4; ++v) A[c * js + t.row(a, v)] = t.x[a][b][v];
      } else if (r0 < N && c0 < N && c < N) {
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (t.row(a, v) < N) A[c * js + t.row(a, v)] = t.x[a][b][v];
      }
    }
}

// Entry (row, col) of the Newton matrix from v = -gamma J_row,col: the direct
// solver's I - gamma J, or the Krylov solver's preconditioner (kIter;
// FormPreconditioner, reactor_nvector_serial.cpp:414-493): the diagonal and,
// unless every entry is kept (pfull), only entries of the Jacobian's pattern
// with |v| > threshold.  Rows and columns < nsp + 1.
template <bool kIter>
__device__ __forceinline__ double newton_entry(double v, int row, int col, bool pfull,
                                               const unsigned long long* __restrict__ jpat,
                                               double threshold) {
  if (row == col) return v + 1.0;
  if (!kIter || pfull) return v;
  const bool in = (jpat[row * 3 + (col >> 6)] >> (col & 63)) & 1ull;
  return (in && fabs(v) > threshold) ? v : 0.0;
}

// The inverse of M = I - gamma J (ng = -gamma; J column-major with column
// stride js) into M (column stride ms), by every thread of the team: J goes
// straight into the register tiles, all of a lane's loads in flight together.
// A function of its own, called and not inlined: its loop runs with its tiles (64 to 144
// registers) alone, where inlined it spilled inside the loop (54 rows: 151,000 cycles
// inlined, 58,000 called).  The integrator's state is saved around the call instead: the
// compiler reports 412 bytes of scratch a lane, 64 registers of them spilled, for one
// wavefront's FP32 kernel (72 and 8 when the tiles stayed in LDS), 600 and 112 for the
// FP32 team of 3, 1,444 and 165 for the FP64 one (40 and 0).
template <class G, class Team, typename T, bool kIter, class MPtr>
__device__ __noinline__ bool newton_inverse(GlobalPtr<const T> J, int js, int N, double ng,
                                            MPtr M, int ms, LdsPtr<T> L, LdsPtr<T> flag,
                                            bool pfull, GlobalPtr<const unsigned long long> jpat,
                                            double threshold) {
  Team team;
  const T* const jg = (const T*)J;
  const unsigned long long* const pat = (const unsigned long long*)jpat;
  GjTiles<G, T> t(Team::kThreads == kWave ? 0 : uni((int)(team.tid() / kWave)));
  gj_load_tiles(t, jg, js, N, [&](T v, int r, int c) {
    return (T)newton_entry<kIter>(ng * (double)v, r, c, pfull, pat, threshold);
  });
  const bool ok = gj_invert_tiles<G>(team, t, (N + 15) >> 4, (T*)L, (T*)flag);
  gj_store_tiles(t, N, ms, (T*)M);
  return ok;
}

// The FP64 inverse of one wavefront: M = I - gamma J (J column-major with stride
// kNP) inverted row per lane in kC registers, stored to M column-major with
// stride N.  kC: the least multiple of 8 (at least 16) that holds the columns -- every
// pivot takes two readlanes and an fma per column held, used or not (N = 11: 29,700
// cycles with 64 columns; 34 species, 4,096 reactors: 36.0 ms with 56, 34.5 ms with 40).
// A call for the same reason as newton_inverse.
template <int kC, bool kIter>
__device__ __forceinline__ bool inverse_rows(const double* __restrict__ jg, int N, double ng,
                                             double* __restrict__ Ml, bool pfull,
                                             const unsigned long long* __restrict__ pat,
                                             double threshold) {
  const int lane = lane_id();
  double R[kC];
#pragma unroll
  for (int c = 0; c < kC; ++c) R[c] = jg[c * kNP + lane];
#pragma unroll
  for (int c = 0; c < kC; ++c) {
    double v = (c < N && lane < N) ? ng * R[c] : 0.0;
    if (c < N && lane < N) v = newton_entry<kIter>(v, lane, c, pfull, pat, threshold);
    else if (c == lane) v += 1.0;
    R[c] = v;
  }
  const bool ok = gj_invert(R, N);
  // register c holds logical column (c + rot) mod kC: keep logical columns < N
  const int rot = gj_rotation<kC>(N);
  if (lane < N) {
#pragma unroll
    for (int c = 0; c < kC; ++c) {
      const int j = c + rot < kC ? c + rot : c + rot - kC;
      if (j < N) Ml[j * N + lane] = R[c];
    }
  }
  return ok;
}

template <int kC, bool kIter>
__device__ __noinline__ bool newton_inverse_rows(GlobalPtr<const double> J, int N, double ng,
                                                 LdsPtr<double> M, bool pfull,
                                                 GlobalPtr<const unsigned long long> jpat,
                                                 double threshold) {
  return inverse_rows<kC, kIter>((const double*)J, N, ng, (double*)M, pfull,
                                 (const unsigned long long*)jpat, threshold);
}

// newton_inverse of at most 16 rows by one wavefront (inlined: one tile).
template <bool kIter>
__device__ __forceinline__ bool inverse_one_tile(const float* __restrict__ J, int N, double ng,
                                                 float* __restrict__ M, int ms, bool pfull,
                                                 const unsigned long long* __restrict__ pat,
                                                 double threshold) {
  const int r = lane_id() & 15, c0 = 4 * (lane_id() >> 4);
  float d[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) d[c] = J[min(c0 + c, N - 1) * kNP + min(r, N - 1)];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const float e = (float)newton_entry<kIter>(ng * (double)d[c], r, c0 + c, pfull, pat, threshold);
    d[c] = (r < N && c0 + c < N) ? e : (r == c0 + c ? 1.0f : 0.0f);
  }
  const bool ok = gj_invert16(d, std::make_integer_sequence<int, 16>{});
#pragma unroll
  for (int c = 0; c < 4; ++c)
    if (r < N && c0 + c < N) M[(c0 + c) * ms + r] = d[c];
  return ok;
}

// The same, called (the variants that do not inline it).
template <bool kIter>
__device__ __noinline__ bool newton_inverse_tile(GlobalPtr<const float> J, int N, double ng,
                                                 LdsPtr<float> M, int ms, bool pfull,
                                                 GlobalPtr<const unsigned long long> jpat,
                                                 double threshold) {
  return inverse_one_tile<kIter>((const float*)J, N, ng, (float*)M, ms, pfull,
                                 (const unsigned long long*)jpat, threshold);
}

}  // namespace zrk
