// HIP kernels for gfx950 (MI355X): matrix-free trilinear-hex operators of
// HPCrack's degraded elasticity and AT2 phase field, the fused Jacobi-PCG
// passes, multigrid transfers, coarse coefficients and Gauss-point updates.
//
// Operator formulation.  On a uniform voxel grid the gradient of a trilinear
// field at the 2x2x2 Gauss points is sum-factorised: d/dx at Gauss point
// (gx,gy,gz) does not depend on gx and equals the x-edge differences of the
// element interpolated bilinearly in y and z.  The transposed contraction
// B^T sigma is factorised the same way.  This needs ~1.2 kflop per element
// instead of ~8 kflop for the reference's per-Gauss-point loops
// (mechanical_pcg.cpp:114-172), and gives the same operator up to rounding.
//
// Tiling.  A block of 256 threads owns a 32x8 column of elements (one per
// thread) and marches up a chunk of z-layers.  Each step evaluates one
// element layer from two node planes held in LDS (u and, on the finest level,
// K, G, d) while the global loads of the plane after next are in flight.  The
// 8 corner contributions of every element are exchanged so that each node
// sums its 4 in-plane neighbours in a fixed order: the x-neighbour is the
// adjacent lane (DPP row shift), the y-neighbour goes through LDS.  The node
// plane below the layer is then complete and handed to the fused epilogue
// (residual, PCG update, diagonal ...); the plane above is carried in
// registers.  No atomics: results are deterministic.  Tiles overlap by one
// element so that the 31x7 interior node columns are owned by one block.
//
// Small levels.  A level of at most SMALL_NODES nodes and SMALL_ELEMS
// elements runs a whole Jacobi-PCG smoother call in one workgroup
// (small_pcg_kernel): vectors in registers, p and the element contributions
// in LDS, block-wide reductions, no launches between iterations.
//
// Reductions.  Every block reduces its partial sums with wavefront shuffles
// in a fixed tree, writes them to a partials array, and the last block to
// finish (ticket counter) reduces the partials in fixed order and updates the
// device scalars (alpha, beta, r.z ...).  Deterministic, one launch per pass.
// The smoother passes of small levels leave the partials to the next pass
// instead (OpenRed).
#include <hip/hip_runtime.h>
#include <cfloat>
#include <cmath>
#include <type_traits>

#include "hpcr_internal.h"
#include "hpcr_tile.h"
#include "hpcr_multi.h"

namespace hpcr {

thread_local Recorder* t_recorder = nullptr;

// ---- mechanical tile ops --------------------------------------------------
enum MechMode { M_APPLY = 0, M_RESID = 1, M_PCGA = 2, M_DIAG = 3 };

// FOLD: the grid is cubic (hx = hy = hz = h), so the gradient's 1/h and the
// transposed contraction's w_g/h fold into the moduli (times w_g/h^2, once
// per node plane on the finest level, once per element on coarse levels);
// with a power-of-two h this gives the same bits as the scaled form.
// GAUSS: a coarse level's element by the Gauss-point sums instead of the mode
// form, for the residual and pass A of the mixed solve's coarsest level
// (MIX_SMALL_NODES).  A template parameter and not a run-time flag: a kernel
// with both forms holds the registers of both (pass A 241, with one of them
// 170 or 142).
template <int MODE, bool FINE, bool FOLD = false, bool GAUSS = false>
struct MechOp {
  using T = double;
  using TR = double;
  static constexpr int NC = 3;
  static constexpr int NU = (MODE == M_DIAG) ? 0 : 3;  // vector values per node in LDS
  static constexpr int NK = FINE ? 3 : 0;              // K, G, d
  static constexpr int NV = (NU + NK) > 0 ? NU + NK : 1;
  static constexpr int NR = (MODE == M_PCGA) ? 6 + NK : NV;  // PCGA fetches z and p_old
  using Raw = double[NR];
  static constexpr int NSL = NSLOT, MIN_WAVES = HPCR_MECH_WAVES;  // LDS plane slots, occupancy target
  struct Acc {
    double a[3];
    __device__ Acc() { a[0] = a[1] = a[2] = 0.0; }
  };
  struct State {
    double beta;
  };
  // per-element data, staged through LDS with the node planes: the split
  // flag on the finest level, K_e and G_e on coarse levels
  using TE = std::conditional_t<FINE, int, double>;
  static constexpr int NE = FINE ? 1 : 2;
  MechCoef C;
  const double* x;      // APPLY/RESID: input vector; PCGA: z
  const double* invD;   // RESID
  const double* p_old;  // PCGA
  double* out;          // APPLY: y; RESID: r; PCGA: w; DIAG: invD
  double* out2;         // RESID: f; PCGA: p_new (null: the first direction is x itself, in place); DIAG: diag (or null)
  double* out3;         // RESID: z
  int flag;             // RESID: t0fine; PCGA: first
  double sx, sy, sz, tx_, ty_, tz_, wg, ihx2, ihy2, ihz2;
  double fs;            // FOLD: w_g / h^2
  HexScale<double> hs;  // not FOLD: scales of the constant-moduli element
  Reduce R;
  size_t N;
  static constexpr bool OPEN = MODE == M_PCGA;
  OpenRed O;  // PCGA: open reductions of a small level's call
  static_assert(!(FOLD && MODE == M_DIAG), "the diagonal keeps its own scaling");
  static_assert(!GAUSS || (!FINE && (MODE == M_RESID || MODE == M_PCGA)), "a coarse smoother call's passes");

  __device__ __forceinline__ State state() const {
    State s;
    s.beta = (MODE == M_PCGA && !flag && !O.out) ? R.scal[S_BETA] : 0.0;
    return s;
  }

  // node values through buffer resources: a node outside the grid (or past
  // the chunk) reads zeros without a branch
  __device__ __forceinline__ void fetch(const LevelGeom& L, int gx, int gy, int gz, bool ok, const State& st,
                                        double (&r)[NR]) const {
#pragma unroll
    for (int k = 0; k < NR; k++) r[k] = 0.0;
    const unsigned ob = ok ? nid32(L, gx, gy, gz) * 8u : BOFF_NONE;
    const size_t nb = N * 8;
    if constexpr (MODE == M_APPLY || MODE == M_RESID || MODE == M_PCGA) {
#pragma unroll
      for (int c = 0; c < 3; c++) r[c] = bld(brsrc(x + c * N, nb), ob);
    }
    if constexpr (MODE == M_PCGA) {
      if (!flag) {
#pragma unroll
        for (int c = 0; c < 3; c++) r[3 + c] = bld(brsrc(p_old + c * N, nb), ob);
      }
    }
    if constexpr (FINE) {
      constexpr int o = NR - 3;
      r[o + 0] = bld(brsrc(C.K, nb), ob);
      r[o + 1] = bld(brsrc(C.G, nb), ob);
      r[o + 2] = bld(brsrc(C.d, nb), ob);
    }
  }

  __device__ __forceinline__ void efetch(const LevelGeom& L, int ex, int ey, int ez, bool ok, TE (&e)[NE]) const {
    const unsigned q = nid32(L, ex, ey, ez);
    if constexpr (FINE) {
      e[0] = bld_i8(brsrc(C.flag, N), ok ? q : BOFF_NONE);
    } else {
      const unsigned ob = ok ? 8u * q : BOFF_NONE;
      e[0] = bld(brsrc(C.Ke, N * 8), ob);
      e[1] = bld(brsrc(C.Ge, N * 8), ob);
    }
  }

  __device__ __forceinline__ void commit(const double (&r)[NR], const State& st, double (&v)[NV]) const {
    if constexpr (MODE == M_PCGA) {
#pragma unroll
      for (int c = 0; c < 3; c++) v[c] = r[c] + st.beta * r[3 + c];
#pragma unroll
      for (int k = 0; k < NK; k++) v[3 + k] = r[6 + k];
    } else {
#pragma unroll
      for (int k = 0; k < NV; k++) v[k] = r[k];
    }
    if constexpr (FINE && FOLD) {
      // K and G times w_g/h^2 (zero stays zero: the zero rule is unchanged)
      v[NU + 0] *= fs;
      v[NU + 1] *= fs;
    }
  }

  __device__ __forceinline__ void lame(const double (&sN)[NSL][NV][PLANE], int s0, int tx, int ty, const TE (&e)[NE],
                                       double (&lam)[2][2][2], double (&mu)[2][2][2], double& lam0,
                                       double& mu0) const {
    if constexpr (FINE) {
      double Kn[2][2][2], Gn[2][2][2], dn[2][2][2];
      gather8(sN, s0, tx, ty, NU + 0, Kn);
      gather8(sN, s0, tx, ty, NU + 1, Gn);
      gather8(sN, s0, tx, ty, NU + 2, dn);
      fine_lame(Kn, Gn, dn, e[0], C.small_k, lam, mu);
      lam0 = mu0 = 0.0;
    } else {
      lam0 = e[0] - (2.0 / 3.0) * e[1];
      mu0 = e[1];
      if constexpr (FOLD) {
        lam0 *= fs;
        mu0 *= fs;
      }
#pragma unroll
      for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
          for (int c = 0; c < 2; c++) {
            lam[a][b][c] = lam0;
            mu[a][b][c] = mu0;
          }
    }
  }

  __device__ __forceinline__ void element(const LevelGeom& L, const double (&sN)[NSL][NV][PLANE], int s0, int tx,
                                          int ty, int ex, int ey, int ez, const State& st, const TE (&e)[NE],
                                          double (&f)[3][2][2][2]) const {
    double lam[2][2][2], mu[2][2][2], lam0, mu0;
    lame(sN, s0, tx, ty, e, lam, mu, lam0, mu0);
    if constexpr (MODE == M_DIAG) {
      mech_element_diag(lam, mu, ihx2, ihy2, ihz2, wg, f);
    } else {
      double u[3][2][2][2];
#pragma unroll
      for (int c = 0; c < 3; c++) gather8(sN, s0, tx, ty, c, u[c]);
      if constexpr (FINE)
        mech_element<false, !FOLD>(u, lam, mu, 0.0, 0.0, sx, sy, sz, tx_, ty_, tz_, f);
      else if constexpr (GAUSS)
        mech_element<true, !FOLD>(u, lam, mu, lam0, mu0, sx, sy, sz, tx_, ty_, tz_, f);
      else
        hex_element(u, lam0, mu0, FOLD ? hex_unit<double>() : hs, f);
    }
  }

  // finest-level operator passes: each element takes its bottom node plane's
  // interpolated moduli and in-plane gradient parts from the element below
  using Carry = std::conditional_t<FINE && MODE != M_DIAG && kDelta<double>, FineCarry<double>, void>;
  template <class C_, int PL>
  __device__ __forceinline__ void element_planes(const LevelGeom& L, const double (&sN)[NSL][NV][PL], int s0,
                                                 int tx, int ty, int ex, int ey, int ez, const State& st,
                                                 const TE (&e)[NE], double (&f)[3][2][2][2], C_& cr,
                                                 bool first) const {
    double Kn[2][2][2], Gn[2][2][2], dn[2][2][2];
    gather8(sN, s0, tx, ty, NU + 0, Kn);
    gather8(sN, s0, tx, ty, NU + 1, Gn);
    gather8(sN, s0, tx, ty, NU + 2, dn);
    double lam[2][2][2], mu[2][2][2];
    fine_lame_planes(Kn, Gn, dn, e[0], C.small_k, cr, first, lam, mu);
    double u[3][2][2][2];
#pragma unroll
    for (int c = 0; c < 3; c++) gather8(sN, s0, tx, ty, c, u[c]);
    mech_element_planes<!FOLD>(u, lam, mu, cr, first, sx, sy, sz, tx_, ty_, tz_, f);
  }

  static constexpr bool NEEDS_OWN = (MODE == M_PCGA);
  // RESID: f and 1/D of the owner's node, read one plane ahead
  struct NData {
    double f[MODE == M_RESID ? 3 : 1], iD[MODE == M_RESID ? 3 : 1];
  };
  __device__ __forceinline__ void nfetch(const LevelGeom& L, int i, int j, int k, NData& n) const {
    if constexpr (MODE == M_RESID) {
      const unsigned ob = nid32(L, i, j, k) * 8u;
#pragma unroll
      for (int c = 0; c < 3; c++) {
        n.f[c] = ldo(out2 + c * N, ob);
        n.iD[c] = ldo(invD + c * N, ob);
      }
    }
  }
  // v: assembled values of node (i, j, k); own: the node's LDS values (p)
  __device__ __forceinline__ void epilogue(const LevelGeom& L, const double (&own)[3], int i, int j, int k, int dm,
                                           const double (&v)[3], const State& st, const NData& nd,
                                           Acc& acc) const {
    const unsigned ob = nid32(L, i, j, k) * 8u;
    if constexpr (MODE == M_APPLY) {
#pragma unroll
      for (int c = 0; c < 3; c++) sto(out + c * N, ob, v[c]);
    } else if constexpr (MODE == M_RESID) {
#pragma unroll
      for (int c = 0; c < 3; c++) {
        double fv = nd.f[c];
        const bool dir = (dm >> c) & 1;
        if (flag && dir) {
          fv = v[c];
          sto(out2 + c * N, ob, fv);
        }
        const double r = dir ? 0.0 : fv - v[c];
        const double z = r * nd.iD[c];
        sto(out + c * N, ob, r);
        sto(out3 + c * N, ob, z);
        acc.a[0] += r * z;
        acc.a[1] += r * r;
        acc.a[2] += fv * fv;
      }
    } else if constexpr (MODE == M_PCGA) {
#pragma unroll
      for (int c = 0; c < 3; c++) {
        const double p = own[c];
        if (out2) sto(out2 + c * N, ob, p);
        sto(out + c * N, ob, v[c]);
        acc.a[0] += p * v[c];
      }
    } else {  // M_DIAG
#pragma unroll
      for (int c = 0; c < 3; c++) {
        if (out2) sto(out2 + c * N, ob, v[c]);
        sto(out + c * N, ob, 1.0 / v[c]);
        acc.a[0] += (v[c] == 0.0) ? 1.0 : 0.0;
      }
    }
  }

  // split-output pass A (tile_body_split): node (i, j, k) of the tile's own
  // region, written to p_new and w as by epilogue()
  __device__ __forceinline__ void epilogue_split(const LevelGeom& L, const double (&p)[3], int i, int j, int k,
                                                 const double (&v)[3], Acc& acc) const {
    static_assert(MODE == M_PCGA, "split outputs are pass A's");
    const unsigned ob = nid32(L, i, j, k) * 8u;
#pragma unroll
    for (int c = 0; c < 3; c++) {
      if (out2) sto(out2 + c * N, ob, p[c]);
      sto(out + c * N, ob, v[c]);
      acc.a[0] += p[c] * v[c];
    }
  }
  // one component c of a side node's part, at byte offset so of the side
  // arrays; where no tile has the node in its own region (own_p: the last
  // node column or row of the grid) also p_new, and w = 0, at the node's byte
  // offset ob, so that pass B reads w at every node
  __device__ __forceinline__ void side1(const SplitW& S, unsigned so, double p, double v, bool own_p, unsigned ob,
                                        int c, Acc& acc) const {
    static_assert(MODE == M_PCGA, "split outputs are pass A's");
    sto(S.ws, so, v);
    acc.a[0] += p * v;
    if (own_p) {
      if (out2) sto(out2 + c * N, ob, p);
      sto(out + c * N, ob, 0.0);
    }
  }

  __device__ __forceinline__ void finish(Acc& acc, const Blk& bk) const {
    if constexpr (MODE == M_APPLY) return;
    double* scal = R.scal;
    if constexpr (MODE == M_RESID) {
      const int t0 = flag;
      reduce_finalize<RED_SUM, 3>(bk, acc.a, R, 0.0, [=](double (&s)[3]) {
        scal[S_RZ] = s[0];
        scal[S_RR] = s[1];
        if (t0) scal[S_FF] = s[2];
      });
    } else if constexpr (MODE == M_PCGA) {
      double v1[1] = {acc.a[0]};
      if (O.out) return open_store(bk, v1, O);
      reduce_finalize<RED_SUM, 1>(bk, v1, R, 0.0, [=](double (&s)[1]) {
        scal[S_PW] = s[0];
        scal[S_ALPHA] = scal[S_RZ] / s[0];
      });
    } else {
      double v1[1] = {acc.a[0]};
      reduce_finalize<RED_SUM, 1>(bk, v1, R, 0.0, [=](double (&s)[1]) { scal[S_ZERO] = s[0]; });
    }
  }
};

// ---- phase-field tile ops -------------------------------------------------
// OPENR: pass A of an open call (OpenRed).  A parameter, because four waves per
// SIMD leave 128 registers, which each of the two passes A fits and one kernel
// with both ends of the reduction does not: with 4 registers spilled in the
// march a smoother iteration took 258 us at 257x129x257 (now 231; spheres of a
// second phase), 81 at 129^3 (74) and 21.7 at 65^3 (20.9).  At three waves
// instead 65^3, 990 blocks, takes 22.3 and the others the same.
template <int MODE, bool OPENR = false>
struct PfOp {
  using T = double;
  using TR = double;
  static constexpr int NC = 1;
  static constexpr int NU = (MODE == M_DIAG) ? 0 : 1;
  static constexpr int NV = NU + 1;  // + gc
  static constexpr int NR = (MODE == M_PCGA) ? 3 : NV;
  using Raw = double[NR];
  static constexpr int NSL = NSLOT, MIN_WAVES = 4;
  struct Acc {
    double a[3];
    __device__ Acc() { a[0] = a[1] = a[2] = 0.0; }
  };
  struct State {
    double beta;
  };
  // the element's strain history H, staged through LDS with the node planes
  using TE = double;
  static constexpr int NE = 1;
  __device__ __forceinline__ void efetch(const LevelGeom& L, int ex, int ey, int ez, bool ok, double (&e)[1]) const {
    e[0] = bld(brsrc(C.H, N * 8), ok ? nid32(L, ex, ey, ez) * 8u : BOFF_NONE);
  }
  PfCoef C;
  const double* x;      // APPLY/RESID: d; PCGA: z
  const double* invD;   // RESID
  const double* p_old;  // PCGA
  double* out;          // APPLY: y; RESID: R; PCGA: w; DIAG: invD
  double* out2;         // RESID: fd (read); PCGA: p_new (null as in MechOp); DIAG: diag or null
  double* out3;         // RESID: z
  int flag;             // PCGA: first
  double sx, sy, sz, wg, ihx2, ihy2, ihz2;
  Reduce R;
  size_t N;
  static constexpr bool OPEN = OPENR;
  OpenRed O;  // as MechOp's

  __device__ __forceinline__ State state() const {
    State s;
    s.beta = (MODE == M_PCGA && !flag && !OPENR) ? R.scal[S_BETA] : 0.0;
    return s;
  }

  // through buffer resources, as MechOp's
  __device__ __forceinline__ void fetch(const LevelGeom& L, int gx, int gy, int gz, bool ok, const State& st,
                                        double (&r)[NR]) const {
#pragma unroll
    for (int k = 0; k < NR; k++) r[k] = 0.0;
    const unsigned ob = ok ? nid32(L, gx, gy, gz) * 8u : BOFF_NONE;
    const size_t nb = N * 8;
    if constexpr (MODE != M_DIAG) r[0] = bld(brsrc(x, nb), ob);
    if constexpr (MODE == M_PCGA) {
      if (!flag) r[1] = bld(brsrc(p_old, nb), ob);
    }
    r[NR - 1] = bld(brsrc(C.gc, nb), ob);
  }

  __device__ __forceinline__ void commit(const double (&r)[NR], const State& st, double (&v)[NV]) const {
    if constexpr (MODE == M_PCGA) {
      v[0] = r[0] + st.beta * r[1];
      v[1] = r[2];
    } else {
#pragma unroll
      for (int k = 0; k < NV; k++) v[k] = r[k];
    }
  }

  __device__ __forceinline__ void element(const LevelGeom& L, const double (&sN)[NSL][NV][PLANE], int s0, int tx,
                                          int ty, int ex, int ey, int ez, const State& st, const double (&e)[1],
                                          double (&f)[1][2][2][2]) const {
    double gcn[2][2][2];
    gather8(sN, s0, tx, ty, NU, gcn);
    if constexpr (MODE != M_DIAG) {
      // Where every element of the wave has one gc at its nodes (inside one
      // phase of an image), or a 0 among them (the zero rule: gc = 0 at every
      // Gauss point, an element outside the grid too), its coefficients are
      // constant and the wave takes the mode form: 7 compares decide, by the
      // values alone.
      const bool z = any_zero(gcn);
      const bool one = all_equal4(gcn[0]) & all_equal4(gcn[1]) & (gcn[0][0][0] == gcn[1][0][0]);
      if (__all(one | z)) {
        asm volatile("" ::: "memory");  // the nodal values are read in each branch
        double v[2][2][2];
        gather8(sN, s0, tx, ty, 0, v);
        const double g = z ? 0.0 : gcn[0][0][0];
        const double m = wg * (2.0 * e[0] + div_uniform(g, C.lc, C.rlc)), k = wg * g * C.lc;
        pf_hex_element(v, m, k, ihx2, ihy2, ihz2, f[0]);
        return;
      }
    }
    double m[2][2][2], k[2][2][2];
    pf_coefs(gcn, e[0], C.lc, C.rlc, wg, m, k);
    if constexpr (MODE == M_DIAG) {
      pf_element_diag(m, k, ihx2, ihy2, ihz2, f[0]);
    } else {
      double v[2][2][2];
      gather8(sN, s0, tx, ty, 0, v);
      pf_element(v, m, k, sx, sy, sz, f[0]);
    }
  }

  static constexpr bool NEEDS_OWN = (MODE == M_PCGA);
  struct NData {
    double f, iD;
  };
  __device__ __forceinline__ void nfetch(const LevelGeom& L, int i, int j, int k, NData& n) const {
    if constexpr (MODE == M_RESID) {
      const size_t q = nidx(L, i, j, k);
      n.f = out2[q];
      n.iD = invD[q];
    }
  }
  __device__ __forceinline__ void epilogue(const LevelGeom& L, const double (&own)[1], int i, int j, int k, int dm,
                                           const double (&v)[1], const State& st, const NData& nd,
                                           Acc& acc) const {
    const size_t q = nidx(L, i, j, k);
    if constexpr (MODE == M_APPLY) {
      out[q] = v[0];
    } else if constexpr (MODE == M_RESID) {
      const double fv = nd.f;
      const double r = fv - v[0];
      const double z = r * nd.iD;
      out[q] = r;
      out3[q] = z;
      acc.a[0] += r * z;
      acc.a[1] += r * r;
      acc.a[2] += fv * fv;
    } else if constexpr (MODE == M_PCGA) {
      const double p = own[0];
      if (out2) out2[q] = p;
      out[q] = v[0];
      acc.a[0] += p * v[0];
    } else {
      if (out2) out2[q] = v[0];
      out[q] = 1.0 / v[0];
      acc.a[0] += (v[0] == 0.0) ? 1.0 : 0.0;
    }
  }

  __device__ __forceinline__ void finish(Acc& acc, const Blk& bk) const {
    if constexpr (MODE == M_APPLY) return;
    double* scal = R.scal;
    if constexpr (MODE == M_RESID) {
      reduce_finalize<RED_SUM, 3>(bk, acc.a, R, 0.0, [=](double (&s)[3]) {
        scal[S_RZ] = s[0];
        scal[S_RR] = s[1];
        scal[S_FF] = s[2];
      });
    } else if constexpr (MODE == M_PCGA) {
      double v1[1] = {acc.a[0]};
      if constexpr (OPENR) return open_store(bk, v1, O);
      reduce_finalize<RED_SUM, 1>(bk, v1, R, 0.0, [=](double (&s)[1]) {
        scal[S_PW] = s[0];
        scal[S_ALPHA] = scal[S_RZ] / s[0];
      });
    } else {
      double v1[1] = {acc.a[0]};
      reduce_finalize<RED_SUM, 1>(bk, v1, R, 0.0, [=](double (&s)[1]) { scal[S_ZERO] = s[0]; });
    }
  }
};

static dim3 tile_grid(const LevelGeom& L) { return dim3((unsigned)tile_blocks(L.nx, L.ny, L.nz, L.zc)); }

template <class Op>
static Op mech_op(const LevelGeom& L, const MechCoef& C) {
  Op op{};
  op.C = C;
  op.N = (size_t)L.nx * L.ny * L.nz;
  op.sx = 1.0 / L.hx;
  op.sy = 1.0 / L.hy;
  op.sz = 1.0 / L.hz;
  op.wg = 0.125 * L.hx * L.hy * L.hz;
  op.tx_ = op.wg / L.hx;
  op.ty_ = op.wg / L.hy;
  op.tz_ = op.wg / L.hz;
  op.ihx2 = 1.0 / (L.hx * L.hx);
  op.ihy2 = 1.0 / (L.hy * L.hy);
  op.ihz2 = 1.0 / (L.hz * L.hz);
  op.fs = op.tx_ * op.sx;
  op.hs = HexScale<double>(L.hx, L.hy, L.hz);
  return op;
}

template <int MODE, bool FINE, bool FOLD, bool GAUSS = false>
static void run_mech_op(hipStream_t s, const LevelGeom& L, const MechCoef& C, const double* x, const double* invD,
                        const double* p_old, double* out, double* out2, double* out3, int flag, const Reduce& R,
                        const SplitW* S, const OpenRed* O) {
  using Op = MechOp<MODE, FINE, FOLD, GAUSS>;
  auto op = mech_op<Op>(L, C);
  op.x = x; op.invD = invD; op.p_old = p_old; op.out = out; op.out2 = out2; op.out3 = out3;
  op.flag = flag; op.R = R;
  if (O) op.O = *O;
  if constexpr (MODE == M_PCGA && FINE) {
    if (S) {
      const dim3 g((unsigned)split_blocks(L, *S));
      if (record<TileSplitK<Op>>(g, {L, op, *S})) return;
      tile_split_kernel<Op><<<g, dim3(TPB), 0, s>>>(L, op, *S);
      return;
    }
  }
  if (record<TileK<Op>>(tile_grid(L), {L, op})) return;
  tile_kernel<Op><<<tile_grid(L), dim3(TPB), 0, s>>>(L, op);
}

template <int MODE>
static void run_mech(hipStream_t s, const LevelGeom& L, const MechCoef& C, const double* x, const double* invD,
                     const double* p_old, double* out, double* out2, double* out3, int flag, const Reduce& R,
                     const SplitW* S = nullptr, const OpenRed* O = nullptr) {
  constexpr bool CAN_FOLD = (MODE != M_DIAG);
  const bool fold = CAN_FOLD && cubic_grid(L);
  if (C.fine) {
    if (fold)
      run_mech_op<MODE, true, CAN_FOLD>(s, L, C, x, invD, p_old, out, out2, out3, flag, R, S, O);
    else
      run_mech_op<MODE, true, false>(s, L, C, x, invD, p_old, out, out2, out3, flag, R, S, O);
  } else {
    if constexpr (MODE == M_RESID || MODE == M_PCGA) {
      if (C.gauss) {
        if (fold)
          run_mech_op<MODE, false, true, true>(s, L, C, x, invD, p_old, out, out2, out3, flag, R, S, O);
        else
          run_mech_op<MODE, false, false, true>(s, L, C, x, invD, p_old, out, out2, out3, flag, R, S, O);
        return;
      }
    }
    if (fold)
      run_mech_op<MODE, false, CAN_FOLD>(s, L, C, x, invD, p_old, out, out2, out3, flag, R, S, O);
    else
      run_mech_op<MODE, false, false>(s, L, C, x, invD, p_old, out, out2, out3, flag, R, S, O);
  }
}

void launch_mech_apply(hipStream_t s, const LevelGeom& L, const MechCoef& C, const double* x, double* y) {
  Reduce R{};
  run_mech<M_APPLY>(s, L, C, x, nullptr, nullptr, y, nullptr, nullptr, 0, R);
}
void launch_mech_resid(hipStream_t s, const LevelGeom& L, const MechCoef& C, const double* u, double* f,
                       double* r, double* z, const double* invD, int t0fine, const Reduce& R) {
  run_mech<M_RESID>(s, L, C, u, invD, nullptr, r, f, z, t0fine, R);
}
void launch_mech_pcg_a(hipStream_t s, const LevelGeom& L, const MechCoef& C, const double* z,
                       const double* p_old, double* p_new, double* w, int first, const Reduce& R,
                       const SplitW* S, const OpenRed* O) {
  run_mech<M_PCGA>(s, L, C, z, nullptr, p_old, w, p_new, nullptr, first, R, (S && S->ws && C.fine) ? S : nullptr, O);
}
void launch_mech_diag(hipStream_t s, const LevelGeom& L, const MechCoef& C, double* diag_or_null,
                      double* invD, const Reduce& R) {
  run_mech<M_DIAG>(s, L, C, nullptr, nullptr, nullptr, invD, diag_or_null, nullptr, 0, R);
}

template <int MODE, bool OPENR = false>
static void run_pf(hipStream_t s, const LevelGeom& L, const PfCoef& C, const double* x, const double* invD,
                   const double* p_old, double* out, double* out2, double* out3, int flag, const Reduce& R,
                   const OpenRed* O = nullptr) {
  using Op = PfOp<MODE, OPENR>;
  Op op{};
  op.C = C;
  op.x = x; op.invD = invD; op.p_old = p_old; op.out = out; op.out2 = out2; op.out3 = out3;
  op.flag = flag; op.R = R;
  if (O) op.O = *O;
  op.N = Nof(L);
  op.sx = 1.0 / L.hx;
  op.sy = 1.0 / L.hy;
  op.sz = 1.0 / L.hz;
  op.wg = 0.125 * L.hx * L.hy * L.hz;
  op.ihx2 = 1.0 / (L.hx * L.hx);
  op.ihy2 = 1.0 / (L.hy * L.hy);
  op.ihz2 = 1.0 / (L.hz * L.hz);
  if (record<TileK<Op>>(tile_grid(L), {L, op})) return;
  tile_kernel<Op><<<tile_grid(L), dim3(TPB), 0, s>>>(L, op);
}

void launch_pf_apply(hipStream_t s, const LevelGeom& L, const PfCoef& C, const double* x, double* y) {
  Reduce R{};
  run_pf<M_APPLY>(s, L, C, x, nullptr, nullptr, y, nullptr, nullptr, 0, R);
}
void launch_pf_resid(hipStream_t s, const LevelGeom& L, const PfCoef& C, const double* d, const double* fd,
                     double* r, double* z, const double* invD, const Reduce& R) {
  run_pf<M_RESID>(s, L, C, d, invD, nullptr, r, const_cast<double*>(fd), z, 0, R);
}
void launch_pf_pcg_a(hipStream_t s, const LevelGeom& L, const PfCoef& C, const double* z, const double* p_old,
                     double* p_new, double* w, int first, const Reduce& R, const OpenRed* O) {
  if (O)
    run_pf<M_PCGA, true>(s, L, C, z, nullptr, p_old, w, p_new, nullptr, first, R, O);
  else
    run_pf<M_PCGA>(s, L, C, z, nullptr, p_old, w, p_new, nullptr, first, R);
}
void launch_pf_diag(hipStream_t s, const LevelGeom& L, const PfCoef& C, double* diag_or_null, double* invD,
                    const Reduce& R) {
  run_pf<M_DIAG>(s, L, C, nullptr, nullptr, nullptr, invD, diag_or_null, nullptr, 0, R);
}

// ---------------------------------------------------------------------------
// Pointwise PCG pass B
// ---------------------------------------------------------------------------
constexpr int PW_TPB = 256;
static int pw_blocks(size_t n) {
  size_t b = (n + PW_TPB - 1) / PW_TPB;
  return (int)(b < 2048 ? (b == 0 ? 1 : b) : 2048);
}
// grid of the PCG pass-B kernels (at most HPCR_PASSB_MAX_BLOCKS blocks,
// grid-stride beyond)
#ifndef HPCR_PASSB_MAX_BLOCKS
#define HPCR_PASSB_MAX_BLOCKS 512
#endif
int passb_blocks(size_t n) {
  const size_t b = (n + PW_TPB - 1) / PW_TPB;
  const size_t cap = HPCR_PASSB_MAX_BLOCKS;
  return (int)(b == 0 ? 1 : (b < cap ? b : cap));
}

// Tuning macros of the pass-B kernels: HPCR_PASSB_NT (non-temporal loads and
// stores of the streamed vectors), HPCR_PASSB_UNROLL2 (two nodes per thread
// and iteration).
#ifdef HPCR_PASSB_NT
#define PB_LD(x) __builtin_nontemporal_load(&(x))
#define PB_ST(v, x) __builtin_nontemporal_store((v), &(x))
#else
#define PB_LD(x) (x)
#define PB_ST(v, x) ((x) = (v))
#endif

// Reductions of a pass B: r.z -> beta (not after the last iteration), r.r, and
// with slot >= 0 the alpha of an update left to a later pass B
template <bool LAST>
__device__ __forceinline__ void passb_reduce(const Blk& bk, double (&acc)[2], const Reduce& R, int slot) {
  double* scal = R.scal;
  if constexpr (LAST) {
    double rr[1] = {acc[1]};
    reduce_finalize<RED_SUM, 1>(bk, rr, R, 0.0, [=](double (&s)[1]) { scal[S_RR] = s[0]; });
  } else {
    reduce_finalize<RED_SUM, 2>(bk, acc, R, 0.0, [=](double (&s)[2]) {
      scal[S_BETA] = s[0] / scal[S_RZ];
      scal[S_RZ] = s[0];
      scal[S_RR] = s[1];
      if (slot >= 0) scal[S_AH + slot] = scal[S_ALPHA];
    });
  }
}

// LDSF: the Dirichlet axis flags are staged in LDS (levels with
// nx + ny + nz <= DIRF_MAX), so a node's mask needs no dependent global load,
// which would also wait on the stores still in flight.
// NP: x updates of the CG group applied here (0: this iteration's is left
// out and its alpha kept in scal[S_AH + slot]).  A group's updates come in
// iteration order, each as the one fma of the undeferred form.
template <int NP>
struct GroupAlpha {
  double a[NP > 0 ? NP : 1];
  __device__ __forceinline__ GroupAlpha(const double* scal) {
#pragma unroll
    for (int m = 0; m + 1 < NP; m++) a[m] = scal[S_AH + m];
    a[NP > 0 ? NP - 1 : 0] = scal[S_ALPHA];
  }
  __device__ __forceinline__ double apply(const PGroup& P, size_t o, double x) const {
#pragma unroll
    for (int m = 0; m < NP; m++) x = fma(a[m], PB_LD(P.p[m][o]), x);
    return x;
  }
};

// w of node (i, j, k), component c, from the parts of a split-output pass A
// (SplitW), added in a fixed order: the part of the tile whose own region
// holds the node, of the tile below (top row), of the tile to its left (right
// column), of the tile below-left (corner).  A part is taken where that
// tile exists: none has the last node column x = 64 ntx or row y = 4 nty in
// its own region, nor a right column in row 4 nty, nor a top row in column
// 64 ntx.
__device__ __forceinline__ double split_w(const LevelGeom& L, const SplitW& S, const double* __restrict__ w, int c,
                                          size_t o, unsigned i, unsigned j, unsigned k) {
  const bool col = i < (unsigned)(STX * S.ntx), row = j < (unsigned)(STY * S.nty);
  const bool xe = i > 0 && i % STX == 0, ye = j > 0 && j % STY == 0;
  const unsigned kx = i / STX - 1, ky = j / STY - 1;
  // the own-region part is loaded unconditionally (pass A stores 0 at the
  // nodes past every own region); the right-column and corner parts, which
  // one lane in 64 needs, without a branch: an absent one from an offset past
  // the side arrays' resource, which reads 0 (and v + 0 = v)
  const auto rs = brsrc(S.ws, S.count() * 8);
  const unsigned ot = (3u * S.nr + c * S.nt + (k * (unsigned)S.nty + ky) * (unsigned)L.nx + i) * 8u;
  const unsigned orr = (c * S.nr + (k * (unsigned)L.ny + j) * (unsigned)S.ntx + kx) * 8u;
  const unsigned oc = (3u * (S.nr + S.nt) + c * S.nc + (k * (unsigned)S.nty + ky) * (unsigned)S.ntx + kx) * 8u;
  const double v = PB_LD(w[o]);
  double t = 0.0;
  if (ye && col) t = ldo(S.ws, ot);  // whole rows: a branch that waves mostly take or skip together
  const double r = bld(rs, (xe && row) ? orr : BOFF_NONE);
  const double q = bld(rs, (xe && ye) ? oc : BOFF_NONE);
  return ((v + t) + r) + q;
}

// LAST: the call's last iteration, after which neither z nor beta is used: z is
// not stored, 1/D not read and r.z not summed.  That is 48 of the 264 B per
// node that a pass B closing a group of four moves (of 216 B closing two);
// at 257^3 978 -> 778 us and 791 -> 602 us.
template <bool LDSF, int NP, bool WPARTS, bool LAST>
__device__ __forceinline__ void mech_pcg_b_body(const LevelGeom& L, double* __restrict__ u, double* __restrict__ r,
                                                double* __restrict__ z, const PGroup& P,
                                                const double* __restrict__ w, const double* __restrict__ invD,
                                                int slot, const Reduce& R, const SplitW& S, const Blk& bk) {
  __shared__ unsigned char sflags[LDSF ? DIRF_MAX : 1];
  const DirFlags F{sflags};
  if constexpr (LDSF) {
    F.stage(L);
    __syncthreads();
  }
  // node counts stay below 2^32 (a 1625^3 grid would not fit in HBM)
  const unsigned N = (unsigned)Nof(L);
  const unsigned plane = (unsigned)L.nx * (unsigned)L.ny;
  const double alpha = R.scal[S_ALPHA];
  const GroupAlpha<NP> ga(R.scal);
  double acc[2] = {0.0, 0.0};
  auto node = [&](unsigned q) {
    const unsigned k = q / plane;
    int dm = 0;
    unsigned i = 0, j = 0;
    if constexpr (LDSF || WPARTS) {
      const unsigned rem = q - k * plane;
      j = rem / (unsigned)L.nx;
      i = rem - j * (unsigned)L.nx;
    }
    if constexpr (LDSF) {
      dm = F.mask(L, (int)i, (int)j, (int)k);
    } else if (L.fz[k]) {
      const unsigned rem = q - k * plane;
      const unsigned jj = rem / (unsigned)L.nx, ii = rem - jj * (unsigned)L.nx;
      dm = dir_mask(L, (int)ii, (int)jj, (int)k);
    }
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const size_t o = (size_t)c * N + q;
      if constexpr (NP > 0) PB_ST(ga.apply(P, o, PB_LD(u[o])), u[o]);
      double wv;
      if constexpr (WPARTS)
        wv = split_w(L, S, w, c, o, i, j, k);
      else
        wv = PB_LD(w[o]);
      double rv = PB_LD(r[o]) - alpha * wv;
      if ((dm >> c) & 1) rv = 0.0;
      PB_ST(rv, r[o]);
      if constexpr (!LAST) {
        const double zv = rv * PB_LD(invD[o]);
        PB_ST(zv, z[o]);
        acc[0] += rv * zv;
      }
      acc[1] += rv * rv;
    }
  };
  const unsigned stride = bk.gx * PW_TPB;
#ifdef HPCR_PASSB_UNROLL2
  for (unsigned q = bk.x * PW_TPB + threadIdx.x; q < N; q += 2 * stride) {
    node(q);
    if (q + stride < N) node(q + stride);
  }
#else
  for (unsigned q = bk.x * PW_TPB + threadIdx.x; q < N; q += stride) node(q);
#endif
  passb_reduce<LAST>(bk, acc, R, NP == 0 ? slot : -1);
}

template <bool LDSF, int NP, bool WPARTS, bool LAST>
__global__ __launch_bounds__(PW_TPB) void mech_pcg_b_kernel(const LevelGeom L, double* __restrict__ u,
                                                            double* __restrict__ r, double* __restrict__ z,
                                                            const PGroup P, const double* __restrict__ w,
                                                            const double* __restrict__ invD, int slot,
                                                            const Reduce R, const SplitW S) {
  mech_pcg_b_body<LDSF, NP, WPARTS, LAST>(L, u, r, z, P, w, invD, slot, R, S, Blk::hw());
}

struct PassBArgs {
  LevelGeom L;
  size_t N;
  double* x;  // u or d
  double* r;
  double* z;
  PGroup P;
  const double* w;
  const double* invD;
  int slot;
  Reduce R;
  SplitW S;   // mechanics: the parts of a split-output pass A (S.ws null: w whole)
};
template <bool LDSF, int NP, bool WPARTS, bool LAST>
struct MechPassBK {
  using Args = PassBArgs;
  static constexpr int NT = PW_TPB, MINW = 1;
  static dim3 block() { return dim3(PW_TPB); }
  __device__ __forceinline__ static void run(const Args& a, const Blk& bk) {
    mech_pcg_b_body<LDSF, NP, WPARTS, LAST>(a.L, a.x, a.r, a.z, a.P, a.w, a.invD, a.slot, a.R, a.S, bk);
  }
};

template <int NP, bool LAST>
__device__ __forceinline__ void pf_pcg_b_body(size_t N, double* __restrict__ d, double* __restrict__ r,
                                              double* __restrict__ z, const PGroup& P, const double* __restrict__ w,
                                              const double* __restrict__ invD, int slot, const Reduce& R,
                                              const Blk& bk) {
  const double alpha = R.scal[S_ALPHA];
  const GroupAlpha<NP> ga(R.scal);
  double acc[2] = {0.0, 0.0};
  for (size_t q = (size_t)bk.x * PW_TPB + threadIdx.x; q < N; q += (size_t)bk.gx * PW_TPB) {
    if constexpr (NP > 0) d[q] = ga.apply(P, q, d[q]);
    const double rv = r[q] - alpha * w[q];
    r[q] = rv;
    if constexpr (!LAST) {
      const double zv = rv * invD[q];
      z[q] = zv;
      acc[0] += rv * zv;
    }
    acc[1] += rv * rv;
  }
  passb_reduce<LAST>(bk, acc, R, NP == 0 ? slot : -1);
}

template <int NP, bool LAST>
__global__ __launch_bounds__(PW_TPB) void pf_pcg_b_kernel(size_t N, double* __restrict__ d, double* __restrict__ r,
                                                          double* __restrict__ z, const PGroup P,
                                                          const double* __restrict__ w,
                                                          const double* __restrict__ invD, int slot,
                                                          const Reduce R) {
  pf_pcg_b_body<NP, LAST>(N, d, r, z, P, w, invD, slot, R, Blk::hw());
}
template <int NP, bool LAST>
struct PfPassBK {
  using Args = PassBArgs;
  static constexpr int NT = PW_TPB, MINW = 1;
  static dim3 block() { return dim3(PW_TPB); }
  __device__ __forceinline__ static void run(const Args& a, const Blk& bk) {
    pf_pcg_b_body<NP, LAST>(a.N, a.x, a.r, a.z, a.P, a.w, a.invD, a.slot, a.R, bk);
  }
};

// f(NP, LAST) of an iteration: only the pass B that closes a group or the
// call applies updates, and one that closes a group inside the call closes
// CG_GROUP of them.  KEEP: calls whose last iteration keeps z and r.z
// (the phase field's), where LAST is false at every group position.
template <bool KEEP, class F>
static void passb_dispatch(int np, bool last, F f) {
  static_assert(CG_GROUP == 4, "one instantiation per group position");
  using std::integral_constant;
  if (np == 0) return f(integral_constant<int, 0>(), std::false_type());
  auto go = [&](auto n) {
    if constexpr (KEEP || decltype(n)::value == CG_GROUP) {
      if (!last) return f(n, std::false_type());
    }
    f(n, std::true_type());
  };
  switch (np) {
    case 1: go(integral_constant<int, 1>()); break;
    case 2: go(integral_constant<int, 2>()); break;
    case 3: go(integral_constant<int, 3>()); break;
    default: go(integral_constant<int, 4>()); break;
  }
}
void launch_mech_pcg_b(hipStream_t s, const LevelGeom& L, double* u, double* r, double* z, const PGroup& P,
                       const double* w, const double* invD, int np, int slot, bool last, const Reduce& R,
                       const SplitW* S) {
  const bool parts = S && S->ws;
  const SplitW none{};
  const SplitW& SW = parts ? *S : none;
  const dim3 g(passb_blocks(Nof(L))), b(PW_TPB);
  const PassBArgs a{L, Nof(L), u, r, z, P, w, invD, slot, R, SW};
  auto go = [&](auto ldsf, auto wparts) {
    passb_dispatch<false>(np, last, [&](auto n, auto l) {
      constexpr bool LDSF = decltype(ldsf)::value, WPARTS = decltype(wparts)::value, LAST = decltype(l)::value;
      constexpr int NP = decltype(n)::value;
      if (record<MechPassBK<LDSF, NP, WPARTS, LAST>>(g, a)) return;
      hipLaunchKernelGGL((mech_pcg_b_kernel<LDSF, NP, WPARTS, LAST>), g, b, 0, s, L, u, r, z, P, w, invD, slot, R,
                         SW);
    });
  };
  if (L.nx + L.ny + L.nz <= DIRF_MAX) {
    if (parts)
      go(std::true_type(), std::true_type());
    else
      go(std::true_type(), std::false_type());
  } else {
    if (parts)
      go(std::false_type(), std::true_type());
    else
      go(std::false_type(), std::false_type());
  }
}
void launch_pf_pcg_b(hipStream_t s, const LevelGeom& L, double* d, double* r, double* z, const PGroup& P,
                     const double* w, const double* invD, int np, int slot, bool last, const Reduce& R) {
  const size_t N = Nof(L);
  const dim3 g(passb_blocks(N)), b(PW_TPB);
  const PassBArgs a{L, N, d, r, z, P, w, invD, slot, R};
  passb_dispatch<true>(np, last, [&](auto n, auto l) {
    constexpr bool LAST = decltype(l)::value;
    constexpr int NP = decltype(n)::value;
    if (record<PfPassBK<NP, LAST>>(g, a)) return;
    hipLaunchKernelGGL((pf_pcg_b_kernel<NP, LAST>), g, b, 0, s, N, d, r, z, P, w, invD, slot, R);
  });
}

// Pass B of an open call on a small level (OpenRed): all of a thread's first
// loads go out before the sum of p.Ap that alpha waits for.  The values and
// the order of the sums are mech_pcg_b_body's and pf_pcg_b_body's.
template <int NC, int NP, bool LAST>
__device__ __forceinline__ void open_pcg_b_body(const LevelGeom& L, double* __restrict__ x, double* __restrict__ r,
                                                double* __restrict__ z, const PGroup& P,
                                                const double* __restrict__ w, const double* __restrict__ invD,
                                                int slot, bool rr, const Reduce& R, const OpenRed& O,
                                                const Blk& bk) {
  const unsigned N = (unsigned)Nof(L), plane = (unsigned)L.nx * (unsigned)L.ny;
  const OpenShare sh(O);
  double* scal = R.scal;
  const double rz = scal[(O.it & 1) ? S_RZ1 : S_RZ];
  double ah[NP > 1 ? NP - 1 : 1];
#pragma unroll
  for (int m = 0; m + 1 < NP; m++) ah[m] = scal[S_AH + m];
  struct Node {
    double r[NC], w[NC], iD[NC], x[NC], p[NP > 0 ? NP : 1][NC];
    int dm;
  } d;
  auto load = [&](unsigned q) {
#pragma unroll
    for (int c = 0; c < NC; c++) {
      const size_t o = (size_t)c * N + q;
      d.r[c] = r[o];
      d.w[c] = w[o];
      if constexpr (!LAST) d.iD[c] = invD[o];
      if constexpr (NP > 0) {
        d.x[c] = x[o];
#pragma unroll
        for (int m = 0; m < NP; m++) d.p[m][c] = P.p[m][o];
      }
    }
    d.dm = 0;
    if constexpr (NC == 3) {
      const unsigned k = q / plane, rem = q - k * plane;
      const unsigned j = rem / (unsigned)L.nx, i = rem - j * (unsigned)L.nx;
      d.dm = dir_mask_flat(L, (int)i, (int)j, (int)k);
    }
  };
  unsigned q = bk.x * PW_TPB + threadIdx.x;
  const unsigned stride = bk.gx * PW_TPB;
  load(min(q, N - 1));
  const double pw = sh.total();
  const double alpha = rz / pw;
  if (bk.x == 0 && threadIdx.x == 0) {
    scal[S_PW] = pw;
    scal[S_ALPHA] = alpha;
    if (NP == 0) scal[S_AH + slot] = alpha;
  }
  double acc[1] = {0.0};
  while (q < N) {
#pragma unroll
    for (int c = 0; c < NC; c++) {
      const size_t o = (size_t)c * N + q;
      if constexpr (NP > 0) {
        double xv = d.x[c];
#pragma unroll
        for (int m = 0; m + 1 < NP; m++) xv = fma(ah[m], d.p[m][c], xv);
        x[o] = fma(alpha, d.p[NP - 1][c], xv);
      }
      double rv = d.r[c] - alpha * d.w[c];
      if ((d.dm >> c) & 1) rv = 0.0;
      r[o] = rv;
      if constexpr (!LAST) {
        const double zv = rv * d.iD[c];
        z[o] = zv;
        acc[0] += rv * zv;
      } else {
        acc[0] += rv * rv;
      }
    }
    q += stride;
    if (q < N) load(q);
  }
  if constexpr (!LAST)
    open_store(bk, acc, O);
  else if (rr)
    reduce_finalize<RED_SUM, 1>(bk, acc, R, 0.0, [=](double (&s)[1]) { scal[S_RR] = s[0]; });
}
struct OpenPassBArgs {
  LevelGeom L;
  double* x;
  double* r;
  double* z;
  PGroup P;
  const double* w;
  const double* invD;
  int slot, rr;
  Reduce R;
  OpenRed O;
};
template <int NC, int NP, bool LAST>
struct OpenPassBK {
  using Args = OpenPassBArgs;
  static constexpr int NT = PW_TPB, MINW = 1;
  static dim3 block() { return dim3(PW_TPB); }
  __device__ __forceinline__ static void run(const Args& a, const Blk& bk) {
    open_pcg_b_body<NC, NP, LAST>(a.L, a.x, a.r, a.z, a.P, a.w, a.invD, a.slot, a.rr != 0, a.R, a.O, bk);
  }
};
template <int NC, int NP, bool LAST>
__global__ __launch_bounds__(PW_TPB) void open_pcg_b_kernel(const OpenPassBArgs a) {
  OpenPassBK<NC, NP, LAST>::run(a, Blk::hw());
}
static_assert(HPCR_PASSB_MAX_BLOCKS <= OPEN_BLOCKS, "pass A adds up every partial of an open pass B");
void launch_open_pcg_b(hipStream_t s, const LevelGeom& L, int ncomp, double* x, double* r, double* z,
                       const PGroup& P, const double* w, const double* invD, int np, int slot, bool last, bool rr,
                       const Reduce& R, const OpenRed& O) {
  const dim3 g(passb_blocks(Nof(L))), b(PW_TPB);
  const OpenPassBArgs a{L, x, r, z, P, w, invD, slot, rr ? 1 : 0, R, O};
  auto go = [&](auto nc) {
    passb_dispatch<false>(np, last, [&](auto n, auto l) {
      constexpr int NC = decltype(nc)::value, NP = decltype(n)::value;
      constexpr bool LAST = decltype(l)::value;
      if (record<OpenPassBK<NC, NP, LAST>>(g, a)) return;
      hipLaunchKernelGGL((open_pcg_b_kernel<NC, NP, LAST>), g, b, 0, s, a);
    });
  };
  if (ncomp == 3)
    go(std::integral_constant<int, 3>());
  else
    go(std::integral_constant<int, 1>());
}

// ---------------------------------------------------------------------------
// Dirichlet boundary conditions (boundary_conditions.cpp:28-111)
// ---------------------------------------------------------------------------
struct Planes {
  int k[4];
  int n;
};

__device__ __forceinline__ void dirichlet_bd_body(const LevelGeom& L, double* u, double Ut, const Planes& P,
                                                  const Blk& bk) {
  const size_t N = Nof(L);
  const int i = bk.x * blockDim.x + threadIdx.x;
  const int j = bk.y;
  if (i >= L.nx) return;
  // unrolled: the plane list is indexed with constants (no private copy)
#pragma unroll
  for (int t = 0; t < 4; t++) {
    if (t >= P.n) break;
    const int k = P.k[t];
    const int dm = dir_mask(L, i, j, k);
    const size_t q = nidx(L, i, j, k);
    if (dm & 1) u[q] = 0.0;
    if (dm & 2) u[N + q] = 0.0;
    if (dm & 4) u[2 * N + q] = (dm & 8) ? Ut : 0.0;
  }
}
__global__ void dirichlet_bd_kernel(const LevelGeom L, double* u, double Ut, Planes P) {
  dirichlet_bd_body(L, u, Ut, P, Blk::hw());
}
struct DirichletBdK {
  struct Args {
    LevelGeom L;
    double* u;
    double Ut;
    Planes P;
  };
  static constexpr int NT = 64, MINW = 1;
  static dim3 block() { return dim3(64); }
  __device__ __forceinline__ static void run(const Args& a, const Blk& bk) {
    dirichlet_bd_body(a.L, a.u, a.Ut, a.P, bk);
  }
};
__global__ void dirichlet_copy_kernel(const LevelGeom L, double* f, const double* Fi, Planes P) {
  const size_t N = Nof(L);
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y;
  if (i >= L.nx) return;
  for (int t = 0; t < P.n; t++) {
    const int k = P.k[t];
    const int dm = dir_mask(L, i, j, k);
    const size_t q = nidx(L, i, j, k);
#pragma unroll
    for (int c = 0; c < 3; c++)
      if ((dm >> c) & 1) f[c * N + q] = Fi[c * N + q];
  }
}
static Planes planes_of(const int* kp, int n) {
  Planes P{};
  P.n = n > 4 ? 4 : n;
  for (int t = 0; t < P.n; t++) P.k[t] = kp[t];
  return P;
}
void launch_dirichlet_bd(hipStream_t s, const LevelGeom& L, double* u, double Ut, const int* kp, int n) {
  if (n <= 0) return;
  if (record<DirichletBdK>(dim3((L.nx + 63) / 64, L.ny), {L, u, Ut, planes_of(kp, n)})) return;
  hipLaunchKernelGGL(dirichlet_bd_kernel, dim3((L.nx + 63) / 64, L.ny), dim3(64), 0, s, L, u, Ut, planes_of(kp, n));
}
void launch_dirichlet_copy(hipStream_t s, const LevelGeom& L, double* f, const double* Fi, const int* kp, int n) {
  if (n <= 0) return;
  hipLaunchKernelGGL(dirichlet_copy_kernel, dim3((L.nx + 63) / 64, L.ny), dim3(64), 0, s, L, f, Fi,
                     planes_of(kp, n));
}

// ---------------------------------------------------------------------------
// Whole smoother call of a small coarse level in one workgroup
// (pcg_u, mechanical_pcg.cpp:223-330; pcg_d, phase_field_pcg.cpp:133-214)
// ---------------------------------------------------------------------------
// x, r, p and 1/D of a thread's nodes stay in registers (p in LDS from 512
// threads on).  Per operator apply:
// p -> LDS, barrier, every element writes its corner contributions to LDS,
// barrier, every node sums the contributions of its (up to) 8 elements in a
// fixed order, from slots found once (an absent element reads a slot of
// zeros).  Reductions are block-wide in a fixed order.  The fused
// multiply-adds are written out (see hex_force_modes).  The recurrence is
// that of the two-pass path: p = z + beta p, alpha = r.z / p.Ap,
// beta = r.z_new / r.z.
//
// What bounds it is one iteration's chain of dependent steps: the element's
// arithmetic, two LDS round trips, two block sums and two divisions; at most
// 16 of the chip's 1024 SIMD waves run.  So the element is the
// constant-moduli mode form (hex_force: ~190 operations instead of ~430), and
// on levels of at most 256 nodes a thread has one displacement component
// (SPLIT: the wave's component is uniform, ~95 operations), which also
// spreads the vector updates and the node sums over three times the waves.
//
// Layouts (threads; nodes a thread), by the level's nodes and elements:
//   mechanics     <= 128 / 128: SPLIT 3 x 128;   <= 256 / 256: SPLIT 3 x 256
//   phase field   <= 128 / 128: 128; 1           <= 256 / 256: 256; 1
//   both          <= 1024 / 512: 512; 2          <= 1536 / 1024: 1024; 2
// The upper line is the workgroup: one element per thread, 1024 threads; there
// the contributions go through LDS one component at a time (BYC: 8 of 24 for
// 1024 elements are 64 KiB), and p and x stay in LDS.  Its 128 registers a
// thread do not suffice all the same: mechanics spills 165 (212 B a lane), the
// phase field 12.  A level beyond it runs the tile passes, two launches an
// iteration.
// us of a call's 50 iterations (its start left out), first with the levels up to
// 512 nodes and 256 elements in one workgroup with the eight-Gauss-point element
// and shuffle sums and larger ones by the tile passes with ticketed reductions:
//   mechanics     5x5x5 135 -> 61.5 (float vectors the same), 5x5x9 148 -> 86
//                 9x9x9 755 -> 157, 7x11x8 750 -> 147, 11x11x11 755 -> 670,
//                 17x9x9 767 -> 664
//   phase field   9x9x9 624 -> 99, 11x11x11 619 -> 183, 17x9x9 620 -> 180
// and the same by the tile passes with open reductions (OpenRed), which came
// later: mechanics 9x9x9 560, 11x11x11 560 to 590, 17x9x9 560; phase field 490
// to 540.  So the 512-thread layout is well inside its line, and the 1024-thread
// one of mechanics saves launches (one for 2 to 100) but not time on a GPU that
// has nothing else to run.
static_assert(SMALL_NODES == 1536 && SMALL_ELEMS == 1024, "small-level layouts");

// Sum over a wavefront into lane 63: an inclusive scan by DPP row shifts and
// row broadcasts (registers only; a shuffle would go through the LDS
// crossbar, ~100 cycles a step).
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_part(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffLL), CTRL, ROWS, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ double wave_sum63(double v) {
  v += dpp_part<0x111, 0xf>(v);  // row_shr:1
  v += dpp_part<0x112, 0xf>(v);  // row_shr:2
  v += dpp_part<0x114, 0xf>(v);  // row_shr:4
  v += dpp_part<0x118, 0xf>(v);  // row_shr:8
  v += dpp_part<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  v += dpp_part<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
  return v;
}

// Block-wide sums, every thread receiving the total: wavefront sums to LDS,
// one barrier, then every thread adds the NW partials in wavefront order.  Consecutive calls alternate between the two halves of sh, so a half
// is written again only after the barrier of the call in between, which every
// thread reaches after its reads of that half.
template <int NW, int NV>
__device__ __forceinline__ void block_sum_all(double (&v)[NV], double* sh, int& half) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  double* h = sh + half * (3 * 16);
#pragma unroll
  for (int k = 0; k < NV; k++) v[k] = wave_sum63(v[k]);
  if (lane == 63)
#pragma unroll
    for (int k = 0; k < NV; k++) h[k * 16 + wid] = v[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; k++) {
    double a = h[k * 16];
#pragma unroll
    for (int w = 1; w < NW; w++) a = a + h[k * 16 + w];
    v[k] = a;
  }
  half ^= 1;
}

template <class TIO>
struct SmallArgsT {
  LevelGeom L;
  // mechanics: element K_e, G_e; phase field: element H, nodal gc
  const double* Ke;
  const double* Ge;
  const double* H;
  const double* gc;
  double lc, rlc;      // lc and 1 / lc
  HexScale<double> hs; // mechanics
  TIO* x;              // u (3 comps) or d
  const TIO* f;        // right-hand side
  const double* invD;  // inverse Jacobi diagonal
  TIO* r;              // final residual (optional)
  TIO* p;              // final search direction (optional)
  TIO* w;              // final A p (optional)
  double Ut;
  int NB;
  double* scal;
};
using SmallArgs = SmallArgsT<double>;

// NP: nodes (and elements) the block's threads cover at a time; NPT: nodes
// per thread; SPLIT: mechanics with one component per thread, 3 NP threads
template <int NC_, int NP_, int NPT_, bool SPLIT_>
struct SmallLayout {
  static constexpr int NC = NC_, NP = NP_, NPT = NPT_;
  static constexpr bool SPLIT = SPLIT_;
  static constexpr int THREADS = SPLIT ? 3 * NP : NP;
  static_assert(!SPLIT || (NC == 3 && NPT == 1 && NP % 64 == 0), "a wave has one component");
};

// TIO: type of the vectors in HBM; the iteration itself is FP64
template <class Lay, class TIO>
__device__ __forceinline__ void small_pcg_body(const SmallArgsT<TIO>& a) {
  constexpr int NC = Lay::NC, NP = Lay::NP, NPT = Lay::NPT;
  constexpr bool SPLIT = Lay::SPLIT;
  constexpr int NCT = SPLIT ? 1 : NC;             // components of a thread
  constexpr int NW = Lay::THREADS / 64;
  constexpr int EST = NP + 1;                     // contribution slots: NP elements and the zeros
  constexpr bool BYC = NC * 8 * EST * 8 > 112 * 1024;  // contributions through LDS one component at a time
  constexpr int NCE = BYC ? 1 : NC;               // components in LDS at a time
  constexpr bool PLDS = NPT > 1;                  // a thread reads its own p back from LDS
  constexpr bool XLDS = NP == 1024;               // and keeps its own x there
  constexpr int NN = XLDS ? SMALL_NODES : NP * NPT;
  const LevelGeom& L = a.L;
  __shared__ double sP[NC][NN];
  __shared__ double sX[XLDS ? NC : 1][XLDS ? NN : 1];
  __shared__ double sE[NCE * 8][EST];
  __shared__ double sh[2 * 3 * 16];
  int half = 0;
  const int tid = threadIdx.x;
  const int c0 = SPLIT ? __builtin_amdgcn_readfirstlane(tid / NP) : 0;
  const int tn = SPLIT ? tid - c0 * NP : tid;     // node and element slot of the thread
  const int N = L.nx * L.ny * L.nz;
  const int ex_n = L.nx - 1, ey_n = L.ny - 1;
  const int E = ex_n * ey_n * (L.nz - 1);

  // Element of this thread and its constant coefficients.  A level has about
  // half as many elements as nodes, so half of a component's waves have none;
  // waves go to the four SIMDs in turn, and with the elements of one component
  // on its upper half of the threads the waves that have some share no SIMD
  // (3 x 128: waves 0, 2, 5 instead of 0, 2, 4) or two at most (3 x 256:
  // 0 1, 6 7, 8 9 instead of 0 1, 4 5, 8 9).
  const bool upper = SPLIT && c0 == (NP == 128 ? 2 : 1);
  const int te = upper ? tn ^ (NP / 2) : tn;
  const bool has_e = te < E;
  int eb = 0;  // its lowest node
  double lam0 = 0.0, mu0 = 0.0;
  double pm[2][2][2], pk[2][2][2];
  if (has_e) {
    const int ei = te % ex_n, ej = (te / ex_n) % ey_n, ek = te / (ex_n * ey_n);
    eb = ei + L.nx * (ej + L.ny * ek);
    if constexpr (NC == 3) {
      lam0 = fma(-2.0 / 3.0, a.Ge[eb], a.Ke[eb]);
      mu0 = a.Ge[eb];
    } else {
      double gcn[2][2][2];
#pragma unroll
      for (int iz = 0; iz < 2; iz++)
#pragma unroll
        for (int iy = 0; iy < 2; iy++)
#pragma unroll
          for (int ix = 0; ix < 2; ix++) gcn[iz][iy][ix] = a.gc[eb + ix + L.nx * (iy + L.ny * iz)];
      pf_coefs(gcn, a.H[eb], a.lc, a.rlc, 0.125 * L.hx * L.hy * L.hz, pm, pk);
    }
  }
  const HexScale<double> hsr = SPLIT ? a.hs.rotated(c0) : a.hs;
  if (tid < NCE * 8) sE[tid][NP] = 0.0;

  // nodes of this thread; their values in sP, and x
  int qn[NPT], dm[NPT];
  double xv[XLDS ? 1 : NPT][NCT], r[NPT][NCT], iD[NPT][NCT], p[PLDS ? 1 : NPT][NCT], w[NPT][NCT];
  auto own = [&](int s, int c) -> double& { return sP[SPLIT ? c0 : c][tn + s * NP]; };
  auto xval = [&](int s, int c) -> double& {
    if constexpr (XLDS)
      return sX[c][tn + s * NP];
    else
      return xv[s][c];
  };
  unsigned eo[NPT][4];  // contribution slots of the node's 8 elements, two per word
#pragma unroll
  for (int s = 0; s < NPT; s++) {
    const int q = tn + s * NP;
    qn[s] = q < N ? q : -1;
    dm[s] = 0;
#pragma unroll
    for (int t = 0; t < 4; t++) eo[s][t] = (unsigned)NP * 0x10001u;
#pragma unroll
    for (int c = 0; c < NCT; c++) r[s][c] = iD[s][c] = 0.0;
    if (q < N) {
      const int i = q % L.nx, j = (q / L.nx) % L.ny, k = q / (L.nx * L.ny);
      if constexpr (NC == 3) {
        dm[s] = dir_mask(L, i, j, k);
        if constexpr (SPLIT) dm[s] = (dm[s] >> c0) & 1 ? (1 | (c0 == 2 ? dm[s] & 8 : 0)) : 0;
      }
#pragma unroll
      for (int t = 0; t < 8; t++) {
        const int e_i = i - (t & 1), e_j = j - ((t >> 1) & 1), e_k = k - (t >> 2);
        const bool in = e_i >= 0 && e_j >= 0 && e_k >= 0 && e_i < ex_n && e_j < ey_n && e_k < L.nz - 1;
        const unsigned e = in ? (unsigned)(e_i + ex_n * (e_j + ey_n * e_k)) : (unsigned)NP;
        eo[s][t >> 1] = (t & 1) ? ((eo[s][t >> 1] & 0xffffu) | (e << 16)) : e;
      }
#pragma unroll
      for (int c = 0; c < NCT; c++) {
        const size_t o = (size_t)(SPLIT ? c0 : c) * N + q;
        double x = (double)a.x[o];
        r[s][c] = (double)a.f[o];
        iD[s][c] = a.invD[o];
        // Dirichlet_BD (boundary_conditions.cpp:28-66)
        if (NC == 3 && ((dm[s] >> c) & 1)) x = (dm[s] & 8) && (SPLIT || c == 2) ? a.Ut : 0.0;
        xval(s, c) = x;
        own(s, c) = x;
      }
    }
  }

  // a thread's contributions of local component c to LDS, and its nodes' sums
  auto hand_over = [&](const double (&f)[2][2][2], int c) {
#pragma unroll
    for (int t = 0; t < 8; t++) {
      const int iz = t >> 2, iy = (t >> 1) & 1, ix = t & 1;
      if constexpr (SPLIT) {
        // corner (ix, iy, iz) of the rotated axes
        const int slot = c0 == 0 ? t : (c0 == 1 ? 2 * ix + 4 * iy + iz : 4 * ix + iy + 2 * iz);
        sE[c0 * 8 + slot][te] = f[iz][iy][ix];
      } else {
        sE[(BYC ? 0 : c) * 8 + t][te] = f[iz][iy][ix];
      }
    }
  };
  auto sum_up = [&](int c) {
#pragma unroll
    for (int s = 0; s < NPT; s++) {
      double v[8];
#pragma unroll
      for (int t = 0; t < 8; t++) {
        const unsigned e = (t & 1) ? eo[s][t >> 1] >> 16 : eo[s][t >> 1] & 0xffffu;
        v[t] = sE[(BYC ? 0 : (SPLIT ? c0 : c)) * 8 + t][e];
      }
      // element pairs across z first (every order of the 8 is as good)
      w[s][c] = ((v[0] + v[4]) + (v[1] + v[5])) + ((v[2] + v[6]) + (v[3] + v[7]));
    }
  };
  // w = A v for v in sP: element contributions, then node sums
  auto apply = [&]() {
    __syncthreads();
    const int sy = L.nx, sz = L.nx * L.ny;
    if constexpr (NP == 1024) {
      // with 128 registers a thread, LDS addresses and the products of the
      // moduli and the grid scales are formed again in every apply, not kept
      // across the loop
      asm volatile("" : "+v"(lam0), "+v"(mu0), "+v"(eb));
#pragma unroll
      for (int s = 0; s < NPT; s++)
#pragma unroll
        for (int t = 0; t < 4; t++) asm volatile("" : "+v"(eo[s][t]));
    }
    if constexpr (SPLIT) {
      if (has_e) {
        // the wave's component leads: axes and components rotated by c0
        const int st0 = c0 == 0 ? 1 : (c0 == 1 ? sy : sz), st1 = c0 == 0 ? sy : (c0 == 1 ? sz : 1),
                  st2 = c0 == 0 ? sz : (c0 == 1 ? 1 : sy);
        double v[3][2][2][2], f[2][2][2];
#pragma unroll
        for (int c = 0; c < 3; c++) {
          const double* P = &sP[c0 + c < 3 ? c0 + c : c0 + c - 3][eb];
#pragma unroll
          for (int t = 0; t < 8; t++)
            v[c][t >> 2][(t >> 1) & 1][t & 1] = P[(t & 1) * st0 + ((t >> 1) & 1) * st1 + (t >> 2) * st2];
        }
        hex_force_lead(v, lam0, mu0, hsr, f);
        hand_over(f, 0);
      }
      __syncthreads();
      sum_up(0);
    } else if constexpr (NC == 3) {
      double U[3][8];
      if (has_e) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
          double u[2][2][2];
#pragma unroll
          for (int t = 0; t < 8; t++)
            u[t >> 2][(t >> 1) & 1][t & 1] = sP[c][eb + (t & 1) + ((t >> 1) & 1) * sy + (t >> 2) * sz];
          hex_modes(u, U[c]);
        }
      }
      auto comp = [&](auto cc) {
        constexpr int c = decltype(cc)::value;
        if (BYC && c > 0) __syncthreads();  // the last component's contributions have been read
        if (has_e) {
          double f[2][2][2];
          hex_force_of<c>(U, lam0, mu0, hsr, f);
          hand_over(f, c);
        }
        if constexpr (BYC) {
          __syncthreads();
          sum_up(c);
        }
      };
      comp(std::integral_constant<int, 0>());
      comp(std::integral_constant<int, 1>());
      comp(std::integral_constant<int, 2>());
      if constexpr (!BYC) {
        __syncthreads();
#pragma unroll
        for (int c = 0; c < 3; c++) sum_up(c);
      }
    } else {
      if (has_e) {
        double v[2][2][2], f[2][2][2];
#pragma unroll
        for (int t = 0; t < 8; t++)
          v[t >> 2][(t >> 1) & 1][t & 1] = sP[0][eb + (t & 1) + ((t >> 1) & 1) * sy + (t >> 2) * sz];
        pf_element(v, pm, pk, 1.0 / L.hx, 1.0 / L.hy, 1.0 / L.hz, f);
        hand_over(f, 0);
      }
      __syncthreads();
      sum_up(0);
    }
  };

  // initial residual r = f - A x (masked)
  apply();
  double acc[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int s = 0; s < NPT; s++)
#pragma unroll
    for (int c = 0; c < NCT; c++) {
      acc[2] = fma(r[s][c], r[s][c], acc[2]);  // r still holds f
      r[s][c] = (qn[s] < 0 || ((dm[s] >> c) & 1)) ? 0.0 : r[s][c] - w[s][c];
      acc[0] = fma(r[s][c], mul_nc(r[s][c], iD[s][c]), acc[0]);
      acc[1] = fma(r[s][c], r[s][c], acc[1]);
    }
  block_sum_all<NW, 3>(acc, sh, half);
  // the phase-field smoother resets fd_norm on every call (phase_field_pcg.cpp:163)
  if (NC == 1 && tid == 0) a.scal[S_FF] = acc[2];
  double rz = acc[0], rr = acc[1], beta = 0.0, pw = 0.0, alpha = 0.0;

  for (int it = 0; it < a.NB; it++) {
    // pass A: p = z + beta p (first: p = z); w = A p; p.w
#pragma unroll
    for (int s = 0; s < NPT; s++)
#pragma unroll
      for (int c = 0; c < NCT; c++) {
        if (PLDS && qn[s] < 0) continue;
        double& pl = own(s, c);
        const double z = mul_nc(r[s][c], iD[s][c]);
        const double pv = it == 0 ? z : fma(beta, PLDS ? pl : p[PLDS ? 0 : s][c], z);
        if constexpr (!PLDS) p[s][c] = pv;
        pl = pv;
      }
    apply();
    double pa[1] = {0.0};
#pragma unroll
    for (int s = 0; s < NPT; s++)
#pragma unroll
      for (int c = 0; c < NCT; c++) {
        if (PLDS && qn[s] < 0) continue;
        pa[0] = fma(PLDS ? own(s, c) : p[PLDS ? 0 : s][c], w[s][c], pa[0]);
      }
    block_sum_all<NW, 1>(pa, sh, half);
    pw = pa[0];
    alpha = rz / pw;
    // pass B: x += alpha p; r -= alpha w; mask; r.z, r.r
    double ab[2] = {0.0, 0.0};
#pragma unroll
    for (int s = 0; s < NPT; s++)
#pragma unroll
      for (int c = 0; c < NCT; c++) {
        if (PLDS && qn[s] < 0) continue;
        xval(s, c) = fma(alpha, PLDS ? own(s, c) : p[PLDS ? 0 : s][c], xval(s, c));
        double rv = fma(-alpha, w[s][c], r[s][c]);
        if ((dm[s] >> c) & 1) rv = 0.0;
        r[s][c] = rv;
        ab[0] = fma(rv, mul_nc(rv, iD[s][c]), ab[0]);
        ab[1] = fma(rv, rv, ab[1]);
      }
    block_sum_all<NW, 2>(ab, sh, half);
    beta = ab[0] / rz;
    rz = ab[0];
    rr = ab[1];
  }

#pragma unroll
  for (int s = 0; s < NPT; s++) {
    if (qn[s] < 0) continue;
#pragma unroll
    for (int c = 0; c < NCT; c++) {
      const size_t o = (size_t)(SPLIT ? c0 : c) * N + qn[s];
      a.x[o] = (TIO)xval(s, c);
      if (a.r) a.r[o] = (TIO)r[s][c];
      if (a.NB > 0 && a.p) {
        a.p[o] = (TIO)(PLDS ? own(s, c) : p[PLDS ? 0 : s][c]);
        a.w[o] = (TIO)w[s][c];
      }
    }
  }
  if (tid == 0) {
    a.scal[S_RZ] = rz;
    a.scal[S_RR] = rr;
    if (a.NB > 0) {
      a.scal[S_BETA] = beta;
      a.scal[S_PW] = pw;
      a.scal[S_ALPHA] = alpha;
    }
  }
}

template <class Lay, class TIO>
__global__ __launch_bounds__(Lay::THREADS) void small_pcg_kernel(const SmallArgsT<TIO> a) {
  small_pcg_body<Lay, TIO>(a);
}
template <class Lay, class TIO>
struct SmallPcgK {
  using Args = SmallArgsT<TIO>;
  static constexpr int NT = Lay::THREADS, MINW = 1;
  static dim3 block() { return dim3(Lay::THREADS); }
  __device__ __forceinline__ static void run(const Args& a, const Blk&) { small_pcg_body<Lay, TIO>(a); }
};
template <class Lay, class TIO>
static void launch_small_layout(hipStream_t s, const SmallArgsT<TIO>& a) {
  if (record<SmallPcgK<Lay, TIO>>(dim3(1), a)) return;
  small_pcg_kernel<Lay, TIO><<<dim3(1), dim3(Lay::THREADS), 0, s>>>(a);
}
template <int NC, class TIO>
static void launch_small(hipStream_t s, const LevelGeom& L, const SmallArgsT<TIO>& a) {
  const long n = (long)L.nx * L.ny * L.nz;
  const long e = (long)(L.nx - 1) * (L.ny - 1) * (L.nz - 1);
  if (n <= 128 && e <= 128)
    launch_small_layout<SmallLayout<NC, 128, 1, NC == 3>>(s, a);
  else if (n <= 256 && e <= 256)
    launch_small_layout<SmallLayout<NC, 256, 1, NC == 3>>(s, a);
  else if (n <= 1024 && e <= 512)
    launch_small_layout<SmallLayout<NC, 512, 2, false>>(s, a);
  else
    launch_small_layout<SmallLayout<NC, 1024, 2, false>>(s, a);
}

// coarsest solve of the FP32 preconditioner: zero start, homogeneous
// Dirichlet values, FP64 iteration on float right-hand side and result
void launch_small_pcg_u_f32(hipStream_t s, const LevelGeom& L, const double* Ke, const double* Ge, float* x,
                            const float* b, const double* invD, int NB, double* scal) {
  SmallArgsT<float> a{};
  a.L = L;
  a.Ke = Ke;
  a.Ge = Ge;
  a.hs = HexScale<double>(L.hx, L.hy, L.hz);
  a.x = x;
  a.f = b;
  a.invD = invD;
  a.Ut = 0.0;
  a.NB = NB;
  a.scal = scal;
  launch_small<3, float>(s, L, a);
}

bool small_level(const LevelGeom& L) {
  const long n = (long)L.nx * L.ny * L.nz;
  const long e = (long)(L.nx - 1) * (L.ny - 1) * (L.nz - 1);
  return n <= SMALL_NODES && e <= SMALL_ELEMS && L.nx >= 2 && L.ny >= 2 && L.nz >= 2;
}

void launch_small_pcg_u(hipStream_t s, const LevelGeom& L, const double* Ke, const double* Ge, double* u,
                        const double* f, const double* invD, double* r, double* p, double* w, double Ut, int NB,
                        double* scal) {
  SmallArgs a{};
  a.L = L;
  a.Ke = Ke;
  a.Ge = Ge;
  a.hs = HexScale<double>(L.hx, L.hy, L.hz);
  a.x = u;
  a.f = f;
  a.invD = invD;
  a.r = r;
  a.p = p;
  a.w = w;
  a.Ut = Ut;
  a.NB = NB;
  a.scal = scal;
  launch_small<3, double>(s, L, a);
}

void launch_small_pcg_d(hipStream_t s, const LevelGeom& L, const double* H, const double* gc, double lc, double* d,
                        const double* fd, const double* invD, double* r, double* p, double* w, int NB, double* scal) {
  SmallArgs a{};
  a.L = L;
  a.H = H;
  a.gc = gc;
  a.lc = lc;
  a.rlc = 1.0 / lc;
  a.x = d;
  a.f = fd;
  a.invD = invD;
  a.r = r;
  a.p = p;
  a.w = w;
  a.NB = NB;
  a.scal = scal;
  launch_small<1, double>(s, L, a);
}

// ---------------------------------------------------------------------------
// image_MP on the device (image_input.cpp:120-142)
// ---------------------------------------------------------------------------
// gray level -> (K, G, gc) with the reference's integer-division
// interpolation between table rows, the same FP64 operations in the same
// order as the host restatement (no contraction), so results are identical
__global__ __launch_bounds__(256) void image_mp_kernel(size_t n, const unsigned char* __restrict__ img,
                                                       const MatTable* __restrict__ tab, double vs,
                                                       double* __restrict__ K, double* __restrict__ G,
                                                       double* __restrict__ gc, int* __restrict__ bad) {
#pragma clang fp contract(off)
  __shared__ int sg[MAT_MAX];
  __shared__ double sE[MAT_MAX], snu[MAT_MAX], sgc[MAT_MAX];
  const int nt = tab->n;
  for (int i = threadIdx.x; i < nt; i += blockDim.x) {
    sg[i] = tab->gray[i];
    sE[i] = tab->E[i];
    snu[i] = tab->nu[i];
    sgc[i] = tab->gc[i];
  }
  __syncthreads();
  for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x) {
    const int x = img[q];
    int pos = -1;
    // findPosition (csv_reader.cpp:74-82)
    for (int i = 0; i < nt - 1; ++i)
      if (x >= sg[i] && x <= sg[i + 1]) {
        pos = i;
        break;
      }
    if (pos < 0 || sg[pos + 1] == sg[pos]) {
      bad[0] = 1;
      continue;
    }
    const int fac = (x - sg[pos]) / (sg[pos + 1] - sg[pos]);
    double E = sE[pos] + (double)fac * (sE[pos + 1] - sE[pos]);
    const double nu = snu[pos] + (double)fac * (snu[pos + 1] - snu[pos]);
    gc[q] = sgc[pos] + (double)fac * (sgc[pos + 1] - sgc[pos]);
    E = vs * E;
    K[q] = 1.0 / (3.0 * (1.0 - 2.0 * nu)) * E;
    G[q] = 1.0 / (2.0 * (1.0 + nu)) * E;
  }
}
void launch_image_mp(hipStream_t s, size_t n, const unsigned char* img, const MatTable* tab, double vs, double* K,
                     double* G, double* gc, int* bad) {
  hipLaunchKernelGGL(image_mp_kernel, dim3(pw_blocks(n)), dim3(256), 0, s, n, img, tab, vs, K, G, gc, bad);
}

// ---------------------------------------------------------------------------
// Transfers (multigrid_intergrid.cpp)
// ---------------------------------------------------------------------------
// solution_injection + Dirichlet_BD + copy to uold (multigrid_intergrid.cpp:25-121)
__device__ __forceinline__ void inject_body(const LevelGeom& Lc, const LevelGeom& Lf, int ncomp,
                                            const double* __restrict__ uf, double* __restrict__ uc,
                                            double* __restrict__ ucold, int apply_bc, double Ut, const Blk& bk) {
  const int i = bk.x * 64 + threadIdx.x;
  const int j = bk.y * 4 + threadIdx.y, k = bk.z;
  if (i >= Lc.nx || j >= Lc.ny) return;
  const size_t Nc = Nof(Lc), Nf = Nof(Lf);
  const size_t qc = nidx(Lc, i, j, k), qf = nidx(Lf, 2 * i, 2 * j, 2 * k);
  const int dm = apply_bc ? dir_mask(Lc, i, j, k) : 0;
  for (int c = 0; c < ncomp; c++) {
    double v = uf[c * Nf + qf];
    if ((dm >> c) & 1) v = (c == 2 && (dm & 8)) ? Ut : 0.0;
    uc[c * Nc + qc] = v;
    if (ucold) ucold[c * Nc + qc] = v;
  }
}
__global__ __launch_bounds__(256) void inject_kernel(const LevelGeom Lc, const LevelGeom Lf, int ncomp,
                                                     const double* __restrict__ uf, double* __restrict__ uc,
                                                     double* __restrict__ ucold, int apply_bc, double Ut) {
  inject_body(Lc, Lf, ncomp, uf, uc, ucold, apply_bc, Ut, Blk::hw());
}
struct InjectK {
  struct Args {
    LevelGeom Lc;
    LevelGeom Lf;
    int ncomp;
    const double* uf;
    double* uc;
    double* ucold;
    int apply_bc;
    double Ut;
  };
  static constexpr int NT = 256, MINW = 1;
  static dim3 block() { return dim3(64, 4); }
  __device__ __forceinline__ static void run(const Args& a, const Blk& bk) {
    inject_body(a.Lc, a.Lf, a.ncomp, a.uf, a.uc, a.ucold, a.apply_bc, a.Ut, bk);
  }
};
void launch_inject(hipStream_t s, const LevelGeom& Lc, const LevelGeom& Lf, int ncomp, const double* uf,
                   double* uc, double* ucold, int apply_bc, double Ut) {
  if (record<InjectK>(dim3((Lc.nx + 63) / 64, (Lc.ny + 3) / 4, Lc.nz), {Lc, Lf, ncomp, uf, uc, ucold, apply_bc, Ut}))
    return;
  hipLaunchKernelGGL(inject_kernel, dim3((Lc.nx + 63) / 64, (Lc.ny + 3) / 4, Lc.nz), dim3(64, 4), 0, s, Lc, Lf,
                     ncomp, uf, uc, ucold, apply_bc, Ut);
}

// 2-D blocks of 64 x 4 threads over (x, y), one z-plane per blockIdx.z
constexpr int XB = 64, YB = 4;

// coarsen_f_standard_routine (multigrid_intergrid.cpp:124-342): full weighting
// with out-of-range neighbours counted as 0, written in its separable form
// (1-D weights 1/2, 1, 1/2 per axis)
// one thread per node, x fastest: (i, j, k) of node q of a level
__device__ __forceinline__ void node_ijk(const LevelGeom& L, unsigned q, int& i, int& j, int& k) {
  const unsigned plane = (unsigned)L.nx * (unsigned)L.ny;
  const unsigned kk = q / plane, rem = q - kk * plane;
  const unsigned jj = rem / (unsigned)L.nx;
  i = (int)(rem - jj * (unsigned)L.nx);
  j = (int)jj;
  k = (int)kk;
}

// f_c = A u_c + R r_f (Fic = A u_c).  START: also the residual that the coarse
// smoother starts from.  With u_c the injected iterate, r_c = f_c - A u_c is
// R r_f itself (zero on Dirichlet DOFs), so r_c, z_c = r_c / D and the sums r.z
// and r.r come with the restriction and the smoother's own residual pass (and
// its Dirichlet launch) is left out.  Onto 129^3 nodes: restriction
// 142 -> 219 us for a residual of 98 us left out; 65^3: 20 -> 37 for 32 + 4;
// 33^3 and 17^3: 5.4 -> 9 for 10 to 13 + 4.
// One component of a node per thread; with START at most RESTRICT_BLOCKS blocks, whose
// partials the last one adds.
constexpr int RESTRICT_BLOCKS = 1024;
template <int NC, bool START>
__device__ __forceinline__ void restrict_body(const LevelGeom& Lc, const LevelGeom& Lf, const double* __restrict__ rf,
                                              const double* __restrict__ Fic, double* __restrict__ fc,
                                              double* __restrict__ rc, double* __restrict__ zc,
                                              const double* __restrict__ invD, const Reduce& Rd, const Blk& bk) {
  // one component of a node per thread (see mix_restrict_body)
  const unsigned Nc = (unsigned)Nof(Lc);
  const size_t Nf = Nof(Lf);
  double sum[2] = {0.0, 0.0};
  for (unsigned t = bk.x * 256 + threadIdx.x; t < NC * Nc; t += bk.gx * 256) {
    const int c = NC == 1 ? 0 : (t >= 2 * Nc ? 2 : (t >= Nc ? 1 : 0));
    int i, j, k;
    node_ijk(Lc, t - c * Nc, i, j, k);
    const double fi = Fic[t], iD = START ? invD[t] : 0.0;
    const int dm = START && NC == 3 ? dir_mask_flat(Lc, i, j, k) : 0;
    const Restrict27<double> R(Lf, i, j, k);
    const double acc = R(rf + c * Nf);
    fc[t] = fi + acc;
    if constexpr (START) {
      const double r = ((dm >> c) & 1) ? 0.0 : acc;
      const double z = r * iD;
      rc[t] = r;
      zc[t] = z;
      sum[0] += r * z;
      sum[1] += r * r;
    }
  }
  if constexpr (START) {
    double* scal = Rd.scal;
    reduce_finalize<RED_SUM, 2>(bk, sum, Rd, 0.0, [=](double (&s)[2]) {
      scal[S_RZ] = s[0];
      scal[S_RR] = s[1];
    });
  }
}
struct RestrictArgs {
  LevelGeom Lc;
  LevelGeom Lf;
  const double* rf;
  const double* Fic;
  double* fc;
  double* rc;
  double* zc;
  const double* invD;
  Reduce R;
};
template <int NC, bool START>
__global__ __launch_bounds__(256) void restrict_kernel(const RestrictArgs a) {
  restrict_body<NC, START>(a.Lc, a.Lf, a.rf, a.Fic, a.fc, a.rc, a.zc, a.invD, a.R, Blk::hw());
}
template <int NC, bool START>
struct RestrictK {
  using Args = RestrictArgs;
  static constexpr int NT = 256, MINW = 1;
  static dim3 block() { return dim3(256); }
  __device__ __forceinline__ static void run(const Args& a, const Blk& bk) {
    restrict_body<NC, START>(a.Lc, a.Lf, a.rf, a.Fic, a.fc, a.rc, a.zc, a.invD, a.R, bk);
  }
};
void launch_restrict(hipStream_t s, const LevelGeom& Lc, const LevelGeom& Lf, int ncomp, const double* rf,
                     const double* Fic, double* fc, double* rc, double* zc, const double* invD, const Reduce& R) {
  const RestrictArgs a{Lc, Lf, rf, Fic, fc, rc, zc, invD, R};
  const unsigned nb = (unsigned)((ncomp * Nof(Lc) + 255) / 256);
  auto go = [&](auto nc, auto start) {
    constexpr int NC = decltype(nc)::value;
    constexpr bool START = decltype(start)::value;
    const dim3 g(START ? std::min<unsigned>(nb, RESTRICT_BLOCKS) : nb);
    if (record<RestrictK<NC, START>>(g, a)) return;
    hipLaunchKernelGGL((restrict_kernel<NC, START>), g, dim3(256), 0, s, a);
  };
  if (ncomp == 3) {
    if (rc)
      go(std::integral_constant<int, 3>(), std::true_type());
    else
      go(std::integral_constant<int, 3>(), std::false_type());
  } else {
    if (rc)
      go(std::integral_constant<int, 1>(), std::true_type());
    else
      go(std::integral_constant<int, 1>(), std::false_type());
  }
}

// e_c = u_c - u_c,old (the coarse-grid correction, multigrid_intergrid.cpp:484-518)
__device__ __forceinline__ void diff_body(size_t n, const double* __restrict__ a, const double* __restrict__ b,
                                          double* __restrict__ e, const Blk& bk) {
  for (size_t q = (size_t)bk.x * blockDim.x + threadIdx.x; q < n; q += (size_t)bk.gx * blockDim.x)
    e[q] = a[q] - b[q];
}
__global__ void diff_kernel(size_t n, const double* __restrict__ a, const double* __restrict__ b,
                            double* __restrict__ e) {
  diff_body(n, a, b, e, Blk::hw());
}
struct DiffK {
  struct Args {
    size_t n;
    const double* a;
    const double* b;
    double* e;
  };
  static constexpr int NT = 256, MINW = 1;
  static dim3 block() { return dim3(256); }
  __device__ __forceinline__ static void run(const Args& a, const Blk& bk) {
    diff_body(a.n, a.a, a.b, a.e, bk);
  }
};

// refine_standard_routine + Dirichlet_BD (multigrid_intergrid.cpp:416-549):
// trilinear interpolation of the correction e_c, one writer per fine node,
// two x-adjacent fine nodes per thread (ProlongPair)
__device__ __forceinline__ void prolong_body(const LevelGeom& Lf, const LevelGeom& Lc, int ncomp,
                                             double* __restrict__ uf, const double* __restrict__ e,
                                             const double* __restrict__ eold, int apply_bc, double Ut,
                                             const Blk& bk) {
  const unsigned q = bk.x * 256 + threadIdx.x;
  if (q >= (unsigned)prolong_pairs(Lf)) return;
  int ip, y, z;
  bool has1;
  pair_ijk(Lf, q, ip, has1, y, z);
  const size_t Nc = Nof(Lc), Nf = Nof(Lf);
  // separable trilinear weights (0.5 on each odd axis); identical to the
  // reference's averages of 2, 4 or 8 corrections up to rounding order
  const ProlongPair<double> Pr(Lc, ip, has1, y, z);
  const int x = 2 * ip;
  const unsigned of = nid32(Lf, x, y, z) * 8u;
  const int dm0 = apply_bc ? dir_mask_flat(Lf, x, y, z) : 0;
  const int dm1 = apply_bc ? dir_mask_flat(Lf, has1 ? x + 1 : x, y, z) : 0;
  auto comps = [&](auto nc) {
    constexpr int NC = decltype(nc)::value;
    double c0[NC], c1[NC];
    if (eold) {
#pragma unroll
      for (int c = 0; c < NC; c++) Pr.diff(e + c * Nc, eold + c * Nc, c0[c], c1[c]);
    } else {
#pragma unroll
      for (int c = 0; c < NC; c++) Pr(e + c * Nc, c0[c], c1[c]);
    }
#pragma unroll
    for (int c = 0; c < NC; c++) {
      double v = ldo(uf + c * Nf, of) + c0[c];
      if ((dm0 >> c) & 1) v = (c == 2 && (dm0 & 8)) ? Ut : 0.0;
      sto(uf + c * Nf, of, v);
      if (has1) {
        double v1 = ldo(uf + c * Nf, of + 8u) + c1[c];
        if ((dm1 >> c) & 1) v1 = (c == 2 && (dm1 & 8)) ? Ut : 0.0;
        sto(uf + c * Nf, of + 8u, v1);
      }
    }
  };
  if (ncomp == 3)
    comps(std::integral_constant<int, 3>());
  else
    comps(std::integral_constant<int, 1>());
}
__global__ __launch_bounds__(256) void prolong_kernel(const LevelGeom Lf, const LevelGeom Lc, int ncomp,
                                                      double* __restrict__ uf, const double* __restrict__ e,
                                                      const double* __restrict__ eold, int apply_bc, double Ut) {
  prolong_body(Lf, Lc, ncomp, uf, e, eold, apply_bc, Ut, Blk::hw());
}
struct ProlongK {
  struct Args {
    LevelGeom Lf;
    LevelGeom Lc;
    int ncomp;
    double* uf;
    const double* e;
    const double* eold;
    int apply_bc;
    double Ut;
  };
  static constexpr int NT = 256, MINW = 1;
  static dim3 block() { return dim3(256); }
  __device__ __forceinline__ static void run(const Args& a, const Blk& bk) {
    prolong_body(a.Lf, a.Lc, a.ncomp, a.uf, a.e, a.eold, a.apply_bc, a.Ut, bk);
  }
};
void launch_prolong(hipStream_t s, const LevelGeom& Lf, const LevelGeom& Lc, int ncomp, double* uf,
                    const double* uc, const double* ucold, int apply_bc, double Ut, double* scratch) {
  const size_t n = (size_t)ncomp * Nof(Lc);
  const bool own_diff = Nof(Lf) <= PROLONG_DIFF_NODES;
  const double* e = own_diff ? uc : scratch;
  const double* eold = own_diff ? ucold : nullptr;
  const dim3 g((unsigned)((prolong_pairs(Lf) + 255) / 256));
  if (!own_diff && !record<DiffK>(dim3(pw_blocks(n)), {n, uc, ucold, scratch}))
    hipLaunchKernelGGL(diff_kernel, dim3(pw_blocks(n)), dim3(256), 0, s, n, uc, ucold, scratch);
  if (record<ProlongK>(g, {Lf, Lc, ncomp, uf, e, eold, apply_bc, Ut})) return;
  hipLaunchKernelGGL(prolong_kernel, g, dim3(256), 0, s, Lf, Lc, ncomp, uf, e, eold, apply_bc, Ut);
}

// ---------------------------------------------------------------------------
// Per-element Gauss-point kernels on the finest level
// ---------------------------------------------------------------------------
__device__ __forceinline__ void load8(const LevelGeom& L, const double* f, int i, int j, int k,
                                      double (&v)[2][2][2]) {
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
      for (int c = 0; c < 2; c++) v[a][b][c] = f[nidx(L, i + c, j + b, k + a)];
}

struct Strain {
  double xx, yy, zz, xy, xz, yz;  // tensor components (xy = gamma_xy / 2)
};
__device__ __forceinline__ Strain strain_at(const double (&dx)[3][2][2], const double (&dy)[3][2][2],
                                            const double (&dz)[3][2][2], int gx, int gy, int gz) {
  Strain e;
  e.xx = dx[0][gz][gy];
  e.yy = dy[1][gz][gx];
  e.zz = dz[2][gy][gx];
  e.xy = 0.5 * (dx[1][gz][gy] + dy[0][gz][gx]);
  e.xz = 0.5 * (dx[2][gz][gy] + dz[0][gy][gx]);
  e.yz = 0.5 * (dy[2][gz][gx] + dz[1][gy][gx]);
  return e;
}
// epsilon_dev (mechanical_strain.cpp:47-61) and Phi_positive/negative
// (strain_history.cpp:134-159)
__device__ __forceinline__ double dev2(const Strain& e) {
  const double t = (1.0 / 3.0) * (e.xx + e.yy + e.zz);
  const double a = e.xx - t, b = e.yy - t, c = e.zz - t;
  return a * a + b * b + c * c + 2.0 * (e.xy * e.xy + e.xz * e.xz + e.yz * e.yz);
}
__device__ __forceinline__ double phi_pos(double K, double G, const Strain& e) {
  const double tr = e.xx + e.yy + e.zz;
  const double d2 = dev2(e);
  return (tr >= 0) ? 0.5 * K * tr * tr + G * d2 : G * d2;
}
__device__ __forceinline__ double phi_neg(double K, const Strain& e) {
  const double tr = e.xx + e.yy + e.zz;
  return (tr >= 0) ? 0.0 : 0.5 * K * tr * tr;
}

struct ElemArgs {
  const double* u;
  const double* K;
  const double* G;
  const double* d;
  const double* gc;
};

__device__ __forceinline__ void elem_grads(const LevelGeom& L, const double* u, int i, int j, int k,
                                           double (&dx)[3][2][2], double (&dy)[3][2][2], double (&dz)[3][2][2]) {
  const size_t N = Nof(L);
#pragma unroll
  for (int c = 0; c < 3; c++) {
    double v[2][2][2];
    load8(L, u + c * N, i, j, k, v);
    grad8(v, 1.0 / L.hx, 1.0 / L.hy, 1.0 / L.hz, dx[c], dy[c], dz[c]);
  }
}

// MP_choice_element + MP_element (material_selection.cpp:19-45, 67-81)
__global__ void flag_means_kernel(const LevelGeom L, const double* __restrict__ u, const double* __restrict__ K,
                                  const double* __restrict__ G, const double* __restrict__ d,
                                  signed char* __restrict__ flag, double* __restrict__ Ke, double* __restrict__ Ge,
                                  double small_k, int compute_flag) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y, k = blockIdx.z;
  if (i > L.nx - 2) return;
  double Kn[2][2][2], Gn[2][2][2], dn[2][2][2], Kg[2][2][2], Gg[2][2][2], dg[2][2][2];
  load8(L, K, i, j, k, Kn);
  load8(L, G, i, j, k, Gn);
  gp_mp(Kn, Kg);
  gp_mp(Gn, Gg);
  const size_t e = nidx(L, i, j, k);
  int fl;
  if (compute_flag) {
    double dx[3][2][2], dy[3][2][2], dz[3][2][2];
    elem_grads(L, u, i, j, k, dx, dy, dz);
    double tr = 0.0, pp = 0.0, pn = 0.0;
    for (int gz = 0; gz < 2; gz++)
      for (int gy = 0; gy < 2; gy++)
        for (int gx = 0; gx < 2; gx++) {
          const Strain s = strain_at(dx, dy, dz, gx, gy, gz);
          tr += s.xx + s.yy + s.zz;
          pp += phi_pos(Kg[gz][gy][gx], Gg[gz][gy][gx], s);
          pn += phi_neg(Kg[gz][gy][gx], s);
        }
    fl = 0;
    if (tr >= 0.0) fl = 0;
    if (tr < 0.0) fl = 1;
    if (pp < pn) fl = 2;
    flag[e] = (signed char)fl;
  } else {
    fl = flag[e];
  }
  load8(L, d, i, j, k, dn);
  gp_mp(dn, dg);
  double sK = 0.0, sG = 0.0;
  for (int gz = 0; gz < 2; gz++)
    for (int gy = 0; gy < 2; gy++)
      for (int gx = 0; gx < 2; gx++) {
        const double g = degr(dg[gz][gy][gx], small_k);
        sK += (fl == 0) ? g * Kg[gz][gy][gx] : Kg[gz][gy][gx];
        sG += (fl == 2) ? Gg[gz][gy][gx] : g * Gg[gz][gy][gx];
      }
  Ke[e] = 0.125 * sK;
  Ge[e] = 0.125 * sG;
}
void launch_flag_means(hipStream_t s, const LevelGeom& L, const double* u, const double* K, const double* G,
                       const double* d, signed char* flag, double* Ke, double* Ge, double small_k,
                       int compute_flag) {
  hipLaunchKernelGGL(flag_means_kernel, dim3((L.nx - 1 + 63) / 64, L.ny - 1, L.nz - 1), dim3(64), 0, s, L, u, K, G,
                     d, flag, Ke, Ge, small_k, compute_flag);
}

// strain_history (strain_history.cpp:162-210)
__global__ void strain_history_kernel(const LevelGeom L, const double* __restrict__ u, const double* __restrict__ K,
                                      const double* __restrict__ G, const double* __restrict__ gc,
                                      double* __restrict__ H, double lc, double u_prop) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y, k = blockIdx.z;
  if (i > L.nx - 2) return;
  double Kn[2][2][2], Gn[2][2][2], cn[2][2][2], Kg[2][2][2], Gg[2][2][2], cg[2][2][2];
  load8(L, K, i, j, k, Kn);
  load8(L, G, i, j, k, Gn);
  load8(L, gc, i, j, k, cn);
  gp_mp(Kn, Kg);
  gp_mp(Gn, Gg);
  gp_mp(cn, cg);
  double dx[3][2][2], dy[3][2][2], dz[3][2][2];
  elem_grads(L, u, i, j, k, dx, dy, dz);
  double tmp = 0.0;
  for (int gz = 0; gz < 2; gz++)
    for (int gy = 0; gy < 2; gy++)
      for (int gx = 0; gx < 2; gx++) {
        Strain s = strain_at(dx, dy, dz, gx, gy, gz);
        s.xx *= u_prop; s.yy *= u_prop; s.zz *= u_prop;
        s.xy *= u_prop; s.xz *= u_prop; s.yz *= u_prop;
        tmp += phi_pos(Kg[gz][gy][gx], Gg[gz][gy][gx], s) - 0.5 * cg[gz][gy][gx] / lc;
      }
  const double Ht = 0.125 * tmp;
  const size_t e = nidx(L, i, j, k);
  if (H[e] < Ht) H[e] = Ht;
}
void launch_strain_history(hipStream_t s, const LevelGeom& L, const double* u, const double* K, const double* G,
                           const double* gc, double* H, double lc, double u_prop) {
  hipLaunchKernelGGL(strain_history_kernel, dim3((L.nx - 1 + 63) / 64, L.ny - 1, L.nz - 1), dim3(64), 0, s, L, u,
                     K, G, gc, H, lc, u_prop);
}

// U_e (strain_history.cpp:86-131): min over Gauss points of sqrt(phi_c / W)
__global__ __launch_bounds__(256) void elastic_limit_kernel(const LevelGeom L, const double* __restrict__ u,
                                                            const double* __restrict__ K,
                                                            const double* __restrict__ G,
                                                            const double* __restrict__ gc, double lc,
                                                            const Reduce R) {
  const size_t ne = (size_t)(L.nx - 1) * (L.ny - 1) * (L.nz - 1);
  double m[1] = {1e10};
  for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < ne; q += (size_t)gridDim.x * blockDim.x) {
    const int i = (int)(q % (L.nx - 1));
    const size_t r = q / (L.nx - 1);
    const int j = (int)(r % (L.ny - 1));
    const int k = (int)(r / (L.ny - 1));
    double Kn[2][2][2], Gn[2][2][2], cn[2][2][2], Kg[2][2][2], Gg[2][2][2], cg[2][2][2];
    load8(L, K, i, j, k, Kn);
    load8(L, G, i, j, k, Gn);
    load8(L, gc, i, j, k, cn);
    gp_mp(Kn, Kg);
    gp_mp(Gn, Gg);
    gp_mp(cn, cg);
    double dx[3][2][2], dy[3][2][2], dz[3][2][2];
    elem_grads(L, u, i, j, k, dx, dy, dz);
    for (int gz = 0; gz < 2; gz++)
      for (int gy = 0; gy < 2; gy++)
        for (int gx = 0; gx < 2; gx++) {
          const Strain e = strain_at(dx, dy, dz, gx, gy, gz);
          const double Kv = Kg[gz][gy][gx], Gv = Gg[gz][gy][gx];
          const double tr = e.xx + e.yy + e.zz;
          const double sxx = Kv * tr + 2.0 * Gv * (e.xx - 1.0 / 3.0 * tr);
          const double syy = Kv * tr + 2.0 * Gv * (e.yy - 1.0 / 3.0 * tr);
          const double szz = Kv * tr + 2.0 * Gv * (e.zz - 1.0 / 3.0 * tr);
          const double W = 0.5 * (sxx * e.xx + syy * e.yy + szz * e.zz +
                                  2.0 * (2.0 * Gv) * (e.xy * e.xy + e.xz * e.xz + e.yz * e.yz));
          const double phic = 0.5 * cg[gz][gy][gx] / lc;
          const double ut = sqrt(phic / W);
          if (ut < m[0]) m[0] = ut;
        }
  }
  double* scal = R.scal;
  reduce_finalize<RED_MIN, 1>(m, R, 1e10, [=](double (&s)[1]) { scal[S_RED] = s[0]; });
}
void launch_elastic_limit(hipStream_t s, const LevelGeom& L, const double* u, const double* K, const double* G,
                          const double* gc, double lc, const Reduce& R) {
  const size_t ne = (size_t)(L.nx - 1) * (L.ny - 1) * (L.nz - 1);
  hipLaunchKernelGGL(elastic_limit_kernel, dim3(pw_blocks(ne)), dim3(256), 0, s, L, u, K, G, gc, lc, R);
}

// ---------------------------------------------------------------------------
// Coarse coefficients (material_coarse_element.cpp, image_input.cpp)
// ---------------------------------------------------------------------------
__global__ void elem_vr_kernel(const LevelGeom Lc, const LevelGeom Lf, const double* __restrict__ Hf,
                               double* __restrict__ Hc, int voigt_only) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y, k = blockIdx.z;
  if (i >= Lc.nx) return;
  const size_t qc = nidx(Lc, i, j, k);
  const bool inside = i <= Lc.nx - 2 && j <= Lc.ny - 2 && k <= Lc.nz - 2;
  double V = 0.0, Rm = 0.0;
  if (inside) {
    const int x = 2 * i, y = 2 * j, z = 2 * k;
    const double h0 = Hf[nidx(Lf, x, y, z)], h1 = Hf[nidx(Lf, x + 1, y, z)];
    const double h2 = Hf[nidx(Lf, x, y + 1, z)], h3 = Hf[nidx(Lf, x + 1, y + 1, z)];
    const double h4 = Hf[nidx(Lf, x, y, z + 1)], h5 = Hf[nidx(Lf, x + 1, y, z + 1)];
    const double h6 = Hf[nidx(Lf, x, y + 1, z + 1)], h7 = Hf[nidx(Lf, x + 1, y + 1, z + 1)];
    V = 0.125 * (h0 + h1 + h2 + h3 + h4 + h5 + h6 + h7);
    if (!voigt_only)
      Rm = 8. / (1. / h0 + 1. / h1 + 1. / h2 + 1. / h3 + 1. / h4 + 1. / h5 + 1. / h6 + 1. / h7);
  }
  if (voigt_only) {
    if (inside) Hc[qc] = V;
  } else {
    Hc[qc] = 0.5 * (0.5 * (V + Rm) + sqrt(V * Rm));
  }
}
void launch_elem_vr(hipStream_t s, const LevelGeom& Lc, const LevelGeom& Lf, const double* Hf, double* Hc,
                    int voigt_only) {
  hipLaunchKernelGGL(elem_vr_kernel, dim3((Lc.nx + 63) / 64, Lc.ny, Lc.nz), dim3(64), 0, s, Lc, Lf, Hf, Hc,
                     voigt_only);
}

// voight / reuss / coarse_VR (image_input.cpp:144-273)
__global__ void nodal_vr_kernel(const LevelGeom Lc, const LevelGeom Lf, const double* __restrict__ M,
                                double* __restrict__ Mc) {
  const int ic = blockIdx.x * blockDim.x + threadIdx.x;
  const int jc = blockIdx.y, kc = blockIdx.z;
  if (ic >= Lc.nx) return;
  const int x = 2 * ic, y = 2 * jc, z = 2 * kc;
  const int xm = max(x - 1, 0), xp = min(x + 1, Lf.nx - 1);
  const int ym = max(y - 1, 0), yp = min(y + 1, Lf.ny - 1);
  const int zm = max(z - 1, 0), zp = min(z + 1, Lf.nz - 1);
  const int P[27][3] = {{xm, ym, zm}, {xm, ym, zp}, {xm, yp, zm}, {xm, yp, zp}, {xp, ym, zm}, {xp, ym, zp},
                        {xp, yp, zm}, {xp, yp, zp}, {xm, ym, z},  {xm, yp, z},  {xp, ym, z},  {xp, yp, z},
                        {xm, y, zm},  {xm, y, zp},  {xp, y, zm},  {xp, y, zp},  {x, ym, zm},  {x, ym, zp},
                        {x, yp, zm},  {x, yp, zp},  {x, y, zm},   {x, y, zp},   {x, ym, z},   {x, yp, z},
                        {xm, y, z},   {xp, y, z},   {x, y, z}};
  double sv = 0.0, sr = 0.0;
  for (int t = 0; t < 27; t++) {
    const double v = M[nidx(Lf, P[t][0], P[t][1], P[t][2])];
    sv += v;
    sr += 1. / v;
  }
  const double V = 1.0 / 27.0 * sv;
  const double R = 27.0 / sr;
  Mc[nidx(Lc, ic, jc, kc)] = 0.5 * (0.5 * (V + R) + sqrt(V * R));
}
void launch_nodal_vr(hipStream_t s, const LevelGeom& Lc, const LevelGeom& Lf, const double* Mf, double* Mc) {
  hipLaunchKernelGGL(nodal_vr_kernel, dim3((Lc.nx + 63) / 64, Lc.ny, Lc.nz), dim3(64), 0, s, Lc, Lf, Mf, Mc);
}

// fd_h (phase_field_right_hand_side.cpp:14-47) as a node gather
__global__ void fd_h_kernel(const LevelGeom L, const double* __restrict__ H, double* __restrict__ fd) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y, k = blockIdx.z;
  if (i >= L.nx) return;
  const double wg = 0.125 * L.hx * L.hy * L.hz;
  const double S = (GA + GB) * (GA + GB) * (GA + GB);  // sum_g N_a(g)
  double acc = 0.0;
  for (int dz = 1; dz >= 0; dz--)
    for (int dy = 1; dy >= 0; dy--)
      for (int dx = 1; dx >= 0; dx--) {
        const int ei = i - dx, ej = j - dy, ek = k - dz;
        if (ei < 0 || ej < 0 || ek < 0 || ei > L.nx - 2 || ej > L.ny - 2 || ek > L.nz - 2) continue;
        acc += wg * 2.0 * H[nidx(L, ei, ej, ek)] * S;
      }
  fd[nidx(L, i, j, k)] = acc;
}
void launch_fd_h(hipStream_t s, const LevelGeom& L, const double* H, double* fd) {
  hipLaunchKernelGGL(fd_h_kernel, dim3((L.nx + 63) / 64, L.ny, L.nz), dim3(64), 0, s, L, H, fd);
}

// externe_force_sum (mechanical_right_hnd.cpp:40-59)
__global__ __launch_bounds__(256) void top_sum_kernel(const LevelGeom L, const double* __restrict__ fz,
                                                      const Reduce R) {
  const size_t plane = (size_t)L.nx * L.ny;
  const size_t base = (size_t)(L.nz - 1) * plane;
  double a[1] = {0.0};
  for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < plane; q += (size_t)gridDim.x * blockDim.x)
    a[0] += fz[base + q];
  double* scal = R.scal;
  reduce_finalize<RED_SUM, 1>(a, R, 0.0, [=](double (&s)[1]) { scal[S_RED] = s[0]; });
}
void launch_top_sum(hipStream_t s, const LevelGeom& L, const double* fz, const Reduce& R) {
  const size_t plane = (size_t)L.nx * L.ny;
  hipLaunchKernelGGL(top_sum_kernel, dim3(pw_blocks(plane)), dim3(256), 0, s, L, fz, R);
}

// delta_d_max / d_max (phase_field_max_search.cpp:17-53): max(0, max(a - b))
__global__ __launch_bounds__(256) void max_diff_kernel(size_t n, const double* __restrict__ a,
                                                       const double* __restrict__ b, const Reduce R) {
  double m[1] = {0.0};
  for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x) {
    const double v = b ? a[q] - b[q] : a[q];
    if (m[0] < v) m[0] = v;
  }
  double* scal = R.scal;
  reduce_finalize<RED_MAX, 1>(m, R, 0.0, [=](double (&s)[1]) { scal[S_RED] = s[0]; });
}
void launch_max_diff(hipStream_t s, size_t n, const double* a, const double* b_or_null, const Reduce& R) {
  hipLaunchKernelGGL(max_diff_kernel, dim3(pw_blocks(n)), dim3(256), 0, s, n, a, b_or_null, R);
}

// stiffness contrast of a nodal modulus field: max(a) into scal[S_RED] and
// max(1/a) over a > 0 into scal[S_SCRATCH] (a = 0 nodes are the zero-node
// rule's, not a phase)
__global__ __launch_bounds__(256) void contrast_kernel(size_t n, const double* __restrict__ a, const Reduce R) {
  double m[2] = {0.0, 0.0};
  for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x) {
    const double v = a[q];
    if (m[0] < v) m[0] = v;
    if (v > 0.0 && m[1] < 1.0 / v) m[1] = 1.0 / v;
  }
  double* scal = R.scal;
  reduce_finalize<RED_MAX, 2>(m, R, 0.0, [=](double (&s)[2]) {
    scal[S_RED] = s[0];
    scal[S_SCRATCH] = s[1];
  });
}
void launch_contrast(hipStream_t s, size_t n, const double* a, const Reduce& R) {
  hipLaunchKernelGGL(contrast_kernel, dim3(pw_blocks(n)), dim3(256), 0, s, n, a, R);
}

// squared norm of ncomp*N values into scal[S_RR] (grid_norm, pcg_utilities.cpp:35-58)
__global__ __launch_bounds__(256) void norm2_kernel(size_t n, const double* __restrict__ a, const Reduce R) {
  double m[1] = {0.0};
  for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x)
    m[0] += a[q] * a[q];
  double* scal = R.scal;
  reduce_finalize<RED_SUM, 1>(m, R, 0.0, [=](double (&s)[1]) { scal[S_RR] = s[0]; });
}
void launch_norm2(hipStream_t s, size_t n, const double* a, const Reduce& R) {
  hipLaunchKernelGGL(norm2_kernel, dim3(pw_blocks(n)), dim3(256), 0, s, n, a, R);
}

__global__ void flag_to_double_kernel(size_t n, const signed char* f, double* o) {
  for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x)
    o[q] = (double)f[q];
}
__global__ void double_to_flag_kernel(size_t n, const double* in, signed char* f) {
  for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x)
    f[q] = (signed char)in[q];
}
__device__ __forceinline__ void fill_body(size_t n, double* p, double v, const Blk& bk) {
  for (size_t q = (size_t)bk.x * blockDim.x + threadIdx.x; q < n; q += (size_t)bk.gx * blockDim.x)
    p[q] = v;
}
__global__ void fill_kernel(size_t n, double* p, double v) {
  fill_body(n, p, v, Blk::hw());
}
struct FillK {
  struct Args {
    size_t n;
    double* p;
    double v;
  };
  static constexpr int NT = 256, MINW = 1;
  static dim3 block() { return dim3(256); }
  __device__ __forceinline__ static void run(const Args& a, const Blk& bk) {
    fill_body(a.n, a.p, a.v, bk);
  }
};
void launch_flag_to_double(hipStream_t s, size_t n, const signed char* f, double* out) {
  hipLaunchKernelGGL(flag_to_double_kernel, dim3(pw_blocks(n)), dim3(256), 0, s, n, f, out);
}
void launch_double_to_flag(hipStream_t s, size_t n, const double* in, signed char* f) {
  hipLaunchKernelGGL(double_to_flag_kernel, dim3(pw_blocks(n)), dim3(256), 0, s, n, in, f);
}
void launch_fill(hipStream_t s, size_t n, double* p, double v) {
  if (record<FillK>(dim3(pw_blocks(n)), {n, p, v})) return;
  hipLaunchKernelGGL(fill_kernel, dim3(pw_blocks(n)), dim3(256), 0, s, n, p, v);
}

}  // namespace hpcr
