// The fused stage on tiles of one material (gfx950): the same stage as
// stage_tile of m2c_stage.h, bit for bit, for tiles whose cells and the two
// cells around them along each axis all hold one active material
// (k_tile_mixed), with linear reconstruction on a uniform mesh and an HLLC,
// Roe or LLF flux.  That is nearly every tile of a run.
#pragma once
#include "m2c_exactdiv.h"
#include "m2c_stage.h"

namespace m2c {

// Limited slopes of a cell from the one-sided differences d0, d1 along an axis,
// with the coefficients of a uniform mesh, A = B = 1 and (van Albada) K = 2: lim_gmm and lim_va with the multiplications by one left out.
// The divisions of the five components are formed side by side, and not at
// all where no lane of the wave has a slope to limit.
__device__ __forceinline__ void limited(const Scheme& s, const double* d0, const double* d1, double* h) {
  if (s.limiter == M2CX_LIM_VANALBADA) {
    bool z[5], any = false;
#pragma unroll
    for (int p = 0; p < 5; p++) {
      const double pr = d0[p] * d1[p];
      z[p] = (pr <= 0) | (fabs(pr) < 1e-16);
      any |= !z[p];
      h[p] = 0.0;
    }
    if (any) {
      // where a slope is formed d0 d1 >= 1e-16, so that a + b >= 2e-16 and the
      // numerator d0 d1 (d0 + d1) >= 2e-24: with a + b <= 2^600 the quotient is
      // in range
      bool ok = true;
#pragma unroll
      for (int p = 0; p < 5; p++) {
        const double a = d0[p] * d0[p], b = d1[p] * d1[p], n = d1[p] * a + d0[p] * b;
        const double r = Recip(a + b).quot(n);
        ok &= z[p] | (a + b <= 0x1p600);
        h[p] = z[p] ? 0.0 : r;
      }
      if (!__all(ok)) {
#pragma unroll
        for (int p = 0; p < 5; p++) {
          const double a = d0[p] * d0[p], b = d1[p] * d1[p];
          const double r = (d1[p] * a + d0[p] * b) / (a + b);
          h[p] = z[p] ? 0.0 : r;
        }
      }
    }
  } else if (s.limiter == M2CX_LIM_GENERALIZED_MINMOD) {
#pragma unroll
    for (int p = 0; p < 5; p++) h[p] = lim_gmm(1.0, 1.0, s.gmm, d0[p], d1[p]);
  } else {
#pragma unroll
    for (int p = 0; p < 5; p++) h[p] = 0.5 * (d0[p] + d1[p]);
  }
}

// half the slopes, from the cell's state v and its neighbours'
__device__ __forceinline__ void half_slopes(const Scheme& s, const double* v, const double* vm, const double* vp,
                                            double* h) {
  double d0[5], d1[5];
#pragma unroll
  for (int p = 0; p < 5; p++) {
    d0[p] = v[p] - vm[p];
    d1[p] = vp[p] - v[p];
  }
  limited(s, d0, d1, h);
#pragma unroll
  for (int p = 0; p < 5; p++) h[p] *= 0.5;
}

// The cell value where a face state fails CheckState or would be clipped
// (face_state); returns bit 0 fail, bit 1 fail that clipping would not mend.
// The tests are combined without short cuts: a branch each would cost more.
__device__ __forceinline__ int keep_or_revert(const DevEos& E, const double* v, double* f) {
  if (E.type == M2CX_EOS_DUMMY) return 0;
  bool bad = false;
#pragma unroll
  for (int p = 0; p < 5; p++) bad |= !(fabs(f[p]) <= DBL_MAX);
  if (E.type == M2CX_EOS_MG) bad |= eos_check(E, f[0], f[4]);
  else bad |= (f[0] <= 0.0) | (f[4] + E.pc <= 0.0);
  const bool clip = (f[0] < E.rhomin) | (f[4] < E.pmin) | (f[0] > E.rhomax) | (f[4] > E.pmax);
  if (bad | clip) {
#pragma unroll
    for (int p = 0; p < 5; p++) f[p] = v[p];
  }
  return (bad ? 1 : 0) | ((bad & !clip) ? 2 : 0);
}

// The cell value q0 and half the limited slopes h of a cell along axis D in the
// scheme's reconstruction variables (recon_slope; uniform mesh, one material;
// x, y, z order).  v is the cell's state, vm and vp its neighbours'.  Returns
// whether the eigenvectors exist (c^2 >= 0).
__device__ __forceinline__ bool slopes_in_vars(const DevEos& E, const Scheme& s, int D, const double* v,
                                               const double* vm, const double* vp, double* q0, double* h) {
  const int vtype = s.var_type;
  const bool cons = (vtype == M2CX_VAR_CONSERVATIVE || vtype == M2CX_VAR_CONSERVATIVE_CHARACTERISTIC);
  const bool chr = vtype != M2CX_VAR_CONSERVATIVE;
  double d0[5], d1[5];
  if (cons) {
    double t[5];
    eos_p2c(E, v, q0);
    eos_p2c(E, vm, t);
#pragma unroll
    for (int p = 0; p < 5; p++) d0[p] = q0[p] - t[p];
    eos_p2c(E, vp, t);
#pragma unroll
    for (int p = 0; p < 5; p++) d1[p] = t[p] - q0[p];
  } else {
#pragma unroll
    for (int p = 0; p < 5; p++) {
      q0[p] = v[p];
      d0[p] = v[p] - vm[p];
      d1[p] = vp[p] - v[p];
    }
  }
  CharBasis b;
  bool ok = true;
  if (chr) {
    ok = char_setup(E, v, D, b);
    double w[5];
    if (cons) char_left(b, v, d0, w);
    else char_from_prim(b, v, d0, w);
#pragma unroll
    for (int p = 0; p < 5; p++) d0[p] = w[p];
    if (cons) char_left(b, v, d1, w);
    else char_from_prim(b, v, d1, w);
#pragma unroll
    for (int p = 0; p < 5; p++) d1[p] = w[p];
  }
  limited(s, d0, d1, h);
  if (chr) {
    double w[5];
    if (cons) char_right(b, v, h, w);
    else char_to_prim(b, v, h, w);
#pragma unroll
    for (int p = 0; p < 5; p++) h[p] = w[p];
  }
#pragma unroll
  for (int p = 0; p < 5; p++) h[p] *= 0.5;
  return ok;
}
// the minus or plus face itself (recon_face)
__device__ __forceinline__ void face_from_vars(const DevEos& E, const Scheme& s, const double* q0, const double* h,
                                               bool minus, double* f) {
  double u[5];
#pragma unroll
  for (int p = 0; p < 5; p++) u[p] = f[p] = minus ? q0[p] - h[p] : q0[p] + h[p];
  if (s.var_type != M2CX_VAR_PRIMITIVE_CHARACTERISTIC) eos_c2p(E, u, f);
}
// The minus or plus face of a cell whose six faces pass CheckState (it is not
// in s.rflag); one that would be clipped reverts to the cell's state.
__device__ __forceinline__ void face_in_vars(const DevEos& E, const Scheme& s, const double* v, const double* q0,
                                             const double* h, bool minus, double* out) {
  double f[5];
  face_from_vars(E, s, q0, h, minus, f);
  const bool clip = eos_would_clip(E, f);
#pragma unroll
  for (int p = 0; p < 5; p++) out[p] = clip ? v[p] : f[p];
}

// States along an axis: {rho, normal velocity, first and second tangential
// velocity, p}, the tangential ones in x, y, z order.
__device__ __forceinline__ void to_axis(int D, const double* v, double* w) {
  // the empty asm keeps the selects from becoming an indexed load (see vsel)
  double a = v[1], b = v[2], c = v[3];
  asm("" : "+v"(a), "+v"(b), "+v"(c));
  w[0] = v[0];
  w[1] = D == 0 ? a : (D == 1 ? b : c);
  w[2] = D == 0 ? b : a;
  w[3] = D == 2 ? b : c;
  w[4] = v[4];
}
// component of a state or flux array that holds entry q of the order above
__device__ __forceinline__ int axis_comp(int D, int q) {
  if (q == 1) return 1 + D;
  if (q == 2) return D == 0 ? 2 : 1;
  if (q == 3) return D == 2 ? 2 : 3;
  return q;
}

// (u^2 + v^2) + w^2 of a state in axis order
__device__ __forceinline__ double speed2(bool z, const double* w) {
  const double n2 = w[1] * w[1], a2 = w[2] * w[2], b2 = w[3] * w[3];
  return (a2 + (z ? b2 : n2)) + (z ? n2 : b2);
}

// e, c^2 and p / rho of a state (eos_e, eos_c2) from the reciprocal of rho
template <class A>
struct PointState {
  double e, c2, prho, dpdrho;
};
template <class A>
__device__ __forceinline__ PointState<A> point_state(const DevEos& E, double rho, const typename A::R& irho, double p) {
  PointState<A> r;
  r.prho = irho.quot(p);
  if (E.type == M2CX_EOS_SG) {
    r.e = typename A::R(E.gam1 * rho).quot(p + E.gam * E.pc);
    r.dpdrho = E.gam1 * r.e;
    r.c2 = r.dpdrho + irho.quot(E.gam1 * rho * r.e - E.gam * E.pc) * E.gam1;
  } else {
    r.e = eos_e(E, rho, p);
    r.dpdrho = eos_dpdrho(E, rho, r.e);
    r.c2 = E.type == M2CX_EOS_DUMMY ? DBL_MIN : r.dpdrho + irho.quot(eos_p(E, rho, r.e)) * eos_Gamma(E, rho);
  }
  return r;
}

// flux_hllc in axis order (z: the axis is z): every quantity of the two
// states is formed once, the quotients by rho, by the Roe weights' sum and by
// the squares of the averages share a reciprocal, and the star state is
// formed for the side the contact leaves in the face.  `ok` is cleared where
// an operand is outside the range of the fast arithmetic; the result is then
// not to be used.
// Bounds, for rho in [2^-100, 2^100], p and the normal velocity zero or in
// [2^-600, 2^100..200], e and its average in [2^-150, 2^150]: differences of
// such numbers are zero or at least an ulp of them, so every numerator below
// is zero or above 2^-750 and every denominator within [2^-400, 2^600].
template <class A>
__device__ __forceinline__ void hllc_axis(const DevEos& E, bool z, const double* Wm, const double* Wp, double* F,
                                          int& err, bool& ok) {
  using R = typename A::R;
  const double eps = 1e-10;
  const double rm = Wm[0], um = Wm[1], pm = Wm[4], rp = Wp[0], up = Wp[1], pp = Wp[4];
  const double rho_hat = A::root(rm * rp), srm = A::root(rm), srp = A::root(rp);
  const R irm(rm), irp(rp), isum(srm + srp);
  const PointState<A> m = point_state<A>(E, rm, irm, pm), q = point_state<A>(E, rp, irp, pp);
  const double drho = rp - rm, dp = pp - pm;
  const double diff = isum.quot(up - um);
  const double pr = isum.quot(srm * m.prho + srp * q.prho) + 0.5 * diff * diff;
  const double de = q.e - m.e;
  const double e_hat = isum.quot(srm * m.e + srp * q.e);
  const R irh2(rho_hat * rho_hat);
  const double w_rho = irh2.quot(drho * drho);
  const double w_e = R(e_hat * e_hat).quot(de * de);
  const R iden(w_rho + w_e + eps);
  const double dpdrho_avg = isum.quot(srm * m.dpdrho + srp * q.dpdrho);
  const double Gamma_avg = isum.quot(srm * eos_Gamma(E, rm) + srp * eos_Gamma(E, rp));
  const double t1 = (w_e + eps) * dpdrho_avg;
  const double t2 = irh2.quot((dp - Gamma_avg * rho_hat * de) * drho);
  const double dpdrho_hat = iden.quot(t1 + t2);
  const double g1 = (w_rho + eps) * Gamma_avg;
  const double g2 = R(rho_hat * e_hat * e_hat).quot((dp - dpdrho_avg * drho) * de);
  const double Gamma_hat = iden.quot(g1 + g2);
  const double c2_hat = dpdrho_hat + Gamma_hat * pr;
  const bool neg = c2_hat <= 0;
  const double c_hat = neg ? eps : A::root(c2_hat);
  if (m.c2 < 0 || q.c2 < 0) err |= 1;
  const double cm = A::root(m.c2), cp = A::root(q.c2);
  ok = in_range(rm, 0x1p-100, 0x1p100) & in_range(rp, 0x1p-100, 0x1p100) & in_range(m.e, 0x1p-150, 0x1p150) &
       in_range(q.e, 0x1p-150, 0x1p150) & in_range(e_hat, 0x1p-150, 0x1p150) & (fabs(pm) <= 0x1p200) &
       (fabs(pp) <= 0x1p200) & ((fabs(pm) >= 0x1p-600) | (pm == 0)) & ((fabs(pp) >= 0x1p-600) | (pp == 0)) &
       (fabs(um) <= 0x1p100) & (fabs(up) <= 0x1p100) & ((fabs(um) >= 0x1p-600) | (um == 0)) &
       ((fabs(up) >= 0x1p-600) | (up == 0)) & (neg | in_range(c2_hat, 0x1p-300, 0x1p300)) &
       in_range(m.c2, 0x1p-300, 0x1p300) & in_range(q.c2, 0x1p-300, 0x1p300);
  const double un_hat = isum.quot(srm * um + srp * up);
  const double a = um - cm, b = un_hat - c_hat;
  const double Sm = (b < a) ? b : a;  // std::min
  const double a2 = up + cp, b2 = un_hat + c_hat;
  const double Sp = (a2 < b2) ? b2 : a2;  // std::max
  const double gm = Sm - um, gp = Sp - up;
  const double qm = rm * gm, qp = rp * gp;
  const double Ss = (pp - pm + rm * um * gm - rp * up * gp) / (qm - qp);
  const bool below = 0.0 <= Sm, above = !below & (0.0 >= Sp), star = !below & !above;
  const bool minus = below | (star & (Ss >= 0.0));
  if (star && !(Ss >= 0.0) && !(Ss <= 0.0)) err |= 1;
  double W[5];
#pragma unroll
  for (int k = 0; k < 5; k++) W[k] = minus ? Wm[k] : Wp[k];
  const double S = minus ? Sm : Sp, e = minus ? m.e : q.e, rg = minus ? qm : qp, prho = minus ? m.prho : q.prho;
  const double ek = e + 0.5 * speed2(z, W);
  // the physical flux, then the jump across the outer wave
  const double mom = W[0] * W[1];
  F[0] = mom;
  F[1] = mom * W[1] + W[4];
  F[2] = mom * W[2];
  F[3] = mom * W[3];
  F[4] = mom * (ek + prho);
  if (star) {
    R ir = irm;
    if (!minus) ir = irp;
    const double U4 = W[0] * ek;
    const double rs = rg / (S - Ss);
    const double us4 = ir.quot(U4) + (Ss - W[1]) * (Ss + W[4] / rg);
    F[0] += S * (rs - W[0]);
    F[1] += S * (Ss * rs - mom);
    F[2] += S * (W[2] * rs - W[0] * W[2]);
    F[3] += S * (W[3] * rs - W[0] * W[3]);
    F[4] += S * (us4 * rs - U4);
  }
}
__device__ __forceinline__ void flux_hllc_axis(const DevEos& E, bool z, const double* Wm, const double* Wp, double* F,
                                               int& err) {
  int e1 = 0;
  bool ok = true;
  hllc_axis<FastMath>(E, z, Wm, Wp, F, e1, ok);
  if (!__all(ok)) {
    e1 = 0;
    hllc_axis<GeneralMath>(E, z, Wm, Wp, F, e1, ok);
  }
  err |= e1;
}

// Roe and LLF keep the x, y, z order (their sums run over it).  HLLC: compiled
// for that flux alone; with the Roe flux's eigenvectors the kernel takes 197 to
// 199 registers, two waves per SIMD, without them 167, three (256^3 water: 2.42
// ms per launch against 1.86 ms).
template <bool HLLC>
__device__ __forceinline__ void flux_axis(const DevEos& E, const Scheme& s, int D, const double* Wm, const double* Wp,
                                          double* F, int& err) {
  if (HLLC) {
    flux_hllc_axis(E, D == 2, Wm, Wp, F, err);
    return;
  }
  double Vm[5], Vp[5], f[5];
  auto back = [D](const double* w, double* v) {
    v[0] = w[0];
    v[1] = D == 0 ? w[1] : w[2];
    v[2] = D == 0 ? w[2] : (D == 1 ? w[1] : w[3]);
    v[3] = D == 2 ? w[1] : w[3];
    v[4] = w[4];
  };
  back(Wm, Vm);
  back(Wp, Vp);
  flux_num(E, s.flux, s.del, D, Vm, Vp, f, err);
  to_axis(D, f, F);
}

// ghost_face in axis order
__device__ __forceinline__ void ghost_axis(int bc, const CF5& V, long cg, int D, const double* img, double* out) {
  if (bc == M2CX_BC_INLET || bc == M2CX_BC_INLET2 || bc == M2CX_BC_OVERSET) {
#pragma unroll
    for (int q = 0; q < 5; q++) out[q] = V(axis_comp(D, q), cg);
    return;
  }
  const bool n = bc == M2CX_BC_SYMMETRY || bc == M2CX_BC_SLIPWALL || bc == M2CX_BC_STICKWALL;
  const bool t = bc == M2CX_BC_STICKWALL;
  out[0] = img[0];
  out[1] = n ? -img[1] : img[1];
  out[2] = t ? -img[2] : img[2];
  out[3] = t ? -img[3] : img[3];
  out[4] = img[4];
}

// One tile.  Phase A: each thread limits the slopes of its cell along the
// three axes once, keeps the three minus-face states in registers and leaves
// the plus-face states in LDS, in the slot of the face they belong to; the
// cells around the tile are shared out over the threads (plus side: the state
// stays with the thread that will do that face; minus side: to LDS).  Phase
// B: each thread computes the flux of its minus faces and of one plus face of
// the tile's last layers, in place over the state it read from the slot.
// Phase C: residual and Runge-Kutta combination, as in stage_tile.
//
// The material is the same for the whole tile, so its parameters sit in
// scalar registers and the type of equation of state is a scalar branch: no
// lane loads a material table, and one pass of straight-line code follows per
// face.
//
// Bound by FP64 issue and the latency of its chains, not by memory (200 B per
// cell and launch are 0.7 ms of a 256^3 launch).  256^3 water, RK3 launches:
// 4.24 ms with stage_tile, 1.86 ms here (VALU issue on 64% of the cycles at
// three waves per SIMD; held to 128 registers for four it spills: 2.88 ms);
// 128x32x32 gas: 53 -> 24 us.  GEN (any reconstruction variables; a cell that
// s.rflag marks is reconstructed in primitive ones): the slopes' eigenvectors
// set the cost, formed once per cell and axis instead of for each of its two
// faces (191x97x61 water, Roe, conservative-characteristic: 737 -> 330 us).
template <int MODE, int BX, int BY, int BZ, bool HLLC, bool GEN>
__device__ __forceinline__ void ustage_body(const StageArgs& a, int tile, const DevEos E,
                                            double (*sF)[TileShape<BX, BY, BZ>::NFACE]) {
  using TS = TileShape<BX, BY, BZ>;
  constexpr int NE = TS::EX + TS::EY + TS::EZ;
  const DevGrid& g = a.g;
  const Scheme& s = a.s;
  const int t = threadIdx.x;
  const int tx = t % BX, ty = (t / BX) % BY, tz = t / (BX * BY);
  const int ntx = (g.NX + BX - 1) / BX, nty = (g.NY + BY - 1) / BY;
  const int ib = (tile % ntx) * BX, jb = ((tile / ntx) % nty) * BY, kb = (tile / (ntx * nty)) * BZ;
  const int i = ib + tx, j = jb + ty, k = kb + tz;
  const bool inside = (i < g.NX) && (j < g.NY) && (k < g.NZ);
  const long c = gidx(g, i, j, k);
  int err = 0;

  double lo[4][5];  // minus-face states, in axis order: own x, y, z; the plus neighbour's
#pragma unroll
  for (int q = 0; q < 4; q++)
#pragma unroll
    for (int p = 0; p < 5; p++) lo[q][p] = 0.0;

  if (inside) {
    double v[5];
    load5(a.Vin, c, v);
    int fails = 0, unf = 0;
#pragma unroll
    for (int D = 0; D < 3; D++) {
      const long st = axis_stride(g, D);
      double vm[5], vp[5], h[5], l[5], r[5];
      load5(a.Vin, c - st, vm);
      load5(a.Vin, c + st, vp);
      if (GEN && !s.rflag[c]) {
        double q0[5];
        slopes_in_vars(E, s, D, v, vm, vp, q0, h);
        face_in_vars(E, s, v, q0, h, true, l);
        face_in_vars(E, s, v, q0, h, false, r);
      } else {
        half_slopes(s, v, vm, vp, h);
#pragma unroll
        for (int p = 0; p < 5; p++) {
          l[p] = v[p] - h[p];
          r[p] = v[p] + h[p];
        }
        const int bl = keep_or_revert(E, v, l), br = keep_or_revert(E, v, r);
        fails |= ((bl & 1) | ((br & 1) << 1)) << (2 * D);
        unf |= ((bl >> 1) | ((br >> 1) << 1)) << (2 * D);
      }
      const int slot = TS::slot(D, tx + (D == 0), ty + (D == 1), tz + (D == 2));
#pragma unroll
      for (int p = 0; p < 5; p++) sF[p][slot] = r[p];
      to_axis(D, l, lo[D]);
    }
    // a failing face besides the first that clipping would not mend aborts
    if (fails & (fails - 1) & unf) err = 1;
  }
#pragma unroll 1
  for (int e = t; e < 2 * NE; e += TS::NT) {
    const bool plus = e < NE;
    const int q = plus ? e : e - NE;
    int D, li, lj, lk;
    if (q < TS::EZ) {
      D = 2; li = q % BX; lj = q / BX; lk = plus ? BZ : -1;
    } else if (q < TS::EZ + TS::EY) {
      const int r = q - TS::EZ;
      D = 1; li = r % BX; lk = r / BX; lj = plus ? BY : -1;
    } else {
      const int r = q - TS::EZ - TS::EY;
      D = 0; lj = r % BY; lk = r / BY; li = plus ? BX : -1;
    }
    const int fi = ib + li, fj = jb + lj, fk = kb + lk;
    if (fi < 0 || fj < 0 || fk < 0 || fi >= g.NX || fj >= g.NY || fk >= g.NZ) continue;
    const long cc = gidx(g, fi, fj, fk), st = axis_stride(g, D);
    double v[5], vm[5], vp[5], h[5], f[5];
    if (GEN && !s.rflag[cc]) {
      double q0[5], x[5];
      load5(a.Vin, cc, v);
      load5(a.Vin, cc - st, vm);
      load5(a.Vin, cc + st, vp);
      slopes_in_vars(E, s, D, v, vm, vp, q0, h);
      face_in_vars(E, s, v, q0, h, plus, x);
      to_axis(D, x, f);
    } else {
#pragma unroll
      for (int p = 0; p < 5; p++) {
        const int w = axis_comp(D, p);
        v[p] = a.Vin(w, cc);
        vm[p] = a.Vin(w, cc - st);
        vp[p] = a.Vin(w, cc + st);
      }
      half_slopes(s, v, vm, vp, h);
#pragma unroll
      for (int p = 0; p < 5; p++) f[p] = plus ? v[p] - h[p] : v[p] + h[p];
      keep_or_revert(E, v, f);
    }
    if (plus) {
#pragma unroll
      for (int p = 0; p < 5; p++) lo[3][p] = f[p];
    } else {
      const int slot = TS::slot(D, li + (D == 0), lj + (D == 1), lk + (D == 2));
#pragma unroll
      for (int p = 0; p < 5; p++) sF[axis_comp(D, p)][slot] = f[p];
    }
  }
  __syncthreads();

  const int njobs = (t < NE) ? 4 : 3;
#pragma unroll 1
  for (int job = 0; job < njobs; job++) {
    double Wp[5], Wm[5], F[5];
#pragma unroll
    for (int p = 0; p < 5; p++) {
      Wp[p] = lo[0][p];
      lo[0][p] = lo[1][p];
      lo[1][p] = lo[2][p];
      lo[2][p] = lo[3][p];
    }
    int D = job, li = tx, lj = ty, lk = tz;
    if (job == 3) {
      if (t < TS::EZ) {
        D = 2; li = t % BX; lj = t / BX; lk = BZ;
      } else if (t < TS::EZ + TS::EY) {
        const int r = t - TS::EZ;
        D = 1; li = r % BX; lk = r / BX; lj = BY;
      } else {
        const int r = t - TS::EZ - TS::EY;
        D = 0; lj = r % BY; lk = r / BY; li = BX;
      }
    }
    const int fi = ib + li, fj = jb + lj, fk = kb + lk;
    const int pos = D == 0 ? fi : (D == 1 ? fj : fk);
    const int N = D == 0 ? g.NX : (D == 1 ? g.NY : g.NZ);
    const bool ok = fi < g.NX + (D == 0) && fj < g.NY + (D == 1) && fk < g.NZ + (D == 2);
    if (!ok) continue;
    const int slot = TS::slot(D, li, lj, lk);
    if (pos != 0) {
#pragma unroll
      for (int q = 0; q < 5; q++) Wm[q] = sF[axis_comp(D, q)][slot];
    }
    if (pos == 0 || pos == N) {
      const long cf = gidx(g, fi, fj, fk);
      if (pos == 0) ghost_axis(g.bc[2 * D], a.Vin, cf - axis_stride(g, D), D, Wp, Wm);
      else ghost_axis(g.bc[2 * D + 1], a.Vin, cf, D, Wm, Wp);
    }
    flux_axis<HLLC>(E, s, D, Wm, Wp, F, err);
#pragma unroll
    for (int q = 0; q < 5; q++) sF[axis_comp(D, q)][slot] = F[q];
  }
  // the conserved states that the combination reads, on their way while the
  // other waves finish their fluxes
  StageIn in;
  if (inside) stage_load<MODE>(a, c, in);
  __syncthreads();
  if (err) atomicOr(&a.cnt->error, 1);
  if (!inside) return;

  const double dxi = g_axis(g, 3)[i + 1], dyj = g_axis(g, 4)[j + 1], dzk = g_axis(g, 5)[k + 1];
  const double ax = dyj * dzk, ay = dxi * dzk, az = dxi * dyj;
  const int fxm = TS::slot(0, tx, ty, tz), fxp = TS::slot(0, tx + 1, ty, tz);
  const int fym = TS::slot(1, tx, ty, tz), fyp = TS::slot(1, tx, ty + 1, tz);
  const int fzm = TS::slot(2, tx, ty, tz), fzp = TS::slot(2, tx, ty, tz + 1);
  const double cst = 1.0 / (-(dxi * dyj * dzk));
  double r[5];
#pragma unroll
  for (int p = 0; p < 5; p++) {
    double acc = 0.0 - ax * sF[p][fxm];
    acc = acc - ay * sF[p][fym];
    acc = acc - az * sF[p][fzm];
    acc = acc + ax * sF[p][fxp];
    acc = acc + ay * sF[p][fyp];
    acc = acc + az * sF[p][fzp];
    r[p] = acc * cst;
  }
  stage_update<MODE>(a, E, in, i, j, k, c, r);
}

template <int MODE, int BX, int BY, int BZ, bool HLLC, bool GEN>
__device__ __forceinline__ void ustage_tile(const StageArgs& a, int tile) {
  __shared__ double sF[5][TileShape<BX, BY, BZ>::NFACE];
  if (a.tflag && a.tflag[tile]) return;
  const DevGrid& g = a.g;
  const int ntx = (g.NX + BX - 1) / BX, nty = (g.NY + BY - 1) / BY;
  const long c0 = gidx(g, (tile % ntx) * BX, ((tile / ntx) % nty) * BY, (tile / (ntx * nty)) * BZ);
  const int id = __builtin_amdgcn_readfirstlane((int)a.ID[c0]);
  const DevEos E = c_mats[a.s.mset].m[id];
  // one copy of the tile's code per type of equation of state, each without
  // the others' branches
  if (E.type == M2CX_EOS_SG) ustage_body<MODE, BX, BY, BZ, HLLC, GEN>(a, tile, E, sF);
  else if (E.type == M2CX_EOS_NASG) ustage_body<MODE, BX, BY, BZ, HLLC, GEN>(a, tile, E, sF);
  else ustage_body<MODE, BX, BY, BZ, HLLC, GEN>(a, tile, E, sF);
}

// Waves per SIMD the compiler keeps the kernel's registers to: three for HLLC and
// primitive variables (168 registers at most), two, as they are, for the
// eigenvectors of the others (185 to 199).
constexpr int ustage_waves(bool hllc, bool gen) { return hllc && !gen ? 3 : 2; }

template <int MODE, int BX, int BY, int BZ, bool HLLC, bool GEN>
__global__ void __launch_bounds__(BX * BY * BZ, ustage_waves(HLLC, GEN)) k_stage_u(StageArgs a) {
  // read in place, as in k_stage
  const StageArgs& ar = *(const StageArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  const DevGrid& g = ar.g;
  const int ntiles = ((g.NX + BX - 1) / BX) * ((g.NY + BY - 1) / BY) * ((g.NZ + BZ - 1) / BZ);
  const int tile = xcd_tile(ntiles);
  if (tile >= ntiles) return;
  ustage_tile<MODE, BX, BY, BZ, HLLC, GEN>(ar, tile);
}

// The members of an ensemble in one launch, as k_stage_multi.  Two waves per SIMD,
// also where three would fit: the launch runs beside the batched Riemann launch,
// four waves per SIMD of 320 registers of which one is resident, and stage waves
// that take the room a finished one leaves hold the next one back.  At three the
// stage launches of 12 members of 48^3 to 128^3 were shorter (2.42 -> 1.36 ms) and
// their steps were not (271 / 268 ms, within the spread); 64 members of 64^3 to
// 192^3 took 259 to 291 ms per step, by tile shape, instead of 245.
template <int MODE, int BX, int BY, int BZ, bool HLLC, bool GEN>
__global__ void __launch_bounds__(BX * BY * BZ) __attribute__((amdgpu_waves_per_eu(2, 2)))
    k_stage_u_multi(const StageArgs* __restrict__ tab, const int* __restrict__ toff, int nm) {
  const int total = toff[nm];
  const int t = xcd_tile(total);
  if (t >= total) return;
  const int m = multi_member(toff, nm, t);
  ustage_tile<MODE, BX, BY, BZ, HLLC, GEN>(tab[m], t - toff[m]);
}

}  // namespace m2c
