// The hydro arithmetic in the arrangement of the reference's shaders (src/hydro/*.wgsl, riemann/
// *.wgsl): limiters, half step, face solve and signal rate. Block grids with per-block timesteps
// use it, where the other paths use hydro.hpp's arrangement of the same formulas.
//
// The two differ by rounding, and the scheme magnifies that. The shock flag asks whether the
// velocities around a cell converge; at the rim of a face beside a coarser block one of its
// neighbours is an empty edge texel, whose pressure jump is always over the threshold, so in gas close
// to rest the sign of a difference at the rounding level picks HLL or HLLC for the cell's
// faces there. After eight cycles of eight substeps of the 3D blast (root 4, two refinements) the
// two arrangements' states are 3e-7 to 1.2e-5 apart in the L2 norm, by seed, and up to 3e-3 in single
// cells; in FP64, where no less is rounding, 1e-6 and 4e-4. Neither is the nearer one to FP64 (3.5e-6
// both). A cycle's values are therefore kept to the bit as they have been; its passes are bound by
// the atlases' latency and bandwidth, so the cheaper arrangement gains little there.
#pragma once
#include "hydro.hpp"

namespace shx {
// (calls among these functions are qualified: hydro.hpp has the same names, and its structs would
// bring them in by argument)
namespace ref {

// Koren's smoothness measure of a channel against its natural scale s = 0.01 scale: the
// difference energy over s^2 (koren.wgsl:274-292), or, where s^2 over- or underflows, the
// differences scaled by 1/|s| first. What depends on the scale alone is formed once per scale
// (a cell's six channels have four: rho, c_s three times, p, none) and shared by its edges.
template <typename T>
struct EdgeScale { T s2inv; T k; bool as_is; };

template <typename T>
__device__ __forceinline__ EdgeScale<T> edge_scale(T scale) {
  const T SMOOTH = T(0.01);
  T s = SMOOTH * scale;
  T s2 = s * s;
  EdgeScale<T> e;
  e.as_is = (s2 >= T(1e-30) && s2 < T(1e30)) || (s == T(0));
  e.s2inv = tmax(s2, T(1e-30));
  if constexpr (sizeof(T) == 4) e.s2inv = trcp(e.s2inv);   // tdiv(q, ss) = q rcp(ss) in FP32
  e.k = trcp(tmax(tabs(s), T(1e-37)));
  return e;
}

// Twice the edge increment from the differences (far, near) and the channel's scale.
// Koren (koren.wgsl:274-292): its early return gives exactly the blend's value per channel
// (the blend weight is 1 for a smooth channel), so each channel is formed on its own.
template <typename T, int LIM>
__device__ __forceinline__ T edge1(T far, T near, const EdgeScale<T>& sc) {
  if constexpr (LIM == LIM_KOREN) {
    T fr = (far + T(2) * near) * T(1.0 / 3.0);
    T q = far * far + near * near;
    T eta;
    if (sc.as_is) {
      // FP32: q times the reciprocal (tdiv's form); FP64: the quotient (s2inv holds ss)
      if constexpr (sizeof(T) == 4) eta = q * sc.s2inv;
      else eta = tdiv(q, sc.s2inv);
    } else {
      T fk = far * sc.k, nk = near * sc.k;
      eta = fk * fk + nk * nk;
    }
    // sign(near) min(2|far|, 2|near|, |fr|) where far and near share a sign (fr then does too)
    T lim = minmod(T(2) * far, minmod(T(2) * near, fr));
    T w = tclamp(T(1.5) - eta, T(0), T(1));
    return (w == T(1)) ? fr : tmix(lim, fr, w);
  } else if constexpr (LIM == LIM_MC) {
    // sign(far) min(2|far|, 2|near|, |far + near| / 2) where far and near share a sign
    return minmod(T(2) * far, minmod(T(2) * near, T(0.5) * (far + near)));
  } else if constexpr (LIM == LIM_MINMOD) {
    return minmod(far, near);
  } else {
    return same_sign(far, near) ? T(2) * far * tdiv(near, far + near) : T(0);
  }
}

// isen_inc / isen_blend (hydro/q.wgsl:183-213) with no reference state and no potential, in two
// parts: what depends only on the three cells (the densities along the adiabat through the
// centre, the smoothness, adiabat and shear switches), shared by a cell's up and down edges, and
// the edge's own blend.
template <typename T>
struct IsenCommon { bool ok; T gi, tl, tr, room; };

template <typename T>
__device__ __forceinline__ IsenCommon<T> isen_common(const Params<T>& P, const Prim<T>& l, const Prim<T>& c,
                                                     const Prim<T>& r) {
  const T ISEN_SMOOTH = T(0.2), ISEN_ADIABAT = T(0.01), ISEN_SHEAR = T(0.1), ISEN_ROOM = T(0.01);
  IsenCommon<T> k;
  k.ok = l.rho > T(0) && l.p > T(0) && c.rho > T(0) && c.p > T(0) && r.rho > T(0) && r.p > T(0);
  k.gi = trcp(P.gamma);
  k.tl = l.rho * tpow(tdiv(c.p, l.p), k.gi) - c.rho;
  k.tr = r.rho * tpow(tdiv(c.p, r.p), k.gi) - c.rho;
  T ks = tclamp(T(2) - tdiv(tmax(tabs(l.p - c.p), tabs(r.p - c.p)), ISEN_SMOOTH * c.p), T(0), T(1));
  T ka = tclamp(T(2) - tdiv(tmax(tabs(k.tl), tabs(k.tr)), ISEN_ADIABAT * c.rho), T(0), T(1));
  T dxr = r.vx - c.vx, dyr = r.vy - c.vy, dzr = r.vz - c.vz;
  T dxl = c.vx - l.vx, dyl = c.vy - l.vy, dzl = c.vz - l.vz;
  T dvr = tsqrt(dxr * dxr + dyr * dyr + dzr * dzr);
  T dvl = tsqrt(dxl * dxl + dyl * dyl + dzl * dzl);
  T kv = tclamp(T(2) - tdiv(tmax(dvr, dvl), ISEN_SHEAR * tmax(c.cs, T(1e-30))), T(0), T(1));
  k.room = ISEN_ROOM * c.rho * ks * ka * kv;
  return k;
}

template <typename T, int LIM>
__device__ __forceinline__ T isen_blend(const IsenCommon<T>& k, const EdgeScale<T>& srho, const Prim<T>& l,
                                        const Prim<T>& c, const Prim<T>& r, T x, T bx, T sgn) {
  const T ISEN_CAP = T(0.25);
  if (!k.ok) return x + tclamp(T(0) - x, T(0), T(0));
  T far = sgn > T(0) ? -k.tl : k.tr;
  T near = sgn > T(0) ? k.tr : -k.tl;
  T d = ref::edge1<T, LIM>(far, near, srho);
  T pf = c.p + T(0.5) * sgn * bx;
  T wn = sgn > T(0) ? r.rho : l.rho;
  T rf = tclamp((c.rho + T(0.5) * sgn * d) * tpow(tdiv(tmax(pf, T(1e-30)), c.p), k.gi), tmin(c.rho, wn),
                tmax(c.rho, wn));
  T bound = tmax(ISEN_CAP * tmin(tabs(c.rho - l.rho), tabs(r.rho - c.rho)), k.room);
  T i0 = T(2) * sgn * (rf - c.rho);
  return x + tclamp(i0 - x, -bound, bound);
}

// edge_up (UP) / edge_dn (hydro/q.wgsl:214-239), no potential.
template <typename T, int LIM, bool ISEN, bool UP>
__device__ __forceinline__ Inc<T> edge_k(const Params<T>& P, const Prim<T>& l, const Prim<T>& c, const Prim<T>& r,
                                         const IsenCommon<T>& k) {
  Inc<T> o;
  constexpr bool fwd = UP || lim_symmetric<LIM>();
  auto e = [&](T lo, T mid, T hi, const EdgeScale<T>& sc) {
    T below = mid - lo, above = hi - mid;
    return fwd ? ref::edge1<T, LIM>(below, above, sc) : ref::edge1<T, LIM>(above, below, sc);
  };
  EdgeScale<T> srho{}, sv{}, sp{}, s0{};
  if constexpr (LIM == LIM_KOREN) {
    srho = ref::edge_scale(c.rho); sv = ref::edge_scale(c.cs); sp = ref::edge_scale(c.p); s0 = ref::edge_scale(T(0));
  }
  o.rho = e(l.rho, c.rho, r.rho, srho);
  o.vx = e(l.vx, c.vx, r.vx, sv);
  o.vy = e(l.vy, c.vy, r.vy, sv);
  o.vz = e(l.vz, c.vz, r.vz, sv);
  o.p = e(l.p, c.p, r.p, sp);
  o.s = e(l.s, c.s, r.s, s0);
  if constexpr (ISEN) o.rho = ref::isen_blend<T, LIM>(k, srho, l, c, r, o.rho, o.p, UP ? T(1) : T(-1));
  return o;
}
template <typename T, int LIM, bool ISEN, bool UP>
__device__ __forceinline__ Inc<T> edge(const Params<T>& P, const Prim<T>& l, const Prim<T>& c, const Prim<T>& r) {
  IsenCommon<T> k{};
  if constexpr (ISEN) k = ref::isen_common(P, l, c, r);
  return ref::edge_k<T, LIM, ISEN, UP>(P, l, c, r, k);
}

// One axis's contribution to the predictor: the face-to-face slope and the positivity terms.
template <typename T, int LIM, bool ISEN>
__device__ __forceinline__ AxisSlope<T> axis_slope(const Params<T>& P, const Prim<T>& m, const Prim<T>& q,
                                                   const Prim<T>& p) {
  AxisSlope<T> r;
  // a cell's up and down edges share the isentropic terms of its three cells
  IsenCommon<T> k{};
  if constexpr (ISEN) k = ref::isen_common(P, m, q, p);
  Inc<T> u = ref::edge_k<T, LIM, ISEN, true>(P, m, q, p, k);
  if constexpr (lim_symmetric<LIM>()) {
    r.s = u;
    r.big = tabs(u.p);
    r.fall = T(-0.5) * tabs(u.rho);
  } else {
    Inc<T> d = ref::edge_k<T, LIM, ISEN, false>(P, m, q, p, k);
    r.s.rho = T(0.5) * (u.rho + d.rho);
    r.s.vx = T(0.5) * (u.vx + d.vx);
    r.s.vy = T(0.5) * (u.vy + d.vy);
    r.s.vz = T(0.5) * (u.vz + d.vz);
    r.s.p = T(0.5) * (u.p + d.p);
    r.s.s = T(0.5) * (u.s + d.s);
    r.big = tmax(tabs(u.p), tabs(d.p));
    r.fall = tmin(T(0.5) * u.rho, T(-0.5) * d.rho);
  }
  return r;
}

// The Hancock half step from the cell, its six neighbours' pressures and normal velocities
// (for the shock detector) and the three axis slopes.
template <typename T>
__device__ __forceinline__ Half<T> hancock(const Params<T>& P, const Prim<T>& q, const AxisSlope<T> sl[3],
                                           T conv, T jump, T dt) {
  Half<T> o;
  T big = tmax(tmax(tmax(T(0), sl[0].big), sl[1].big), sl[2].big);
  T fall = tmin(tmin(tmin(T(0), sl[0].fall), sl[1].fall), sl[2].fall);
  T shock = (conv < T(0) && jump > P.shock_thresh) ? T(1) : T(0);
  T h = T(0.5) * dt / P.dx;
  T rho = q.rho;
  const Inc<T>& sx = sl[0].s;
  const Inc<T>& sy = sl[1].s;
  const Inc<T>& sz = sl[2].s;
  T dv = sx.vx + sy.vy + sz.vz;
  T da0 = q.vx * sx.rho + q.vy * sy.rho + q.vz * sz.rho;
  T da1 = q.vx * sx.vx + q.vy * sy.vx + q.vz * sz.vx;
  T da2 = q.vx * sx.vy + q.vy * sy.vy + q.vz * sz.vy;
  T da3 = q.vx * sx.vz + q.vy * sy.vz + q.vz * sz.vz;
  T db0 = q.vx * sx.p + q.vy * sy.p + q.vz * sz.p;
  T db1 = q.vx * sx.s + q.vy * sy.s + q.vz * sz.s;
  T ir = trcp(rho);
  o.rho = rho - h * (da0 + rho * dv);
  o.vx = q.vx - h * (da1 + sx.p * ir);
  o.vy = q.vy - h * (da2 + sy.p * ir);
  o.vz = q.vz - h * (da3 + sz.p * ir);
  o.p = q.p - h * (db0 + rho * q.cs * q.cs * dv);
  o.s = q.s - h * db1;
  o.shock = shock;
  T rmin = o.rho + fall;
  T pmin = o.p - T(0.5) * big;
  o.fo = T(0);
  if (!(rmin > T(0) && pmin > T(0))) {
    o.rho = q.rho; o.vx = q.vx; o.vy = q.vy; o.vz = q.vz; o.p = q.p; o.s = q.s;
    o.fo = T(1);
  }
  return o;
}

// Shock detector (predictor.wgsl:114-134): converging flow and the largest relative pressure
// jump across the cell.
template <typename T>
__device__ __forceinline__ T jump_of(T pm, T pp) {
  return tdiv(tabs(pp - pm), tmin(pp, pm));
}

// One side of a face (to_side, flux.wgsl:60-85) in the face frame: n normal, t1/t2 the
// cyclically following components (rot, flux.wgsl:37-41).
template <typename T>
struct Side { T rho, vn, vt1, vt2, p, s, cs, eint; };

template <typename T>
__device__ __forceinline__ Side<T> make_side(const Params<T>& P, T rho, T vn, T vt1, T vt2, T p, T s,
                                             T lo_rho, T lo_p) {
  Side<T> o;
  o.rho = tmax(rho, tmax(lo_rho, P.rho_floor));
  o.vn = vn; o.vt1 = vt1; o.vt2 = vt2;
  o.s = s;
  o.p = tmax(p, tmax(lo_p, P.p_floor));
  o.cs = tsqrt(tdiv(P.gamma * o.p, o.rho));
  o.eint = o.p * P.igm1;
  return o;
}

// A side's total energy, momentum and normal flux (hllc.wgsl:7-28), each from the side's own
// primitives in one fixed expression
template <typename T>
struct SideFlux { T E, m0, m1, m2, f0, f1, f2, fe; };
template <typename T>
__device__ __forceinline__ SideFlux<T> side_flux(T rho, T vn, T vt1, T vt2, T p, T eint) {
  SideFlux<T> o;
  o.E = eint + T(0.5) * rho * (vn * vn + vt1 * vt1 + vt2 * vt2);
  o.m0 = rho * vn; o.m1 = rho * vt1; o.m2 = rho * vt2;
  o.f0 = o.m0 * vn + p; o.f1 = o.m1 * vn; o.f2 = o.m2 * vn;
  o.fe = (o.E + p) * vn;
  return o;
}

// HLLC blended toward HLL by w (riemann/hllc.wgsl:4-85), or HLL (riemann/hll.wgsl:87-121).
// Each branch forms only the side quantities it uses: the upwind side's on a supersonic face,
// the star side's on a subsonic one, both where the HLL state is needed.
template <typename T, int RS>
__device__ __forceinline__ Flux<T> riemann(const Side<T>& l, const Side<T>& r, T w_hll) {
  T sl = tmin(l.vn - l.cs, r.vn - r.cs);
  T sr = tmax(l.vn + l.cs, r.vn + r.cs);
  Flux<T> o;
  if (sl >= T(0) || sr <= T(0)) {
    // supersonic: the upwind side's own flux
    const bool up_l = sl >= T(0);
    const SideFlux<T> u = ref::side_flux(up_l ? l.rho : r.rho, up_l ? l.vn : r.vn, up_l ? l.vt1 : r.vt1,
                                    up_l ? l.vt2 : r.vt2, up_l ? l.p : r.p, up_l ? l.eint : r.eint);
    o.m = u.m0; o.mx = u.f0; o.my = u.f1; o.mz = u.f2; o.e = u.fe; o.vn = up_l ? l.vn : r.vn;
  } else {
    T ql = l.rho * (sl - l.vn);
    T qr = r.rho * (sr - r.vn);
    const bool star = RS != RS_HLL && ql < T(0) && qr > T(0);
    // The HLL state between the waves: the flux itself where the star densities are not
    // positive (and for HLL), the blend's other end where the face is flagged; a subsonic
    // unflagged face (w = 0: the blend is the star flux exactly) skips it.
    T hm, hp0, hp1, hp2, he;
    if (!star || w_hll != T(0)) {
      const SideFlux<T> a = ref::side_flux(l.rho, l.vn, l.vt1, l.vt2, l.p, l.eint);
      const SideFlux<T> b = ref::side_flux(r.rho, r.vn, r.vt1, r.vt2, r.p, r.eint);
      T inv = trcp(sr - sl);
      T slsr = sl * sr;
      hm = (sr * a.m0 - sl * b.m0 + slsr * (r.rho - l.rho)) * inv;
      hp0 = (sr * a.f0 - sl * b.f0 + slsr * (b.m0 - a.m0)) * inv;
      hp1 = (sr * a.f1 - sl * b.f1 + slsr * (b.m1 - a.m1)) * inv;
      hp2 = (sr * a.f2 - sl * b.f2 + slsr * (b.m2 - a.m2)) * inv;
      he = (sr * a.fe - sl * b.fe + slsr * (b.E - a.E)) * inv;
    }
    if constexpr (RS == RS_HLL) {
      o.m = hm; o.mx = hp0; o.my = hp1; o.mz = hp2; o.e = he;
      o.vn = tdiv(r.p - l.p + l.vn * ql - r.vn * qr, ql - qr);
    } else {
      if (!star) {
        o.m = hm; o.mx = hp0; o.my = hp1; o.mz = hp2; o.e = he;
        o.vn = T(0.5) * (l.vn + r.vn);
      } else {
        T sm = tdiv(r.p - l.p + l.vn * ql - r.vn * qr, ql - qr);
        // the star state as differences from the outer state (hllc.wgsl:52-74)
        bool left = sm >= T(0);
        T S = left ? sl : sr;
        T rho = left ? l.rho : r.rho;
        T un = left ? l.vn : r.vn;
        T u1 = left ? l.vt1 : r.vt1;
        T u2 = left ? l.vt2 : r.vt2;
        T p = left ? l.p : r.p;
        T q = left ? ql : qr;
        const SideFlux<T> c = ref::side_flux(rho, un, u1, u2, p, left ? l.eint : r.eint);
        T k = tdiv(sm - un, S - sm);
        T dr = rho * k;
        T f = rho + dr;
        T cm = c.m0 + S * dr;
        T c0 = c.f0 + S * (sm * dr + rho * (sm - un));
        T c1 = c.f1 + S * (dr * u1);
        T c2 = c.f2 + S * (dr * u2);
        T ce = c.fe + S * (c.E * k + f * (sm - un) * (sm + tdiv(p, q)));
        if (w_hll != T(0)) {
          o.m = tmix(cm, hm, w_hll);
          o.mx = tmix(c0, hp0, w_hll);
          o.my = tmix(c1, hp1, w_hll);
          o.mz = tmix(c2, hp2, w_hll);
          o.e = tmix(ce, he, w_hll);
        } else {
          o.m = cm; o.mx = c0; o.my = c1; o.mz = c2; o.e = ce;
        }
        o.vn = sm;
      }
    }
  }
  // internal energy and the scalar ride on the mass flux, upwinded
  bool up = o.m >= T(0);
  o.ei = o.m * tdiv(up ? l.eint : r.eint, up ? l.rho : r.rho);
  o.s = o.m * (up ? l.s : r.s);
  return o;
}

// One cell's side of a face before the face's own lower bound and floors: the half-step state plus
// half the edge increment toward the face (to_side, flux.wgsl:60-63; zero increment for a
// first-order cell), with its half-step density and pressure and its shock flag.
// sgn = +1 for the cell's upper face (il its up increment), -1 for its lower face.
template <typename T>
__device__ __forceinline__ SideData<T> side_of(const Half<T>& h, const Inc<T>& inc, T sgn) {
  T hs = T(0.5) * sgn * (T(1) - h.fo);
  SideData<T> o;
  o.rho = h.rho + hs * inc.rho;
  o.vx = h.vx + hs * inc.vx;
  o.vy = h.vy + hs * inc.vy;
  o.vz = h.vz + hs * inc.vz;
  o.p = h.p + hs * inc.p;
  o.s = h.s + hs * inc.s;
  o.hrho = h.rho;
  o.hp = h.p;
  o.shock = h.shock;
  return o;
}

// face_flux (flux.wgsl:92-125) between the half-step states hl (left) and hr (right), given twice
// the increments from each cell toward the face (il: the left cell's up increment, ir: the right
// cell's down increment), along a run-time axis: the velocities are rotated into the face frame
// (flux.wgsl:37-41) and the momentum back (the empty asm as in face_from_sides_rt).
template <typename T, int RS>
__device__ __forceinline__ Flux<T> face_flux(const Params<T>& P, const Half<T>& hl, const Inc<T>& il,
                                             const Half<T>& hr, const Inc<T>& ir, int axis) {
  const SideData<T> L = ref::side_of(hl, il, T(1)), R = ref::side_of(hr, ir, T(-1));
  T w = tmax(L.shock, R.shock);
  T lo_rho = T(0.5) * tmin(L.hrho, R.hrho);
  T lo_p = T(0.5) * tmin(L.hp, R.hp);
  T lx = L.vx, ly = L.vy, lz = L.vz, rx = R.vx, ry = R.vy, rz = R.vz;
  asm("" : "+v"(lx), "+v"(ly), "+v"(lz), "+v"(rx), "+v"(ry), "+v"(rz));
  const bool a0 = axis == 0, a1 = axis == 1;
  Side<T> sl = ref::make_side(P, L.rho, a0 ? lx : (a1 ? ly : lz), a0 ? ly : (a1 ? lz : lx), a0 ? lz : (a1 ? lx : ly),
                              L.p, L.s, lo_rho, lo_p);
  Side<T> sr = ref::make_side(P, R.rho, a0 ? rx : (a1 ? ry : rz), a0 ? ry : (a1 ? rz : rx), a0 ? rz : (a1 ? rx : ry),
                              R.p, R.s, lo_rho, lo_p);
  Flux<T> F = ref::riemann<T, RS>(sl, sr, w);
  T n = F.mx, t1 = F.my, t2 = F.mz;
  asm("" : "+v"(n), "+v"(t1), "+v"(t2));
  F.mx = a0 ? n : (a1 ? t2 : t1); F.my = a0 ? t1 : (a1 ? n : t2); F.mz = a0 ? t2 : (a1 ? t1 : n);
  return F;
}

// The signal rate of a cell (hydro/rates.wgsl:60-62).
template <typename T>
__device__ __forceinline__ T rate_of(const Params<T>& P, const Prim<T>& w) {
  T signal = tsqrt(w.cs * w.cs);
  return tabs(w.vx) + tabs(w.vy) + tabs(w.vz) + P.ndim * signal;
}

}  // namespace ref
}  // namespace shx
