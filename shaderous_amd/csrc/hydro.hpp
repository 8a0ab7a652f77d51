// Device core of the MUSCL-Hancock + HLLC hydro update: primitives, boundary mapping, limited
// reconstruction, the Hancock predictor, the face Riemann solve and the conservative update.
// Shared by every kernel (uniform plain, uniform fused, blocks, ensemble) so that all of them
// compute each quantity with the same instructions. Templated on the arithmetic type T (float
// for the production path, double for the all-FP64 precision twin), the limiter, the Riemann
// solver and the density-along-the-adiabat option.
//
// The arithmetic follows the reference's WGSL with every optional module off; each function
// cites the file and lines it follows (paths under the reference's src/).
//
// The fused kernels are bound by VALU issue, and a reciprocal, root, log or exp takes the issue
// slots of four other instructions, so the formulas here are arranged for few of both: one set of
// expressions for every state a face can have (riemann), Koren's weight once per channel for both
// edges, increments kept at the size they are used at, no root or quotient where a product tells
// the same. Against the reference's own arrangement, with the same tiles and launches: turbulence
// 256^3 (MC) 0.578 -> 0.52 ms per step, KH 2048^2 (Koren + isentropic) 0.182 -> 0.146, Sedov 128^3
// (the same scheme) 0.157 -> 0.121, turbulence 96^3 in FP64 0.316 -> 0.275; the error against 64
// bits after 100 to 200 steps as before (2e-7 to 3e-7), half for Sedov.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace shx {

enum { LIM_KOREN = 0, LIM_MC = 1, LIM_VANLEER = 2, LIM_MINMOD = 3 };
enum { RS_HLLC = 0, RS_HLL = 1 };
enum { BC_PERIODIC = 0, BC_OUTFLOW = 1, BC_REFLECT = 2, BC_OUTFLOW_ONLY = 3 };

template <typename T> struct Vec4;
template <> struct Vec4<float> { using type = float4; };
template <> struct Vec4<double> { using type = double4; };
template <typename T> using T4 = typename Vec4<T>::type;

// The Params values the hydro path reads (hydro/common.wgsl:4-79), in the run's precision.
template <typename T>
struct Params {
  int n[3];
  int bc_lo[3];
  int bc_hi[3];
  int flat;            // one layer along z (2D): z neighbours are the cell itself
  T ndim;              // P.geom.y
  T gamma, gm1, igm1;  // P.eos.x, P.eos.x - 1, 1 / (P.eos.x - 1)
  T dx, cfl, rho_floor, p_floor, eta_dual, shock_thresh, t_end, dt_max;
  T fluff[3];
};

// min/max/abs as single instructions (v_min_f32, v_max_f32, the |x| source modifier); a NaN
// operand yields the other one.
__device__ __forceinline__ float tmin(float a, float b) { return __builtin_fminf(a, b); }
__device__ __forceinline__ double tmin(double a, double b) { return __builtin_fmin(a, b); }
__device__ __forceinline__ float tmax(float a, float b) { return __builtin_fmaxf(a, b); }
__device__ __forceinline__ double tmax(double a, double b) { return __builtin_fmax(a, b); }
__device__ __forceinline__ float tabs(float a) { return __builtin_fabsf(a); }
__device__ __forceinline__ double tabs(double a) { return __builtin_fabs(a); }
// The same for operands that come from memory or LDS, where the compiler would first quiet each
// one (v_max x, x) in case it is a signaling NaN: arithmetic makes none, and states are checked
// finite when they are set. (The compiler's hazard pass does not look at inline assembly's operands:
// a test of the built code holds that none is a transcendental's result of the slot before.)
__device__ __forceinline__ float raw_min(float a, float b) {
  float r;
  asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double raw_min(double a, double b) { return tmin(a, b); }
__device__ __forceinline__ float raw_max(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double raw_max(double a, double b) { return tmax(a, b); }
template <typename T> __device__ __forceinline__ T tsign(T a) { return a > T(0) ? T(1) : (a < T(0) ? T(-1) : T(0)); }
// x held to [lo, hi] (lo <= hi; a NaN x gives lo): in FP32 the median, one instruction, and between
// the constants 0 and 1 the output modifier of the instruction that forms x
__device__ __forceinline__ float tclamp(float x, float lo, float hi) { return __builtin_amdgcn_fmed3f(x, lo, hi); }
__device__ __forceinline__ double tclamp(double x, double lo, double hi) { return tmin(tmax(x, lo), hi); }
// x held between a and b, whichever is the smaller
__device__ __forceinline__ float tbetween(float x, float a, float b) { return __builtin_amdgcn_fmed3f(x, a, b); }
__device__ __forceinline__ double tbetween(double x, double a, double b) { return tclamp(x, tmin(a, b), tmax(a, b)); }
// Single precision: the hardware reciprocal and square root (v_rcp_f32, v_sqrt_f32, ~1 ulp;
// WGSL allows 2.5 ulp for division). Double precision: correctly rounded.
__device__ __forceinline__ float trcp(float b) { return __builtin_amdgcn_rcpf(b); }
__device__ __forceinline__ double trcp(double b) { return 1.0 / b; }
__device__ __forceinline__ float tdiv(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
__device__ __forceinline__ double tdiv(double a, double b) { return a / b; }
// A quotient that several kernels form for themselves and that has to be the same in each (a step
// over a cell size): spelled out, as the compiler lowers a plain a / b to a correctly rounded or an
// approximate form by what stands around it. To half an ulp and a little.
__device__ __forceinline__ float tratio(float a, float b) {
  const float r = __builtin_amdgcn_rcpf(b), q = a * r;
  return __builtin_fmaf(__builtin_fmaf(-q, b, a), r, q);
}
__device__ __forceinline__ double tratio(double a, double b) { return a / b; }
// The quotients that decide the step, a rate over a cell size and cfl dx over the largest rate: formed
// in several kernels, with the same need. Spelled out in the form the compiler gives a plain a / b
// in them today (mantissas by the approximate reciprocal, exponents apart; about an ulp), which never
// falls as a rises, so that a quotient of the largest rate is the largest quotient.
__device__ __forceinline__ float tquot(float a, float b) {
  return __builtin_ldexpf(__builtin_amdgcn_frexp_mantf(a) * __builtin_amdgcn_rcpf(__builtin_amdgcn_frexp_mantf(b)),
                          __builtin_amdgcn_frexp_expf(a) - __builtin_amdgcn_frexp_expf(b));
}
__device__ __forceinline__ double tquot(double a, double b) { return a / b; }
__device__ __forceinline__ float tsqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
__device__ __forceinline__ double tsqrt(double x) { return __builtin_sqrt(x); }
// Single-precision pow as WGSL defines it, exp2(b log2 a) (every base here is positive), by the
// hardware's log2 and exp2 (v_log_f32, v_exp_f32): the library powf's exact-case handling costs
// ~40 instructions a call, and the isentropic reconstruction makes six calls per axis.
__device__ __forceinline__ float tpow(float a, float b) { return __builtin_amdgcn_exp2f(b * __builtin_amdgcn_logf(a)); }
// Double precision: the library's, as a call. Inlined at its 24 uses of a plane it made kernels of up
// to 348 KB, several times the instruction cache; the largest (k_fused_r, isentropic reconstruction
// beside walls) gave wrong values, where the same source with the call gives the plain path's. What
// in that build was wrong is not known, so the kernels' sizes are bounded by a test. Turbulence 96^3 in
// FP64, Koren + isentropic: 0.78 -> 0.50 ms per step with the call.
__device__ __attribute__((noinline)) inline double tpow(double a, double b) { return pow(a, b); }
// WGSL mix(x, y, a) = x (1 - a) + y a
template <typename T> __device__ __forceinline__ T tmix(T x, T y, T a) { return x * (T(1) - a) + y * a; }
// sign(a) * sign(b) > 0, formed from the signs so that small products do not underflow
// (limiters/koren.wgsl:287-289)
template <typename T> __device__ __forceinline__ bool same_sign(T a, T b) {
  return (a > T(0) && b > T(0)) || (a < T(0) && b < T(0));
}
// minmod(x, y) = sign(x) min(|x|, |y|) when sign(x) sign(y) > 0, else 0: in FP32 the median of
// (0, x, y), one instruction (a zero result may carry the sign of x or y)
__device__ __forceinline__ float minmod(float x, float y) { return __builtin_amdgcn_fmed3f(0.0f, x, y); }
__device__ __forceinline__ double minmod(double x, double y) {
  return same_sign(x, y) ? (x > 0.0 ? tmin(x, y) : tmax(x, y)) : 0.0;
}

// Primitive record (hydro/q.wgsl:56): rho, v, p, scalar s, sound speed c.
template <typename T>
struct Prim {
  T rho, vx, vy, vz, p, s, cs;
};

// prim_from_cons (hydro/prim.wgsl:131-156), ideal gas (eos/ideal.wgsl:235-267), pressure floor
// without a Jeans floor (hydro/pfloor.wgsl:169-171).
template <typename T>
__device__ __forceinline__ Prim<T> prim_from_cons(const Params<T>& P, T4<T> u1, T4<T> u2) {
  Prim<T> q;
  T rho = raw_max(u1.x, P.rho_floor);
  T p = P.gm1 * u2.y;
  if (!(p >= P.p_floor)) p = P.p_floor;
  T ir = trcp(rho);
  q.rho = rho;
  q.vx = u1.y * ir;
  q.vy = u1.z * ir;
  q.vz = u1.w * ir;
  q.p = p;
  q.s = u2.z * ir;
  q.cs = tsqrt(P.gamma * p * ir);
  return q;
}

// ---- boundary mapping: hydro/common.wgsl:433-539, hydro/boundary.wgsl:47-84 ----
// One axis: the in-range index standing for i, the velocity sign along that axis and the
// outflow-only side (+-1, 0 for none).
struct AxisMap { int i; int flip; int side; };
__device__ __forceinline__ AxisMap map_axis(int i, int n, int lo, int hi) {
  AxisMap m{i, 1, 0};
  if (i >= 0 && i < n) return m;
  bool up = i >= n;
  int k = up ? hi : lo;
  if (k == BC_PERIODIC) {
    int v = up ? i - n : i + n;
    m.i = v < 0 ? 0 : (v > n - 1 ? n - 1 : v);
  } else if (k == BC_REFLECT) {
    m.i = up ? 2 * n - 1 - i : -1 - i;
    m.flip = -1;
  } else {
    m.i = up ? n - 1 : 0;
    if (k == BC_OUTFLOW_ONLY) m.side = up ? 1 : -1;
  }
  // (a reflecting axis of one or two cells, or a ragged tile's rim, can reach further than n
  // beyond the face: keep every index in range)
  m.i = m.i < 0 ? 0 : (m.i > n - 1 ? n - 1 : m.i);
  return m;
}
// bc_velocity (common.wgsl:536-539) on one component
template <typename T>
__device__ __forceinline__ T bc_vel(T v, int flip, int side) {
  T w = flip < 0 ? -v : v;
  if (side != 0) {
    T sd = T(side);
    w = tmax(w * sd, T(0)) * sd;
  }
  return w;
}

// ---- limiters: hydro/limiters/*.wgsl, per channel ----
// Increments are kept as the step from a cell's centre to its face, half of the reference's
// (which halves them at each use): every factor left out is a power of two, so the values are
// the same, and the symmetric limiters lose two doublings per channel.
//
// Koren's smoothness measure of a channel (koren.wgsl:274-292) is the difference energy over the
// square of its natural scale s = 0.01 scale. Here the differences are scaled by 1/|s| and then
// squared, which neither over- nor underflows; a zero scale stands for 1e-15, the root of the
// reference's smallest s^2. It depends on the scale alone and is formed once per scale (a cell's
// six channels have four: rho, c_s three times, p, none).
template <typename T>
__device__ __forceinline__ T edge_scale(T scale) {
  const T s = tabs(T(0.01) * scale);
  return s == T(0) ? T(1e15) : trcp(tmax(s, T(1e-37)));
}

// Koren's blend weight of a channel from its two differences: the same for the cell's up and
// down edges, so a pair of edges forms it once.
template <typename T>
__device__ __forceinline__ T koren_weight(T below, T above, T k) {
  const T b = below * k, a = above * k;
  const T e = T(1.5) - b * b;
  return tclamp(e - a * a, T(0), T(1));
}
// Koren's increment toward the face `near` lies on (least: the minmod of the two), blended by w from
// the limited value to the plain one (w = 1 gives the plain one exactly: the limited value is no
// larger). The early return of koren.wgsl gives the blend's value per channel, so each channel is formed on its own.
template <typename T>
__device__ __forceinline__ T koren_edge(T far, T near, T least, T w) {
  const T fr = (far + T(2) * near) * T(1.0 / 6.0);
  // sign(near) min(|far|, |near|, |fr|) where far and near share a sign (fr then does too)
  return tmix(minmod(least, fr), fr, w);
}
// The symmetric limiters' increment from the two differences, the same toward both faces
template <typename T, int LIM>
__device__ __forceinline__ T sym_edge(T below, T above) {
  if constexpr (LIM == LIM_MC) {
    // sign min(|below|, |above|, |below + above| / 4) where the two share a sign
    return minmod(below, minmod(above, T(0.25) * (below + above)));
  } else if constexpr (LIM == LIM_MINMOD) {
    return T(0.5) * minmod(below, above);
  } else {
    return same_sign(below, above) ? below * tdiv(above, below + above) : T(0);
  }
}
template <int LIM> constexpr bool lim_symmetric() { return LIM != LIM_KOREN; }

// The increment of one channel toward the upper (UP) or lower face; k: edge_scale of the
// channel's scale (Koren)
template <typename T, int LIM, bool UP>
__device__ __forceinline__ T edge1(T below, T above, T k) {
  if constexpr (LIM == LIM_KOREN) {
    const T w = koren_weight(below, above, k);
    const T least = minmod(below, above);
    return UP ? koren_edge(below, above, least, w) : koren_edge(above, below, least, w);
  } else {
    return sym_edge<T, LIM>(below, above);
  }
}

// The increment of each reconstructed channel (rho, vx, vy, vz, p, s) toward a face.
template <typename T>
struct Inc { T rho, vx, vy, vz, p, s; };

// isen_inc / isen_blend (hydro/q.wgsl:183-213) with no reference state and no potential, in two
// parts: what depends only on the three cells (the densities along the adiabat through the
// centre, the smoothness, adiabat and shear switches), shared by a cell's up and down edges, and
// the edge's own blend. Everything that divides by the centre's pressure shares one reciprocal:
// (p_c / p)^(1/gamma) is taken as (p / p_c)^(-1/gamma).
template <typename T>
struct IsenCommon { bool ok; T gi, ipc, tl, tr, bound; };

template <typename T>
__device__ __forceinline__ IsenCommon<T> isen_common(const Params<T>& P, const Prim<T>& l, const Prim<T>& c,
                                                     const Prim<T>& r) {
  const T ISEN_SMOOTH = T(0.2), ISEN_ADIABAT = T(0.01), ISEN_SHEAR = T(0.1), ISEN_ROOM = T(0.01), ISEN_CAP = T(0.25);
  IsenCommon<T> k;
  // (the unassembled edge texels of a block are zeros)
  k.ok = raw_min(raw_min(raw_min(l.rho, l.p), raw_min(c.rho, c.p)), raw_min(r.rho, r.p)) > T(0);
  k.gi = trcp(P.gamma);
  k.ipc = trcp(c.p);
  k.tl = l.rho * tpow(l.p * k.ipc, -k.gi) - c.rho;
  k.tr = r.rho * tpow(r.p * k.ipc, -k.gi) - c.rho;
  T ks = tclamp(T(2) - tmax(tabs(l.p - c.p), tabs(r.p - c.p)) * (k.ipc * T(1.0 / ISEN_SMOOTH)), T(0), T(1));
  T ka = tclamp(T(2) - tdiv(tmax(tabs(k.tl), tabs(k.tr)), ISEN_ADIABAT * c.rho), T(0), T(1));
  T dxr = r.vx - c.vx, dyr = r.vy - c.vy, dzr = r.vz - c.vz;
  T dxl = c.vx - l.vx, dyl = c.vy - l.vy, dzl = c.vz - l.vz;
  T dv = tsqrt(tmax(dxr * dxr + dyr * dyr + dzr * dzr, dxl * dxl + dyl * dyl + dzl * dzl));
  T kv = tclamp(T(2) - tdiv(dv, ISEN_SHEAR * tmax(c.cs, T(1e-30))), T(0), T(1));
  // how far the blend may move the density, as an increment
  const T room = (T(0.5) * ISEN_ROOM) * c.rho * ks * ka * kv;
  k.bound = tmax((T(0.5) * ISEN_CAP) * tmin(tabs(c.rho - l.rho), tabs(r.rho - c.rho)), room);
  return k;
}

// x, bx: the increments of density and pressure toward the face; d: the limited increment of the
// densities along the adiabat; wn: the density beyond the face
template <typename T, bool UP>
__device__ __forceinline__ T isen_blend(const IsenCommon<T>& k, const Prim<T>& c, T wn, T x, T bx, T d) {
  const T sgn = UP ? T(1) : T(-1);
  const T pf = c.p + sgn * bx;
  const T rf = tbetween((c.rho + sgn * d) * tpow(tmax(pf, T(1e-30)) * k.ipc, k.gi), c.rho, wn);
  const T i0 = sgn * (rf - c.rho);
  return k.ok ? x + tclamp(i0 - x, -k.bound, k.bound) : x;
}

// What one axis's edges of a cell share: the differences to its two neighbours, Koren's scales,
// the isentropic terms.
template <typename T>
struct EdgeTerms {
  Inc<T> below, above;
  T krho, kv, kp, k0;
  IsenCommon<T> isen;
};

template <typename T, int LIM, bool ISEN>
__device__ __forceinline__ EdgeTerms<T> edge_terms(const Params<T>& P, const Prim<T>& l, const Prim<T>& c,
                                                   const Prim<T>& r) {
  EdgeTerms<T> e{};
  e.below = Inc<T>{c.rho - l.rho, c.vx - l.vx, c.vy - l.vy, c.vz - l.vz, c.p - l.p, c.s - l.s};
  e.above = Inc<T>{r.rho - c.rho, r.vx - c.vx, r.vy - c.vy, r.vz - c.vz, r.p - c.p, r.s - c.s};
  if constexpr (LIM == LIM_KOREN) {
    e.krho = edge_scale(c.rho); e.kv = edge_scale(c.cs); e.kp = edge_scale(c.p); e.k0 = edge_scale(T(0));
  }
  if constexpr (ISEN) e.isen = isen_common(P, l, c, r);
  return e;
}

// edge_up (UP) / edge_dn (hydro/q.wgsl:214-239), no potential.
template <typename T, int LIM, bool ISEN, bool UP>
__device__ __forceinline__ Inc<T> edge_of(const EdgeTerms<T>& e, const Prim<T>& l, const Prim<T>& c, const Prim<T>& r) {
  Inc<T> o;
  o.rho = edge1<T, LIM, UP>(e.below.rho, e.above.rho, e.krho);
  o.vx = edge1<T, LIM, UP>(e.below.vx, e.above.vx, e.kv);
  o.vy = edge1<T, LIM, UP>(e.below.vy, e.above.vy, e.kv);
  o.vz = edge1<T, LIM, UP>(e.below.vz, e.above.vz, e.kv);
  o.p = edge1<T, LIM, UP>(e.below.p, e.above.p, e.kp);
  o.s = edge1<T, LIM, UP>(e.below.s, e.above.s, e.k0);
  if constexpr (ISEN) {
    const T d = edge1<T, LIM, UP>(-e.isen.tl, e.isen.tr, e.krho);
    o.rho = isen_blend<T, UP>(e.isen, c, UP ? r.rho : l.rho, o.rho, o.p, d);
  }
  return o;
}
template <typename T, int LIM, bool ISEN, bool UP>
__device__ __forceinline__ Inc<T> edge(const Params<T>& P, const Prim<T>& l, const Prim<T>& c, const Prim<T>& r) {
  return edge_of<T, LIM, ISEN, UP>(edge_terms<T, LIM, ISEN>(P, l, c, r), l, c, r);
}

// Half-step state (hydro/predictor.wgsl:46-209): rho, v, p, s at t + dt/2, the shock flag and
// the first-order flag.
template <typename T>
struct Half { T rho, vx, vy, vz, p, s, shock, fo; };

// One axis's contribution to the predictor: the slope (the up increment of a symmetric limiter,
// half of the face-to-face slope; the sum of Koren's two, all of it: slope_step takes the factor)
// and the positivity terms.
template <typename T>
struct AxisSlope { Inc<T> s; T big; T fall; };

template <typename T, int LIM, bool ISEN>
__device__ __forceinline__ AxisSlope<T> axis_slope(const Params<T>& P, const Prim<T>& m, const Prim<T>& q,
                                                   const Prim<T>& p, Inc<T>* up_out, Inc<T>* dn_out) {
  AxisSlope<T> r;
  // a cell's up and down edges share their differences, Koren's weights and the isentropic terms
  const EdgeTerms<T> e = edge_terms<T, LIM, ISEN>(P, m, q, p);
  const Inc<T> u = edge_of<T, LIM, ISEN, true>(e, m, q, p);
  if constexpr (lim_symmetric<LIM>()) {
    r.s = u;
    r.big = tabs(u.p);
    r.fall = -tabs(u.rho);
    if (up_out) *up_out = u;
    if (dn_out) *dn_out = u;
  } else {
    const Inc<T> d = edge_of<T, LIM, ISEN, false>(e, m, q, p);
    r.s.rho = u.rho + d.rho;
    r.s.vx = u.vx + d.vx;
    r.s.vy = u.vy + d.vy;
    r.s.vz = u.vz + d.vz;
    r.s.p = u.p + d.p;
    r.s.s = u.s + d.s;
    r.big = tmax(tabs(u.p), tabs(d.p));
    r.fall = tmin(u.rho, -d.rho);
    if (up_out) *up_out = u;
    if (dn_out) *dn_out = d;
  }
  return r;
}
// What the half step multiplies an axis's slope by: half a step's dt / dx for a whole slope
template <typename T, int LIM>
__device__ __forceinline__ T slope_step(const Params<T>& P, T dt) {
  return lim_symmetric<LIM>() ? tratio(dt, P.dx) : tratio(T(0.5) * dt, P.dx);
}

// Shock detector (predictor.wgsl:114-134): converging flow and a relative pressure jump across
// the cell above the threshold, |p+ - p-| / min(p+, p-) > thresh. jump_over is positive where
// that holds along an axis (the product form: no reciprocal).
template <typename T>
__device__ __forceinline__ T jump_over(const Params<T>& P, T pm, T pp) {
  return tabs(pp - pm) - P.shock_thresh * raw_min(pp, pm);
}

// The Hancock half step from the cell, the three axis slopes, and for the shock detector the
// convergence and the largest jump_over; h: slope_step. gamma p is the rho c_s^2 of
// predictor.wgsl, without the sound speed's root.
template <typename T, int LIM>
__device__ __forceinline__ Half<T> hancock(const Params<T>& P, const Prim<T>& q, const AxisSlope<T> sl[3],
                                           T conv, T jump, T h) {
  Half<T> o;
  T big = tmax(tmax(sl[0].big, sl[1].big), sl[2].big);
  T fall = tmin(tmin(tmin(T(0), sl[0].fall), sl[1].fall), sl[2].fall);
  T shock = (conv < T(0) && jump > T(0)) ? T(1) : T(0);
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
  o.p = q.p - h * (db0 + P.gamma * q.p * dv);
  o.s = q.s - h * db1;
  o.shock = shock;
  T rmin = o.rho + fall;
  T pmin = o.p - big;
  o.fo = T(0);
  if (!(rmin > T(0) && pmin > T(0))) {
    o.rho = q.rho; o.vx = q.vx; o.vy = q.vy; o.vz = q.vz; o.p = q.p; o.s = q.s;
    o.fo = T(1);
  }
  return o;
}

// The half step of a cell of a flat grid (one layer along z) from its four neighbours: hancock
// without the z axis, whose neighbours are the cell itself (predictor.wgsl:46-209 with a zero
// z slope, no z convergence and no z jump). The terms left out are zeros, so the result is
// hancock's but for the sign of a zero. ixu .. iyd (may be null) receive the x and y edge
// increments.
template <typename T, int LIM, bool ISEN>
__device__ __forceinline__ Half<T> half_flat(const Params<T>& P, const Prim<T>& q, const Prim<T>& xm,
                                             const Prim<T>& xp, const Prim<T>& ym, const Prim<T>& yp, T h,
                                             Inc<T>* ixu, Inc<T>* ixd, Inc<T>* iyu, Inc<T>* iyd) {
  const AxisSlope<T> ax = axis_slope<T, LIM, ISEN>(P, xm, q, xp, ixu, ixd);
  const AxisSlope<T> ay = axis_slope<T, LIM, ISEN>(P, ym, q, yp, iyu, iyd);
  const T conv = (xp.vx - xm.vx) + (yp.vy - ym.vy);
  const T jump = tmax(jump_over(P, xm.p, xp.p), jump_over(P, ym.p, yp.p));
  Half<T> o;
  T big = tmax(ax.big, ay.big);
  T fall = tmin(tmin(T(0), ax.fall), ay.fall);
  T shock = (conv < T(0) && jump > T(0)) ? T(1) : T(0);
  T rho = q.rho;
  const Inc<T>& sx = ax.s;
  const Inc<T>& sy = ay.s;
  T dv = sx.vx + sy.vy;
  T da0 = q.vx * sx.rho + q.vy * sy.rho;
  T da1 = q.vx * sx.vx + q.vy * sy.vx;
  T da2 = q.vx * sx.vy + q.vy * sy.vy;
  T da3 = q.vx * sx.vz + q.vy * sy.vz;
  T db0 = q.vx * sx.p + q.vy * sy.p;
  T db1 = q.vx * sx.s + q.vy * sy.s;
  T ir = trcp(rho);
  o.rho = rho - h * (da0 + rho * dv);
  o.vx = q.vx - h * (da1 + sx.p * ir);
  o.vy = q.vy - h * (da2 + sy.p * ir);
  o.vz = q.vz - h * da3;
  o.p = q.p - h * (db0 + P.gamma * q.p * dv);
  o.s = q.s - h * db1;
  o.shock = shock;
  T rmin = o.rho + fall;
  T pmin = o.p - big;
  o.fo = T(0);
  if (!(rmin > T(0) && pmin > T(0))) {
    o.rho = q.rho; o.vx = q.vx; o.vy = q.vy; o.vz = q.vz; o.p = q.p; o.s = q.s;
    o.fo = T(1);
  }
  return o;
}

// ---- face: hydro/flux.wgsl:60-125, riemann/hllc.wgsl, riemann/hll.wgsl ----
template <typename T>
struct Flux { T m, mx, my, mz, e, ei, s, vn; };

// One side of a face (to_side, flux.wgsl:60-85) in the face frame: n normal, t1/t2 the
// cyclically following components (rot, flux.wgsl:37-41); pr = p / rho. lo_rho, lo_p: the face's
// lower bounds, floors included.
template <typename T>
struct Side { T rho, vn, vt1, vt2, p, s, cs, pr; };

template <typename T>
__device__ __forceinline__ Side<T> make_side(const Params<T>& P, T rho, T vn, T vt1, T vt2, T p, T s, T lo_rho, T lo_p) {
  Side<T> o;
  o.rho = raw_max(rho, lo_rho);
  o.vn = vn; o.vt1 = vt1; o.vt2 = vt2;
  o.s = s;
  o.p = raw_max(p, lo_p);
  o.pr = tdiv(o.p, o.rho);
  o.cs = tsqrt(P.gamma * o.pr);
  return o;
}

// A side's total energy, momentum and normal flux (hllc.wgsl:7-28), for the HLL state
template <typename T>
struct SideFlux { T E, m0, m1, m2, f0, f1, f2, fe; };
template <typename T>
__device__ __forceinline__ SideFlux<T> side_flux(const Params<T>& P, const Side<T>& q) {
  SideFlux<T> o;
  o.E = q.p * P.igm1 + T(0.5) * q.rho * (q.vn * q.vn + q.vt1 * q.vt1 + q.vt2 * q.vt2);
  o.m0 = q.rho * q.vn; o.m1 = q.rho * q.vt1; o.m2 = q.rho * q.vt2;
  o.f0 = o.m0 * q.vn + q.p; o.f1 = o.m1 * q.vn; o.f2 = o.m2 * q.vn;
  o.fe = (o.E + q.p) * q.vn;
  return o;
}

// HLLC, taken to HLL where w is not zero (riemann/hllc.wgsl:4-85, whose blend weight is a flag), or
// HLL (riemann/hll.wgsl:87-121).
//
// The supersonic and the two star states go through one set of expressions, so that a wave whose
// faces differ in them does not run each in turn: the side K the face's fluxes come from, its
// wave speed S, and u the normal velocity of the state at the face, which is the contact's speed
// sm between the waves and K's own where K is supersonic (the star state is then K's state itself,
// taken as it is). With d = S - u_K and 1/(S - u),
//   rho* = rho d / (S - u),  p* = p + rho d (u - u_K),  E* = (E d - p u_K + p* u) / (S - u)
// and the flux is (rho* u, rho* u^2 + p*, rho* u v_t, (E* + p*) u): the star flux of
// hllc.wgsl:52-74 by the jump conditions, with one reciprocal where that form takes three. The
// mass flux has the sign of u, which is also what K was picked by, so the internal energy and the
// scalar it carries are K's.
template <typename T, int RS>
__device__ __forceinline__ Flux<T> riemann(const Params<T>& P, const Side<T>& l, const Side<T>& r, T w_hll) {
  const T sl = tmin(l.vn - l.cs, r.vn - r.cs);
  const T sr = tmax(l.vn + l.cs, r.vn + r.cs);
  const T ql = l.rho * (sl - l.vn);
  const T qr = r.rho * (sr - r.vn);
  const T sm = tdiv(r.p - l.p + l.vn * ql - r.vn * qr, ql - qr);
  const bool up_l = sl >= T(0), up_r = sr <= T(0), super = up_l || up_r;
  const bool left = up_l || (!up_r && sm >= T(0));
  const T S = left ? sl : sr;
  const T rho = left ? l.rho : r.rho;
  const T un = left ? l.vn : r.vn;
  const T u1 = left ? l.vt1 : r.vt1;
  const T u2 = left ? l.vt2 : r.vt2;
  const T p = left ? l.p : r.p;
  const T E = p * P.igm1 + T(0.5) * rho * (un * un + u1 * u1 + u2 * u2);
  const T u = super ? un : sm;
  const T d = S - un;
  const T inv = trcp(S - u);
  const T ps = p + (rho * d) * (u - un);
  const T rs = super ? rho : rho * d * inv;
  const T es = super ? E : (E * d - p * un + ps * u) * inv;
  Flux<T> o;
  o.m = rs * u;
  o.mx = o.m * u + ps;
  o.my = o.m * u1;
  o.mz = o.m * u2;
  o.e = (es + ps) * u;
  o.ei = o.m * ((left ? l.pr : r.pr) * P.igm1);
  o.s = o.m * (left ? l.s : r.s);
  o.vn = u;
  // The HLL state between the waves: the flux itself where the star densities are not positive (a
  // sound speed of zero, or below the rounding of the velocity: else ql < 0 < qr), for HLL, and
  // where the face is flagged.
  const bool star = ql < T(0) && qr > T(0);
  if (!super && (RS == RS_HLL || !star || w_hll != T(0))) {
    const SideFlux<T> a = side_flux(P, l);
    const SideFlux<T> b = side_flux(P, r);
    const T ih = trcp(sr - sl);
    const T slsr = sl * sr;
    o.m = (sr * a.m0 - sl * b.m0 + slsr * (r.rho - l.rho)) * ih;
    o.mx = (sr * a.f0 - sl * b.f0 + slsr * (b.m0 - a.m0)) * ih;
    o.my = (sr * a.f1 - sl * b.f1 + slsr * (b.m1 - a.m1)) * ih;
    o.mz = (sr * a.f2 - sl * b.f2 + slsr * (b.m2 - a.m2)) * ih;
    o.e = (sr * a.fe - sl * b.fe + slsr * (b.E - a.E)) * ih;
    if (RS != RS_HLL && !star) o.vn = T(0.5) * (l.vn + r.vn);
    const bool up = o.m >= T(0);
    o.ei = o.m * ((up ? l.pr : r.pr) * P.igm1);
    o.s = o.m * (up ? l.s : r.s);
  }
  return o;
}

// One cell's side of a face before the face's own lower bound and floors: the half-step state
// plus the edge increment toward the face (to_side, flux.wgsl:60-63; zero increment for a
// first-order cell), with the cell's share of the face's lower bounds, half its half-step density
// and pressure and at least the floors (flux.wgsl:109-117), and its shock flag (flux.wgsl:93).
template <typename T>
struct SideData { T rho, vx, vy, vz, p, s, hrho, hp, shock; };

// sgn = +1 for the cell's upper face (il its up increment), -1 for its lower face.
template <typename T>
__device__ __forceinline__ SideData<T> side_of(const Params<T>& P, const Half<T>& h, const Inc<T>& inc, T sgn) {
  T hs = sgn * (T(1) - h.fo);
  SideData<T> o;
  o.rho = h.rho + hs * inc.rho;
  o.vx = h.vx + hs * inc.vx;
  o.vy = h.vy + hs * inc.vy;
  o.vz = h.vz + hs * inc.vz;
  o.p = h.p + hs * inc.p;
  o.s = h.s + hs * inc.s;
  o.hrho = tmax(T(0.5) * h.rho, P.rho_floor);
  o.hp = tmax(T(0.5) * h.p, P.p_floor);
  o.shock = h.shock;
  return o;
}

// face_flux (flux.wgsl:92-125) from the left cell's upper side and the right cell's lower side
// along `axis`. Momentum comes back in grid components.
template <typename T, int RS>
__device__ __forceinline__ Flux<T> face_from_sides(const Params<T>& P, const SideData<T>& L, const SideData<T>& R,
                                                   int axis) {
  T w = L.shock + R.shock;   // flags: zero where neither cell has one
  T lo_rho = raw_min(L.hrho, R.hrho);
  T lo_p = raw_min(L.hp, R.hp);
  // rot (flux.wgsl:37-41): axis 0 -> (x, y, z), 1 -> (y, z, x), 2 -> (z, x, y)
  T ln, l1, l2, rn, r1, r2;
  if (axis == 0) { ln = L.vx; l1 = L.vy; l2 = L.vz; rn = R.vx; r1 = R.vy; r2 = R.vz; }
  else if (axis == 1) { ln = L.vy; l1 = L.vz; l2 = L.vx; rn = R.vy; r1 = R.vz; r2 = R.vx; }
  else { ln = L.vz; l1 = L.vx; l2 = L.vy; rn = R.vz; r1 = R.vx; r2 = R.vy; }
  Side<T> sl = make_side(P, L.rho, ln, l1, l2, L.p, L.s, lo_rho, lo_p);
  Side<T> sr = make_side(P, R.rho, rn, r1, r2, R.p, R.s, lo_rho, lo_p);
  Flux<T> F = riemann<T, RS>(P, sl, sr, w);
  // unrot: the face frame's (n, t1, t2) back to grid components
  T n = F.mx, t1 = F.my, t2 = F.mz;
  if (axis == 0) { F.mx = n; F.my = t1; F.mz = t2; }
  else if (axis == 1) { F.mx = t2; F.my = n; F.mz = t1; }
  else { F.mx = t1; F.my = t2; F.mz = n; }
  return F;
}

// face_from_sides for an axis known only at run time: the velocities are rotated into the face
// frame here and the face solved as one along x, the same values in the same order as
// face_from_sides(axis). The components are picked from registers (the empty asm makes them
// opaque values): picking them from the side structs lets the compiler select by address, which
// puts both sides in scratch memory.
template <typename T, int RS>
__device__ __forceinline__ Flux<T> face_from_sides_rt(const Params<T>& P, SideData<T> L, SideData<T> R, int axis) {
  T lx = L.vx, ly = L.vy, lz = L.vz, rx = R.vx, ry = R.vy, rz = R.vz;
  asm("" : "+v"(lx), "+v"(ly), "+v"(lz), "+v"(rx), "+v"(ry), "+v"(rz));
  const bool a0 = axis == 0, a1 = axis == 1;
  L.vx = a0 ? lx : (a1 ? ly : lz); L.vy = a0 ? ly : (a1 ? lz : lx); L.vz = a0 ? lz : (a1 ? lx : ly);
  R.vx = a0 ? rx : (a1 ? ry : rz); R.vy = a0 ? ry : (a1 ? rz : rx); R.vz = a0 ? rz : (a1 ? rx : ry);
  Flux<T> F = face_from_sides<T, RS>(P, L, R, 0);
  T n = F.mx, t1 = F.my, t2 = F.mz;
  asm("" : "+v"(n), "+v"(t1), "+v"(t2));
  F.mx = a0 ? n : (a1 ? t2 : t1); F.my = a0 ? t1 : (a1 ? n : t2); F.mz = a0 ? t2 : (a1 ? t1 : n);
  return F;
}

// face_flux between the half-step states hl (left) and hr (right), given the increments
// from each cell toward the face (il: the left cell's up increment, ir: the right cell's down
// increment), along a run-time axis.
template <typename T, int RS>
__device__ __forceinline__ Flux<T> face_flux(const Params<T>& P, const Half<T>& hl, const Inc<T>& il,
                                             const Half<T>& hr, const Inc<T>& ir, int axis) {
  return face_from_sides_rt<T, RS>(P, side_of(P, hl, il, T(1)), side_of(P, hr, ir, T(-1)), axis);
}

// advance (hydro/advance.wgsl:31-52), dual_energy (hydro/dual_energy.wgsl:73-87) and the
// tenuous-gas limits (hydro/fluff.wgsl:195-205). net is the net inflow per unit dt/dx.
template <typename T>
__device__ __forceinline__ void advance(const Params<T>& P, T4<T> u1, T4<T> u2, const Flux<T>& net, T p_half, T dtdx,
                                        T4<T>& o1, T4<T>& o2) {
  T rho = tmax(u1.x + dtdx * net.m, P.rho_floor);
  T mx = u1.y + dtdx * net.mx;
  T my = u1.z + dtdx * net.my;
  T mz = u1.w + dtdx * net.mz;
  T E = u2.x + dtdx * net.e;
  T pdv = tmax(p_half, P.p_floor) * net.vn;
  T eint = u2.y + dtdx * (net.ei + pdv);
  T sc = u2.z + dtdx * net.s;
  T ke = tdiv(T(0.5) * (mx * mx + my * my + mz * mz), rho);
  T eth = E - ke;
  T emin = P.p_floor * P.igm1;
  T en0, en1;
  if (eth > P.eta_dual * E && eth >= emin && eth >= T(0)) {
    en0 = E; en1 = eth;
  } else {
    T ei = eint;
    if (!(ei >= emin)) ei = emin;
    en0 = ke + ei; en1 = ei;
  }
  if (rho < P.fluff[0]) {
    bool changed = false;
    T emax = rho * P.fluff[1];
    if (en1 > emax) { en1 = emax; changed = true; }
    T pmax = rho * P.fluff[2];
    T pm = tsqrt(mx * mx + my * my + mz * mz);
    if (pm > pmax) { T f = tdiv(pmax, pm); mx *= f; my *= f; mz *= f; changed = true; }
    if (changed) en0 = tdiv(T(0.5) * (mx * mx + my * my + mz * mz), rho) + en1;
  }
  o1.x = rho; o1.y = mx; o1.z = my; o1.w = mz;
  o2.x = en0; o2.y = en1; o2.z = sc; o2.w = T(0);
}

// Net inflow (flux.wgsl:385-394) from the lower and upper face of each axis.
template <typename T>
__device__ __forceinline__ Flux<T> net_of(const Flux<T>& xl, const Flux<T>& xh, const Flux<T>& yl, const Flux<T>& yh,
                                          const Flux<T>& zl, const Flux<T>& zh) {
  Flux<T> n;
  n.m = ((xl.m - xh.m) + (yl.m - yh.m)) + (zl.m - zh.m);
  n.mx = ((xl.mx - xh.mx) + (yl.mx - yh.mx)) + (zl.mx - zh.mx);
  n.my = ((xl.my - xh.my) + (yl.my - yh.my)) + (zl.my - zh.my);
  n.mz = ((xl.mz - xh.mz) + (yl.mz - yh.mz)) + (zl.mz - zh.mz);
  n.e = ((xl.e - xh.e) + (yl.e - yh.e)) + (zl.e - zh.e);
  n.ei = ((xl.ei - xh.ei) + (yl.ei - yh.ei)) + (zl.ei - zh.ei);
  n.s = ((xl.s - xh.s) + (yl.s - yh.s)) + (zl.s - zh.s);
  n.vn = ((xl.vn - xh.vn) + (yl.vn - yh.vn)) + (zl.vn - zh.vn);
  return n;
}

// The signal rate of a cell (hydro/rates.wgsl:60-62).
template <typename T>
__device__ __forceinline__ T rate_of(const Params<T>& P, const Prim<T>& w) {
  return tabs(w.vx) + tabs(w.vy) + tabs(w.vz) + P.ndim * w.cs;
}

// Non-negative floats order as their bit patterns: the reductions compare those.
__device__ __forceinline__ uint32_t order_bits(float x) { return __float_as_uint(x); }
__device__ __forceinline__ unsigned long long order_bits(double x) { return (unsigned long long)__double_as_longlong(x); }

// The clock pass (hydro/clock.wgsl:132-242) on one thread: bank the step just taken
// (Kahan-summed t), then dt = cfl dx / max rate, clamped by dt_max and the end time.
// clk = (dt, t, tc, steps, ...11 entries).
template <typename T>
__device__ __forceinline__ void clock_pass(const Params<T>& P, T* clk, T max_rate) {
  T prev = clk[0];
  if (prev > T(0)) {
    T y = prev - clk[2];
    T t = clk[1] + y;
    T d = t - clk[1];
    clk[2] = d - y;
    clk[1] = t;
    clk[3] = clk[3] + T(1);
  }
  T dt = tquot(P.cfl * P.dx, tmax(max_rate, T(1e-30)));
  dt = tmin(dt, P.dt_max);
  T remaining = P.t_end - clk[1];
  if (remaining <= T(1e-6) * tabs(P.t_end)) dt = T(0);
  else dt = tmin(dt, remaining);
  if (T(1e30) - clk[1] < T(0.5) * dt) dt = T(0);
  if (clk[10] != T(0)) dt = T(0);
  clk[0] = dt;
}

}  // namespace shx
