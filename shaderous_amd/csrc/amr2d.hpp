// The step of 2D block grids (quadtrees of 16^2-cell blocks): the leaves' ghosts in one kernel,
// then one in which a workgroup takes a leaf's cells and ghosts into LDS, predicts, solves the
// faces and updates, where the passes (amr_impl.hpp) carry the cells' texels (W) and half steps
// (PA, PB) through HBM, ten times the state's own bytes. The ghosts stay apart: their chain of table
// and cell reads needs more waves in flight than a workgroup with a leaf in LDS leaves room for
// (formed inside, the two launches for 3136 leaves took 72 and 34 us against 21 + 34 and 16). The
// values are the passes':
//  - threads 0-255 the cells, 256-319 the first layer of face ghosts, 320-383 the second
//    (af_column);
//  - a ghost's half step "at source" (amr/predict.wgsl:183-221): beside a same-level leaf the
//    texels here are the ones that leaf's own predictor reads, but for a ghost at a face's end,
//    whose stencil reaches past the face: that texel, as the leaf across assembles it, is formed
//    besides (two per face, kept in PA's and PB's corners, which nothing else uses); beside a
//    coarser block in place with masked slopes; a boundary image's from the cell it images;
//  - coarse-fine faces through a flux register, as the fused 3D march's: a leaf writes the fluxes
//    of its faces on a coarser block, and the leaves with a refined neighbour, in a second launch,
//    take the means of the two fine fluxes (match_faces). The first launch steps the other leaves,
//    and of the second's those with a coarser neighbour run up to their register fluxes.
// The step's rate is taken from the cells in the ghosts' launch, as the assembly takes it.
#pragma once
#include "amr_fused.hpp"

namespace shx {

// LDS: the columns of the 20 x 20 plane and the eight texels at the faces' ends; the fluxes take
// the primitives' place. 54 KB: three workgroups per CU.
constexpr int FL_ENDS = AF_NT, FL_NT = AF_NT + 8;
template <typename T>
struct FlatLds : ColumnLds<T, FL_NT> {
  static constexpr int Q = 0, FX = 0, FY = 8 * FL_NT, SX = 16 * FL_NT, SY = 24 * FL_NT, SK = 32 * FL_NT,
                       SIZE = 33 * FL_NT;
};

template <typename T>
__device__ __forceinline__ Inc<T> pick_inc(bool k, const Inc<T>& a, const Inc<T>& b) {
  Inc<T> o;
  o.rho = k ? a.rho : b.rho; o.vx = k ? a.vx : b.vx; o.vy = k ? a.vy : b.vy;
  o.vz = k ? a.vz : b.vz; o.p = k ? a.p : b.p; o.s = k ? a.s : b.s;
  return o;
}

// The mean of the two fine fluxes through the face of cell (x, y) on side k, from the register of
// the refined neighbour np's child (fine_face's order)
template <typename T, bool COMP>
__device__ __forceinline__ Flux<T> reg_mean_flat(const int* __restrict__ tab, const int* __restrict__ reg_of,
                                                 const T* __restrict__ R, int np, int k, int x, int y,
                                                 const Flux<T>& fallback) {
  const int upper = !(k & 1), l = k < 2 ? y : x, half = l >= AMR_BS / 2;
  const int ch = bt(tab, np, BT_CHILD + (k < 2 ? (upper | (half << 1)) : (half | (upper << 1))));
  const int reg = ch >= 0 ? reg_of[ch * 6 + (k ^ 1)] : -1;
  if (reg < 0) return fallback;   // not reached in a 2:1-balanced tree (checked at creation)
  const T4<T>* p = reinterpret_cast<const T4<T>*>(R + ((size_t)reg * AMR_BS + 2 * (l - (AMR_BS / 2) * half)) * 8);
  T sum[8], err[8];
#pragma unroll
  for (int q = 0; q < 8; q++) { sum[q] = T(0); err[q] = T(0); }
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const T4<T> a = p[2 * i], b = p[2 * i + 1];
    const T fv[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int q = 0; q < 8; q++) {
      if constexpr (COMP) {
        T e;
        two_sum(sum[q], fv[q], sum[q], e);
        err[q] = err[q] + e;
      } else {
        sum[q] = sum[q] + fv[q];
      }
    }
  }
  const T w = T(0.5);
  Flux<T> F;
  F.m = (sum[0] + err[0]) * w; F.mx = (sum[1] + err[1]) * w;
  F.my = (sum[2] + err[2]) * w; F.mz = (sum[3] + err[3]) * w;
  F.e = (sum[4] + err[4]) * w; F.ei = (sum[5] + err[5]) * w;
  F.s = (sum[6] + err[6]) * w; F.vn = (sum[7] + err[7]) * w;
  return F;
}

// The ghosts of the listed leaves into W (the texels the assembly leaves there), the texels past
// their faces' ends into the corners of PA and PB, and the largest rate / dx of their cells. The
// first workgroups take two leaves' 128 ghosts each, the next 32 leaves' eight end texels, the last
// (at most FL_RATES, so as many atomics) the cells in turn. Bound by the latency of the ghosts'
// reads.
constexpr int FL_RATES = 512;
__device__ __forceinline__ int flat_end(int e) {
  const int i = e & 1, j = (e >> 1) & 1;   // the corner at (i, j), its texel e / 4
  return (j * (AMR_BS + AMR_NG) + (e >> 2)) * AMR_PAD + i * (AMR_BS + AMR_NG);
}
template <typename T, int LIM>
__global__ __launch_bounds__(256) void k_amr_flat_ghosts(Params<T> P, const int* __restrict__ tab,
                                                         const int* __restrict__ list, int count,
                                                         const T4<T>* __restrict__ U1, const T4<T>* __restrict__ U2,
                                                         T4<T>* __restrict__ W1, T4<T>* __restrict__ W2,
                                                         T4<T>* __restrict__ PA, T4<T>* __restrict__ PB,
                                                         unsigned long long* slot) {
  constexpr int TEXELS = AmrGeo<2>::TEXELS;
  const int ghosts = (count + 1) / 2, ends = (count + 31) / 32;
  const int wg = blockIdx.x, tid = threadIdx.x;
  if (wg < ghosts + ends) {
    const bool ring = wg < ghosts;
    const int b = ring ? 2 * wg + (tid >> 7) : 32 * (wg - ghosts) + (tid >> 3);
    if (b >= count) return;
    const int s = list[b];
    int src = s, x, y;
    if (ring) {
      const int g = tid & 127, f = g >> 5, layer = (g >> 4) & 1, i = g & 15;
      const int a = (f & 1) ? AMR_BS + layer : -1 - layer;
      x = f < 2 ? a : i;
      y = f < 2 ? i : a;
    } else {
      // face f's lower and upper end, as the same-level leaf across assembles them
      const int e = tid & 7, f = e >> 1, end = (e & 1) ? AMR_BS : -1, in = (f & 1) ? 0 : AMR_BS - 1;
      src = same_leaf(tab, s, f);
      if (src < 0) return;
      x = f < 2 ? in : end;
      y = f < 2 ? end : in;
    }
    Prim<T> w;
    if (!amr_texel<T, LIM, 2>(P, tab, U1, U2, src, x, y, 0, w)) return;
    const size_t o = (size_t)s * TEXELS + (ring ? texd<2>(x, y, 0) : flat_end(tid & 7));
    (ring ? W1 : PA)[o] = v4<T>(w.rho, w.vx, w.vy, w.vz);
    (ring ? W2 : PB)[o] = v4<T>(w.p, w.cs, w.s, T(0));
    return;
  }
  T r = T(0);
  for (int b = wg - ghosts - ends; b < count; b += gridDim.x - ghosts - ends) {
    const int s = list[b];
    const size_t o = (size_t)s * AmrGeo<2>::CELLS + tid;
    r = tmax(r, tquot(rate_of(P, prim_from_cons(P, U1[o], U2[o])), level_dx(P, bt(tab, s, BT_LEVEL))));
  }
  block_max_to(r, slot);
}

// The rest of the step. Bound by VALU issue with the barriers between its three phases; three
// workgroups per CU (at most 96 VGPRs; at 100, two, the step below takes 5% longer). The adaptive
// shear layer's 3136 leaves (Koren, HLLC; 2176 plain, 896 of the others with a coarser neighbour):
// 106 us per step in passes (29 assembly, 30 half steps, 41
// updates, clock), 75 so (21 ghosts, 34 and 16 the two launches, clock); 352 leaves (MC) 38 -> 28 us.
template <typename T, int LIM, int RS, bool ISEN, bool MATCH, bool COMP>
__global__ __launch_bounds__(AF_THREADS, 5) void k_amr_flat(
    Params<T> G, const int* __restrict__ tab, const int* __restrict__ list, int nfull, const int* __restrict__ reg_of,
    T* __restrict__ R, const T4<T>* __restrict__ U1, const T4<T>* __restrict__ U2, const T4<T>* __restrict__ W1,
    const T4<T>* __restrict__ W2, const T4<T>* __restrict__ PA, const T4<T>* __restrict__ PB, T4<T>* __restrict__ O1,
    T4<T>* __restrict__ O2, const T* __restrict__ clk) {
  using FL = FlatLds<T>;
  constexpr int BX = AF_SIDE;
  __shared__ T4<T> LL[FL::SIZE / 4];
  T* const L = reinterpret_cast<T*>(LL);
  const int s = __builtin_amdgcn_readfirstlane(list[blockIdx.x]);
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid) >> 6;
  const bool cells = wave < 4;
  int x, y;
  af_column(tid, x, y);
  const typename FL::At t = FL::at((y + 2) * BX + (x + 2));
  const size_t o = (size_t)s * (AMR_BS * AMR_BS) + (cells ? y * AMR_BS + x : 0);
  T4<T> u1, u2;
  Prim<T> none, w;
  none.rho = none.vx = none.vy = none.vz = none.p = none.s = none.cs = T(0);
  if (cells) {
    u1 = U1[o];
    u2 = U2[o];
    // the corner columns are edges: zero, as in the atlas
    if (tid < 16) {
      const int i = tid & 3, j = tid >> 2;
      FL::put_prim(L, FL::Q, FL::at((j < 2 ? j : AMR_BS + j) * BX + (i < 2 ? i : AMR_BS + i)), none);
    }
    w = prim_from_cons(G, u1, u2);
  } else {
    const size_t g = (size_t)s * AmrGeo<2>::TEXELS;
    w = load_w<T>(W1, W2, g + texd<2>(x, y, 0));
    if (tid < 264) FL::put_prim(L, FL::Q, FL::at(FL_ENDS + tid - 256), load_w<T>(PA, PB, g + flat_end(tid - 256)));
  }
  FL::put_prim(L, FL::Q, t, w);
  const T dt = clk[0];
  Params<T> P = G;   // this block's
  P.dx = level_dx(G, bt(tab, s, BT_LEVEL));
  const T dtdx = wave_uniform(tratio(dt, P.dx)), hstep = wave_uniform(slope_step<T, LIM>(P, dt));
  __syncthreads();

  Half<T> h;
  SideData<T> xl, yl;   // the cell's lower sides; a ghost's one side in xl
  const int side = (tid >> 4) & 3, axis = side >> 1;
  const bool ring1 = wave == 4;
  if (cells) {
    const Prim<T> xm = FL::prim(L, FL::Q, t.off(-1)), xp = FL::prim(L, FL::Q, t.off(1));
    const Prim<T> ym = FL::prim(L, FL::Q, t.off(-BX)), yp = FL::prim(L, FL::Q, t.off(BX));
    Inc<T> xu, xd, yu, yd;
    h = half_flat<T, LIM, ISEN>(P, w, xm, xp, ym, yp, hstep, &xu, &xd, &yu, &yd);
    FL::put_side(L, FL::SX, t, side_of(P, h, xu, T(1)));
    FL::put_side(L, FL::SY, t, side_of(P, h, yu, T(1)));
    xl = side_of(P, h, xd, T(-1));
    yl = side_of(P, h, yd, T(-1));
    FL::put_shock(L, FL::SK, t, h.shock);
  } else if (ring1) {
    const int nb = bt(tab, s, BT_NB + side);
    const bool coarse = nb == -1, image = nb < -1, same = nb >= 0 && is_leaf(tab, nb);
    const int i = side < 2 ? y : x;
    // the texel whose half step it is (an image's cell), and its stencil
    const typename FL::At c = image ? FL::at((min(max(y, 0), AMR_BS - 1) + 2) * BX + min(max(x, 0), AMR_BS - 1) + 2) : t;
    const bool low = same && i == 0, high = same && i == AMR_BS - 1;   // a stencil past the face's end
    const typename FL::At e0 = FL::at(FL_ENDS + 2 * side), e1 = FL::at(FL_ENDS + 2 * side + 1);
    auto pick = [](bool k, const typename FL::At& m, const typename FL::At& n) {
      return typename FL::At{k ? m.a : n.a, k ? m.b : n.b, k ? m.c : n.c};
    };
    const Prim<T> xm = FL::prim(L, FL::Q, pick(low && axis == 1, e0, c.off(-1)));
    const Prim<T> xp = FL::prim(L, FL::Q, pick(high && axis == 1, e1, c.off(1)));
    const Prim<T> ym = FL::prim(L, FL::Q, pick(low && axis == 0, e0, c.off(-BX)));
    const Prim<T> yp = FL::prim(L, FL::Q, pick(high && axis == 0, e1, c.off(BX)));
    Prim<T> q = FL::prim(L, FL::Q, c);
    q.cs = w.cs;   // (an image's is its cell's)
    AxisSlope<T> sl[3];
    Inc<T> xu, xd, yu, yd;
    sl[0] = axis_slope<T, LIM, ISEN>(P, xm, q, xp, &xu, &xd);
    sl[1] = axis_slope<T, LIM, ISEN>(P, ym, q, yp, &yu, &yd);
    sl[2].s.rho = sl[2].s.vx = sl[2].s.vy = sl[2].s.vz = sl[2].s.p = sl[2].s.s = T(0);
    sl[2].big = sl[2].fall = T(0);
    if (coarse) {
      const T cut = (i == 0 || i == AMR_BS - 1) ? T(0) : T(1);
      scale_inc(sl[0].s, axis == 1 ? cut : T(1));
      scale_inc(sl[1].s, axis == 0 ? cut : T(1));
    }
    const T conv = (xp.vx - xm.vx) + (yp.vy - ym.vy);
    const T jump = tmax(jump_over(P, xm.p, xp.p), jump_over(P, ym.p, yp.p));
    h = hancock<T, LIM>(P, q, sl, conv, jump, hstep);
    const bool dn = side & 1;
    Inc<T> e = pick_inc(axis == 0, pick_inc(dn, xd, xu), pick_inc(dn, yd, yu));
    if (image) {
      const GSrc g = ghost_src(tab, s, x, y, 0);
      h.vx = bc_vel(h.vx, g.fx, g.sx);
      h.vy = bc_vel(h.vy, g.fy, g.sy);
      const int d = axis == 0 ? 1 : BX;
      Inc<T> eu, ed;
      (void)axis_slope<T, LIM, ISEN>(P, FL::prim(L, FL::Q, t.off(-d)), w, FL::prim(L, FL::Q, t.off(d)), &eu, &ed);
      e = pick_inc(dn, ed, eu);
    }
    xl = side_of(P, h, e, dn ? T(-1) : T(1));
    if (!dn) FL::put_side(L, axis == 0 ? FL::SX : FL::SY, t, xl);
    FL::put_shock(L, FL::SK, t, h.shock);
  }
  __syncthreads();

  // the first launch writes the register, for every leaf with a coarser neighbour; the second only
  // reads it (a store there, though of the same flux, would race with the coarser leaf's read)
  auto face = [&](int k, Flux<T> F) {
    if constexpr (!MATCH) {
      const int r = reg_of[s * 6 + k];
      if (r >= 0) {
        T4<T>* p = reinterpret_cast<T4<T>*>(R + ((size_t)r * AMR_BS + (k < 2 ? y : x)) * 8);
        p[0] = v4<T>(F.m, F.mx, F.my, F.mz);
        p[1] = v4<T>(F.e, F.ei, F.s, F.vn);
      }
    } else {
      const int np = bt(tab, s, BT_NB + k);
      if (np >= 0 && !is_leaf(tab, np))
        return reg_mean_flat<T, COMP>(tab, reg_of, R, np, k, min(max(x, 0), AMR_BS - 1), min(max(y, 0), AMR_BS - 1), F);
    }
    return F;
  };
  Flux<T> Fx, Fy;
  if (cells) {
    Fx = face_from_sides<T, RS>(P, FL::side(L, FL::SX, FL::SK, t.off(-1)), xl, 0);
    if (x == 0) Fx = face(0, Fx);
    FL::put_flux(L, FL::FX, t, Fx);
    Fy = face_from_sides<T, RS>(P, FL::side(L, FL::SY, FL::SK, t.off(-BX)), yl, 1);
    if (y == 0) Fy = face(2, Fy);
    FL::put_flux(L, FL::FY, t, Fy);
  } else if (ring1 && (side & 1)) {
    Flux<T> F = face_from_sides_rt<T, RS>(
        P, FL::side(L, axis == 0 ? FL::SX : FL::SY, FL::SK, t.off(axis == 0 ? -1 : -BX)), xl, axis);
    F = face(side, F);
    FL::put_flux(L, axis == 0 ? FL::FX : FL::FY, t, F);
  }
  if ((int)blockIdx.x >= nfull) return;   // its register fluxes alone
  __syncthreads();
  if (cells) {
    const Flux<T> net = net_of(Fx, FL::flux(L, FL::FX, t.off(1)), Fy, FL::flux(L, FL::FY, t.off(BX)), zero_flux<T>(),
                               zero_flux<T>());
    T4<T> o1, o2;
    advance(P, u1, u2, net, h.p, dtdx, o1, o2);
    O1[o] = o1;
    O2[o] = o2;
  }
}

template <typename T, int LIM, int RS, bool ISEN, int D>
void AmrImpl<T, LIM, RS, ISEN, D>::flat_ghosts(const AmrLaunch& L, const int* list, int count, const void* u1,
                                               const void* u2, void* w1, void* w2, void* pa, void* pb,
                                               unsigned long long* slot) {
  static_assert(D == 2, "the flat step is for 2D blocks");
  if (count <= 0) return;
  const int grid = (count + 1) / 2 + (count + 31) / 32 + (count < FL_RATES ? count : FL_RATES);
  hipLaunchKernelGGL((k_amr_flat_ghosts<T, LIM>), dim3(grid), dim3(256), 0, L.stream, P(L), L.tab, list, count,
                     (const T4<T>*)u1, (const T4<T>*)u2, (T4<T>*)w1, (T4<T>*)w2, (T4<T>*)pa, (T4<T>*)pb, slot);
}

template <typename T, int LIM, int RS, bool ISEN, int D>
void AmrImpl<T, LIM, RS, ISEN, D>::flat(const AmrLaunch& L, const int* list, int nfull, int count, bool match,
                                        bool compensated, const int* reg_of, void* reg, const void* u1,
                                        const void* u2, const void* w1, const void* w2, const void* pa,
                                        const void* pb, void* o1, void* o2, const void* clk) {
  static_assert(D == 2, "the flat step is for 2D blocks");
  if (count <= 0) return;
#define SHX_FLAT(M, C)                                                                                              \
  hipLaunchKernelGGL((k_amr_flat<T, LIM, RS, ISEN, M, C>), dim3(count), dim3(AF_THREADS), 0, L.stream, P(L), L.tab, \
                     list, nfull, reg_of, (T*)reg, (const T4<T>*)u1, (const T4<T>*)u2, (const T4<T>*)w1,            \
                     (const T4<T>*)w2, (const T4<T>*)pa, (const T4<T>*)pb, (T4<T>*)o1, (T4<T>*)o2, (const T*)clk)
  if (!match) SHX_FLAT(false, false);
  else if (compensated) SHX_FLAT(true, true);
  else SHX_FLAT(true, false);
#undef SHX_FLAT
}

}  // namespace shx
