// The fused block-AMR step for gfx950: two batched kernels over device lists of leaves compute
// what the reference's assemble, predict and update passes compute (src/amr/assemble.wgsl,
// predict.wgsl, update.wgsl), with no W, PA or PB atlas of the blocks' cells in HBM:
//
//  - k_amr_shell, twice: per leaf, the ghost texels of its 20^3 region, formed from U (boundary
//    images, prolongation from a coarser leaf, restriction of refined children: amr_texel); then
//    the half steps of its first ghost layer where those are another block's cells ("at source",
//    amr/predict.wgsl:183-221): beside boundary images, and on the rims of faces beside same-level
//    leaves, once per source cell;
//  - k_amr_fused, one persistent kernel per launch: a workgroup owns one 16^3 block at a time
//    and marches along z: its cells from U, its ghosts from the shell; the half step of every
//    cell and of the ghosts beside a coarser block (masked transverse slopes), in LDS;
//  - every face once; the conservative update of each cell; the next step's rate / dx;
//  - coarse-fine faces through a flux register: a leaf writes the fluxes of its faces on a
//    coarser block (as it computed them), and the coarser leaf reads the four fine fluxes of
//    each of its faces there and takes their mean (TwoSum-compensated when asked), which is
//    what match_faces (amr/update.wgsl:207-290) recomputes from the finer block's atlas.
//  - one launch for all leaves: workgroups take pairs from a device queue (level by level from the
//    finest the leaves with a coarse-fine face, those that only supply a coarser leaf before those
//    that wait for finer ones, with leaves that do neither between and at the end: build_lists in
//    api_amr.cpp); a leaf with a refined neighbour first waits for the finer leaves across it (a done flag per slot, set
//    with release order after their march). The queue hands out pairs in order and a leaf only
//    waits for leaves earlier in it, all of which are held by running workgroups, so the waits
//    end; each is bounded besides, and a wait that runs out sets an error flag the host reports.
//
// Thread layout: 384 threads (6 waves) own the columns of the block's 20 x 20 texel plane that
// ever hold a value: threads 0-255 the 16 x 16 cell columns, 256-319 the 64 face-ghost columns
// of ring 1, 320-383 the 64 of ring 2 (x or y = -2 or 17, the other in range). The 16 remaining
// columns (both x and y outside the cells) are edges or corners at every plane: zero, as in the
// atlas. So the cell waves never diverge on ghost work, and each role runs its own loop over the
// planes (the uniform march's form, uniform_roles.hpp, with its LDS layout: 72 KB per block in
// FP32), with two barriers per plane: after the half steps, after the fluxes. The ghost planes
// z = -1 and 16 concern the cell waves alone. Two blocks share a 12-wave workgroup (one per CU at
// up to 168 VGPRs), whose waves go to the SIMDs in turn: two cell waves and one ghost or load wave
// on each.
#pragma once
#include "amr_impl.hpp"

namespace shx {

constexpr int AF_SIDE = AMR_PAD;              // 20 columns per side
constexpr int AF_NT = AF_SIDE * AF_SIDE;      // 400 columns
constexpr int AF_THREADS = 384;             // one block's march
// blocks marched side by side per workgroup: two in FP32 (2 x 72 KB of LDS), one in FP64
template <typename T>
constexpr int af_pair() { return sizeof(T) == 4 ? 2 : 1; }
constexpr int AF_RING = 128;                  // ghost columns with a value: 64 of ring 1, 64 of ring 2

// thread -> column (x, y) in block coordinates, [-2, 18). A cell wave holds a 4-wide strip of the
// 16 rows: with the LDS rows 20 columns apart its lanes reach distinct banks (4 rows of 16 would
// meet in a third of them).
__device__ __forceinline__ void af_column(int t, int& x, int& y) {
  if (t < 256) { x = 4 * (t >> 6) + (t & 3); y = (t & 63) >> 2; return; }
  const int ring = t < 320 ? 1 : 2;
  t = (t - 256) & 63;
  const int side = t >> 4, i = t & 15;
  const int lo = -ring, hi = AMR_BS - 1 + ring;
  x = side == 0 ? lo : (side == 1 ? hi : i);
  y = side == 2 ? lo : (side == 3 ? hi : i);
}

// Flux register: per coarse-fine face of a leaf, its 16 x 16 faces' fluxes (8 values each), in
// the face's transverse order (t2 * 16 + t1, t1 = (axis + 1) % 3, t2 = (axis + 2) % 3)
template <typename T>
__device__ __forceinline__ void reg_put(T* __restrict__ R, int reg, int idx, const Flux<T>& F) {
  T4<T>* p = reinterpret_cast<T4<T>*>(R + ((size_t)reg * 256 + idx) * 8);
  p[0] = v4<T>(F.m, F.mx, F.my, F.mz);
  p[1] = v4<T>(F.e, F.ei, F.s, F.vn);
}

// The mean of the four fine fluxes through the face of cell (x, y, z) on side k, read from the
// register of the refined neighbour's child; summed in match_faces' order (t2 outer, t1 inner)
template <typename T, bool COMP, bool COHERENT>
__device__ __forceinline__ Flux<T> reg_mean(const int* __restrict__ tab, const int* __restrict__ reg_of,
                                            const T* __restrict__ R, int np, int k, int x, int y, int z,
                                            const Flux<T>& fallback) {
  const int axis = k >> 1, upper = !(k & 1);
  const int hx = x >= AMR_BS / 2, hy = y >= AMR_BS / 2, hz = z >= AMR_BS / 2;
  const int bx = axis == 0 ? upper : hx, by = axis == 1 ? upper : hy, bz = axis == 2 ? upper : hz;
  const int ch = bt(tab, np, BT_CHILD + (bx | (by << 1) | (bz << 2)));
  const int reg = ch >= 0 ? reg_of[ch * 6 + (k ^ 1)] : -1;
  if (reg < 0) return fallback;   // not reached in a 2:1-balanced tree (checked at creation)
  // transverse fine coordinates of the first of the four faces
  const int fx = 2 * (x - (AMR_BS / 2) * hx), fy = 2 * (y - (AMR_BS / 2) * hy), fz = 2 * (z - (AMR_BS / 2) * hz);
  const int u0 = axis == 0 ? fy : (axis == 1 ? fz : fx);   // t1
  const int v0 = axis == 0 ? fz : (axis == 1 ? fx : fy);   // t2
  T sum[8], err[8];
#pragma unroll
  for (int q = 0; q < 8; q++) { sum[q] = T(0); err[q] = T(0); }
#pragma unroll
  for (int j = 0; j < 2; j++)
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const T* p = R + ((size_t)reg * 256 + (v0 + j) * 16 + (u0 + i)) * 8;
      T fv[8];
      if constexpr (COHERENT) {
        // device-coherent loads: written by another workgroup of this launch
#pragma unroll
        for (int q = 0; q < 8; q++) fv[q] = __hip_atomic_load(p + q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      } else {
        const T4<T> a = reinterpret_cast<const T4<T>*>(p)[0], b = reinterpret_cast<const T4<T>*>(p)[1];
        fv[0] = a.x; fv[1] = a.y; fv[2] = a.z; fv[3] = a.w; fv[4] = b.x; fv[5] = b.y; fv[6] = b.z; fv[7] = b.w;
      }
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
  Flux<T> F;
  F.m = (sum[0] + err[0]) * T(0.25); F.mx = (sum[1] + err[1]) * T(0.25);
  F.my = (sum[2] + err[2]) * T(0.25); F.mz = (sum[3] + err[3]) * T(0.25);
  F.e = (sum[4] + err[4]) * T(0.25); F.ei = (sum[5] + err[5]) * T(0.25);
  F.s = (sum[6] + err[6]) * T(0.25); F.vn = (sum[7] + err[7]) * T(0.25);
  return F;
}

// Coarse-fine faces of the march, by a per-(slot, face) action: act >= 0 even: the neighbour is
// coarser, write this face's fluxes to register act / 2; odd: the neighbour is refined, take
// the face's fluxes from coarse-face buffer act / 2 (the means its march formed first); -1:
// neither.
template <typename T>
__device__ __forceinline__ Flux<T> boundary_face(int act, T* __restrict__ R, const T* __restrict__ CF, int idx,
                                                 Flux<T> F) {
  if (act < 0) return F;
  if (act & 1) {
    const T4<T>* p = reinterpret_cast<const T4<T>*>(CF + ((size_t)(act >> 1) * 256 + idx) * 8);
    const T4<T> a = p[0], b = p[1];
    F.m = a.x; F.mx = a.y; F.my = a.z; F.mz = a.w;
    F.e = b.x; F.ei = b.y; F.s = b.z; F.vn = b.w;
  } else {
    reg_put(R, act >> 1, idx, F);
  }
  return F;
}

template <typename T>
__device__ __forceinline__ void scale_inc(Inc<T>& q, T m) {
  q.rho *= m; q.vx *= m; q.vy *= m; q.vz *= m; q.p *= m; q.s *= m;
}

// ---------------- the ghost shell ----------------
// Per leaf, what its march needs from outside its own cells, formed in one batched pass with
// every lane busy: the ghost texels of its 20^3 region (the four ghost planes z = -2, -1, 16, 17
// whole, then the 128 ghost columns with a value over the 16 cell planes) and the half steps of its first
// ghost layer where they are another block's cells (64 face-ghost columns x 16 planes, then the
// two z-face ghost planes). 32 bytes per item.
constexpr int SH_TEXELS = 4 * AF_NT + AF_RING * AMR_BS;                     // 1600 + 128 * 16 = 3648
constexpr int SH_HALVES = 64 * AMR_BS + 2 * AMR_BS * AMR_BS;                 // 1024 + 512 = 1536
constexpr int SH_ITEMS = SH_TEXELS + SH_HALVES;                               // 5184

__device__ __forceinline__ int ghost_plane_slot(int z) { return z == -2 ? 0 : (z == -1 ? 1 : (z == AMR_BS ? 2 : 3)); }

// The same-level leaf across face k of block s (0 -x, 1 +x, 2 -y, 3 +y, 4 -z, 5 +z), or -1. Its
// cells are the block's ghost texels there as they are (no image, no interpolation), so the
// march reads them directly, and the shell forms nothing for that face but the half steps of
// its rim.
__device__ __forceinline__ int same_leaf(const int* __restrict__ tab, int s, int k) {
  const int nb = bt(tab, s, BT_NB + k);
  return (nb >= 0 && is_leaf(tab, nb)) ? nb : -1;
}
// Away from the face's rim (both coordinates along the face in [1, 14]), the half step of a
// first-layer ghost of a same-level leaf uses only texels the march holds, the same ones the
// source block's own predictor uses: the march forms it in place, exactly as at its source.
__device__ __forceinline__ bool off_rim(int i, int j) {
  return i >= 1 && i <= AMR_BS - 2 && j >= 1 && j <= AMR_BS - 2;
}

// a shell texel
template <typename T>
__device__ __forceinline__ Prim<T> shell_prim(T4<T> a, T4<T> b) {
  Prim<T> w;
  w.rho = a.x; w.vx = a.y; w.vy = a.z; w.vz = a.w;
  w.p = b.x; w.s = b.y; w.cs = b.z;
  return w;
}
// the item of ghost texel (x, y, z), out of the block along one axis
__device__ __forceinline__ int shell_texel(int x, int y, int z) {
  if (z < 0 || z >= AMR_BS) return ghost_plane_slot(z) * AF_NT + (y + 2) * AF_SIDE + (x + 2);
  const bool ox = x < 0 || x >= AMR_BS;
  const int c = ox ? x : y, i = ox ? y : x;
  const int ring = c < 0 ? -1 - c : c - AMR_BS, side = (ox ? 0 : 2) + (c >= AMR_BS);
  return 4 * AF_NT + z * AF_RING + ring * 64 + side * 16 + i;
}

// The shell's texels, one wave per item (shell index, slot, face k, code), listed on the host from
// the static mesh: the two layers (512 texels) beyond a face whose neighbour is not a same-level
// leaf. Beside a coarser block (code 8) a lane takes one of the face's 64 coarse cells and forms
// its eight fine texels from one set of slopes; else the wave takes 64 texels (code 0-7), images
// and means. Bound by latency: a chain of table and cell reads.
// On the 3D blast's 1618 leaves 43 us with a wave per 64 texels, slopes formed for each texel by
// seven calls; 28 us as now.
template <typename T, int LIM>
__device__ __forceinline__ void shell_texels(const Params<T>& P, const int* __restrict__ tab,
                                             const int4* __restrict__ work, int nwork, const T4<T>* __restrict__ U1,
                                             const T4<T>* __restrict__ U2, T4<T>* __restrict__ SH) {
  const int wv = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (wv >= nwork) return;
  const int4 wk = work[wv];
  // (the wave's own: the table reads of a face are scalar)
  const int li = __builtin_amdgcn_readfirstlane(wk.x), s = __builtin_amdgcn_readfirstlane(wk.y);
  const int k = __builtin_amdgcn_readfirstlane(wk.z), code = __builtin_amdgcn_readfirstlane(wk.w);
  const int lane = threadIdx.x & 63, axis = k >> 1;
  T4<T>* const sh = SH + (size_t)li * SH_ITEMS * 2;
  auto put = [&](int x, int y, int z, const Prim<T>& w) {
    T4<T>* out = sh + (size_t)shell_texel(x, y, z) * 2;
    out[0] = v4<T>(w.rho, w.vx, w.vy, w.vz);
    out[1] = v4<T>(w.p, w.s, w.cs, T(0));
  };
  if (code == 8) {
    // the coarse cell's first fine texel: even along every axis
    const int n = (k & 1) ? AMR_BS : -2, i = 2 * (lane & 7), j = 2 * (lane >> 3);
    const int x = axis == 0 ? n : i, y = axis == 1 ? n : (axis == 0 ? i : j), z = axis == 2 ? n : j;
    int par[3];
    const Prolong<T> g = coarse_cell<T, LIM, 3>(P, tab, U1, U2, s, x, y, z, bt(tab, s, BT_COARSE + k), par);
#pragma unroll
    for (int c = 0; c < 8; c++) {
      const Cons<T> u = g.child(c & 1, (c >> 1) & 1, c >> 2);
      put(x + (c & 1), y + ((c >> 1) & 1), z + (c >> 2), prim_from_cons(P, u.a, u.b));
    }
    return;
  }
  const int e = code * 64 + lane, layer = e >> 8, i = e & 15, j = (e >> 4) & 15;
  const int n = (k & 1) ? AMR_BS + layer : -1 - layer;
  const int x = axis == 0 ? n : i, y = axis == 1 ? n : (axis == 0 ? i : j), z = axis == 2 ? n : j;
  Prim<T> w;
  if (amr_texel<T, LIM, 3, false>(P, tab, U1, U2, s, x, y, z, w)) put(x, y, z, w);
}

// The half step of cell (x, y, z) of leaf `slot` (predict_cell on the source block,
// amr/predict.wgsl:90-181): its texels from U where they are stored cells, else from the leaf's
// own shell, all in one batch of loads; P carries the block's dx
template <typename T, int LIM, bool ISEN>
__device__ __forceinline__ Half<T> half_at_source(const Params<T>& P, const int* __restrict__ tab,
                                                  const int* __restrict__ shell_of, const T4<T>* __restrict__ U1,
                                                  const T4<T>* __restrict__ U2, const T4<T>* __restrict__ SH, int slot,
                                                  int x, int y, int z, T dt) {
  Spot sp[7];
  spots(tab, slot, x, y, z, sp);
  const T4<T>* sh = SH + (size_t)shell_of[slot] * SH_ITEMS * 2;
  T4<T> a[7], b[7];
#pragma unroll
  for (int k = 0; k < 7; k++) {
    int c[3];
    stencil_at(k, x, y, z, c);
    const T4<T>* g = sh + 2 * (k > 0 && !sp[k].ok ? shell_texel(c[0], c[1], c[2]) : 0);
    a[k] = *(sp[k].ok ? U1 + sp[k].cell : g);
    b[k] = *(sp[k].ok ? U2 + sp[k].cell : g + 1);
  }
  __builtin_amdgcn_sched_barrier(0);
  Prim<T> w[7];
#pragma unroll
  for (int k = 0; k < 7; k++) {
    w[k] = prim_from_cons(P, a[k], b[k]);
    if (!sp[k].ok) w[k] = shell_prim<T>(a[k], b[k]);
  }
  const Prim<T>&q = w[0], &xm = w[1], &xp = w[2], &ym = w[3], &yp = w[4], &zm = w[5], &zp = w[6];
  AxisSlope<T> sl[3];
  sl[0] = axis_slope<T, LIM, ISEN>(P, xm, q, xp, nullptr, nullptr);
  sl[1] = axis_slope<T, LIM, ISEN>(P, ym, q, yp, nullptr, nullptr);
  sl[2] = axis_slope<T, LIM, ISEN>(P, zm, q, zp, nullptr, nullptr);
  const T conv = (xp.vx - xm.vx) + (yp.vy - ym.vy) + (zp.vz - zm.vz);
  const T jump = tmax(jump_over(P, xm.p, xp.p), tmax(jump_over(P, ym.p, yp.p), jump_over(P, zm.p, zp.p)));
  return hancock<T, LIM>(P, q, sl, conv, jump, slope_step<T, LIM>(P, dt));
}

// The shell's half steps (after its texels). The first nrim lanes: the rims of faces beside
// same-level leaves. A rim ghost's source is a cell on an edge of the leaf across the face, whose
// transverse stencil reaches past the face (the march holds only the face itself). One lane per
// source cell, from records listed on the host (source slot, cell x | y << 4 | z << 8, then up to
// three (shell index, half-step item) destinations, -1 for none): an edge cell feeds the shells of
// the leaves across both its faces, a corner cell three, so each is predicted once, and the lanes
// of a wave take the edge cells of one block. A same-level face maps no velocity.
// The other blocks: the first layer beside a boundary image, one wave per item (shell index, slot,
// face k, chunk 0-3). Faces on a coarser block have no half steps here (the march predicts those
// ghosts in place).
// Bound by bandwidth: an edge cell's stencil along y and z touches a cache line per texel, nearly
// the blocks' whole state in all (5.2 TB/s on the 3D blast: 81 us with the ghosts formed anew for
// each stencil, 41 us read from the shell).
template <typename T, int LIM, bool ISEN>
__device__ __forceinline__ void shell_halves(const Params<T>& P, const int* __restrict__ tab,
                                             const int* __restrict__ shell_of, const int4* __restrict__ rim, int nrim,
                                             const int4* __restrict__ work, int nwork, const T4<T>* __restrict__ U1,
                                             const T4<T>* __restrict__ U2, T4<T>* SH, const T* __restrict__ clk) {
  const int rim_blocks = (nrim + 255) >> 8;
  int slot, x, y, z;
  int li[3], h[3];
  GSrc g;
  g.fx = g.fy = g.fz = 1;
  g.sx = g.sy = g.sz = 0;
  if ((int)blockIdx.x < rim_blocks) {
    const int w = blockIdx.x * 256 + threadIdx.x;
    if (w >= nrim) return;
    const int4 a = rim[2 * w], b = rim[2 * w + 1];
    slot = a.x;
    x = a.y & 15;
    y = (a.y >> 4) & 15;
    z = (a.y >> 8) & 15;
    li[0] = a.z; li[1] = b.x; li[2] = b.z;
    h[0] = a.w; h[1] = b.y; h[2] = b.w;
  } else {
    const int wv = ((int)blockIdx.x - rim_blocks) * 4 + (threadIdx.x >> 6);
    if (wv >= nwork) return;
    const int4 wk = work[wv];
    const int s = wk.y, k = wk.z, e = wk.w * 64 + (threadIdx.x & 63), i = e & 15, j = e >> 4;
    if (k < 4) {
      const int col = k * 16 + i;
      af_column(256 + col, x, y);
      z = j;
      h[0] = col * AMR_BS + z;
    } else {
      x = i;
      y = j;
      z = k == 4 ? -1 : AMR_BS;
      h[0] = 64 * AMR_BS + (k == 4 ? 0 : AMR_BS * AMR_BS) + y * AMR_BS + x;
    }
    li[0] = wk.x;
    li[1] = li[2] = -1;
    h[1] = h[2] = 0;
    g = ghost_src(tab, s, x, y, z);
    if (g.kind != 0) return;
    slot = g.slot;
    x = g.x;
    y = g.y;
    z = g.z;
  }
  Params<T> Pl = P;
  Pl.dx = level_dx(P, bt(tab, slot, BT_LEVEL));
  Half<T> hc = half_at_source<T, LIM, ISEN>(Pl, tab, shell_of, U1, U2, SH, slot, x, y, z, clk[0]);
  hc.vx = bc_vel(hc.vx, g.fx, g.sx);
  hc.vy = bc_vel(hc.vy, g.fy, g.sy);
  hc.vz = bc_vel(hc.vz, g.fz, g.sz);
  const T4<T> v0 = v4<T>(hc.rho, hc.vx, hc.vy, hc.vz), v1 = v4<T>(hc.p, hc.s, hc.shock, hc.fo);
#pragma unroll
  for (int d = 0; d < 3; d++) {
    if (li[d] < 0) continue;
    T4<T>* out = SH + ((size_t)li[d] * SH_ITEMS + SH_TEXELS + h[d]) * 2;
    out[0] = v0;
    out[1] = v1;
  }
}

// PART 0 the texels, PART 1 (a launch later: it reads them) the half steps
template <typename T, int LIM, bool ISEN, int PART>
__global__ __launch_bounds__(256, 4) void k_amr_shell(Params<T> P, const int* __restrict__ tab,
                                                      const int* __restrict__ shell_of, const int4* __restrict__ rim,
                                                      int nrim, const int4* __restrict__ work, int nwork,
                                                      const T4<T>* __restrict__ U1, const T4<T>* __restrict__ U2,
                                                      T4<T>* SH, const T* __restrict__ clk) {
  if constexpr (PART == 0)
    shell_texels<T, LIM>(P, tab, work, nwork, U1, U2, SH);
  else
    shell_halves<T, LIM, ISEN>(P, tab, shell_of, rim, nrim, work, nwork, U1, U2, SH, clk);
}

// ---------------- the march ----------------
// Before each march: the queue starts at pair 0 and the step's epoch (the value done flags are
// set to) moves on.
template <typename T>
__global__ void k_amr_queue_start(int* qctl) {
  qctl[AMR_Q_NEXT] = 0;
  qctl[AMR_Q_EPOCH] = qctl[AMR_Q_EPOCH] + 1;
}

// Launch bound: twelve waves per workgroup (two blocks), one workgroup per CU in FP32 (three
// waves per SIMD: up to 168 VGPRs); six waves (one block) in FP64.
// Bound by VALU issue and, on a few hundred leaves, by how evenly the pairs divide among the CUs.
// On the 3D blast (8^3 root blocks, two refinements, 1618 leaves, MC, HLLC): 462 us with one loop
// for all roles, ghost cases chosen by lane in it; 342 us with a loop per role (-26%). The rate's
// division is by the block (tquot by one dx keeps the order, so the maximum has the same bits).
template <typename T, int LIM, int RS, bool ISEN>
__global__ __launch_bounds__((sizeof(T) == 4 ? 2 : 1) * AF_THREADS, (sizeof(T) == 4 ? 3 : 1)) void k_amr_fused(
    Params<T> P, const int* __restrict__ tab, const int* __restrict__ list, int count,
    const int* __restrict__ shell_of, const T4<T>* __restrict__ SH, const int* __restrict__ act,
    T* __restrict__ R, T* __restrict__ CF, const int* __restrict__ reg_of, int comp, const int* __restrict__ dep_off,
    const int* __restrict__ dep, int* __restrict__ qctl, int* __restrict__ done, const T4<T>* __restrict__ U1,
    const T4<T>* __restrict__ U2, T4<T>* __restrict__ O1, T4<T>* __restrict__ O2, const T* __restrict__ clk,
    unsigned long long* next_slot) {
  constexpr int NT = AF_NT, BX = AF_SIDE, AF_PAIR = af_pair<T>();
  using PL = PlaneLds<T, NT>;
  __shared__ T4<T> LL[AF_PAIR * PL::SIZE / 4];
  __shared__ T red[AF_PAIR * AF_THREADS / 64];
  __shared__ int q_pair;
  const int epoch = qctl[AMR_Q_EPOCH];
  // which of the workgroup's two blocks this wave marches (a scalar), and its thread index there
  const int gwave = __builtin_amdgcn_readfirstlane(threadIdx.x) >> 6;
  const int half = gwave >= AF_THREADS / 64;
  const int tid = threadIdx.x - AF_THREADS * half;
  T* const L = reinterpret_cast<T*>(LL) + half * PL::SIZE;
  int x, y;
  af_column(tid, x, y);
  const typename PL::At t = PL::at((y + 2) * BX + (x + 2));   // the column, in raster order
  // the columns no thread owns are edges at every plane: zero in both plane slots, for good
  for (int i = tid; i < 12 * NT; i += AF_THREADS) L[i] = T(0);
  // roles by wave: 0-3 the cell columns, 4 the face ghosts of ring 1, 5 ring 2 (loads only)
  const int wave = gwave - (AF_THREADS / 64) * half;
  const bool cells = wave < 4, ghosts = wave == 4;
  // a ghost lane's side: 0 -x, 1 +x, 2 -y, 3 +y
  const int side = (tid >> 4) & 3;
  const T dt = clk[0];
  const T dx0 = P.dx;
  T rate_max = T(0);

  for (;;) {
    // the next pair from the queue (every thread has passed a barrier since it last read q_pair)
    if (threadIdx.x == 0) q_pair = atomicAdd(&qctl[AMR_Q_NEXT], 1);
    __syncthreads();
    const int wp = __builtin_amdgcn_readfirstlane(q_pair);
    __syncthreads();   // every thread has read q_pair before thread 0 takes the next ticket
    if (AF_PAIR * wp >= count) break;
    // -1 pads a queue part of odd length. With pairs it is always a pair's second entry (parts
    // start at even positions): that half takes part in the barriers only. A one-block
    // workgroup skips it.
    if (list[AF_PAIR * wp] < 0) continue;
    const int wi = AF_PAIR * wp + half;
    const bool act_blk = wi < count && list[wi] >= 0;
    const int s = __builtin_amdgcn_readfirstlane(list[act_blk ? wi : AF_PAIR * wp]);
    // a leaf with a refined neighbour: wait for the finer leaves across it (one lane each), then
    // form the means of their fluxes on its coarse-fine faces
    const int d0 = act_blk ? dep_off[s] : 0, nd = act_blk ? dep_off[s + 1] - d0 : 0;
    // The flags are read with agent-scope acquire loads, pairing with the writers' release
    // fence: what a finer leaf wrote before its flag (its register fluxes) is visible to the
    // reads after the barrier below, which are device-coherent loads as well
    if (tid < nd) {
      int* flag = done + dep[d0 + tid];
      int spins = 0;
      while (__hip_atomic_load(flag, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT) != epoch) {
        if (++spins > AMR_WAIT_SPINS) {
          __hip_atomic_store(&qctl[AMR_Q_ERROR], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          break;
        }
        __builtin_amdgcn_s_sleep(2);
      }
    }
    __syncthreads();
    if (nd > 0) {
      for (int k = 0; k < 6; k++) {
        const int a = act[s * 6 + k];
        if (a < 0 || !(a & 1) || tid >= 256) continue;
        const int axis = k >> 1, t1 = tid & 15, t2 = tid >> 4;
        const int n = (k & 1) ? AMR_BS - 1 : 0;
        const int fx = axis == 0 ? n : (axis == 1 ? t2 : t1);
        const int fy = axis == 1 ? n : (axis == 2 ? t2 : t1);
        const int fz = axis == 2 ? n : (axis == 0 ? t2 : t1);
        const int np = bt(tab, s, BT_NB + k);
        const Flux<T> F = comp ? reg_mean<T, true, true>(tab, reg_of, R, np, k, fx, fy, fz, zero_flux<T>())
                               : reg_mean<T, false, true>(tab, reg_of, R, np, k, fx, fy, fz, zero_flux<T>());
        T4<T>* q = reinterpret_cast<T4<T>*>(CF + ((size_t)(a >> 1) * 256 + tid) * 8);
        q[0] = v4<T>(F.m, F.mx, F.my, F.mz);
        q[1] = v4<T>(F.e, F.ei, F.s, F.vn);
      }
    }
    const T4<T>* sh = SH + (size_t)shell_of[s] * SH_ITEMS * 2;
    // this block's cell size (P is the kernel's own copy: its dx is the block's from here on)
    const T dx = dx0 * (T(1) / T(1 << bt(tab, s, BT_LEVEL)));
    P.dx = dx;
    const T dtdx = wave_uniform(tratio(dt, dx)), hstep = wave_uniform(slope_step<T, LIM>(P, dt));
    // the faces' actions (boundary_face)
    int fa[6];
#pragma unroll
    for (int k = 0; k < 6; k++) fa[k] = __builtin_amdgcn_readfirstlane(act[s * 6 + k]);
    __syncthreads();   // the previous block's last LDS reads are done

    const size_t own = (size_t)s * AMR_CELLS;
    // slopes and edge increments of this column in the plane whose primitives are at q (those of
    // the plane below at m, of the plane above in pp), and the shock detector's terms
    struct Edges { Inc<T> xu, xd, yu, yd, zu, zd; };
    auto slopes = [&](int q, int m, Prim<T>& pc, T cs, const Prim<T>& pp, AxisSlope<T> sl[3], Edges& e, T& conv,
                      T& jump) {
      pc = PL::prim(L, q, t);
      pc.cs = cs;
      // (axis by axis, as k_fused_r)
      {
        const Prim<T> xm = PL::prim(L, q, t.off(-1)), xp = PL::prim(L, q, t.off(1));
        sl[0] = axis_slope<T, LIM, ISEN>(P, xm, pc, xp, &e.xu, &e.xd);
        conv = xp.vx - xm.vx;
        jump = jump_over(P, xm.p, xp.p);
      }
      __builtin_amdgcn_sched_barrier(0);
      {
        const Prim<T> ym = PL::prim(L, q, t.off(-BX)), yp = PL::prim(L, q, t.off(BX));
        sl[1] = axis_slope<T, LIM, ISEN>(P, ym, pc, yp, &e.yu, &e.yd);
        conv = conv + (yp.vy - ym.vy);
        jump = tmax(jump, jump_over(P, ym.p, yp.p));
      }
      __builtin_amdgcn_sched_barrier(0);
      const Prim<T> pm = PL::prim(L, m, t);
      sl[2] = axis_slope<T, LIM, ISEN>(P, pm, pc, pp, &e.zu, &e.zd);
      conv = conv + (pp.vz - pm.vz);
      jump = tmax(jump, jump_over(P, pm.p, pp.p));
      __builtin_amdgcn_sched_barrier(0);
    };
    auto shell_half = [&](int h) {
      const T4<T> a = sh[2 * (SH_TEXELS + h)], b = sh[2 * (SH_TEXELS + h) + 1];
      Half<T> hc;
      hc.rho = a.x; hc.vx = a.y; hc.vy = a.z; hc.vz = a.w;
      hc.p = b.x; hc.s = b.y; hc.shock = b.z; hc.fo = b.w;
      return hc;
    };
    // the buffer of plane c's primitives
    auto buf = [](int c) { return (c & 1) ? PL::QN : 0; };

    if (!act_blk) {
      for (int k = 0; k < 2 + 2 * AMR_BS; k++) __syncthreads();
    } else if (cells) {
      const bool kz_lo = bt(tab, s, BT_NB + 4) == -1, kz_hi = bt(tab, s, BT_NB + 5) == -1;
      const int nbz_lo = same_leaf(tab, s, 4), nbz_hi = same_leaf(tab, s, 5);
      const unsigned int at = (unsigned int)(cel(x, y, 0)) * (unsigned int)sizeof(T4<T>);
      T4<T> b1, b2;
      // plane z's texel: this block's cells and a same-level leaf's from U, other ghosts from the
      // shell (a scalar choice per plane)
      auto load = [&](int z) {
        const bool oz = z < 0 || z >= AMR_BS;
        const int src = !oz ? s : (z < 0 ? nbz_lo : nbz_hi);
        if (src >= 0) {
          const size_t o = (size_t)src * AMR_CELLS + (z & (AMR_BS - 1)) * (AMR_BS * AMR_BS);
          b1 = plane_load<T>(U1 + o, at);
          b2 = plane_load<T>(U2 + o, at);
        } else {
          const int g = ghost_plane_slot(z) * AF_NT + (y + 2) * BX + (x + 2);
          b1 = sh[2 * g];
          b2 = sh[2 * g + 1];
        }
      };
      auto prim = [&](int z) {
        const bool oz = z < 0 || z >= AMR_BS;
        return !oz || (z < 0 ? nbz_lo : nbz_hi) >= 0 ? prim_from_cons(P, b1, b2) : shell_prim<T>(b1, b2);
      };
      // a ghost plane's half step (c = -1, 16): in place beside a coarser block, with the slopes
      // along the face dropped where their neighbour is an unassembled edge texel
      // (amr/predict.wgsl:183-221), and where the texel is a same-level leaf's cell away from the
      // face's rim, as at its source; else another block's cell, formed in the shell pass
      auto ghost_plane_half = [&](int c, const Prim<T>& pp, T cs, Edges& e) {
        AxisSlope<T> sl[3];
        Prim<T> pc;
        T conv, jump;
        slopes(buf(c), buf(c - 1), pc, cs, pp, sl, e, conv, jump);
        const bool coarse = c < 0 ? kz_lo : kz_hi;
        if (coarse) {
          scale_inc(sl[0].s, (x == 0 || x == AMR_BS - 1) ? T(0) : T(1));
          scale_inc(sl[1].s, (y == 0 || y == AMR_BS - 1) ? T(0) : T(1));
        }
        Half<T> h = hancock<T, LIM>(P, pc, sl, conv, jump, hstep);
        const bool exact = (c < 0 ? nbz_lo : nbz_hi) >= 0 && off_rim(x, y);
        if (!coarse && !exact) h = shell_half(64 * AMR_BS + (c < 0 ? 0 : AMR_BS * AMR_BS) + y * AMR_BS + x);
        return h;
      };
      load(-2);
      PL::put_prim(L, buf(-2), t, prim(-2));
      load(-1);
      Prim<T> pp = prim(-1);
      PL::put_prim(L, buf(-1), t, pp);
      T cs = pp.cs;            // this column's sound speed in plane c
      load(0);
      __syncthreads();
      SideData<T> zs;          // the upper z side of the plane below, and its half-step pressure
      T hp;
      Flux<T> fz_lo, xy;       // the z face below and the x/y net inflow of that plane
      T rate = T(0);           // the block's largest rate
      auto update = [&](int c, T4<T> u1, T4<T> u2, const Flux<T>& fz) {
        T4<T> o1, o2;
        advance(P, u1, u2, net_z(xy, fz_lo, fz), hp, dtdx, o1, o2);
        const size_t o = own + c * (AMR_BS * AMR_BS);
        plane_store<T>(O1 + o, at, o1);
        plane_store<T>(O2 + o, at, o2);
        rate = tmax(rate, rate_of(P, prim_from_cons(P, o1, o2)));
      };
      {
        pp = prim(0);
        load(1);
        Edges e;
        const Half<T> h = ghost_plane_half(-1, pp, cs, e);
        zs = side_of(P, h, e.zu, T(1));
        PL::put_prim(L, buf(0), t, pp);
        cs = pp.cs;
      }
      __syncthreads();
      for (int c = 0; c < AMR_BS; c++) {
        pp = prim(c + 1);
        Edges e;
        Half<T> h;
        {
          AxisSlope<T> sl[3];
          Prim<T> pc;
          T conv, jump;
          slopes(buf(c), buf(c - 1), pc, cs, pp, sl, e, conv, jump);
          h = hancock<T, LIM>(P, pc, sl, conv, jump, hstep);
        }
        __builtin_amdgcn_sched_barrier(0);
        T4<T> u1, u2;
        if (c > 0) {
          const size_t o = own + (c - 1) * (AMR_BS * AMR_BS);
          u1 = plane_load<T>(U1 + o, at);
          u2 = plane_load<T>(U2 + o, at);
        }
        PL::put_side(L, PL::SX, t, side_of(P, h, e.xu, T(1)));
        PL::put_side(L, PL::SY, t, side_of(P, h, e.yu, T(1)));
        PL::put_shock(L, PL::SK, t, h.shock);
        PL::put_prim(L, buf(c + 1), t, pp);
        cs = pp.cs;
        __builtin_amdgcn_sched_barrier(0);
        Flux<T> fz = face_from_sides<T, RS>(P, zs, side_of(P, h, e.zd, T(-1)), 2);
        if (c == 0) fz = boundary_face<T>(fa[4], R, CF, y * 16 + x, fz);
        __builtin_amdgcn_sched_barrier(0);
        if (c > 0) update(c - 1, u1, u2, fz);
        fz_lo = fz;
        zs = side_of(P, h, e.zu, T(1));
        hp = h.p;
        __builtin_amdgcn_sched_barrier(0);
        load(c + 2);
        __syncthreads();
        Flux<T> Fx = face_from_sides<T, RS>(P, PL::side(L, PL::SX, PL::SK, t.off(-1)), side_of(P, h, e.xd, T(-1)), 0);
        if (fa[0] >= 0 && x == 0) Fx = boundary_face<T>(fa[0], R, CF, c * 16 + y, Fx);
        PL::put_flux(L, PL::FX, t, Fx);
        __builtin_amdgcn_sched_barrier(0);
        Flux<T> Fy = face_from_sides<T, RS>(P, PL::side(L, PL::SY, PL::SK, t.off(-BX)), side_of(P, h, e.yd, T(-1)), 1);
        if (fa[2] >= 0 && y == 0) Fy = boundary_face<T>(fa[2], R, CF, x * 16 + c, Fy);
        PL::put_flux(L, PL::FY, t, Fy);
        __syncthreads();
        xy = net_xy(Fx, PL::flux(L, PL::FX, t.off(1)), Fy, PL::flux(L, PL::FY, t.off(BX)));
      }
      {
        pp = prim(AMR_BS + 1);
        const size_t o = own + (AMR_BS - 1) * (AMR_BS * AMR_BS);
        const T4<T> u1 = plane_load<T>(U1 + o, at), u2 = plane_load<T>(U2 + o, at);
        Edges e;
        const Half<T> h = ghost_plane_half(AMR_BS, pp, cs, e);
        Flux<T> fz = face_from_sides<T, RS>(P, zs, side_of(P, h, e.zd, T(-1)), 2);
        fz = boundary_face<T>(fa[5], R, CF, y * 16 + x, fz);
        update(AMR_BS - 1, u1, u2, fz);
      }
      // the next step's rate / dx (assemble's leaf-cell rate, amr/assemble.wgsl:77-154)
      rate_max = tmax(rate_max, tquot(rate, dx));
    } else {
      // the ghost columns: a same-level leaf's cells from U, others from the shell; edges (the
      // ghost planes' texels beside them) are zero
      const int nbs = same_leaf(tab, s, side);
      const int xs = (x + AMR_BS) & (AMR_BS - 1), ys = (y + AMR_BS) & (AMR_BS - 1);
      const size_t o0 = nbs >= 0 ? (size_t)nbs * AMR_CELLS + cel(xs, ys, 0) : (size_t)0;
      const T4<T>* s1 = nbs >= 0 ? U1 + o0 : sh + 2 * (4 * AF_NT + (tid - 256));
      const T4<T>* s2 = nbs >= 0 ? U2 + o0 : s1 + 1;
      const size_t step = nbs >= 0 ? AMR_BS * AMR_BS : 2 * AF_RING;
      T4<T> b1, b2;
      auto load = [&](int z) {
        b1 = s1[z * step];
        b2 = s2[z * step];
      };
      auto prim = [&] { return nbs >= 0 ? prim_from_cons(P, b1, b2) : shell_prim<T>(b1, b2); };
      Prim<T> none;
      none.rho = none.vx = none.vy = none.vz = none.p = none.s = none.cs = T(0);
      PL::put_prim(L, buf(-1), t, none);
      load(0);
      __syncthreads();
      Prim<T> pp = prim();
      load(1);
      PL::put_prim(L, buf(0), t, pp);
      T cs = pp.cs;
      __syncthreads();
      if (ghosts) {
        // ring 1: beside a coarser block predicted in place; a same-level leaf's cell away from
        // the face's rim as at its source; other half steps from the shell. The +x and +y ghosts'
        // lower faces are the cells' upper ones: one solve along the lane's axis
        const bool gk = bt(tab, s, BT_NB + side) == -1;
        const bool upper = (side & 1) != 0, ax = side == 1;
        const int fk = side == 1 ? fa[1] : fa[3];
        for (int c = 0; c < AMR_BS; c++) {
          if (c + 1 < AMR_BS) pp = prim(); else pp = none;
          Edges e;
          Half<T> h;
          {
            AxisSlope<T> sl[3];
            Prim<T> pc;
            T conv, jump;
            slopes(buf(c), buf(c - 1), pc, cs, pp, sl, e, conv, jump);
            if (gk) {
              scale_inc(sl[0].s, (side >= 2 && (x == 0 || x == AMR_BS - 1)) ? T(0) : T(1));
              scale_inc(sl[1].s, (side < 2 && (y == 0 || y == AMR_BS - 1)) ? T(0) : T(1));
              scale_inc(sl[2].s, (c == 0 || c == AMR_BS - 1) ? T(0) : T(1));
            }
            h = hancock<T, LIM>(P, pc, sl, conv, jump, hstep);
          }
          const bool exact = nbs >= 0 && off_rim(side < 2 ? y : x, c);
          if (!gk && !exact) h = shell_half((tid - 256) * AMR_BS + c);
          if (c + 2 < AMR_BS) load(c + 2);
          PL::put_side(L, PL::SX, t, side_of(P, h, e.xu, T(1)));
          PL::put_side(L, PL::SY, t, side_of(P, h, e.yu, T(1)));
          PL::put_shock(L, PL::SK, t, h.shock);
          const SideData<T> sxl = side_of(P, h, e.xd, T(-1)), syl = side_of(P, h, e.yd, T(-1));
          PL::put_prim(L, buf(c + 1), t, pp);
          cs = pp.cs;
          __syncthreads();
          if (upper) {
            Flux<T> F = face_from_sides_rt<T, RS>(P, PL::side(L, ax ? PL::SX : PL::SY, PL::SK, t.off(ax ? -1 : -BX)),
                                                  ax ? sxl : syl, ax ? 0 : 1);
            F = boundary_face<T>(fk, R, CF, ax ? c * 16 + y : x * 16 + c, F);
            PL::put_flux(L, ax ? PL::FX : PL::FY, t, F);
          }
          __syncthreads();
        }
      } else {
        // ring 2: loads only
        for (int c = 0; c < AMR_BS; c++) {
          if (c + 1 < AMR_BS) PL::put_prim(L, buf(c + 1), t, prim());
          if (c + 2 < AMR_BS) load(c + 2);
          __syncthreads();
          __syncthreads();
        }
      }
    }
    // a leaf on a coarser block: its register fluxes are written (the barrier waits for every
    // wave's stores); one release fence writes them back to device-coherent memory, then its
    // done flag
    __syncthreads();
    bool writes_reg = false;
#pragma unroll
    for (int k = 0; k < 6; k++) writes_reg = writes_reg || (fa[k] >= 0 && !(fa[k] & 1));
    if (tid == 0 && act_blk && writes_reg) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      __hip_atomic_store(done + s, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  // workgroup maximum of the next step's rate, one atomicMax
  const T v = wave_max(rate_max);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    T m = T(0);
    for (int w = 0; w < AF_PAIR * AF_THREADS / 64; w++) m = tmax(m, red[w]);
    max_slot(next_slot, (unsigned long long)order_bits(m));
  }
}

// (3D blocks only: the ops of a 2D grid leave the fused form out)
template <typename T, int LIM, int RS, bool ISEN, int D>
void AmrImpl<T, LIM, RS, ISEN, D>::shell(const AmrLaunch& L, const int* shell_of, const int* work0, int n0,
                                         const int* work1, int n1, const int* work2, int n2, const void* u1,
                                         const void* u2, void* sh, const void* clk) {
  static_assert(D == 3, "the fused form steps 3D blocks");
  if (n0 > 0)
    hipLaunchKernelGGL((k_amr_shell<T, LIM, false, 0>), dim3((n0 + 3) / 4), dim3(256), 0, L.stream, P(L), L.tab,
                       shell_of, nullptr, 0, (const int4*)work0, n0, (const T4<T>*)u1, (const T4<T>*)u2, (T4<T>*)sh,
                       (const T*)clk);
  if (n1 + n2 > 0)
    hipLaunchKernelGGL((k_amr_shell<T, LIM, ISEN, 1>), dim3((n2 + 255) / 256 + (n1 + 3) / 4), dim3(256), 0, L.stream,
                       P(L), L.tab, shell_of, (const int4*)work2, n2, (const int4*)work1, n1, (const T4<T>*)u1,
                       (const T4<T>*)u2, (T4<T>*)sh, (const T*)clk);
}

template <typename T, int LIM, int RS, bool ISEN, int D>
void AmrImpl<T, LIM, RS, ISEN, D>::fused(const AmrLaunch& L, const AmrQueue& Q, const void* sh, const void* u1,
                                         const void* u2, void* o1, void* o2, const void* clk,
                                         unsigned long long* slot) {
  static_assert(D == 3, "the fused form steps 3D blocks");
  if (Q.count <= 0) return;
  constexpr int np = af_pair<T>();
  const int pairs = (Q.count + np - 1) / np;
  const int grid = Q.grid < pairs ? Q.grid : pairs;
  hipLaunchKernelGGL((k_amr_queue_start<T>), dim3(1), dim3(1), 0, L.stream, Q.qctl);
  hipLaunchKernelGGL((k_amr_fused<T, LIM, RS, ISEN>), dim3(grid), dim3(np * AF_THREADS), 0, L.stream, P(L), L.tab,
                     Q.list, Q.count, Q.shell_of, (const T4<T>*)sh, Q.act, (T*)Q.reg, (T*)Q.cf, Q.reg_of, Q.comp,
                     Q.dep_off, Q.dep, Q.qctl, Q.done, (const T4<T>*)u1, (const T4<T>*)u2, (T4<T>*)o1, (T4<T>*)o2,
                     (const T*)clk, slot);
}

}  // namespace shx
