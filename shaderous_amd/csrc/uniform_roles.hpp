// The fused uniform-grid step with threads by role (k_fused_r): the same arithmetic as k_fused,
// with a different map of threads to the tile's columns. A tile is TX x TY cells (32 x 16, 32 x 8
// or 16 x 16, so 256^3 and other power-of-two grids split into whole tiles); of its
// (TX + 4) x (TY + 4) columns, threads own, in this order:
//   [0, TX TY)               the cell columns, x fastest: whole waves of cell work
//   the next 2 TX + 2 TY     ring 1 without its corners (half steps): the top row and the right
//                            column first (they also solve the faces they share with the tile's
//                            cells), then the bottom row and the left column
//   the last 2 TX + 2 TY     ring 2 without its corners (loads only); ring 2's corners are never
//                            read. The last four threads load ring 1's corners as well (their
//                            primitives feed the transverse slopes of ring 1's ends), so that
//                            they take no wave of their own: 16 x 16 cells are six waves.
// Each role runs its own loop over the planes (a scalar branch per wave, the barriers in step): the
// cell waves never carry halo lanes or their registers, and the planes before the first and after
// the last one, which need only the cells' z sides, cost the other waves a conversion.
//
// Bound by VALU issue. Against one loop for every role with its stages behind lane masks, the
// state re-read at its use and single-value LDS accesses, per step: 256^3 MC 0.515 -> 0.342 ms
// (3.1 TB/s of state read and written once), Koren + isentropic 0.795 -> 0.656; 128^3 0.073 ->
// 0.053 and 0.124 -> 0.102; FP64 96^3 MC 0.147 (raster tiles) -> 0.104. 32 x 16 is the tile of large
// grids: its two ring waves land on two SIMDs, beside two cell waves each.
#pragma once

namespace shx {

template <int TX, int TY>
struct RoleTile {
  static constexpr int CX = TX + 4, CY = TY + 4, NC = CX * CY;   // LDS columns
  static constexpr int NCELL = TX * TY;
  static constexpr int NHALF = NCELL + 2 * TX + 2 * TY;          // threads that form half steps
  static constexpr int NFACE = NCELL + TX + TY;                  // threads that solve x/y faces
  static constexpr int NTH = NHALF + 2 * TX + 2 * TY;            // threads with a role
  // At 16 x 16 the ring wave and the load wave are the fifth and sixth of a workgroup, and waves go
  // to a CU's SIMDs in turn: two workgroups would put both ring waves on the first SIMD (0.523
  // against 0.383 ms at 256^3). So a workgroup is launched with eight waves, of which the last
  // four hold those two roles in the fifth and sixth or, in every second run of 256 workgroups (as
  // many as there are CUs), in the seventh and eighth; the other two end at once.
  // (FP64 has the LDS for one workgroup per CU.)
  template <typename T>
  static constexpr bool paired() { return sizeof(T) == 4 && NCELL == 256 && NTH == 384; }
  template <typename T>
  static constexpr int launch() { return paired<T>() ? 512 : NTH; }
  // waves per SIMD the launch bound asks for in FP32: one 11-wave workgroup per CU at 32 x 16 (up
  // to 168 VGPRs), two otherwise (128 VGPRs); one at 16 x 16 where Koren's edges need more
  // registers than that (it serves the grids with too few tiles for two), and in FP64
  template <typename T, int LIM>
  static constexpr int minw() {
    return sizeof(T) == 8 || (paired<T>() && !lim_symmetric<LIM>()) ? 2 : (NCELL > 256 ? 3 : 4);
  }
};

// thread -> column (cx, cy) in cell-tile coordinates, [-2, TX + 2) x [-2, TY + 2)
template <int TX, int TY>
__device__ __forceinline__ void role_column(int t, int& cx, int& cy) {
  using RT = RoleTile<TX, TY>;
  if (t < RT::NCELL) {
    cx = t % TX;
    cy = t / TX;
    return;
  }
  t -= RT::NCELL;
  if (t < TX) { cx = t; cy = TY; return; }             // ring 1: y faces on the top row
  t -= TX;
  if (t < TY) { cx = TX; cy = t; return; }             // x faces on the right column
  t -= TY;
  if (t < TX) { cx = t; cy = -1; return; }             // the bottom row
  t -= TX;
  if (t < TY) { cx = -1; cy = t; return; }             // the left column
  t -= TY;
  if (t < TX) { cx = t; cy = -2; return; }             // ring 2: bottom, top, left, right
  t -= TX;
  if (t < TX) { cx = t; cy = TY + 1; return; }
  t -= TX;
  if (t < TY) { cx = -2; cy = t; return; }
  t -= TY;
  cx = TX + 1; cy = t;
}

// The planes in LDS: per column the primitives of two planes (rho, v | p, s; the centre's sound
// speed stays in a register), the upper x and y sides (rho, v | p, s, half-step rho and p) with the
// cell's shock flag, and the fluxes of the x and y faces below the column: 45 values, kept as
// 4- and 2-vectors so that a neighbour is two or three LDS instructions and not six to nine.
template <typename T> struct Vec2;
template <> struct Vec2<float> { using type = float2; };
template <> struct Vec2<double> { using type = double2; };
// Columns' values in LDS as 4- and 2-vectors (structure of arrays over NT columns; offsets in T)
template <typename T, int NT>
struct ColumnLds {
  using V4 = T4<T>;
  using V2 = typename Vec2<T>::type;
  // A column's byte offsets in the arrays of 4-, 2- and 1-vectors, each kept as a value of its own
  // (the empty asm): the compiler derives one from another by a quarter-rate multiplication per
  // plane otherwise. off: a column so many to the right.
  struct At {
    unsigned int a, b, c;
    __device__ __forceinline__ At off(int d) const {
      return At{a + (unsigned int)(d * (int)sizeof(V4)), b + (unsigned int)(d * (int)sizeof(V2)),
                c + (unsigned int)(d * (int)sizeof(T))};
    }
  };
  static __device__ __forceinline__ At at(int t) {
    At k{(unsigned int)(t * (int)sizeof(V4)), (unsigned int)(t * (int)sizeof(V2)), (unsigned int)(t * (int)sizeof(T))};
    asm("" : "+v"(k.a));
    asm("" : "+v"(k.b));
    asm("" : "+v"(k.c));
    return k;
  }
  template <typename V>
  static __device__ __forceinline__ V& ref(T* L, int base, unsigned int off) {
    return *reinterpret_cast<V*>(reinterpret_cast<char*>(L + base) + off);
  }
  static __device__ __forceinline__ void put_prim(T* L, int q, const At& t, const Prim<T>& w) {
    V4 a; a.x = w.rho; a.y = w.vx; a.z = w.vy; a.w = w.vz;
    V2 b; b.x = w.p; b.y = w.s;
    ref<V4>(L, q, t.a) = a;
    ref<V2>(L, q + 4 * NT, t.b) = b;
  }
  static __device__ __forceinline__ Prim<T> prim(T* L, int q, const At& t) {
    const V4 a = ref<V4>(L, q, t.a);
    const V2 b = ref<V2>(L, q + 4 * NT, t.b);
    Prim<T> w;
    w.rho = a.x; w.vx = a.y; w.vy = a.z; w.vz = a.w; w.p = b.x; w.s = b.y; w.cs = T(0);
    return w;
  }
  static __device__ __forceinline__ void put_side(T* L, int s, const At& t, const SideData<T>& d) {
    V4 a; a.x = d.rho; a.y = d.vx; a.z = d.vy; a.w = d.vz;
    V4 b; b.x = d.p; b.y = d.s; b.z = d.hrho; b.w = d.hp;
    ref<V4>(L, s, t.a) = a;
    ref<V4>(L, s + 4 * NT, t.a) = b;
  }
  static __device__ __forceinline__ void put_shock(T* L, int k, const At& t, T shock) { ref<T>(L, k, t.c) = shock; }
  static __device__ __forceinline__ SideData<T> side(T* L, int s, int k, const At& t) {
    const V4 a = ref<V4>(L, s, t.a), b = ref<V4>(L, s + 4 * NT, t.a);
    SideData<T> d;
    d.rho = a.x; d.vx = a.y; d.vy = a.z; d.vz = a.w; d.p = b.x; d.s = b.y; d.hrho = b.z; d.hp = b.w;
    d.shock = ref<T>(L, k, t.c);
    return d;
  }
  static __device__ __forceinline__ void put_flux(T* L, int f, const At& t, const Flux<T>& F) {
    V4 a; a.x = F.m; a.y = F.mx; a.z = F.my; a.w = F.mz;
    V4 b; b.x = F.e; b.y = F.ei; b.z = F.s; b.w = F.vn;
    ref<V4>(L, f, t.a) = a;
    ref<V4>(L, f + 4 * NT, t.a) = b;
  }
  static __device__ __forceinline__ Flux<T> flux(T* L, int f, const At& t) {
    const V4 a = ref<V4>(L, f, t.a), b = ref<V4>(L, f + 4 * NT, t.a);
    Flux<T> F;
    F.m = a.x; F.mx = a.y; F.my = a.z; F.mz = a.w; F.e = b.x; F.ei = b.y; F.s = b.z; F.vn = b.w;
    return F;
  }
};

// A cell of a plane by its byte offset, through a buffer resource over the plane (a scalar base and
// one 32-bit vector offset; the resource covers 4 GiB, beyond what offsets reach)
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t plane_rsrc(const void* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, 0xffffffff, 0x00020000);
}
template <typename T>
__device__ __forceinline__ T4<T> plane_load(const T4<T>* base, unsigned int off) {
  const __amdgpu_buffer_rsrc_t r = plane_rsrc(base);
  struct Words { u32x4 w[sizeof(T4<T>) / 16]; } k;
#pragma unroll
  for (int i = 0; i < (int)(sizeof(T4<T>) / 16); i++) k.w[i] = __builtin_amdgcn_raw_buffer_load_b128(r, off + 16 * i, 0, 0);
  return __builtin_bit_cast(T4<T>, k);
}
template <typename T>
__device__ __forceinline__ void plane_store(T4<T>* base, unsigned int off, T4<T> v) {
  const __amdgpu_buffer_rsrc_t r = plane_rsrc(base);
  struct Words { u32x4 w[sizeof(T4<T>) / 16]; } k = __builtin_bit_cast(Words, v);
#pragma unroll
  for (int i = 0; i < (int)(sizeof(T4<T>) / 16); i++) __builtin_amdgcn_raw_buffer_store_b128(k.w[i], r, off + 16 * i, 0, 0);
}

// k_fused_r's planes: primitives of two planes (QN apart), sides, shock flags, fluxes
template <typename T, int NT>
struct PlaneLds : ColumnLds<T, NT> {
  static constexpr int QN = 6 * NT, SX = 12 * NT, SY = 20 * NT, SK = 28 * NT, FX = 29 * NT, FY = 37 * NT,
                       SIZE = 45 * NT;
};

// The net inflow of a plane's x and y faces, and with the z faces' (lower lo, upper hi)
template <typename T>
__device__ __forceinline__ Flux<T> net_xy(const Flux<T>& xl, const Flux<T>& xh, const Flux<T>& yl, const Flux<T>& yh) {
  Flux<T> n;
  n.m = (xl.m - xh.m) + (yl.m - yh.m);
  n.mx = (xl.mx - xh.mx) + (yl.mx - yh.mx);
  n.my = (xl.my - xh.my) + (yl.my - yh.my);
  n.mz = (xl.mz - xh.mz) + (yl.mz - yh.mz);
  n.e = (xl.e - xh.e) + (yl.e - yh.e);
  n.ei = (xl.ei - xh.ei) + (yl.ei - yh.ei);
  n.s = (xl.s - xh.s) + (yl.s - yh.s);
  n.vn = (xl.vn - xh.vn) + (yl.vn - yh.vn);
  return n;
}
template <typename T>
__device__ __forceinline__ Flux<T> net_z(const Flux<T>& xy, const Flux<T>& lo, const Flux<T>& hi) {
  Flux<T> n;
  n.m = xy.m + (lo.m - hi.m);
  n.mx = xy.mx + (lo.mx - hi.mx);
  n.my = xy.my + (lo.my - hi.my);
  n.mz = xy.mz + (lo.mz - hi.mz);
  n.e = xy.e + (lo.e - hi.e);
  n.ei = xy.ei + (lo.ei - hi.ei);
  n.s = xy.s + (lo.s - hi.s);
  n.vn = xy.vn + (lo.vn - hi.vn);
  return n;
}

// z: periodic, or through a non-periodic face as k_fused (ZA, ZB: the boundary planes' half steps).
// Columns beyond the grid (a ragged tile's) compute on the cells they map to and store nothing.
// Barriers: the half steps of plane c (sides, and plane c + 1's primitives) are visible after
// the first, its x/y fluxes after the second. The sides of plane c + 1 overwrite those of plane c
// after the second barrier of plane c (the last reads of sides were before it); the fluxes of
// plane c + 1 overwrite those of plane c after the first barrier of plane c + 1; each primitive
// buffer is rewritten a plane after its neighbours were last read from it. The z faces and the
// update of plane c - 1 need nothing of LDS: they go before the first barrier, and the state they
// update is loaded a half step ahead.
// A plane's byte offsets fit 32 bits (the launcher's rule), so a load is a scalar base and one
// vector offset.
template <typename T, int LIM, int RS, bool ISEN, int TX, int TY, bool DEBUG, bool MAPBC>
__global__ __launch_bounds__((RoleTile<TX, TY>::template launch<T>()),
                             (RoleTile<TX, TY>::template minw<T, LIM>())) void k_fused_r(
    Params<T> P, const T4<T>* __restrict__ U1, const T4<T>* __restrict__ U2, T4<T>* __restrict__ O1,
    T4<T>* __restrict__ O2, StepClock<T> C, const T4<T>* __restrict__ ZA, const T4<T>* __restrict__ ZB, int zc) {
  using RT = RoleTile<TX, TY>;
  constexpr int NT = RT::NC, BX = RT::CX, NW = (RT::NTH + 63) / 64;
  using PL = PlaneLds<T, NT>;
  __shared__ T4<T> LV[PL::SIZE / 4];
  __shared__ T red[NW];
  T* const L = reinterpret_cast<T*>(LV);
  const int lin = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
  // the wave's role, a scalar
  int wave = __builtin_amdgcn_readfirstlane(threadIdx.x) >> 6;
  if constexpr (RT::template paired<T>()) {
    if (wave >= 4) {
      if (((wave >> 1) & 1) != ((lin >> 8) & 1)) return;
      wave = 4 | (wave & 1);
    }
  }
  const int tid = wave * 64 + (threadIdx.x & 63);
  const bool cells = wave < RT::NCELL / 64, rings = !cells && wave * 64 < RT::NHALF;
  int cx, cy;
  role_column<TX, TY>(tid, cx, cy);
  const typename PL::At t = PL::at((cy + 2) * BX + (cx + 2));   // the column, in raster order
  const int nx = P.n[0], ny = P.n[1], nz = P.n[2];
  // XCD-aware tile order: the dispatcher deals workgroups to the 8 XCDs in turn (workgroup i to
  // XCD i mod 8), so XCD k takes the k-th of 8 contiguous runs of tiles (the first n mod 8 runs
  // one tile longer) and marches it in order, rows of tiles side by side: the halo columns two
  // tiles share are read through one L2. The same tiles are stepped either way.
  int bx, by, bz;
  {
    const int ntile = gridDim.x * gridDim.y * gridDim.z;
    const int k = lin & 7, q = ntile >> 3, r = ntile & 7;
    const int m = k * q + min(k, r) + (lin >> 3);
    bx = m % gridDim.x;
    by = (m / gridDim.x) % gridDim.y;
    bz = m / (gridDim.x * gridDim.y);
  }
  const int z0 = bz * zc;
  const int z1 = min(z0 + zc, nz);
  const T dt = step_dt(P, C, 0);
  const T dtdx = wave_uniform(tratio(dt, P.dx)), hstep = wave_uniform(slope_step<T, LIM>(P, dt));
  if (blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0 && tid == 0) step_clock_advance(P, C, 0);

  const size_t plane = (size_t)nx * ny;
  // z: periodic, or (ZA given) a non-periodic face that ghost planes map through
  const bool zbc = MAPBC && ZA != nullptr;
  auto plane_of = [&](int z) -> size_t {
    if (zbc) return (size_t)map_axis(z, nz, P.bc_lo[2], P.bc_hi[2]).i * plane;
    while (z < 0) z += nz;
    while (z >= nz) z -= nz;
    return (size_t)z * plane;
  };
  // a column of the tile: the byte offset in a plane of the cell it maps to, and whether that cell
  // is seen through a reflecting x or y face (its velocity turns; outflow-only faces, which clip
  // it, are not run here)
  struct Column { unsigned int at; bool fx, fy; };
  auto column = [&](int cx, int cy) {
    const AxisMap mx = map_axis(bx * TX + cx, nx, P.bc_lo[0], P.bc_hi[0]);
    const AxisMap my = map_axis(by * TY + cy, ny, P.bc_lo[1], P.bc_hi[1]);
    return Column{(unsigned int)(my.i * nx + mx.i) * (unsigned int)sizeof(T4<T>), mx.flip < 0, my.flip < 0};
  };
  auto at = [](const T4<T>* base, unsigned int off) { return plane_load<T>(base, off); };
  auto prim_of = [&](const Column& k, T4<T> u1, T4<T> u2, int z) {
    Prim<T> q = prim_from_cons(P, u1, u2);
    if constexpr (MAPBC) {
      q.vx = k.fx ? -q.vx : q.vx;
      q.vy = k.fy ? -q.vy : q.vy;
    }
    if (zbc && (z < 0 || z >= nz)) {
      const AxisMap mz = map_axis(z, nz, P.bc_lo[2], P.bc_hi[2]);
      q.vz = bc_vel(q.vz, mz.flip, mz.side);
    }
    return q;
  };
  const Column K = column(cx, cy);
  // a ghost column beyond a non-periodic face takes the half step of the cell it maps to
  // (load_pred, hydro/update.wgsl:47-63): that cell's stencil sits inward in the tile
  int sx = cx, sy = cy;
  {
    const int x = bx * TX + cx, y = by * TY + cy;
    if ((x < 0 && P.bc_lo[0] != BC_PERIODIC) || (x >= nx && P.bc_hi[0] != BC_PERIODIC))
      sx = cx + (map_axis(x, nx, P.bc_lo[0], P.bc_hi[0]).i - x);
    if ((y < 0 && P.bc_lo[1] != BC_PERIODIC) || (y >= ny && P.bc_hi[1] != BC_PERIODIC))
      sy = cy + (map_axis(y, ny, P.bc_lo[1], P.bc_hi[1]).i - y);
  }
  const bool mapped = MAPBC && ((sx != cx) || (sy != cy));
  const bool any_mapped = MAPBC && __ballot(mapped) != 0;
  const typename PL::At ts = PL::at((min(max(sy, -1), TY) + 2) * BX + (min(max(sx, -1), TX) + 2));

  // the half step of this column in the plane whose primitives are at q (those of the plane below
  // at m, of the plane above in pp), and its edge increments (hydro/predictor.wgsl:46-209)
  struct Edges { Inc<T> xu, xd, yu, yd, zu, zd; };
  auto half_at = [&](int q, const typename PL::At& at, Prim<T> pc, const Prim<T>& pm, const Prim<T>& pp, Edges& e) {
    AxisSlope<T> sl[3];
    // axis by axis: the scheduler would read every neighbour first, at 12 more registers an axis
    T conv, jump;
    {
      const Prim<T> xm = PL::prim(L, q, at.off(-1)), xp = PL::prim(L, q, at.off(1));
      sl[0] = axis_slope<T, LIM, ISEN>(P, xm, pc, xp, &e.xu, &e.xd);
      conv = xp.vx - xm.vx;
      jump = jump_over(P, xm.p, xp.p);
    }
    __builtin_amdgcn_sched_barrier(0);
    {
      const Prim<T> ym = PL::prim(L, q, at.off(-BX)), yp = PL::prim(L, q, at.off(BX));
      sl[1] = axis_slope<T, LIM, ISEN>(P, ym, pc, yp, &e.yu, &e.yd);
      conv = conv + (yp.vy - ym.vy);
      jump = tmax(jump, jump_over(P, ym.p, yp.p));
    }
    __builtin_amdgcn_sched_barrier(0);
    sl[2] = axis_slope<T, LIM, ISEN>(P, pm, pc, pp, &e.zu, &e.zd);
    __builtin_amdgcn_sched_barrier(0);
    conv = conv + (pp.vz - pm.vz);
    return hancock<T, LIM>(P, pc, sl, conv, tmax(jump, jump_over(P, pm.p, pp.p)), hstep);
  };
  auto half_of = [&](int q, int m, T cs, const Prim<T>& pp, Edges& e) {
    Prim<T> pc = PL::prim(L, q, t);
    pc.cs = cs;
    const Prim<T> pm = PL::prim(L, m, t);
    if constexpr (!MAPBC) {
      return half_at(q, t, pc, pm, pp, e);
    } else {
      // where a lane of the wave is mapped: first every lane's half step at the cell it maps to (the
      // column itself if it maps to none), its centre being this column's primitives seen
      // unflipped, then the increments and the half step here. One body, two turns.
      Half<T> h, hm;
#pragma unroll 1
      for (int k = any_mapped ? 0 : 1; k < 2; k++) {
        const bool first = k == 0;
        Prim<T> qc = pc, qm = pm, qp = pp;
        if (first) {
          qc.vx = K.fx ? -qc.vx : qc.vx; qc.vy = K.fy ? -qc.vy : qc.vy;
          qm.vx = K.fx ? -qm.vx : qm.vx; qm.vy = K.fy ? -qm.vy : qm.vy;
          qp.vx = K.fx ? -qp.vx : qp.vx; qp.vy = K.fy ? -qp.vy : qp.vy;
        }
        h = half_at(q, first ? ts : t, qc, qm, qp, e);
        if (first) {
          hm = h;
          hm.vx = K.fx ? -hm.vx : hm.vx;
          hm.vy = K.fy ? -hm.vy : hm.vy;
        }
      }
      if (mapped) h = hm;
      return h;
    }
  };
  // the buffer of plane c's primitives: plane z0 - 2 and z0 in the first, z0 - 1 and z0 + 1 in the
  // second, and so on
  auto buf = [&](int c) { return ((c - z0) & 1) ? PL::QN : 0; };

  T rate_max = T(0);
  if (cells) {
    const bool upd = bx * TX + cx < nx && by * TY + cy < ny;
    T4<T> b1, b2;
    auto load = [&](int z) {
      const size_t o = plane_of(z);
      b1 = at(U1 + o, K.at);
      b2 = at(U2 + o, K.at);
    };
    load(z0 - 2);
    PL::put_prim(L, buf(z0 - 2), t, prim_of(K, b1, b2, z0 - 2));
    load(z0 - 1);
    Prim<T> pp = prim_of(K, b1, b2, z0 - 1);
    PL::put_prim(L, buf(z0 - 1), t, pp);
    T cs = pp.cs;   // this column's sound speed in plane c
    load(z0);
    __syncthreads();
    SideData<T> zs;           // the upper z side of the plane below
    T hp;                     // and its half-step pressure
    Flux<T> fz_lo, xy;        // the z face below and the x/y net inflow of that plane
    auto update = [&](int c, T4<T> u1, T4<T> u2, const Flux<T>& fz) {
      T4<T> o1, o2;
      if constexpr (DEBUG) {
        o1.x = xy.m; o1.y = xy.mx; o1.z = xy.my; o1.w = xy.mz;
        o2.x = fz_lo.m; o2.y = fz.m; o2.z = T(0); o2.w = T(0);
      } else {
        advance(P, u1, u2, net_z(xy, fz_lo, fz), hp, dtdx, o1, o2);
      }
      if (upd) {
        const size_t o = (size_t)c * plane;
        plane_store<T>(O1 + o, K.at, o1);
        plane_store<T>(O2 + o, K.at, o2);
        if constexpr (!DEBUG) rate_max = tmax(rate_max, rate_of(P, prim_from_cons(P, o1, o2)));
      }
    };
    {
      // plane z0 - 1: its upper z sides
      pp = prim_of(K, b1, b2, z0);
      load(z0 + 1);
      Edges e;
      Half<T> h = half_of(buf(z0 - 1), buf(z0 - 2), cs, pp, e);
      if (zbc && upd) zghost_half(P, ZA, ZB, z0 - 1, K.at / sizeof(T4<T>), h);
      zs = side_of(P, h, e.zu, T(1));
      hp = h.p;
      PL::put_prim(L, buf(z0), t, pp);
      cs = pp.cs;
    }
    __syncthreads();
    for (int c = z0; c < z1; c++) {
      pp = prim_of(K, b1, b2, c + 1);
      Edges e;
      const Half<T> h = half_of(buf(c), buf(c - 1), cs, pp, e);
      __builtin_amdgcn_sched_barrier(0);
      T4<T> u1, u2;
      if (c > z0) {
        const size_t o = (size_t)(c - 1) * plane;
        u1 = at(U1 + o, K.at);
        u2 = at(U2 + o, K.at);
      }
      PL::put_side(L, PL::SX, t, side_of(P, h, e.xu, T(1)));
      PL::put_side(L, PL::SY, t, side_of(P, h, e.yu, T(1)));
      PL::put_shock(L, PL::SK, t, h.shock);
      PL::put_prim(L, buf(c + 1), t, pp);
      cs = pp.cs;
      __builtin_amdgcn_sched_barrier(0);
      const Flux<T> fz = face_from_sides<T, RS>(P, zs, side_of(P, h, e.zd, T(-1)), 2);
      __builtin_amdgcn_sched_barrier(0);
      if (c > z0) update(c - 1, u1, u2, fz);
      fz_lo = fz;
      zs = side_of(P, h, e.zu, T(1));
      hp = h.p;
      __builtin_amdgcn_sched_barrier(0);
      load(c + 2);
      __syncthreads();
      const Flux<T> Fx = face_from_sides<T, RS>(P, PL::side(L, PL::SX, PL::SK, t.off(-1)), side_of(P, h, e.xd, T(-1)), 0);
      PL::put_flux(L, PL::FX, t, Fx);
      __builtin_amdgcn_sched_barrier(0);
      const Flux<T> Fy = face_from_sides<T, RS>(P, PL::side(L, PL::SY, PL::SK, t.off(-BX)), side_of(P, h, e.yd, T(-1)), 1);
      PL::put_flux(L, PL::FY, t, Fy);
      __syncthreads();
      const Flux<T> xh = PL::flux(L, PL::FX, t.off(1)), yh = PL::flux(L, PL::FY, t.off(BX));
      if constexpr (DEBUG) {
        xy.m = Fx.m; xy.mx = xh.m; xy.my = Fy.m; xy.mz = yh.m;
      } else {
        xy = net_xy(Fx, xh, Fy, yh);
      }
    }
    {
      // plane z1: its lower z sides, and the update of plane z1 - 1
      pp = prim_of(K, b1, b2, z1 + 1);
      const size_t o = (size_t)(z1 - 1) * plane;
      const T4<T> u1 = at(U1 + o, K.at), u2 = at(U2 + o, K.at);
      Edges e;
      Half<T> h = half_of(buf(z1), buf(z1 - 1), cs, pp, e);
      if (zbc && upd) zghost_half(P, ZA, ZB, z1, K.at / sizeof(T4<T>), h);
      update(z1 - 1, u1, u2, face_from_sides<T, RS>(P, zs, side_of(P, h, e.zd, T(-1)), 2));
    }
  } else if (rings) {
    // ring 1 (and, in a mixed wave, ring 2's first lanes, which only load)
    const bool ring1 = tid < RT::NHALF, face = tid < RT::NFACE;
    const bool ax = cx == TX;      // the right column's x faces, else the top row's y faces
    T4<T> b1, b2;
    auto load = [&](int z) {
      const size_t o = plane_of(z);
      b1 = at(U1 + o, K.at);
      b2 = at(U2 + o, K.at);
    };
    load(z0 - 1);
    Prim<T> pp = prim_of(K, b1, b2, z0 - 1);
    PL::put_prim(L, buf(z0 - 1), t, pp);
    load(z0);
    __syncthreads();
    pp = prim_of(K, b1, b2, z0);
    load(z0 + 1);
    PL::put_prim(L, buf(z0), t, pp);
    T cs = pp.cs;
    __syncthreads();
    for (int c = z0; c < z1; c++) {
      pp = prim_of(K, b1, b2, c + 1);
      if (c + 2 <= z1) load(c + 2);
      SideData<T> lo;
      if (ring1) {
        Edges e;
        const Half<T> h = half_of(buf(c), buf(c - 1), cs, pp, e);
        PL::put_side(L, PL::SX, t, side_of(P, h, e.xu, T(1)));
        PL::put_side(L, PL::SY, t, side_of(P, h, e.yu, T(1)));
        PL::put_shock(L, PL::SK, t, h.shock);
        const SideData<T> sxl = side_of(P, h, e.xd, T(-1)), syl = side_of(P, h, e.yd, T(-1));
        lo = ax ? sxl : syl;
      }
      PL::put_prim(L, buf(c + 1), t, pp);
      cs = pp.cs;
      __syncthreads();
      if (face) {
        const SideData<T> below = PL::side(L, ax ? PL::SX : PL::SY, PL::SK, t.off(ax ? -1 : -BX));
        const Flux<T> F = face_from_sides_rt<T, RS>(P, below, lo, ax ? 0 : 1);
        PL::put_flux(L, ax ? PL::FX : PL::FY, t, F);
      }
      __syncthreads();
    }
  } else {
    // ring 2, and by the last four threads ring 1's corners
    const int e = tid - (RT::NTH - 4);
    const bool corner = e >= 0;
    const int ex = (e & 1) ? TX : -1, ey = (e & 2) ? TY : -1;
    const typename PL::At te = PL::at((ey + 2) * BX + (ex + 2));
    const Column KE = column(ex, ey);
    T4<T> b1, b2, c1, c2;
    auto load = [&](int z) {
      const size_t o = plane_of(z);
      b1 = at(U1 + o, K.at);
      b2 = at(U2 + o, K.at);
      if (corner) {
        c1 = at(U1 + o, KE.at);
        c2 = at(U2 + o, KE.at);
      }
    };
    auto put = [&](int z) {
      PL::put_prim(L, buf(z), t, prim_of(K, b1, b2, z));
      if (corner) PL::put_prim(L, buf(z), te, prim_of(KE, c1, c2, z));
    };
    load(z0);
    __syncthreads();
    put(z0);
    if (z0 + 1 < z1) load(z0 + 1);
    __syncthreads();
    for (int c = z0; c < z1; c++) {
      if (c + 1 < z1) put(c + 1);
      if (c + 2 < z1) load(c + 2);
      __syncthreads();
      __syncthreads();
    }
  }
  if constexpr (!DEBUG) {
    T v = wave_max(rate_max);
    if ((tid & 63) == 0) red[wave] = v;
    __syncthreads();
    if (tid == 0) {
      T m = T(0);
      for (int w = 0; w < RT::NCELL / 64; w++) m = tmax(m, red[w]);
      max_slot(C.next(0), (unsigned long long)order_bits(m));
    }
  }
}

}  // namespace shx
