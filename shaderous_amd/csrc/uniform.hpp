// Interface between the C-ABI layer and the uniform-grid kernels: type-erased launchers, one
// table per (precision, limiter, Riemann solver, isentropic) combination.
#pragma once
#include <algorithm>
#include <vector>
#include "diag.hpp"
#include "hydro.hpp"

namespace shx {

struct Launch {
  hipStream_t stream;
  const void* params;   // Params<T> of the sim's precision
  size_t ncell;
};

// Column tiles of the fused kernel: k_fused_r's (threads by role, tiles of 32 x 16, 32 x 8 or, as
// FUSED_20x20, 16 x 16 cells: the only one in FP64) and k_fused's (block BX x BY threads in raster
// order, tile (BX - 4) x (BY - 4) cells; FUSED_RASTER20 in FP64 alone, the others in FP32 alone).
// k_fused is slower on every grid measured: it is run on wide planes and on request.
enum { FUSED_20x20 = 0, FUSED_32x16 = 1, FUSED_32x32 = 2, FUSED_R32x16 = 3, FUSED_R32x8 = 4, FUSED_RASTER20 = 5,
       FUSED_NTILES = 6 };
inline bool fused_is_raster(int tile) { return tile == FUSED_32x16 || tile == FUSED_32x32 || tile == FUSED_RASTER20; }
// A plane of 4 GiB or more: k_fused_r addresses a plane with 32 bits
inline bool fused_wide(int nx, int ny, int elem) { return (size_t)nx * ny * 4 * elem >= (size_t)1 << 32; }
// cells per tile along x and y
inline void fused_tile_cells(int tile, int& tx, int& ty) {
  switch (tile) {
    case FUSED_20x20:
    case FUSED_RASTER20: tx = 16; ty = 16; break;
    case FUSED_32x16: tx = 28; ty = 12; break;
    case FUSED_32x32: tx = 28; ty = 28; break;
    case FUSED_R32x16: tx = 32; ty = 16; break;
    default: tx = 32; ty = 8; break;
  }
}

// The k_fused_r or k_fused tile a grid is stepped by where the configuration or the plane's size
// decides it, else -1. FP64 has one tile, 16 x 16 cells, in raster order where a raster tile is
// asked for.
inline int fused_asked(int nx, int ny, int elem, int tx, int ty) {
  int asked = -1;
  for (int k = 0; tx > 0 && k < FUSED_RASTER20; k++) {
    int x, y;
    fused_tile_cells(k, x, y);
    if (x == tx && y == ty) asked = k;
  }
  if (elem == 8) asked = asked >= 0 && fused_is_raster(asked) ? FUSED_RASTER20 : -1;
  if (fused_wide(nx, ny, elem) && !(asked >= 0 && fused_is_raster(asked)))
    asked = elem == 8 ? FUSED_RASTER20 : FUSED_32x16;
  return asked;
}

// A launch of the 3D march: tile and planes per chunk, and what it is expected to cost, in planes of
// a 32 x 16 tile.
struct FusedShape { int tile, zc; double cost; };

// The shapes of k_fused_r for an nx x ny x nz grid on `cus` CUs, cheapest first. A workgroup marches
// zc planes and about 2.5 planes' worth before and after; workgroups fill the chip's slots in turn,
// so the step takes the work of the slot with the most. Per plane of a tile, with as many
// workgroups on a CU as fit (two of 32 x 8 and 16 x 16; one of 32 x 16, and of 16 x 16 with
// Koren's edges) and with one, against one 32 x 16: measured at 256^3 (MC 2.63 us a plane, Koren +
// isentropic 5.05) and at 48^3 to 64^3. tile, zc > 0 (FP64: the tile is given): only those.
inline std::vector<FusedShape> fused_shapes(int nx, int ny, int nz, int cus, bool fp64, bool koren, int tile, int zc) {
  struct Cost { int tile, fit; double alone, full; };
  const Cost sym[3] = {{FUSED_R32x16, 1, 1.0, 1.0}, {FUSED_R32x8, 2, 0.80, 1.09}, {FUSED_20x20, 2, 0.78, 1.09}};
  const Cost asym[3] = {{FUSED_R32x16, 1, 1.0, 1.0}, {FUSED_R32x8, 2, 0.85, 1.5}, {FUSED_20x20, 1, 0.69, 0.69}};
  std::vector<FusedShape> out;
  for (int k = 0; k < 3; k++) {
    Cost c = koren ? asym[k] : sym[k];
    if (fp64) {
      if (c.tile != FUSED_20x20) continue;
      c.fit = 1;
      c.full = c.alone;
    }
    if (tile >= 0 && c.tile != tile) continue;
    int tx, ty, last = 0;
    fused_tile_cells(c.tile, tx, ty);
    const long long tiles = (long long)((nx + tx - 1) / tx) * ((ny + ty - 1) / ty);
    for (int chunks = 1; chunks <= nz; chunks++) {
      const int z = zc > 0 ? std::min(zc, nz) : (nz + chunks - 1) / chunks;
      if (z == last) continue;
      last = z;
      const long long n = tiles * ((nz + z - 1) / z), slots = (long long)cus * c.fit;
      const double each = n <= cus ? c.alone : c.full * (double)((n + slots - 1) / slots);
      out.push_back(FusedShape{c.tile, z, each * (z + 2.5)});
      if (zc > 0) break;
    }
  }
  std::stable_sort(out.begin(), out.end(), [](const FusedShape& a, const FusedShape& b) { return a.cost < b.cost; });
  return out;
}

// The clocks of a fused step (the step kernel takes its own clock pass, StepClock in
// uniform_impl.hpp), per instance: two clocks of 16 values (parity 0, 1), three rate slots, two
// epochs; p: the parity of the state the step reads.
struct ClockRefs {
  void* clk;
  unsigned long long* slot;
  unsigned int* epoch;
  int p;
};
// Bytes of the clock block of n instances: the clocks (2 x 16 values of es bytes each), the
// slots, the epochs (offsets clock_slots_at, clock_epochs_at).
inline size_t clock_slots_at(int n, int es) { return (size_t)n * 32 * es; }
inline size_t clock_epochs_at(int n, int es) { return clock_slots_at(n, es) + (size_t)n * 3 * 8; }
inline size_t clock_block_bytes(int n, int es) { return clock_epochs_at(n, es) + (size_t)n * 2 * 4; }

struct UniformOps {
  void (*rates)(const Launch&, const void* u1, const void* u2, unsigned long long* slot);
  void (*clock)(const Launch&, void* clk, unsigned long long* slot);
  void (*predict)(const Launch&, const void* u1, const void* u2, void* pa, void* pb, const void* clk);
  void (*update)(const Launch&, const void* u1, const void* u2, const void* pa, const void* pb, void* o1, void* o2,
                 const void* clk, bool debug);
  // the fused step; za, zb: the half steps of planes 0 and nz - 1 (zplanes) when a z face is not
  // periodic, else null
  void (*fused)(const Launch&, int tile, const void* u1, const void* u2, void* o1, void* o2, const ClockRefs& ck,
                const void* za, const void* zb, int zc, bool debug);
  void (*zplanes)(const Launch&, const void* u1, const void* u2, void* za, void* zb, const ClockRefs& ck);
  // the 24 diagnostics channels of the state into out (FP64), per-workgroup records in part
  void (*diag)(const Launch&, const DiagGeo&, const void* u1, const void* u2, double* part, int nblocks, double* out);
};

// Each translation unit instantiates a subset; a null table means "not built".
UniformOps uniform_ops_koren32(int rs, int isen);
UniformOps uniform_ops_mc32(int rs, int isen);
UniformOps uniform_ops_other32(int lim, int rs);
UniformOps uniform_ops_f64(int lim, int rs, int isen);

inline UniformOps uniform_ops(int precision, int lim, int rs, int isen) {
  if (precision == 64) return uniform_ops_f64(lim, rs, isen);
  if (lim == LIM_KOREN) return uniform_ops_koren32(rs, isen);
  if (lim == LIM_MC) return uniform_ops_mc32(rs, isen);
  if (isen) return UniformOps{};
  return uniform_ops_other32(lim, rs);
}

}  // namespace shx
