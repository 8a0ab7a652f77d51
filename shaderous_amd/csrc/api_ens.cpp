// C-ABI of libshx for ensembles of independent 2D grids (include/shx.h, shx_ens_*): per-instance
// parameters and offsets, the tile work list, concatenated state, per-instance clocks, graphs.
#include <hip/hip_runtime.h>
#include <math.h>
#include <string.h>

#include <algorithm>
#include <memory>
#include <vector>

#include "common.hpp"
#include "ens_impl.hpp"
#include "state_reader.hpp"

using namespace shx;

struct shx_ens {
  shx_config cfg;
  std::unique_ptr<StateReader> rb{new StateReader};
  int es = 4;
  int count = 0;
  std::vector<int> nx, ny;
  std::vector<long long> off;
  size_t ncell = 0;
  hipStream_t stream = nullptr;
  void* inst = nullptr;        // EnsInst<T>[count]
  void* tiles[ENS_NTILES] = {};   // EnsTile lists per work shape
  int ntiles[ENS_NTILES] = {};
  void* U1[2] = {nullptr, nullptr};
  void* U2[2] = {nullptr, nullptr};
  // the clock block (clock_block_bytes): per instance two clocks (parity 0 and 1, 16 T each),
  // three rate slots and two epochs (StepClock)
  void* clk = nullptr;
  unsigned long long* slot = nullptr;
  unsigned int* epoch = nullptr;
  int cur = 0;
  int tile = ENS_ROWS16;
  int rows_fit = 16;              // the rows of ENS_ROWSFIT
  int grid = 512;
  bool rates_stale = true;
  EnsOps ops{};
  // [parity][1, 2 or 8 steps]: small grids' steps are shorter than a graph launch's host cost
  hipGraphExec_t graph[2][3] = {{nullptr, nullptr, nullptr}, {nullptr, nullptr, nullptr}};
};

namespace {

size_t block_bytes(const shx_ens* e) { return clock_block_bytes(e->count, e->es); }

// The clocks of the step from parity p (its clock pass is in the step kernel).
ClockRefs clock_refs(shx_ens* e, int p) { return ClockRefs{e->clk, e->slot, e->epoch, p}; }

// Instance i's clock that its next step reads.
void* clock_of(shx_ens* e, int i) { return static_cast<char*>(e->clk) + (size_t)(2 * i + e->cur) * 16 * e->es; }

void enqueue_fused(shx_ens* e, int p, int tile) {
  e->ops.fused(e->stream, tile, e->grid, e->inst, e->count, e->tiles[tile], e->ntiles[tile], e->U1[p], e->U2[p],
               e->U1[1 - p], e->U2[1 - p], clock_refs(e, p), nullptr);
}

void enqueue_step(shx_ens* e, int p) { enqueue_fused(e, p, e->tile); }

void destroy_graphs(shx_ens* e) {
  for (int p = 0; p < 2; p++)
    for (int k = 0; k < 3; k++)
      if (e->graph[p][k]) { (void)hipGraphExecDestroy(e->graph[p][k]); e->graph[p][k] = nullptr; }
}

int build_graphs(shx_ens* e) {
  destroy_graphs(e);
  for (int p = 0; p < 2; p++)
    for (int k = 0; k < 3; k++) {
      hipGraph_t g;
      HIPCHK(hipStreamBeginCapture(e->stream, hipStreamCaptureModeThreadLocal));
      const int n = k == 0 ? 1 : (k == 1 ? 2 : 8);
      for (int i = 0; i < n; i++) enqueue_step(e, (p + i) & 1);
      HIPCHK(hipStreamEndCapture(e->stream, &g));
      HIPCHK(hipGraphInstantiate(&e->graph[p][k], g, nullptr, nullptr, 0));
      HIPCHK(hipGraphDestroy(g));
    }
  return SHX_OK;
}

// The slots hold each instance's largest rate of its current state; recomputed before the first
// step after a state change (outside the graphs).
int refresh_rates(shx_ens* e) {
  if (!e->rates_stale) return SHX_OK;
  // every instance's epochs restart at 0: its rate into its slot 0
  HIPCHK(hipMemsetAsync(e->slot, 0, block_bytes(e) - clock_slots_at(e->count, e->es), e->stream));
  int tx, ty;
  ens_tile_cells(e->tile, e->rows_fit, tx, ty);
  e->ops.rates(e->stream, e->inst, e->tiles[e->tile], e->ntiles[e->tile], tx, ty, e->U1[e->cur], e->U2[e->cur],
               e->slot, 3);
  HIPCHK(hipGetLastError());
  e->rates_stale = false;
  return SHX_OK;
}

template <typename T>
int set_state_t(shx_ens* e, int i, const T* u1, const T* u2, size_t ncell) {
  if (!e || i < 0 || i >= e->count) return fail(SHX_EINVAL, "bad instance");
  if ((int)sizeof(T) != e->es) return fail(SHX_EINVAL, "state precision mismatch");
  if (ncell != (size_t)e->nx[i] * e->ny[i]) return fail(SHX_EINVAL, "instance %d holds %d x %d cells", i, e->nx[i], e->ny[i]);
  for (size_t o = 0; o < 4 * ncell; o++)
    if (!isfinite((double)u1[o]) || !isfinite((double)u2[o])) return fail(SHX_ESTATE, "non-finite state at %zu", o / 4);
  // the instance's cells in both parities (the other instances keep theirs)
  for (int p = 0; p < 2; p++) {
    HIPCHK(hipMemcpyAsync((char*)e->U1[p] + e->off[i] * 4 * sizeof(T), u1, ncell * 4 * sizeof(T), hipMemcpyHostToDevice, e->stream));
    HIPCHK(hipMemcpyAsync((char*)e->U2[p] + e->off[i] * 4 * sizeof(T), u2, ncell * 4 * sizeof(T), hipMemcpyHostToDevice, e->stream));
  }
  T clk[16] = {0};
  clk[4] = clk[5] = clk[6] = T(1);
  HIPCHK(hipMemcpyAsync(clock_of(e, i), clk, sizeof clk, hipMemcpyHostToDevice, e->stream));
  HIPCHK(hipStreamSynchronize(e->stream));
  e->rates_stale = true;
  return SHX_OK;
}

template <typename T>
int read_state_t(shx_ens* e, int i, T* u1, T* u2) {
  if (!e || i < 0 || i >= e->count) return fail(SHX_EINVAL, "bad instance");
  if ((int)sizeof(T) != e->es) return fail(SHX_EINVAL, "state precision mismatch");
  const size_t n = (size_t)e->nx[i] * e->ny[i];
  const size_t at = e->off[i] * 4 * sizeof(T);
  HIPCHK(e->rb->read(e->stream, e->cfg.device, u1, (char*)e->U1[e->cur] + at, u2, (char*)e->U2[e->cur] + at, n * 4 * sizeof(T)));
  return SHX_OK;
}

template <typename T>
std::vector<EnsInst<T>> instances(const shx_ens* e) {
  std::vector<EnsInst<T>> v(e->count);
  for (int i = 0; i < e->count; i++) {
    shx_config c = e->cfg;
    c.n[0] = e->nx[i]; c.n[1] = e->ny[i]; c.n[2] = 1;
    c.ndim = 2;
    c.dx = 1.0 / e->nx[i];
    v[i].P = make_params<T>(c);
    v[i].off = e->off[i];
  }
  return v;
}

}  // namespace

extern "C" {

int shx_ens_create(const shx_config* cfg, int count, const int* sizes, shx_ens** out) {
  if (!cfg || !sizes || !out || count < 1) return fail(SHX_EINVAL, "null argument or empty ensemble");
  *out = nullptr;
  const shx_config& c = *cfg;
  if (c.precision != 32 && c.precision != 64) return fail(SHX_EINVAL, "precision %d", c.precision);
  for (int a = 0; a < 2; a++)
    if (c.bc_lo[a] < 0 || c.bc_lo[a] > 3 || c.bc_hi[a] < 0 || c.bc_hi[a] > 3) return fail(SHX_EINVAL, "boundary code on axis %d", a);
  // the tile kernel forms a ghost column's half step from the cell it maps to (outflow,
  // reflecting) or from its own stencil (periodic on both faces); outflow-only clamps and an axis
  // periodic on one face need the cell's own half step as the plain path loads it (load_pred),
  // which a standalone Sim then runs on its plain path
  for (int a = 0; a < 2; a++) {
    if (c.bc_lo[a] == SHX_BC_OUTFLOW_ONLY || c.bc_hi[a] == SHX_BC_OUTFLOW_ONLY)
      return fail(SHX_EINVAL, "ensemble boundaries: outflow-only on axis %d is not supported (periodic, outflow or reflecting)", a);
    if ((c.bc_lo[a] == SHX_BC_PERIODIC) != (c.bc_hi[a] == SHX_BC_PERIODIC))
      return fail(SHX_EINVAL, "ensemble boundaries: axis %d is periodic on one face only", a);
  }
  if (!(c.gamma > 1) || !(c.cfl > 0)) return fail(SHX_EINVAL, "gamma > 1 and cfl > 0 required");
  for (int i = 0; i < count; i++)
    if (sizes[2 * i] < 4 || sizes[2 * i + 1] < 4) return fail(SHX_EINVAL, "instance %d: %d x %d (at least 4 x 4)", i, sizes[2 * i], sizes[2 * i + 1]);
  EnsOps ops = c.precision == 64 ? ens_ops_f64(c.limiter, c.riemann, c.isentropic ? 1 : 0)
                                 : ens_ops_f32(c.limiter, c.riemann, c.isentropic ? 1 : 0);
  if (!ops.fused) return fail(SHX_EINVAL, "no ensemble kernels built for precision %d limiter %d riemann %d isentropic %d", c.precision, c.limiter, c.riemann, c.isentropic);
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= c.device) return fail(SHX_EDEVICE, "no HIP device %d", c.device);
  if (hipSetDevice(c.device) != hipSuccess) return fail(SHX_EDEVICE, "hipSetDevice(%d)", c.device);

  shx_ens* e = new shx_ens();
  e->cfg = c;
  e->es = c.precision == 64 ? 8 : 4;
  e->count = count;
  e->ops = ops;
  for (int i = 0; i < count; i++) {
    e->nx.push_back(sizes[2 * i]);
    e->ny.push_back(sizes[2 * i + 1]);
    e->off.push_back((long long)e->ncell);
    e->ncell += (size_t)sizes[2 * i] * sizes[2 * i + 1];
  }
  int cus = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c.device) != hipSuccess || cus < 1) cus = 256;
  e->grid = 4 * cus;
  e->rows_fit = ens_fit_rows(e->nx.data(), e->ny.data(), count, 4 * cus);
  // untuned: strips from about a million cells on, where they fill the chip, else 28 x 12 tiles
  // (24 grids up to 512^2, 2.4 M cells: 61 against 76 us per step; 12 up to 200^2, 0.16 M: 23 against 16.5)
  e->tile = e->es == 8 ? ENS_20x20 : (e->ncell >= 800000 ? ENS_ROWSFIT : ENS_32x16);
  // a tile asked for by its cells (tile[0] x tile[1]); FP64 has the one
  if (e->es == 4 && c.tile[0] == ENS_STRIP && c.tile[1] > 0) e->rows_fit = c.tile[1];
  for (int k = ENS_NTILES - 1; c.tile[0] > 0 && e->es == 4 && k >= 0; k--) {
    int tx, ty;
    ens_tile_cells(k, e->rows_fit, tx, ty);
    if (tx == c.tile[0] && ty == c.tile[1]) e->tile = k;
  }
  auto alloc = [&](void** p, size_t b) { return hipMalloc(p, b) == hipSuccess; };
  bool ok = hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking) == hipSuccess;
  const size_t bytes = e->ncell * 4 * e->es;
  for (int p = 0; ok && p < 2; p++) ok = alloc(&e->U1[p], bytes) && alloc(&e->U2[p], bytes);
  ok = ok && alloc(&e->clk, block_bytes(e));
  const size_t isz = e->es == 8 ? sizeof(EnsInst<double>) : sizeof(EnsInst<float>);
  ok = ok && alloc(&e->inst, (size_t)count * isz);
  // tile lists, largest instances first (their tiles spread over the device first)
  std::vector<int> order(count);
  for (int i = 0; i < count; i++) order[i] = i;
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return (long long)e->nx[a] * e->ny[a] > (long long)e->nx[b] * e->ny[b]; });
  std::vector<EnsTile> lists[ENS_NTILES];
  for (int k = 0; k < ENS_NTILES; k++) {
    int tx, ty;
    ens_tile_cells(k, e->rows_fit, tx, ty);
    for (int i : order)
      for (int y0 = 0; y0 < e->ny[i]; y0 += ty)
        for (int x0 = 0; x0 < e->nx[i]; x0 += tx) lists[k].push_back(EnsTile{i, x0, y0, std::min(y0 + ty, e->ny[i])});
    e->ntiles[k] = (int)lists[k].size();
    ok = ok && alloc(&e->tiles[k], lists[k].size() * sizeof(EnsTile));
  }
  if (!ok) {
    shx_ens_destroy(e);
    return fail(SHX_ENOMEM, "device allocation failed for %zu cells", e->ncell);
  }
  bool copied = true;
  if (e->es == 8) {
    auto v = instances<double>(e);
    copied = hipMemcpy(e->inst, v.data(), v.size() * sizeof(v[0]), hipMemcpyHostToDevice) == hipSuccess;
  } else {
    auto v = instances<float>(e);
    copied = hipMemcpy(e->inst, v.data(), v.size() * sizeof(v[0]), hipMemcpyHostToDevice) == hipSuccess;
  }
  for (int k = 0; k < ENS_NTILES; k++)
    copied = copied && hipMemcpy(e->tiles[k], lists[k].data(), lists[k].size() * sizeof(EnsTile), hipMemcpyHostToDevice) == hipSuccess;
  e->slot = reinterpret_cast<unsigned long long*>(static_cast<char*>(e->clk) + clock_slots_at(count, e->es));
  e->epoch = reinterpret_cast<unsigned int*>(static_cast<char*>(e->clk) + clock_epochs_at(count, e->es));
  copied = copied && hipMemset(e->clk, 0, block_bytes(e)) == hipSuccess &&
           hipMemset(e->U1[0], 0, bytes) == hipSuccess && hipMemset(e->U2[0], 0, bytes) == hipSuccess &&
           hipMemset(e->U1[1], 0, bytes) == hipSuccess && hipMemset(e->U2[1], 0, bytes) == hipSuccess &&
           hipDeviceSynchronize() == hipSuccess;
  if (!copied) {
    shx_ens_destroy(e);
    return fail(SHX_EDEVICE, "initialising the ensemble's device memory failed");
  }
  int rc = build_graphs(e);
  if (rc) { shx_ens_destroy(e); return rc; }
  size_t least = (size_t)-1, most = 0;
  for (int i = 0; i < count; i++) {
    least = std::min(least, (size_t)e->nx[i] * e->ny[i] * 8 * e->es);
    most = std::max(most, (size_t)e->nx[i] * e->ny[i] * 8 * e->es);
  }
  e->rb->fit(least, most);
  *out = e;
  return SHX_OK;
}

int shx_ens_destroy(shx_ens* e) {
  if (!e) return SHX_OK;
  if (e->stream) (void)hipStreamSynchronize(e->stream);
  destroy_graphs(e);
  for (int p = 0; p < 2; p++) { (void)hipFree(e->U1[p]); (void)hipFree(e->U2[p]); }
  for (int k = 0; k < ENS_NTILES; k++) (void)hipFree(e->tiles[k]);
  (void)hipFree(e->inst); (void)hipFree(e->clk);
  if (e->stream) (void)hipStreamDestroy(e->stream);
  delete e;
  return SHX_OK;
}

int shx_ens_set_state(shx_ens* e, int i, const float* u1, const float* u2, size_t ncell) {
  return set_state_t<float>(e, i, u1, u2, ncell);
}
int shx_ens_set_state_f64(shx_ens* e, int i, const double* u1, const double* u2, size_t ncell) {
  return set_state_t<double>(e, i, u1, u2, ncell);
}
int shx_ens_read_state(shx_ens* e, int i, float* u1, float* u2) { return read_state_t<float>(e, i, u1, u2); }
int shx_ens_read_state_f64(shx_ens* e, int i, double* u1, double* u2) { return read_state_t<double>(e, i, u1, u2); }

int shx_ens_step(shx_ens* e, int count) {
  if (!e || count < 0) return fail(SHX_EINVAL, "bad argument");
  int rc = refresh_rates(e);
  if (rc) return rc;
  for (; count >= 8; count -= 8) HIPCHK(hipGraphLaunch(e->graph[e->cur][2], e->stream));
  for (; count >= 2; count -= 2) HIPCHK(hipGraphLaunch(e->graph[e->cur][1], e->stream));
  if (count == 1) {
    HIPCHK(hipGraphLaunch(e->graph[e->cur][0], e->stream));
    e->cur = 1 - e->cur;
  }
  return SHX_OK;
}

int shx_ens_sync(shx_ens* e) {
  if (!e) return fail(SHX_EINVAL, "null ensemble");
  HIPCHK(hipStreamSynchronize(e->stream));
  return SHX_OK;
}

int shx_ens_read_clock(shx_ens* e, int i, double out[11]) {
  if (!e || !out || i < 0 || i >= e->count) return fail(SHX_EINVAL, "bad argument");
  unsigned char buf[16 * 8];
  HIPCHK(hipMemcpyAsync(buf, clock_of(e, i), 16 * e->es, hipMemcpyDeviceToHost, e->stream));
  HIPCHK(hipStreamSynchronize(e->stream));
  for (int k = 0; k < 11; k++) out[k] = e->es == 8 ? ((double*)buf)[k] : (double)((float*)buf)[k];
  return SHX_OK;
}

int shx_ens_profile(shx_ens* e, int steps, double ms[3]) {
  if (!e || !ms || steps < 1) return fail(SHX_EINVAL, "bad argument");
  int rc = refresh_rates(e);
  if (rc) return rc;
  hipEvent_t ev[3];
  for (int i = 0; i < 3; i++) HIPCHK(hipEventCreate(&ev[i]));
  double acc[3] = {0, 0, 0};
  for (int n = 0; n < steps; n++) {
    const int p = e->cur;
    // the clock pass is inside the step kernel: ms[0] stays 0
    HIPCHK(hipEventRecord(ev[0], e->stream));
    HIPCHK(hipEventRecord(ev[1], e->stream));
    enqueue_fused(e, p, e->tile);
    HIPCHK(hipEventRecord(ev[2], e->stream));
    HIPCHK(hipEventSynchronize(ev[2]));
    HIPCHK(hipGetLastError());
    e->cur = 1 - p;
    float t;
    HIPCHK(hipEventElapsedTime(&t, ev[0], ev[1])); acc[0] += t;
    HIPCHK(hipEventElapsedTime(&t, ev[1], ev[2])); acc[1] += t;
    HIPCHK(hipEventElapsedTime(&t, ev[0], ev[2])); acc[2] += t;
  }
  for (int i = 0; i < 3; i++) ms[i] = acc[i] / steps;
  for (int i = 0; i < 3; i++) (void)hipEventDestroy(ev[i]);
  return SHX_OK;
}

int shx_ens_autotune(shx_ens* e, int reps, int chosen[2]) {
  if (!e) return fail(SHX_EINVAL, "null ensemble");
  if (reps < 1) reps = 3;
  int rc = refresh_rates(e);
  if (rc) return rc;
  // each candidate takes `reps` steps from the current states (clocks and rate slots too), which
  // are restored before the next and at the end
  const size_t bytes = e->ncell * 4 * e->es;
  void *b1 = nullptr, *b2 = nullptr, *cs = nullptr;
  HIPCHK(hipMalloc(&b1, bytes));
  HIPCHK(hipMalloc(&b2, bytes));
  HIPCHK(hipMalloc(&cs, block_bytes(e)));
  const int start = e->cur;
  HIPCHK(hipMemcpyAsync(b1, e->U1[start], bytes, hipMemcpyDeviceToDevice, e->stream));
  HIPCHK(hipMemcpyAsync(b2, e->U2[start], bytes, hipMemcpyDeviceToDevice, e->stream));
  HIPCHK(hipMemcpyAsync(cs, e->clk, block_bytes(e), hipMemcpyDeviceToDevice, e->stream));
  auto restore = [&]() -> int {
    HIPCHK(hipMemcpyAsync(e->U1[start], b1, bytes, hipMemcpyDeviceToDevice, e->stream));
    HIPCHK(hipMemcpyAsync(e->U2[start], b2, bytes, hipMemcpyDeviceToDevice, e->stream));
    HIPCHK(hipMemcpyAsync(e->clk, cs, block_bytes(e), hipMemcpyDeviceToDevice, e->stream));
    return SHX_OK;
  };
  hipEvent_t e0, e1;
  HIPCHK(hipEventCreate(&e0));
  HIPCHK(hipEventCreate(&e1));
  double best = 1e30;
  int bt = e->tile;
  const int cands[] = {ENS_32x32, ENS_32x16, ENS_20x20, ENS_ROWS8, ENS_ROWS16, ENS_ROWS32, ENS_ROWSFIT};
  for (int k : cands) {
    if (e->es == 8 && k != ENS_20x20) continue;
    rc = restore();
    if (rc) return rc;
    // a warm step, then `reps` timed steps
    for (int r = 0, p = start; r <= reps; r++, p = 1 - p) {
      if (r == 1) HIPCHK(hipEventRecord(e0, e->stream));
      enqueue_fused(e, p, k);
    }
    HIPCHK(hipEventRecord(e1, e->stream));
    HIPCHK(hipEventSynchronize(e1));
    HIPCHK(hipGetLastError());
    float t;
    HIPCHK(hipEventElapsedTime(&t, e0, e1));
    if (t < best) { best = t; bt = k; }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  e->tile = bt;
  rc = restore();
  if (rc) return rc;
  HIPCHK(hipStreamSynchronize(e->stream));
  e->cur = start;
  (void)hipFree(b1); (void)hipFree(b2); (void)hipFree(cs);
  rc = build_graphs(e);
  if (rc) return rc;
  if (chosen) ens_tile_cells(bt, e->rows_fit, chosen[0], chosen[1]);
  return SHX_OK;
}

}  // extern "C"
