// Structured-grid HiPIMS step for gfx950.
//
// Layout: every field is a plane of ny rows x pitch elements (pitch is a
// multiple of 64, so each row starts 256-byte aligned in float).  Raster
// (row r, col c) of the reference's input maps to plane element r*pitch + c,
// so the raster's own nodata ring doubles as the stencil apron.
//
// Per step:
//   flux    column walk (swe_walk.hpp): a wave per unit of 60 columns x R
//           rows solves every edge of its cells; listed cells (the
//           reference's fluxMask rule) write dh/dqx/dqy.
//   single-pass step: the walk finishes its own cells (the update below)
//           into a second set of state planes.
//   update  a contiguous chunk of plane elements per block: rain, implicit
//           friction + update, h_max, the CFL minimum (wave64 shuffle + LDS),
//           FP64 volume / flux / rain sums; one partial record per block.
//   finalize one block per domain folds its partials and advances dt, t and
//           the export clamp in the domain's control block (SWE_CUDA.py:818-831);
//           calls of several single-pass steps do so inside the next step's
//           launch instead (FoldState).
// No host synchronisation anywhere in the step.
//
// Each pass is a device function over (domain, tile or chunk).  Single-domain
// launches take the domain descriptor as a kernel argument; ensemble launches
// take a device array of descriptors plus a (domain, local index) map per
// block, so one launch advances every domain of an ensemble by its own dt.
// A domain whose control block has t_stop > 0 and t >= t_stop is skipped
// (the single-pass step copies its state through to the other set).

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <utility>
#include <string>
#include <vector>

#include "../../include/hipims_abi.h"
#include "hp_common.hpp"
#include "swe_physics.hpp"
#include "swe_source.hpp"

namespace hp {

constexpr int kThreads = 256;
constexpr int kMaxStations = 1024;
constexpr int kRateCache = 64;  // station rates kept in LDS per block; further stations are evaluated per cell

__device__ inline bool stopped(const hp_ctrl* c) { return c->t_stop > 0.0 && c->t >= c->t_stop; }

// --- boundary series ------------------------------------------------------
template <class T>
__device__ inline T series_at(const T* tab, int rows, int w, int row, int col) {
  if (tab == nullptr || col < 0 || col >= w || row < 0 || row >= rows) return T(0);
  return tab[row * w + col];
}

template <class T> struct BcValues {
  int type;
  T gd, gwl, gqx, gqy;
};

// --- reductions ------------------------------------------------------------
// The fields of a control block that a step advances, and those they depend on.
struct StepCtrl {
  double t, dt, export_T, export_n, export_pending, steps, t_stop, synced;
  template <class CP> static __device__ StepCtrl of(CP c) {
    return StepCtrl{c->t, c->dt, c->export_T, c->export_n, c->export_pending, c->steps, c->t_stop, c->stopped_synced};
  }
  __device__ bool stopped() const { return t_stop > 0.0 && t >= t_stop; }
  __device__ void put(hp_ctrl* c) const {
    c->t = t;
    c->dt = dt;
    c->export_n = export_n;
    c->export_pending = export_pending;
    c->steps = steps;
    c->stopped_synced = synced;
  }
};

// Time control of one domain from its step's folded CFL minimum: dt = min of
// the candidates (kept when no cell was listed, SWE_CUDA.py:818-822), capped at
// 10x the previous dt, clamped onto the next export time, then t advanced by
// it (SWE_CUDA.py:824-831).  The FP64 sums are the caller's.
__device__ inline StepCtrl next_ctrl(const StepCtrl& c, double mn) {
  double dt = isinf(mn) ? c.dt : mn;
  const double upper = c.dt * 10.0;
  dt = (upper < dt) ? upper : dt;
  const double next_export = (c.export_n + 1.0) * c.export_T;
  const bool at_export = dt + c.t >= next_export;
  const double left = next_export - c.t;
  dt = at_export ? left : dt;
  const double one = at_export ? 1.0 : 0.0;
  return StepCtrl{c.t + dt, dt, c.export_T, c.export_n + one, c.export_pending + one, c.steps + 1.0, c.t_stop, 0.0};
}

// The same for a step the single-pass kernel ran: on a stopped domain that
// step left both sets of planes holding the state.
__device__ inline StepCtrl next_ctrl_single_pass(const StepCtrl& c, double mn) {
  const StepCtrl e = next_ctrl(c, mn);
  const bool s = c.stopped();
  return StepCtrl{s ? c.t : e.t, s ? c.dt : e.dt, c.export_T, s ? c.export_n : e.export_n,
                  s ? c.export_pending : e.export_pending, s ? c.steps : e.steps, c.t_stop, s ? 1.0 : 0.0};
}

// A step's FP64 sums into the control block.
__device__ inline void put_sums(hp_ctrl* ctrl, double vol, double fs, double rs, double dx) {
  const double area = dx * dx;
  ctrl->volume = vol * area;
  ctrl->flux_volume += fs * area;
  ctrl->rain_volume += rs * area;
}

// Per-block results of a pass that ends a step, in the workspace: the CFL
// minimum of every block in one array (all the finalize pass reads when the
// mass sums are off), then, when they are on, one FP64 record per block.
struct Sums {
  double vol, flux, rain, pad;
};

__host__ __device__ constexpr int64_t align256(int64_t x) { return (x + 255) & ~int64_t(255); }
__host__ __device__ constexpr int64_t partials_bytes(int64_t n) { return align256(n * 8) + n * (int64_t)sizeof(Sums); }

struct Partials {
  double* mins;
  Sums* sums;
  __host__ __device__ Partials(void* work, int64_t n)
      : mins((double*)work), sums((Sums*)((char*)work + align256(n * 8))) {}
  __device__ void put(int64_t i, double mn, double vol, double flux, double rain, bool with_sums) const {
    mins[i] = mn;
    if (with_sums) sums[i] = Sums{vol, flux, rain, 0.0};
  }
};

// Minimum over the wave, the same in every lane (all lanes active): lane
// shifts within rows of 16 (row_shr 1, 2, 4, 8: lane 15 holds its row's), then
// row to row, into lane 63; the order does not matter.  A lane that has no
// source keeps its value.  A fraction of the latency of six shuffles through
// LDS, and in float one instruction each (s_nop: a lane shift reads what the
// instruction before it wrote).
template <int CTRL, int ROWS> __device__ inline double shifted(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const int l = (int)(uint32_t)u, h = (int)(uint32_t)(u >> 32);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(l, l, CTRL, ROWS, 0xf, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(h, h, CTRL, ROWS, 0xf, false);
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}
__device__ inline double wave_min(double v) {
  v = fmin(v, shifted<0x111, 0xf>(v));
  v = fmin(v, shifted<0x112, 0xf>(v));
  v = fmin(v, shifted<0x114, 0xf>(v));
  v = fmin(v, shifted<0x118, 0xf>(v));
  v = fmin(v, shifted<0x142, 0xa>(v));  // row_bcast 15 into rows 1 and 3
  v = fmin(v, shifted<0x143, 0xc>(v));  // row_bcast 31 into rows 2 and 3
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, 63);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), 63);
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}
__device__ inline float wave_min(float v) {
  asm("s_nop 1\n\tv_min_f32_dpp %0, %0, %0 row_shr:1 row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\tv_min_f32_dpp %0, %0, %0 row_shr:2 row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\tv_min_f32_dpp %0, %0, %0 row_shr:4 row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\tv_min_f32_dpp %0, %0, %0 row_shr:8 row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\tv_min_f32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
      "s_nop 1\n\tv_min_f32_dpp %0, %0, %0 row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"
      "s_nop 1"
      : "+v"(v));
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}
__device__ inline double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// --- time control inside the step kernel --------------------------------
// A call of several single-pass steps runs no time-control launch between
// them (a launch costs 4 to 5 us whatever it does, and the gap before it 1 to
// 2; a 2048^2 float step takes 60).  Each unit of step k posts its CFL minimum
// into one of kFoldSlots words by an atomic minimum (a non-negative double
// orders like its bits, so the minimum does not depend on the order), and
// every unit of step k + 1 folds the slots and advances the time control for
// itself, from the control block of step k: one load per lane and one wave
// reduction, in the shadow of the unit's first rows.  64 slots: at most one
// load per lane, and 2048^2 in units of 15 rows posts 75 times to each at about
// 36 ns.
// Step k posts to slots[k % 3], reads slots[(k - 1) % 3] and clears
// slots[(k + 1) % 3]; its control block goes from ring[(k - 1) & 1] to
// ring[k & 1], written by the unit 0.  Records of the FP64 sums take turns the
// same way: kFoldSumBlocks further blocks of step k + 1 sum step k's as the
// waves of the time-control kernel do, and the first of them in step k + 2
// adds these up into the control block (one block for all the records took
// longer than the step itself at 6 650 units: 30 us).
constexpr int kFoldSlots = 64;
constexpr int kFoldSumBlocks = 16;
struct FoldState {
  unsigned long long slots[3][kFoldSlots];
  hp_ctrl ring[2];
  double wave_sums[2][3][kFoldSumBlocks];  // of step k (k & 1): volume, flux, rain
  double summed[2];                        // whether step k was one to sum (not stopped)
};
constexpr unsigned long long kNoMinimum = 0x7ff0000000000000ull;  // the bits of +infinity

// What a unit of a folded step works on: st null, a step with a time-control
// launch of its own.
struct WalkFold {
  FoldState* st;
  int k;         // step of the call
  Sums* records;  // this step's records of the domain's units
};

// The sum of n records as wave w of a 1024-thread block takes it (thread i adds
// records i, i + 1024, ... in turn; a wave64 butterfly), by one wave.
__device__ inline void wave_records(const Sums* __restrict__ part, int n, int w, double& vol, double& fs, double& rs) {
  const int lane = threadIdx.x & 63;
  vol = fs = rs = 0.0;
  for (int k = w * 64 + lane; k < n; k += 1024) {
    const Sums p = part[k];
    vol += p.vol;
    fs += p.flux;
    rs += p.rain;
  }
  vol = wave_sum(vol);
  fs = wave_sum(fs);
  rs = wave_sum(rs);
}

// The sixteen waves' sums in turn (one thread).
__device__ inline void add_waves(const double (&s)[3][kFoldSumBlocks], double& vol, double& fs, double& rs) {
  vol = s[0][0];
  fs = s[1][0];
  rs = s[2][0];
  for (int k = 1; k < kFoldSumBlocks; ++k) {
    vol += s[0][k];
    fs += s[1][k];
    rs += s[2][k];
  }
}

// Block w of the sum blocks in the launch of step k: wave w of step k - 1's
// sum; block 0 also brings step k - 2's into the control block (nothing else
// of the launch touches those fields).
__device__ inline void fold_sums_block(hp_ctrl* ctrl, FoldState* f, int k, int w, const Sums* prev, int n, double dx) {
  double vol, fs, rs;
  if (w == 0 && k >= 2 && threadIdx.x == 0 && f->summed[k & 1] != 0.0) {
    add_waves(f->wave_sums[k & 1], vol, fs, rs);
    put_sums(ctrl, vol, fs, rs, dx);
  }
  if (k == 0) return;
  const bool live = !stopped(&f->ring[(k + 1) & 1]);
  if (live) wave_records(prev, n, w, vol, fs, rs);
  if (threadIdx.x == 0) {
    double(&to)[3][kFoldSumBlocks] = f->wave_sums[(k + 1) & 1];
    if (live) {
      to[0][w] = vol;
      to[1][w] = fs;
      to[2][w] = rs;
    }
    if (w == 0) f->summed[(k + 1) & 1] = live ? 1.0 : 0.0;
  }
}

// Fold a block's CFL minimum and FP64 sums into its partial slot.
template <class T>
__device__ inline void block_partial(T mn, double vol, double fsum, double rsum, const Partials& part, int64_t idx,
                                     bool sums) {
  __shared__ double s_red[4][kThreads / 64];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  mn = wave_min(mn);
  if (sums) {
    vol = wave_sum(vol);
    fsum = wave_sum(fsum);
    rsum = wave_sum(rsum);
  }
  if (lane == 0) {
    s_red[0][w] = (double)mn;
    s_red[1][w] = vol;
    s_red[2][w] = fsum;
    s_red[3][w] = rsum;
  }
  __syncthreads();
  if (tid == 0) {
    double m = s_red[0][0], v = s_red[1][0], f = s_red[2][0], r = s_red[3][0];
    for (int k = 1; k < kThreads / 64; ++k) {
      m = fmin(m, s_red[0][k]);
      v += s_red[1][k];
      f += s_red[2][k];
      r += s_red[3][k];
    }
    part.put(idx, m, v, f, r, sums);
  }
}

// Per-cell inputs of the update that do not depend on the fluxes; loaded
// before the flux work so their latency hides behind it.
template <class T> struct CellIn {
  T rain;   // rain rate (m/s)
  T hmax;   // h_max before the step
  T n;      // Manning n of the cell's class
  int cls;  // landuse class
  bool on;  // landuse class != 255 (the reference's update covers the cell)
};

// Rain + implicit friction + update of one cell (HP_UPDATE_STEP semantics,
// SWE_CUDA.py:780-831).  Returns the new state in (h, qx, qy) and the new
// h_max, plus the cell's contributions to the block's reductions: its CFL
// candidate (INFINITY if none), its depth for the volume sum (0 if the cell
// is not covered), and its flux and rain depth increments (0 if not
// updated).  Every output is assigned on every path, so the caller folds
// them in unconditionally and the accumulators stay in registers.
template <class T>
__device__ inline void update_state(const CellIn<T>& in, T& h, T& qx, T& qy, T dhf, T dqx, T dqy, T dF, T dt,
                                    T cfl_dx, T& hmax, T& cand, T& vol_h, T& flux_h, T& rain_h,
                                    bool time_control = true) {
  // one branch (the wet cells' friction) and selects around it: nested
  // branches cost a register copy per output on every side
  const T rdt = in.rain * dt;
  const T dht = (dhf + rdt) - dF;  // flux, + rain, - infiltration (the reference's order)
  const bool upd = both(in.on, either(fabs(dht) > T(0), h >= T(0)));
  T hn = h;
  const bool wet = both(!new_depth_dry(hn, dht), upd);
  T nqx = T(0), nqy = T(0), c = T(60.0);
  if (wet) {
    nqx = qx + dqx;
    nqy = qy + dqy;
    implicit_friction<T>(hn, in.n, dt, nqx, nqy);
    if (time_control) c = cfl_candidate<T>(hn, nqx, nqy, cfl_dx);
  }
  h = upd ? hn : h;
  qx = upd ? nqx : qx;
  qy = upd ? nqy : qy;
  const T hm = Prec<T>::max2(hn, hmax);
  hmax = upd ? hm : hmax;
  cand = upd ? c : T(INFINITY);
  vol_h = in.on ? h : T(0);
  flux_h = upd ? dhf : T(0);
  rain_h = upd ? rdt : T(0);
}

}  // namespace hp

#include "swe_walk.hpp"

namespace hp {

// Infiltration pass over plane elements: a valid cell listed by the flux
// rule of the current state (t == 0, wet, or a wet valid neighbour E, N, W,
// S that is not compact cell 0: the wet list the reference's
// addInfiltrationSource receives from addFlux) takes the Green-Ampt
// increment; dF is written for every element (0 elsewhere) so the update
// pass can subtract it after the rain.
template <class T>
__global__ __launch_bounds__(kThreads) void k_infiltration(hp_grid_desc a) {
  if (stopped(a.ctrl)) return;
  const int64_t pitch = a.pitch, total = pitch * (int64_t)a.ny;
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= total) return;
  const T* __restrict__ h = (const T*)a.h;
  const uint8_t* __restrict__ ty = a.type_slot;
  const int row = (int)(i / pitch), col = (int)(i - row * pitch);
  T dF = T(0);
  if (col < a.nx && ty[i] != 0) {
    // (every neighbour is asked for before any is used: in turn, each would
    // wait for the one before)
    const int nr[4] = {row, row - 1, row, row + 1};
    const int nc[4] = {col + 1, col, col - 1, col};
    bool in[4];
    T hn[4];
    int tn[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      in[k] = both(both(nr[k] >= 0, nr[k] < a.ny), both(nc[k] >= 0, nc[k] < a.nx));
      const int64_t j = in[k] ? (int64_t)nr[k] * pitch + nc[k] : i;
      hn[k] = h[j];
      tn[k] = ty[j];
    }
    bool listed = either(T(a.ctrl->t) == T(0), gt_hs(h[i]));
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const bool other = either(nc[k] != a.cell0_x, nr[k] != a.cell0_y);
      listed = either(listed, both(both(in[k], tn[k] != 0), both(other, gt_hs(hn[k]))));
    }
    if (listed) {
      const int cls = a.landuse[i];
      T* F = (T*)a.infil_F;
      dF = green_ampt<T>(h[i], F[i], ((const T*)a.infil_ks)[cls], ((const T*)a.infil_phi)[cls],
                         ((const T*)a.infil_dtheta)[cls], T(a.ctrl->dt));
      F[i] += dF;
    }
  }
  ((T*)a.infil_dF)[i] = dF;
}

// MODE selects which of the reference driver's update methods the pass is:
//   HP_UPDATE_STEP      time_friction_euler_update_cuda (SWE_CUDA.py:780-831):
//                       cells with |dh| > 0 or h >= 0; friction; CFL + dt/t
//   HP_UPDATE_FRICTION  friction_euler_update_cuda (:766-778): same list, no CFL
//   HP_UPDATE_EULER     euler_update (:712-724): cells with |dh| > 0 or
//                       h > 1e-6; q += dq without friction; no CFL
//   HP_UPDATE_CFL       time_update_cuda (:726-764): cells with h > 1e-6; no
//                       state change and no rain; h_max, CFL + dt/t
// Processes a chunk of kThreads * update_loops() plane elements and writes one
// partial record.  On a small domain a launch lasts as long as one thread's
// chain of loads, divisions and square roots, so a thread has one element
// (with eight, in vectors of four, a 75x75 domain in double took 13.2 us and
// takes 5.6).  Past 1024 blocks the elements per thread grow to eight, so that
// one block can fold the records; from four on they come in accesses of 16
// bytes.  Kernel time with one, two and four elements per access, us: double
// 800^2 17.3, 16.6, -, 2048^2 71, 66, 72, 3000^2 147, 145, 147; float 800^2
// 11.6, -, 11.4, 2048^2 35, 33, 33, 3000^2 72, 67, 64.  (One kernel for vectors
// and single elements cost a 1024^2 float domain a sixth.)
__host__ __device__ inline int update_loops(int64_t total) {
  int n = 1;
  while (n < 8 && total > (int64_t)n * kThreads * 1024) n *= 2;
  return n;
}

// W consecutive elements of the planes.
template <class T, int W> struct UpdateIn {
  T h[W], qx[W], qy[W], hm[W], dh[W], dqx[W], dqy[W], df[W];
  float rain[W];
  uint8_t cls[W];
  int16_t st[W];
};
template <int W, class V> __device__ inline void load_w(V (&to)[W], const V* p) {
  struct alignas(W * sizeof(V)) Vec {
    V x[W];
  };
  const Vec v = *reinterpret_cast<const Vec*>(p);
#pragma unroll
  for (int j = 0; j < W; ++j) to[j] = v.x[j];
}
template <int W, class V> __device__ inline void store_w(V* p, const V (&from)[W]) {
  struct alignas(W * sizeof(V)) Vec {
    V x[W];
  } v;
#pragma unroll
  for (int j = 0; j < W; ++j) v.x[j] = from[j];
  *reinterpret_cast<Vec*>(p) = v;
}

template <class T, int MODE, int W>
__device__ inline void update_elements(const hp_grid_desc& a, int64_t base, int rounds, int64_t total,
                                       const Partials& part, int64_t pidx, T* s_man, T* s_rate) {
  const int tid = threadIdx.x, mode = a.rain_mode;
  // (past the end: the last elements again, which the loop below leaves out.  A
  // class of no cell put in here instead would have every load wait for the
  // classes: 3000^2 in float 64 -> 65 us.)
  auto load = [&](int it) {
    const int64_t at = base + ((int64_t)it * kThreads + tid) * W, i = at < total ? at : total - W;
    UpdateIn<T, W> c{};
    load_w(c.cls, a.landuse + i);
    load_w(c.h, (const T*)a.h + i);
    load_w(c.qx, (const T*)a.qx + i);
    load_w(c.qy, (const T*)a.qy + i);
    load_w(c.hm, (const T*)a.h_max + i);
    if (MODE != HP_UPDATE_CFL) {
      if (a.infil_dF) load_w(c.df, (const T*)a.infil_dF + i);
      load_w(c.dh, (const T*)a.dh + i);
      load_w(c.dqx, (const T*)a.dqx + i);
      load_w(c.dqy, (const T*)a.dqy + i);
      if (mode == HP_RAIN_STATION && a.station) load_w(c.st, a.station + i);
      else if (mode == HP_RAIN_FIELD) load_w(c.rain, a.rain_field + i);
    }
    return c;
  };
  // Single elements are asked for before the tables, whose round trips they
  // overlap; vectors after them, where a launch is bound by memory and the
  // tables, behind them in order, would wait for megabytes (float 1024^2 13.4
  // us the other way round, 13.0 so; double 2048^2 65.3, 63.6).
  UpdateIn<T, W> c{};
  if (W == 1) c = load(0);
  const double times = wave_rain_times(&a);
  const T man = tid < a.n_classes ? ((const T*)a.manning)[tid] : T(0);
  if (stopped(a.ctrl)) {
    if (tid == 0) part.put(pidx, INFINITY, 0.0, 0.0, 0.0, a.mass_sums != 0);
    return;
  }
  const T dt = T(a.ctrl->dt);
  const T cfl_dx = T(a.cfl) * T(a.dx), rscale = T(a.rain_scale);
  if (tid < a.n_classes) s_man[tid] = man;
  const RainRows rr = wave_rain_rows(&a, a.ctrl->t, times);
  if (mode == HP_RAIN_STATION && tid < kRateCache) s_rate[tid] = station_rate<T>(rr, tid, a.rain_scale);
  __syncthreads();
  if (W != 1) c = load(0);
  const bool sums = a.mass_sums != 0;
  T mn = T(INFINITY);
  double vol = 0.0, fsum = 0.0, rsum = 0.0;
  for (int it = 0;; ++it) {
    const bool more = it + 1 < rounds;
    UpdateIn<T, W> next{};
    if (W == 1 && more) next = load(it + 1);  // (vectors ahead would halve the waves in flight)
    const int64_t i = base + ((int64_t)it * kThreads + tid) * W;
    T rate[W] = {};
    if (MODE != HP_UPDATE_CFL) {
      if (mode == HP_RAIN_STATION) {
#pragma unroll
        for (int j = 0; j < W; ++j) {
          const int k = c.st[j];
          rate[j] = (k >= 0 && k < kRateCache) ? s_rate[k] : station_rate<T>(rr, k, a.rain_scale);
        }
      } else if (mode == HP_RAIN_FIELD) {
#pragma unroll
        for (int j = 0; j < W; ++j) rate[j] = T(c.rain[j]) * rscale;
      }
    }
#pragma unroll
    for (int j = 0; j < W; ++j) {
      if (either(c.cls[j] == 255, i >= total)) continue;
      T h = c.h[j];
      if (MODE == HP_UPDATE_CFL) {
        if (gt_hs(h)) {
          c.hm[j] = fmax(h, c.hm[j]);
          mn = fmin(mn, cfl_candidate<T>(h, c.qx[j], c.qy[j], cfl_dx));
        }
      } else {
        const T rdt = rate[j] * dt;
        const T dht = (c.dh[j] + rdt) - c.df[j];  // flux, + rain, - infiltration (the reference's order)
        const bool listed =
            (MODE == HP_UPDATE_EULER) ? (fabs(dht) > T(0) || gt_hs(h)) : (fabs(dht) > T(0) || h >= T(0));
        if (listed) {
          const bool dry = new_depth_dry(h, dht);
          T qx = T(0), qy = T(0);
          if (MODE == HP_UPDATE_EULER || !dry) {
            qx = c.qx[j] + c.dqx[j];
            qy = c.qy[j] + c.dqy[j];
            if (MODE != HP_UPDATE_EULER) implicit_friction<T>(h, s_man[c.cls[j]], dt, qx, qy);
          }
          c.h[j] = h;
          c.qx[j] = qx;
          c.qy[j] = qy;
          if (MODE == HP_UPDATE_STEP) {
            c.hm[j] = fmax(h, c.hm[j]);
            mn = fmin(mn, cfl_candidate<T>(h, qx, qy, cfl_dx));
          }
          if (sums) {
            fsum += (double)c.dh[j];
            rsum += (double)rdt;
          }
        }
      }
      if (sums) vol += (double)h;
    }
    if (i < total) {
      if (MODE != HP_UPDATE_CFL) {
        store_w((T*)a.h + i, c.h);
        store_w((T*)a.qx + i, c.qx);
        store_w((T*)a.qy + i, c.qy);
      }
      if (MODE == HP_UPDATE_STEP || MODE == HP_UPDATE_CFL) store_w((T*)a.h_max + i, c.hm);
    }
    if (!more) break;
    c = W == 1 ? next : load(it + 1);
  }
  block_partial<T>(mn, vol, fsum, rsum, part, pidx, sums);
}

// Elements per access of a domain's update: one, or those of 16 bytes.
template <class T> constexpr int kWide = 16 / sizeof(T);
template <class T> __host__ __device__ inline int update_width(int64_t total) {
  return update_loops(total) >= 4 ? kWide<T> : 1;
}

template <class T, int MODE, int W>
__device__ inline void update_chunk(const hp_grid_desc& a, int64_t chunk, const Partials& part, int64_t pidx, T* s_man,
                                    T* s_rate) {
  const int64_t total = a.pitch * (int64_t)a.ny;  // a multiple of kVec
  const int loops = update_loops(total);
  update_elements<T, MODE, W>(a, chunk * kThreads * loops, loops / W, total, part, pidx, s_man, s_rate);
}

template <class T, int MODE, int W>
__global__ __launch_bounds__(kThreads) void k_update(hp_grid_desc a) {
  __shared__ T s_man[256];
  __shared__ T s_rate[kRateCache];
  update_chunk<T, MODE, W>(a, blockIdx.x, Partials(a.work, gridDim.x), blockIdx.x, s_man, s_rate);
}

// (the domains of an ensemble differ in size: each as it runs alone, so that
// its sums keep their bits)
template <class T, int MODE>
__global__ __launch_bounds__(kThreads) void k_update_multi(const hp_grid_desc* __restrict__ doms,
                                                           const int2* __restrict__ map, void* parts) {
  __shared__ T s_man[256];
  __shared__ T s_rate[kRateCache];
  const int2 m = map[blockIdx.x];
  const hp_grid_desc& a = doms[m.x];
  const Partials part(parts, gridDim.x);
  if (update_width<T>(a.pitch * (int64_t)a.ny) != 1)
    update_chunk<T, MODE, kWide<T>>(a, m.y, part, blockIdx.x, s_man, s_rate);
  else update_chunk<T, MODE, 1>(a, m.y, part, blockIdx.x, s_man, s_rate);
}

// Fold a domain's partials in a fixed order and advance its time control.
// The minima are read 24 per thread before any is used, so one block covers
// 24 576 partials (2048^2 has 4 795 units at its chosen 15 rows, 17 920 at an
// asked height of four) in one memory round trip; the control block is read alongside them rather than ahead of them.
// single_pass: the step just run was the single-pass one.  On a stopped
// domain the time control records whether that step left the second set of
// planes holding the state (the single-pass kernel copies it there on the
// first step past the stop, and no more once this is set).
__device__ inline void finalize_domain(hp_ctrl* ctrl, const double* __restrict__ mins, const Sums* __restrict__ part,
                                       int n, double dx, bool sums, bool single_pass) {
  constexpr int kU = 24;
  __shared__ double s_red[4][16];
  const int tid = threadIdx.x;
  const StepCtrl c = StepCtrl::of(ctrl);
  double mn = INFINITY, vol = 0.0, fs = 0.0, rs = 0.0;
  for (int base = tid; base < n; base += blockDim.x * kU) {
    double v[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int k = base + u * (int)blockDim.x;
      v[u] = k < n ? mins[k] : INFINITY;
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) mn = fmin(mn, v[u]);
  }
  if (c.stopped()) {
    if (threadIdx.x == 0) ctrl->stopped_synced = single_pass ? 1.0 : 0.0;
    return;
  }
  if (sums) {
    for (int k = tid; k < n; k += blockDim.x) {
      const Sums p = part[k];
      vol += p.vol;
      fs += p.flux;
      rs += p.rain;
    }
  }
  mn = wave_min(mn);
  if (sums) {
    vol = wave_sum(vol);
    fs = wave_sum(fs);
    rs = wave_sum(rs);
  }
  const int lane = tid & 63, w = tid >> 6;
  const int nw = (blockDim.x + 63) >> 6;
  if (lane == 0) {
    s_red[0][w] = mn;
    s_red[1][w] = vol;
    s_red[2][w] = fs;
    s_red[3][w] = rs;
  }
  __syncthreads();
  if (tid == 0) {
    mn = s_red[0][0];
    vol = s_red[1][0];
    fs = s_red[2][0];
    rs = s_red[3][0];
    for (int k = 1; k < nw; ++k) {
      mn = fmin(mn, s_red[0][k]);
      vol += s_red[1][k];
      fs += s_red[2][k];
      rs += s_red[3][k];
    }
    next_ctrl(c, mn).put(ctrl);
    if (sums) put_sums(ctrl, vol, fs, rs, dx);
  }
}

__global__ __launch_bounds__(1024) void k_finalize(hp_ctrl* ctrl, void* work, int n, double dx, int sums,
                                                   int single_pass) {
  const Partials P(work, n);
  finalize_domain(ctrl, P.mins, P.sums, n, dx, sums != 0, single_pass != 0);
}

// Before and after the steps of a folded call: the control block into the
// ring, and from it back to the caller's after the last step's fold.
__global__ __launch_bounds__(64) void k_fold_begin(const hp_ctrl* __restrict__ ctrl, FoldState* f) {
  const int lane = threadIdx.x;
  for (int b = 0; b < 3; ++b) f->slots[b][lane] = kNoMinimum;
  if (lane == 0) f->ring[1] = *ctrl;
}
// (k: the number of steps, at least 2; a 1024-thread block with sums)
__device__ inline void fold_end(hp_ctrl* ctrl, const FoldState* f, int k, const Sums* prev, int n, double dx, bool sums) {
  const StepCtrl c = StepCtrl::of(&f->ring[(k + 1) & 1]);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const double mn = wave_min(__builtin_bit_cast(double, (uint64_t)f->slots[(k + 2) % 3][lane]));
  __shared__ double s_sum[3][kFoldSumBlocks];
  const bool add = sums && !c.stopped();
  double vol, fs, rs;
  if (add) {
    wave_records(prev, n, w, vol, fs, rs);
    if (lane == 0) {
      s_sum[0][w] = vol;
      s_sum[1][w] = fs;
      s_sum[2][w] = rs;
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    if (sums && f->summed[k & 1] != 0.0) {
      add_waves(f->wave_sums[k & 1], vol, fs, rs);
      put_sums(ctrl, vol, fs, rs, dx);
    }
    next_ctrl_single_pass(c, mn).put(ctrl);
    if (add) {
      add_waves(s_sum, vol, fs, rs);
      put_sums(ctrl, vol, fs, rs, dx);
    }
  }
}
__global__ __launch_bounds__(1024) void k_fold_end(hp_ctrl* ctrl, const FoldState* f, int k, const Sums* prev, int n,
                                                   double dx, int sums) {
  fold_end(ctrl, f, k, prev, n, dx, sums != 0);
}

// The same for every domain of an ensemble, a block each.
__global__ __launch_bounds__(64) void k_fold_begin_multi(const hp_grid_desc* __restrict__ doms, FoldState* f) {
  const int lane = threadIdx.x;
  FoldState* s = f + blockIdx.x;
  for (int b = 0; b < 3; ++b) s->slots[b][lane] = kNoMinimum;
  if (lane == 0) s->ring[1] = *doms[blockIdx.x].ctrl;
}
__global__ __launch_bounds__(1024) void k_fold_end_multi(const hp_grid_desc* __restrict__ doms,
                                                         const int2* __restrict__ ranges, const FoldState* f, int k,
                                                         const Sums* prev) {
  const int2 r = ranges[blockIdx.x];
  const hp_grid_desc& a = doms[blockIdx.x];
  fold_end(a.ctrl, f + blockIdx.x, k, prev + r.x, r.y, a.dx, a.mass_sums != 0);
}

// k_finalize followed by a calibration step's record (thread 0 wrote the
// control block, so it also reads the next step's t and dt).  The gauge
// depths (one per thread; more are read after the fold) are loaded before
// the fold so that their latency hides behind it.
__global__ __launch_bounds__(1024) void k_finalize_record(hp_ctrl* ctrl, void* work, int n, double dx, int sums,
                                                          StepRecord rec) {
  const Partials P(work, n);
  const int i0 = threadIdx.x;
  double v0 = 0.0;
  if (i0 < rec.n) v0 = rec.f32 ? (double)((const float*)rec.h)[rec.off[i0]] : ((const double*)rec.h)[rec.off[i0]];
  finalize_domain(ctrl, P.mins, P.sums, n, dx, sums != 0, true);
  if (i0 < rec.n) {
    if (rec.f32) ((float*)rec.row)[i0] = (float)v0;
    else ((double*)rec.row)[i0] = v0;
  }
  for (int i = i0 + blockDim.x; i < rec.n; i += blockDim.x) {
    if (rec.f32) ((float*)rec.row)[i] = ((const float*)rec.h)[rec.off[i]];
    else ((double*)rec.row)[i] = ((const double*)rec.h)[rec.off[i]];
  }
  if (rec.sched && threadIdx.x == 0) {
    rec.sched[2 * (int64_t)rec.k_next] = ctrl->t;
    rec.sched[2 * (int64_t)rec.k_next + 1] = ctrl->dt;
  }
}

// One block per domain, with k_finalize's block size, so that a domain's
// partials are folded in the same order as in a standalone run.
__global__ __launch_bounds__(1024) void k_finalize_multi(const hp_grid_desc* __restrict__ doms,
                                                        const int2* __restrict__ ranges, void* parts,
                                                        int n_total, int single_pass) {
  const int2 r = ranges[blockIdx.x];
  const hp_grid_desc& a = doms[blockIdx.x];
  const Partials P(parts, n_total);
  finalize_domain(a.ctrl, P.mins + r.x, P.sums + r.x, r.y, a.dx, a.mass_sums != 0, single_pass != 0);
}

// --- host side -------------------------------------------------------------
static int64_t update_blocks(const hp_grid_desc* g) {
  const int64_t total = g->pitch * (int64_t)g->ny;
  const int64_t chunk = (int64_t)kThreads * update_loops(total);
  return (total + chunk - 1) / chunk;
}

static int64_t units(const hp_grid_desc* g, int cols, int rows) {
  return (int64_t)((g->nx + cols - 1) / cols) * (int64_t)((g->ny + rows - 1) / rows);
}

// Expected time in us of a launch of u units of r rows.  n units on a SIMD
// take row[n - 1] for a row of each (one or two of them run at the latency of
// a row, five in float and three in double fill the SIMD), after start[n - 1]
// for their prologues.  More units than fit at once go in rounds; up to four
// of them, a last round that is nearly empty takes as long as a full one, and
// tall units spread uneven rows (dry ones, nodata) worse, by 0.25 % a row.
// Where every row is wet a launch is one round up to its last slot (4 to 16
// rows: no step in its time before 1.00 of the slots, 11 to 21 % at 1.02).  On
// rain-fed terrain, whose units take unequal times, float ran 4 850 units in
// one round and 5 000 no more, so a first round counts as full 5 % before its
// last slot; double did to 98 % (928^2 8 rows in two rounds 45, 5 in one of
// 97 % 40), but tall units in double count with 5 too, on the evidence of one
// size (2048^2 below: they lose more to uneven rows of a flood than they gain
// under rain).  Later boundaries are no such step (float, 8 rows: 72, 75, 76 us
// at 1.95, 2.00, 2.02 rounds); there 2 % stands in both precisions.  Over many
// rounds only the prologues and a short tail count.  Measured, order 2, height:
// us (units per SIMD): float 256^2 1: 10.1 (1.3), 2: 10.6 (0.6); 500^2 1: 20.1
// (4.4), 2: 16.4 (2.2), 3: 15.4 (1.5), 5: 17.2 (0.9); 1024^2 3: 33.6 (6.0),
// 4: 28.4 (4.5), 5: 27.0 (3.6), 8: 28.4 (2.3); 2048^2 8: 63.2 (8.8), 13: 67.4
// (5.4), 15: 59.0 (4.7), 18: 61.6 (3.9), 24: 68.8 (2.9); 3000^2 15: 119 (9.8),
// 30: 141 (4.9), 31: 122 (4.7), with a flood in a dry plain, order 1, 15: 102,
// 28: 123, 32: 119; 8192^2 8: 814, 16: 752, 24: 744, 32: 737; double 256^2
// 1: 12.7 (1.3), 2: 13.8 (0.6); 700^2 2: 33.0 (4.1), 3: 27.3 (2.7), 5: 29.1
// (1.6), 8: 41.3 (1.0); 2048^2 8: 145 (8.8), 12: 143 (5.8), 14: 158 (5.0),
// 24: 141 (2.9), with a flood in a dry plain 12: 126, 24: 136.
template <class T> static double walk_cost(int64_t u, int r) {
  static const double kRowF[] = {2.05, 2.4, 2.45, 2.85, 3.0}, kStartF[] = {6.3, 8.0, 10.5, 12.0, 16.0};
  static const double kRowD[] = {3.35, 4.1, 5.25}, kStartD[] = {6.7, 8.6, 11.5};
  const double *row = sizeof(T) == 4 ? kRowF : kRowD, *start = sizeof(T) == 4 ? kStartF : kStartD;
  const double x = (double)u / walk_slots<T>();
  const bool many = x > 4.0;
  const double full = x <= 1.0 && (sizeof(T) == 4 || r > 12) ? 0.05 : 0.02;
  const double rounds = many ? x + 0.25 : (double)(1 + (int)(x + full));
  const int i = (int)(rounds > 1.0 ? walk_waves<T>() : (u + kSimds - 1) / kSimds) - 1;
  return start[i] + rounds * row[i] * r * (many ? 1.0 : 1.0 + 0.0025 * r) + 5.0 * (rounds - 1.0);
}

// Rows per flux work unit (60 columns wide): a height asked for by tile_rows
// (2, 4, 6, 8, 10, 12 or 16 in float, 4 or 8 in double), else 0.
static int asked_rows(const hp_grid_desc* g) {
  const int r = g->tile_rows;
  if (g->dtype == HP_F32) return (r == 2 || r == 4 || r == 6 || r == 8 || r == 10 || r == 12 || r == 16) ? r : 0;
  return r == 4 || r == 8 ? r : 0;
}

// What a domain's height counts as where heights are compared and sizes are
// checked (a domain that asks for none: 8 in float, 4 in double).
static int nominal_rows(const hp_grid_desc* g) {
  const int r = asked_rows(g);
  return r ? r : (g->dtype == HP_F32 ? 8 : 4);
}

// The height where none is asked for: the one that a launch of all the n
// domains together is expected to finish first with (see walk_cost).
template <class T> static int chosen_rows(int n, const hp_grid_desc* d) {
  int best = 1;
  double least = 0.0;
  for (int r = 1; r <= 32; ++r) {
    int64_t u = 0;
    for (int k = 0; k < n; ++k) u += (int64_t)((d[k].nx + kWalkOwn - 1) / kWalkOwn) * ((d[k].ny + r - 1) / r);
    const double c = walk_cost<T>(u, r);
    if (r == 1 || c < least) {
      best = r;
      least = c;
    }
  }
  return best;
}
static int chosen_height(int n, const hp_grid_desc* d) {
  return d->dtype == HP_F32 ? chosen_rows<float>(n, d) : chosen_rows<double>(n, d);
}

static int flux_rows(const hp_grid_desc* g) {
  const int r = asked_rows(g);
  return r ? r : chosen_height(1, g);
}

// Flux work units of a domain: one partial record each in the single-pass step.
static int64_t flux_tiles(const hp_grid_desc* g) { return units(g, kWalkOwn, flux_rows(g)); }

// Units a domain of its nominal height has had in every version (64-column
// tiles in double): the records a workspace is sized for hold at least these.
static int64_t nominal_tiles(const hp_grid_desc* g) {
  return units(g, g->dtype == HP_F32 ? kWalkOwn : 64, nominal_rows(g));
}

static int check_desc(const hp_grid_desc* g) {
  if (!g) return fail(HP_EINVAL, "null descriptor");
  if (g->dtype != HP_F32 && g->dtype != HP_F64) return fail(HP_EINVAL, "dtype must be HP_F32 or HP_F64");
  if (g->order != 1 && g->order != 2) return fail(HP_EINVAL, "order must be 1 or 2");
  if (g->nx <= 0 || g->ny <= 0) return fail(HP_EINVAL, "nx and ny must be positive");
  if (g->pitch < g->nx) return fail(HP_EINVAL, "pitch must be >= nx");
  if (g->pitch % kVec != 0) return fail(HP_EINVAL, "pitch must be a multiple of 4");
  if (!(g->dx > 0.0)) return fail(HP_EINVAL, "dx must be positive");
  if (!g->h || !g->qx || !g->qy || !g->z || !g->h_max || !g->dh || !g->dqx || !g->dqy)
    return fail(HP_EINVAL, "a state plane pointer is null");
  if (!g->type_slot || !g->landuse || !g->slot_code || !g->manning || !g->ctrl)
    return fail(HP_EINVAL, "type_slot, landuse, slot_code, manning and ctrl are required");
  if (g->n_classes <= 0 || g->n_classes > 255) return fail(HP_EINVAL, "n_classes must be in 1..255");
  {
    // the update pass moves kVec consecutive elements per access
    const uintptr_t va = (uintptr_t)kVec * (g->dtype == HP_F32 ? 4 : 8);
    const void* planes[] = {g->h, g->qx, g->qy, g->h_max, g->dh, g->dqx, g->dqy};
    for (const void* p : planes)
      if ((uintptr_t)p % va) return fail(HP_EINVAL, "state planes must be aligned to 4 elements");
    if ((uintptr_t)g->landuse % kVec || (uintptr_t)g->station % (2 * kVec) || (uintptr_t)g->rain_field % (4 * kVec))
      return fail(HP_EINVAL, "landuse, station and rain_field planes must be aligned to 4 elements");
  }
  if (g->rain_mode == HP_RAIN_STATION) {
    if (!g->rain_table || g->rain_rows < 1 || g->rain_cols < 2)
      return fail(HP_EINVAL, "station rain needs a table of >= 1 row and >= 2 columns");
    if (g->rain_cols - 1 > kMaxStations) return fail(HP_EINVAL, "at most 1024 rain stations");
  } else if (g->rain_mode == HP_RAIN_FIELD) {
    if (!g->rain_field) return fail(HP_EINVAL, "field rain needs rain_field");
  } else if (g->rain_mode != HP_RAIN_NONE) {
    return fail(HP_EINVAL, "unknown rain_mode");
  }
  if ((g->given_depth && (g->gd_rows < 1 || g->gd_w < 1)) || (g->given_wl && (g->gwl_rows < 1 || g->gwl_w < 1)) ||
      (g->given_q && (g->gq_rows < 1 || g->gq_w < 1)))
    return fail(HP_EINVAL, "boundary series tables need >= 1 row and column");
  if (g->infil_ks && (!g->infil_phi || !g->infil_dtheta || !g->infil_F))
    return fail(HP_EINVAL, "infiltration needs infil_phi, infil_dtheta and infil_F");
  if ((uintptr_t)g->infil_dF % ((uintptr_t)kVec * (g->dtype == HP_F32 ? 4 : 8)))
    return fail(HP_EINVAL, "infil_dF must be aligned to 4 elements");
  if (flux_tiles(g) > 0x7fffffffLL || update_blocks(g) > 0x7fffffffLL) return fail(HP_EINVAL, "domain too large");
  if (g->dtype == HP_F32 && g->pitch * (int64_t)g->ny > 0xffffffffLL)
    return fail(HP_EINVAL, "float planes are limited to 2^32 elements");
  return HP_OK;
}

// A folded step: its place in the call and the record arrays of this step and
// the one before (null without mass sums).  A step that is not folded (st
// null) may take the gauge depths of the state that it starts from.
struct FoldStep {
  FoldState* st;
  int k;
  Sums *records, *prev;
  WalkGauges gauges;
};

template <class T, int ORDER, bool FUSED>
static int launch_walk_t(const hp_grid_desc* g, hipStream_t st, int flags, const FoldStep& f) {
  const int rows = flux_rows(g), ns = (g->nx + kWalkOwn - 1) / kWalkOwn;
  const int n = (int)units(g, kWalkOwn, rows);
  const int extra = f.st && f.records ? kFoldSumBlocks : (f.gauges.n + kWalkLanes - 1) / kWalkLanes;
  hipLaunchKernelGGL((k_walk<T, ORDER, FUSED>), dim3((unsigned)(n + extra)), dim3(kWalkLanes), 0, st, *g,
                     Divisor::of(ns), rows, flags, n, WalkFold{f.st, f.k, f.records}, f.prev, f.gauges);
  return check_launch(FUSED ? "k_walk (single-pass step)" : "k_walk (flux pass)");
}

template <bool FUSED>
static int launch_walk(const hp_grid_desc* g, hipStream_t st, int flags, const FoldStep& f = FoldStep{}) {
  if (g->dtype == HP_F32)
    return (g->order == 2 ? launch_walk_t<float, 2, FUSED> : launch_walk_t<float, 1, FUSED>)(g, st, flags, f);
  return (g->order == 2 ? launch_walk_t<double, 2, FUSED> : launch_walk_t<double, 1, FUSED>)(g, st, flags, f);
}

static int launch_flux(const hp_grid_desc* g, hipStream_t st) { return launch_walk<false>(g, st, 0); }

static int launch_step_fused(const hp_grid_desc* g, hipStream_t st, int flags = 0, const FoldStep& f = FoldStep{}) {
  return launch_walk<true>(g, st, flags, f);
}

static int launch_finalize_fused(const hp_grid_desc* g, hipStream_t st, const StepRecord* rec = nullptr) {
  if (rec) {
    hipLaunchKernelGGL(k_finalize_record, dim3(1), dim3(1024), 0, st, g->ctrl, g->work, (int)flux_tiles(g), g->dx,
                       g->mass_sums, *rec);
    return check_launch("k_finalize_record");
  }
  hipLaunchKernelGGL(k_finalize, dim3(1), dim3(1024), 0, st, g->ctrl, g->work, (int)flux_tiles(g), g->dx,
                     g->mass_sums, 1);
  return check_launch("k_finalize");
}

static int launch_infiltration(const hp_grid_desc* g, hipStream_t st) {
  const int64_t total = g->pitch * (int64_t)g->ny;
  const unsigned nb = (unsigned)((total + kThreads - 1) / kThreads);
  if (g->dtype == HP_F32) hipLaunchKernelGGL(k_infiltration<float>, dim3(nb), dim3(kThreads), 0, st, *g);
  else hipLaunchKernelGGL(k_infiltration<double>, dim3(nb), dim3(kThreads), 0, st, *g);
  return check_launch("k_infiltration");
}

template <class T, int MODE>
static void launch_update_t(const hp_grid_desc* g, int64_t nb, hipStream_t st) {
  if (update_width<T>(g->pitch * (int64_t)g->ny) != 1)
    hipLaunchKernelGGL((k_update<T, MODE, kWide<T>>), dim3((unsigned)nb), dim3(kThreads), 0, st, *g);
  else hipLaunchKernelGGL((k_update<T, MODE, 1>), dim3((unsigned)nb), dim3(kThreads), 0, st, *g);
}

template <int MODE>
static void launch_update_mode(const hp_grid_desc* g, int64_t nb, hipStream_t st) {
  (g->dtype == HP_F32 ? launch_update_t<float, MODE> : launch_update_t<double, MODE>)(g, nb, st);
}

static int launch_update(const hp_grid_desc* g, int mode, hipStream_t st) {
  const int64_t nb = update_blocks(g);
  if (!g->work || g->work_bytes < partials_bytes(nb))
    return fail(HP_ESPACE, "workspace smaller than hp_grid_workspace_bytes()");
  switch (mode) {
    case HP_UPDATE_STEP: launch_update_mode<HP_UPDATE_STEP>(g, nb, st); break;
    case HP_UPDATE_FRICTION: launch_update_mode<HP_UPDATE_FRICTION>(g, nb, st); break;
    case HP_UPDATE_EULER: launch_update_mode<HP_UPDATE_EULER>(g, nb, st); break;
    case HP_UPDATE_CFL: launch_update_mode<HP_UPDATE_CFL>(g, nb, st); break;
    default: return fail(HP_EINVAL, "unknown update mode");
  }
  int rc = check_launch("k_update");
  if (rc) return rc;
  if (mode == HP_UPDATE_STEP || mode == HP_UPDATE_CFL) {
    hipLaunchKernelGGL(k_finalize, dim3(1), dim3(1024), 0, st, g->ctrl, g->work, (int)nb, g->dx,
                       g->mass_sums, 0);
    return check_launch("k_finalize");
  }
  return HP_OK;
}

// ---- ensemble ---------------------------------------------------------------
// Workspace of an ensemble: the descriptors twice (the second copy with the
// two sets of state planes exchanged, for the odd steps of the single-pass
// step), the (domain, unit) and (domain, chunk) maps, the per-domain ranges of
// partial records for the two-pass and the single-pass step, the records, the
// folded time control's states and its two arrays of sum records.
struct EnsembleLayout {
  int64_t off_doms, off_fmap, off_umap, off_fin, off_fin1, off_parts, total;
  int64_t n_ftiles, n_ublocks;
};
static int64_t ensemble_parts_bytes(int64_t n_ftiles, int64_t n_ublocks) {
  return align256(partials_bytes(n_ublocks > n_ftiles ? n_ublocks : n_ftiles));
}
// hp_ensemble::single_pass of a handle: 1, and these
constexpr int kEnsembleFold = 2;  // calls of several steps fold the time control
constexpr int kEnsembleSums = 4;  // a domain keeps mass sums

// The unit height of an ensemble: the one its domains ask for (all the same),
// else by the units of all of them, which share one launch.
static int ensemble_rows(int32_t n, const hp_grid_desc* d) {
  for (int k = 0; k < n; ++k)
    if (asked_rows(&d[k])) return asked_rows(&d[k]);
  return chosen_height(n, d);
}

static EnsembleLayout ensemble_layout(int32_t n, const hp_grid_desc* d) {
  EnsembleLayout L{};
  const int rows = ensemble_rows(n, d);
  for (int k = 0; k < n; ++k) {
    L.n_ftiles += units(&d[k], kWalkOwn, rows);
    L.n_ublocks += update_blocks(&d[k]);
  }
  L.off_doms = 0;
  L.off_fmap = align256(2 * (int64_t)n * (int64_t)sizeof(hp_grid_desc));
  L.off_umap = L.off_fmap + align256(L.n_ftiles * 8);
  L.off_fin = L.off_umap + align256(L.n_ublocks * 8);
  L.off_fin1 = L.off_fin + align256((int64_t)n * 8);
  L.off_parts = L.off_fin1 + align256((int64_t)n * 8);
  L.total = L.off_parts + ensemble_parts_bytes(L.n_ftiles, L.n_ublocks) +
            align256((int64_t)n * (int64_t)sizeof(FoldState)) + 2 * L.n_ftiles * (int64_t)sizeof(Sums);
  return L;
}

template <class T>
static void launch_update_multi(const hp_ensemble* e, hipStream_t st) {
  hipLaunchKernelGGL((k_update_multi<T, HP_UPDATE_STEP>), dim3((unsigned)e->n_update_blocks), dim3(kThreads), 0, st,
                     (const hp_grid_desc*)e->doms, (const int2*)e->update_map, e->partials);
}

template <class T, int ORDER, bool FUSED>
static void launch_walk_multi(const hp_ensemble* e, int parity, hipStream_t st, const FoldStep& f) {
  const int extra = f.st && f.records ? kFoldSumBlocks * e->n_domains : 0;
  hipLaunchKernelGGL((k_walk_multi<T, ORDER, FUSED>), dim3((unsigned)(e->n_flux_tiles + extra)), dim3(kWalkLanes), 0,
                     st, (const hp_grid_desc*)e->doms + (parity ? e->n_domains : 0), (const int2*)e->flux_map,
                     e->partials, (int)e->n_flux_tiles, (int)e->tile_rows, WalkFold{f.st, f.k, f.records},
                     (const Sums*)f.prev, (const int2*)e->fused_finalize_map);
}

template <bool FUSED>
static void launch_walk_multi_any(const hp_ensemble* e, int parity, hipStream_t st, const FoldStep& f = FoldStep{}) {
  if (e->dtype == HP_F32)
    (e->order == 2 ? launch_walk_multi<float, 2, FUSED> : launch_walk_multi<float, 1, FUSED>)(e, parity, st, f);
  else (e->order == 2 ? launch_walk_multi<double, 2, FUSED> : launch_walk_multi<double, 1, FUSED>)(e, parity, st, f);
}

// nsteps single-pass steps of every domain with the time control folded, as
// single_pass_steps does for one: per step of eight 1024^2 scenarios 118 us
// with a time-control launch, 113 folded.
static int ensemble_folded_steps(const hp_ensemble* e, int32_t nsteps, hipStream_t st) {
  uint8_t* base = (uint8_t*)e->partials + ensemble_parts_bytes(e->n_flux_tiles, e->n_update_blocks);
  FoldState* fs = (FoldState*)base;
  Sums* rec = e->single_pass & kEnsembleSums ? (Sums*)(base + align256((int64_t)e->n_domains * (int64_t)sizeof(FoldState))) : nullptr;
  auto records = [&](int k) { return rec ? rec + (int64_t)(k & 1) * e->n_flux_tiles : nullptr; };
  const dim3 nd((unsigned)e->n_domains);
  hipLaunchKernelGGL(k_fold_begin_multi, nd, dim3(64), 0, st, (const hp_grid_desc*)e->doms, fs);
  int rc = check_launch("k_fold_begin_multi");
  for (int32_t k = 0; k < nsteps && !rc; ++k) {
    launch_walk_multi_any<true>(e, k & 1, st, FoldStep{fs, k, records(k), records(k + 1)});
    rc = check_launch("k_walk_multi (single-pass step)");
  }
  if (rc) return rc;
  hipLaunchKernelGGL(k_fold_end_multi, nd, dim3(rec ? 1024 : 64), 0, st, (const hp_grid_desc*)e->doms,
                     (const int2*)e->fused_finalize_map, (const FoldState*)fs, (int)nsteps,
                     (const Sums*)records(nsteps - 1));
  return check_launch("k_fold_end_multi");
}

// One single-pass step of every domain: even steps read the domains' own
// planes and write their second set, odd steps the reverse.
static int ensemble_fused_step_once(const hp_ensemble* e, int parity, hipStream_t st) {
  launch_walk_multi_any<true>(e, parity, st);
  int rc = check_launch("k_walk_multi (single-pass step)");
  if (rc) return rc;
  hipLaunchKernelGGL(k_finalize_multi, dim3((unsigned)e->n_domains), dim3(1024), 0, st,
                     (const hp_grid_desc*)e->doms, (const int2*)e->fused_finalize_map, e->partials,
                     (int)e->n_flux_tiles, 1);
  return check_launch("k_finalize_multi");
}

static int ensemble_step_once(const hp_ensemble* e, hipStream_t st) {
  const bool f32 = e->dtype == HP_F32;
  launch_walk_multi_any<false>(e, 0, st);
  int rc = check_launch("k_walk_multi (flux pass)");
  if (rc) return rc;
  if (f32) launch_update_multi<float>(e, st);
  else launch_update_multi<double>(e, st);
  rc = check_launch("k_update_multi");
  if (rc) return rc;
  hipLaunchKernelGGL(k_finalize_multi, dim3((unsigned)e->n_domains), dim3(1024), 0, st,
                     (const hp_grid_desc*)e->doms, (const int2*)e->finalize_map, e->partials,
                     (int)e->n_update_blocks, 0);
  return check_launch("k_finalize_multi");
}

template <class T>
__global__ void k_gather(const T* __restrict__ plane, const int64_t* __restrict__ off, int64_t n, T* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = plane[off[i]];
}
template <class T>
__global__ void k_scatter(T* __restrict__ plane, const int64_t* __restrict__ off, int64_t n, const T* __restrict__ in) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) plane[off[i]] = in[i];
}

// Single-pass step (h, qx, qy -> h_out, qx_out, qy_out; with save_flux the
// step's flux also into dh, dqx, dqy) and, with finalize, its time control,
// followed by rec when given; without time_control the step computes no
// CFL candidates, sums or partial records (no time control may follow).
// gauges: those of the state before the step.
// Shared with the calibration runs.
int grid_fused_launch(const hp_grid_desc* g, bool save_flux, bool finalize, hipStream_t st, const StepRecord* rec,
                      bool time_control, const WalkGauges& gauges) {
  int rc = check_desc(g);
  if (rc) return rc;
  if (!g->h_out || !g->qx_out || !g->qy_out) return fail(HP_EINVAL, "the fused step needs h_out, qx_out, qy_out");
  if (save_flux && (!g->dh || !g->dqx || !g->dqy)) return fail(HP_EINVAL, "saving the flux needs dh, dqx, dqy");
  if (!g->work || g->work_bytes < partials_bytes(flux_tiles(g)))
    return fail(HP_ESPACE, "workspace smaller than hp_grid_workspace_bytes()");
  if (finalize && !time_control) return fail(HP_EINVAL, "a time control needs the step's CFL candidates");
  FoldStep f{};
  f.gauges = gauges;
  rc = launch_step_fused(g, st, (save_flux ? 1 : 0) | (time_control ? 0 : 2), f);
  if (rc || !finalize) return rc;
  return launch_finalize_fused(g, st, rec);
}

// Flux pass launch shared with the adjoint (which recomputes it).
int grid_flux_launch(const hp_grid_desc* g, hipStream_t st) {
  int rc = check_desc(g);
  if (rc) return rc;
  return launch_flux(g, st);
}

// ---- allocation-free single-pass step ---------------------------------------
// The single-pass step's only scratch memory is its units' partial records
// (CFL minimum, FP64 sums) or, in calls that fold the time control, the fold's
// state and sum records, normally in the caller's workspace.  For callers that
// cannot allocate, a file-scope device array holds them instead: every GPU the
// library runs on keeps its own copy until the process ends.  Nothing in it
// must start at zero: a unit writes its record in every step before the time
// control reads it, a folded call begins with a launch that fills its state,
// and the records that the units of a stopped step leave out are not read.
// Calls that overlap on one GPU share the array and race.
constexpr int64_t kScratchBytes = int64_t(8) << 20;
static __device__ __align__(256) uint8_t scratch[kScratchBytes];
constexpr int kMaxScratchDevices = 64;
static void* g_scratch[kMaxScratchDevices];
static std::mutex g_scratch_mu;

// Device address of the current device's scratch array, looked up once per
// device (hipGetSymbolAddress with that device current).
static int scratch_ptr(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(HP_ELAUNCH, std::string("hipGetDevice: ") + hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxScratchDevices) return fail(HP_EINVAL, "device index beyond the scratch table");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) return fail(HP_ELAUNCH, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    g_scratch[dev] = p;
  }
  *out = g_scratch[dev];
  return HP_OK;
}

// Workspace of a domain: the partial records of the larger of the update
// pass and the flux / single-pass step.
static int64_t workspace_need(const hp_grid_desc* g) {
  return partials_bytes(std::max({flux_tiles(g), nominal_tiles(g), update_blocks(g)}));
}

// Workspace of a call with folded time control: the fold's state, and two
// arrays of sum records when they are kept.  Asked for beside workspace_need;
// where a caller brings less, the time control keeps its own launches.
static int64_t fold_need(const hp_grid_desc* g) {
  return align256(sizeof(FoldState)) + (g->mass_sums ? 2 * flux_tiles(g) * (int64_t)sizeof(Sums) : 0);
}

// The checks every single-pass entry point makes (need: bytes that the
// workspace must have at least).
static int check_fused(const hp_grid_desc* g, int64_t (*need)(const hp_grid_desc*) = workspace_need) {
  int rc = check_desc(g);
  if (rc) return rc;
  if (!g->h_out || !g->qx_out || !g->qy_out) return fail(HP_EINVAL, "the fused step needs h_out, qx_out, qy_out");
  if (!g->work || g->work_bytes < need(g))
    return fail(HP_ESPACE, "workspace smaller than hp_grid_workspace_bytes()");
  return HP_OK;
}

// The records that the single-pass step itself writes.
static int64_t fused_records(const hp_grid_desc* g) { return partials_bytes(flux_tiles(g)); }

// Whether a domain's CFL minima may be folded by the bits of the doubles: a
// negative CFL number, zero included, gives negative ones, which do not order.
static bool ordered_minima(const hp_grid_desc* g) { return g->cfl >= 0.0 && !std::signbit(g->cfl); }

// Calls of at least this many steps fold the time control into the step
// kernel: begin and end are launches too, so below it nothing is saved.
constexpr int kFoldSteps = 3;

// nsteps single-pass steps, each with its time control; the buffers swap every
// step.  before / after are called around every step's kernel.
template <class Before, class After>
static int single_pass_steps(const hp_grid_desc* g, int32_t nsteps, hipStream_t st, Before before, After after) {
  hp_grid_desc d = *g;
  const bool fold = nsteps >= kFoldSteps && ordered_minima(g) && g->work_bytes >= fold_need(g);
  FoldState* fs = fold ? (FoldState*)g->work : nullptr;
  const int64_t n = flux_tiles(g);
  Sums* rec = fold && g->mass_sums ? (Sums*)((char*)g->work + align256(sizeof(FoldState))) : nullptr;
  auto records = [&](int k) { return rec ? rec + (k & 1) * n : nullptr; };
  int rc = HP_OK;
  if (fold) {
    hipLaunchKernelGGL(k_fold_begin, dim3(1), dim3(64), 0, st, (const hp_ctrl*)g->ctrl, fs);
    rc = check_launch("k_fold_begin");
    if (rc) return rc;
  }
  for (int32_t k = 0; k < nsteps; ++k) {
    before(k);
    // the first step of a call copies a stopped domain's state through even
    // if an earlier call left both sets in step: the host may have written
    // the state in between
    rc = launch_step_fused(&d, st, k == 0 ? 4 : 0, FoldStep{fs, k, records(k), records(k + 1)});
    if (rc) return rc;
    after(k);
    if (!fold) {
      rc = launch_finalize_fused(&d, st);
      if (rc) return rc;
    }
    std::swap(d.h, d.h_out);
    std::swap(d.qx, d.qx_out);
    std::swap(d.qy, d.qy_out);
  }
  if (fold) {
    hipLaunchKernelGGL(k_fold_end, dim3(1), dim3(rec ? 1024 : 64), 0, st, g->ctrl, (const FoldState*)fs, (int)nsteps,
                       (const Sums*)records(nsteps - 1), (int)n, g->dx, rec ? 1 : 0);
    rc = check_launch("k_fold_end");
  }
  return rc;
}

// After an odd number of single-pass steps the state sits in the second set
// of planes: bring it back to the caller's (h, qx, qy).
static int copy_state_back(const hp_grid_desc* g, hipStream_t st) {
  const size_t bytes = (size_t)(g->pitch * (int64_t)g->ny) * (g->dtype == HP_F32 ? 4 : 8);
  hipError_t e = hipMemcpyAsync(g->h, g->h_out, bytes, hipMemcpyDeviceToDevice, st);
  if (e == hipSuccess) e = hipMemcpyAsync(g->qx, g->qx_out, bytes, hipMemcpyDeviceToDevice, st);
  if (e == hipSuccess) e = hipMemcpyAsync(g->qy, g->qy_out, bytes, hipMemcpyDeviceToDevice, st);
  if (e != hipSuccess) return fail(HP_ELAUNCH, std::string("state copy: ") + hipGetErrorString(e));
  return HP_OK;
}

// nsteps single-pass steps, the state in the caller's planes at the end.
static int step_fused(const hp_grid_desc* g, int32_t nsteps, hipStream_t st) {
  if (nsteps < 0) return fail(HP_EINVAL, "nsteps must be >= 0");
  int rc = single_pass_steps(g, nsteps, st, [](int) {}, [](int) {});
  if (rc) return rc;
  if (nsteps & 1) return copy_state_back(g, st);
  return HP_OK;
}

}  // namespace hp

using namespace hp;

extern "C" {

int64_t hp_grid_workspace_bytes(const hp_grid_desc* g) {
  if (!g || g->pitch <= 0 || g->ny <= 0 || g->nx <= 0) return 0;
  return std::max(workspace_need(g), fold_need(g));
}

int hp_grid_step_fused(const hp_grid_desc* g, int32_t nsteps, void* stream) {
  int rc = check_fused(g);
  if (rc) return rc;
  return step_fused(g, nsteps, (hipStream_t)stream);
}

int64_t hp_grid_noalloc_max_bytes(void) { return kScratchBytes; }

int hp_grid_step_fused_noalloc(const hp_grid_desc* g, int32_t nsteps, void* stream) {
  int rc = check_desc(g);
  if (rc) return rc;
  const int64_t need = partials_bytes(std::max(nominal_tiles(g), update_blocks(g)));
  if (need > kScratchBytes)
    return fail(HP_ESPACE, "domain needs " + std::to_string(need) + " bytes of per-unit records; the allocation-free "
                           "step holds at most " + std::to_string(kScratchBytes) + " (use hp_grid_step_fused)");
  void* p = nullptr;
  rc = scratch_ptr(&p);
  if (rc) return rc;
  hp_grid_desc d = *g;
  d.work = p;
  d.work_bytes = kScratchBytes;
  // (an asked height whose 60-column units have more records than its
  // nominal tiles gives way to the chosen one, which has fewer)
  if (fused_records(&d) > kScratchBytes) d.tile_rows = 0;
  rc = check_fused(&d, fused_records);
  if (rc) return rc;
  return step_fused(&d, nsteps, (hipStream_t)stream);
}

int hp_grid_step_fused_timed(const hp_grid_desc* g, int32_t nsteps, int32_t sample_every, float* kernel_ms,
                             float* step_ms, void* stream) {
  int rc = check_fused(g);
  if (rc) return rc;
  if (nsteps <= 0 || sample_every <= 0) return fail(HP_EINVAL, "nsteps and sample_every must be positive");
  if (!kernel_ms || !step_ms) return fail(HP_EINVAL, "kernel_ms and step_ms are required");
  hipStream_t st = (hipStream_t)stream;
  // ev[0] / ev[1]: around all nsteps steps; ev[2 + 2j] / ev[3 + 2j]: around
  // the single-pass kernel of the j-th sampled step
  const int32_t samples = (nsteps + sample_every - 1) / sample_every;
  std::vector<hipEvent_t> ev(2 + 2 * (size_t)samples, nullptr);
  auto release = [&]() {
    for (hipEvent_t e : ev)
      if (e) (void)hipEventDestroy(e);
  };
  for (auto& e : ev) {
    if (hipEventCreate(&e) != hipSuccess) {
      release();
      return fail(HP_ELAUNCH, "hipEventCreate failed");
    }
  }
  (void)hipEventRecord(ev[0], st);
  rc = single_pass_steps(
      g, nsteps, st,
      [&](int k) {
        if (k % sample_every == 0) (void)hipEventRecord(ev[2 + 2 * (size_t)(k / sample_every)], st);
      },
      [&](int k) {
        if (k % sample_every == 0) (void)hipEventRecord(ev[3 + 2 * (size_t)(k / sample_every)], st);
      });
  if (rc == HP_OK) {
    (void)hipEventRecord(ev[1], st);
    if (nsteps & 1) rc = copy_state_back(g, st);  // after the timed steps
    if (rc == HP_OK && hipEventSynchronize(ev[1]) != hipSuccess) rc = fail(HP_ELAUNCH, "hipEventSynchronize failed");
  }
  if (rc == HP_OK) {
    float sum = 0.0f, ms = 0.0f;
    for (int32_t j = 0; j < samples; ++j) {
      (void)hipEventElapsedTime(&ms, ev[2 + 2 * (size_t)j], ev[3 + 2 * (size_t)j]);
      sum += ms;
    }
    (void)hipEventElapsedTime(&ms, ev[0], ev[1]);
    *kernel_ms = sum / (float)samples;
    *step_ms = ms;
  }
  release();
  return rc;
}

int hp_grid_flux(const hp_grid_desc* g, void* stream) {
  int rc = check_desc(g);
  if (rc) return rc;
  return launch_flux(g, (hipStream_t)stream);
}

int hp_grid_update(const hp_grid_desc* g, void* stream) { return hp_grid_update_mode(g, HP_UPDATE_STEP, stream); }

int hp_grid_update_mode(const hp_grid_desc* g, int mode, void* stream) {
  int rc = check_desc(g);
  if (rc) return rc;
  return launch_update(g, mode, (hipStream_t)stream);
}

int hp_grid_infiltration(const hp_grid_desc* g, void* stream) {
  int rc = check_desc(g);
  if (rc) return rc;
  if (!g->infil_ks || !g->infil_dF) return fail(HP_EINVAL, "infiltration needs infil_ks and an infil_dF plane");
  return launch_infiltration(g, (hipStream_t)stream);
}

int hp_grid_step(const hp_grid_desc* g, int32_t nsteps, void* stream) {
  int rc = check_desc(g);
  if (rc) return rc;
  if (nsteps < 0) return fail(HP_EINVAL, "nsteps must be >= 0");
  if (g->infil_ks && !g->infil_dF) return fail(HP_EINVAL, "a step with infiltration needs an infil_dF plane");
  hp_grid_desc d = *g;
  if (!d.infil_ks) d.infil_dF = nullptr;  // nothing to subtract
  for (int32_t k = 0; k < nsteps; ++k) {
    rc = launch_flux(&d, (hipStream_t)stream);
    if (rc) return rc;
    if (d.infil_ks) {
      rc = launch_infiltration(&d, (hipStream_t)stream);
      if (rc) return rc;
    }
    rc = launch_update(&d, HP_UPDATE_STEP, (hipStream_t)stream);
    if (rc) return rc;
  }
  return HP_OK;
}

int64_t hp_ensemble_workspace_bytes(int32_t n, const hp_grid_desc* descs) {
  if (n <= 0 || !descs) return 0;
  return ensemble_layout(n, descs).total;
}

int hp_ensemble_init(int32_t n, const hp_grid_desc* descs, int32_t single_pass, void* work, int64_t work_bytes,
                     hp_ensemble* out, void* stream) {
  if (n <= 0 || !descs || !out) return fail(HP_EINVAL, "need n > 0 descriptors and an output handle");
  if (single_pass != 0 && single_pass != 1) return fail(HP_EINVAL, "single_pass must be 0 or 1");
  for (int k = 0; k < n; ++k) {
    if (descs[k].infil_ks) return fail(HP_EINVAL, "infiltration is not supported in an ensemble");
    int rc = check_desc(&descs[k]);
    if (rc) return fail(rc, "domain " + std::to_string(k) + ": " + last_error_slot());
    if (single_pass && (!descs[k].h_out || !descs[k].qx_out || !descs[k].qy_out))
      return fail(HP_EINVAL, "domain " + std::to_string(k) + ": the single-pass step needs h_out, qx_out, qy_out");
    if (descs[k].dtype != descs[0].dtype || descs[k].order != descs[0].order ||
        nominal_rows(&descs[k]) != nominal_rows(&descs[0]))
      return fail(HP_EINVAL, "every domain of an ensemble needs the same dtype, order and tile_rows");
  }
  const EnsembleLayout L = ensemble_layout(n, descs);
  if (!work || work_bytes < L.total) return fail(HP_ESPACE, "workspace smaller than hp_ensemble_workspace_bytes()");
  if (L.n_ftiles > 0x7fffffffLL || L.n_ublocks > 0x7fffffffLL) return fail(HP_EINVAL, "ensemble too large");
  std::vector<uint8_t> host((size_t)L.off_parts, 0);
  std::memcpy(host.data() + L.off_doms, descs, sizeof(hp_grid_desc) * (size_t)n);
  hp_grid_desc* swapped = (hp_grid_desc*)(host.data() + L.off_doms) + n;
  for (int k = 0; k < n; ++k) {
    swapped[k] = descs[k];
    std::swap(swapped[k].h, swapped[k].h_out);
    std::swap(swapped[k].qx, swapped[k].qx_out);
    std::swap(swapped[k].qy, swapped[k].qy_out);
  }
  int32_t* fm = (int32_t*)(host.data() + L.off_fmap);
  int32_t* um = (int32_t*)(host.data() + L.off_umap);
  int32_t* fin = (int32_t*)(host.data() + L.off_fin);
  int32_t* fin1 = (int32_t*)(host.data() + L.off_fin1);
  int64_t fi = 0, ui = 0;
  const int rows = ensemble_rows(n, descs);
  for (int k = 0; k < n; ++k) {
    const int64_t nt = units(&descs[k], kWalkOwn, rows), nu = update_blocks(&descs[k]);
    fin1[2 * k] = (int32_t)fi;
    fin1[2 * k + 1] = (int32_t)nt;
    for (int64_t j = 0; j < nt; ++j, ++fi) {
      fm[2 * fi] = k;
      fm[2 * fi + 1] = (int32_t)j;
    }
    fin[2 * k] = (int32_t)ui;
    fin[2 * k + 1] = (int32_t)nu;
    for (int64_t j = 0; j < nu; ++j, ++ui) {
      um[2 * ui] = k;
      um[2 * ui + 1] = (int32_t)j;
    }
  }
  hipError_t err = hipMemcpyAsync(work, host.data(), host.size(), hipMemcpyHostToDevice, (hipStream_t)stream);
  if (err == hipSuccess) err = hipStreamSynchronize((hipStream_t)stream);
  if (err != hipSuccess) return fail(HP_ELAUNCH, std::string("ensemble table upload: ") + hipGetErrorString(err));
  uint8_t* w = (uint8_t*)work;
  out->n_domains = n;
  out->dtype = descs[0].dtype;
  out->order = descs[0].order;
  out->tile_rows = rows;
  out->n_flux_tiles = (int32_t)L.n_ftiles;
  out->n_update_blocks = (int32_t)L.n_ublocks;
  out->doms = w + L.off_doms;
  out->flux_map = w + L.off_fmap;
  out->update_map = w + L.off_umap;
  out->finalize_map = w + L.off_fin;
  out->partials = w + L.off_parts;
  out->single_pass = single_pass;
  if (single_pass) {
    bool fold = true, sums = false;
    for (int k = 0; k < n; ++k) {
      fold = fold && ordered_minima(&descs[k]);
      sums = sums || descs[k].mass_sums != 0;
    }
    out->single_pass |= (fold ? kEnsembleFold : 0) | (sums ? kEnsembleSums : 0);
  }
  out->fused_finalize_map = w + L.off_fin1;
  return HP_OK;
}

int hp_ensemble_step(const hp_ensemble* e, int32_t nsteps, void* stream) {
  if (!e || e->n_domains <= 0 || !e->doms) return fail(HP_EINVAL, "ensemble handle not initialised");
  if (nsteps < 0) return fail(HP_EINVAL, "nsteps must be >= 0");
  if (e->single_pass) {
    if (nsteps & 1)
      return fail(HP_EINVAL, "a single-pass ensemble advances an even number of steps per call (the state then "
                             "ends in the domains' own planes)");
    if (nsteps >= kFoldSteps && (e->single_pass & kEnsembleFold))
      return ensemble_folded_steps(e, nsteps, (hipStream_t)stream);
    for (int32_t k = 0; k < nsteps; ++k) {
      int rc = ensemble_fused_step_once(e, k & 1, (hipStream_t)stream);
      if (rc) return rc;
    }
    return HP_OK;
  }
  for (int32_t k = 0; k < nsteps; ++k) {
    int rc = ensemble_step_once(e, (hipStream_t)stream);
    if (rc) return rc;
  }
  return HP_OK;
}

int hp_gather(int dtype, const void* plane, const int64_t* offsets, int64_t n, void* out, void* stream) {
  if (dtype != HP_F32 && dtype != HP_F64) return fail(HP_EINVAL, "dtype must be HP_F32 or HP_F64");
  if (n < 0) return fail(HP_EINVAL, "n must be >= 0");
  if (n == 0) return HP_OK;
  if (!plane || !offsets || !out) return fail(HP_EINVAL, "null pointer");
  const unsigned nb = (unsigned)((n + 255) / 256);
  if (dtype == HP_F32)
    hipLaunchKernelGGL(k_gather<float>, dim3(nb), dim3(256), 0, (hipStream_t)stream, (const float*)plane, offsets, n,
                       (float*)out);
  else
    hipLaunchKernelGGL(k_gather<double>, dim3(nb), dim3(256), 0, (hipStream_t)stream, (const double*)plane, offsets,
                       n, (double*)out);
  return check_launch("k_gather");
}

int hp_scatter(int dtype, void* plane, const int64_t* offsets, int64_t n, const void* in, void* stream) {
  if (dtype != HP_F32 && dtype != HP_F64) return fail(HP_EINVAL, "dtype must be HP_F32 or HP_F64");
  if (n < 0) return fail(HP_EINVAL, "n must be >= 0");
  if (n == 0) return HP_OK;
  if (!plane || !offsets || !in) return fail(HP_EINVAL, "null pointer");
  const unsigned nb = (unsigned)((n + 255) / 256);
  if (dtype == HP_F32)
    hipLaunchKernelGGL(k_scatter<float>, dim3(nb), dim3(256), 0, (hipStream_t)stream, (float*)plane, offsets, n,
                       (const float*)in);
  else
    hipLaunchKernelGGL(k_scatter<double>, dim3(nb), dim3(256), 0, (hipStream_t)stream, (double*)plane, offsets, n,
                       (const double*)in);
  return check_launch("k_scatter");
}

}  // extern "C"
