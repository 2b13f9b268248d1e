// Rain source terms and the planes' alignment, shared by the step and its adjoint.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/hipims_abi.h"

namespace hp {

// Planes are aligned to this many elements, and rows hold a multiple of them.
constexpr int kVec = 4;

// Station rain at time t_now (SWE_CUDA.py:472-495): linear in time between
// the table rows that bracket t_now, 0 from the table's last row on, scaled
// by rain_scale.  The bracketing rows are found once per block; the passes
// keep the first stations' rates in LDS and evaluate any further station's
// rate per cell from the two rows.
struct RainRows {
  const double* lo;  // station columns of the rows bracketing t_now
  const double* hi;
  double per;        // interpolation weight
  int n_st;
  bool zero;         // every station rate is 0 (after the table, or one row)
};

// The smallest i in [from, to) for which hit(i), else `to`: the answer of a
// loop from `from` upwards, found 64 candidates at a time by the whole wave
// (all lanes active, the arguments the same in every lane).  Tables of a
// storm hold hundreds of rows (289 rows of five minutes make a day), and a
// loop pays a memory round trip for each: the 37th row of such a table cost a
// block of the update pass about 12 us.
template <class F> __device__ inline int wave_first(int from, int to, F hit) {
  const int lane = (int)(threadIdx.x & 63);
  for (int base = from; base < to; base += 64) {
    const int i = base + lane;
    const uint64_t m = __builtin_amdgcn_ballot_w64(i < to && hit(i));
    if (m) return __builtin_amdgcn_readfirstlane(base + (int)__builtin_ctzll(m));
  }
  return to;
}

// The times of a rain table of at most 64 rows, a row per lane (all the lanes
// of a wave call it): one memory round trip, which a kernel can start before
// it knows its own time.
template <class DP> __device__ inline double wave_rain_times(DP a) {
  if (a->rain_mode != HP_RAIN_STATION || a->rain_table == nullptr || a->rain_rows <= 1 || a->rain_rows > 64) return 0.0;
  const int lane = (int)(threadIdx.x & 63);
  return a->rain_table[(int64_t)(lane < a->rain_rows ? lane : 0) * a->rain_cols];
}

// The bracketing rows at t_now, through any pointer type of the descriptor
// (generic, or the kernel-argument address space); called by whole waves.
// times: wave_rain_times.
template <class DP> __device__ inline RainRows wave_rain_rows(DP a, double t_now, double times) {
  RainRows r{nullptr, nullptr, 0.0, 0, true};
  if (a->rain_mode != HP_RAIN_STATION || a->rain_table == nullptr || a->rain_rows <= 0) return r;
  const int rows = a->rain_rows, cols = a->rain_cols;
  const double* tab = a->rain_table;
  r.n_st = cols - 1;
  if (rows <= 1) return r;
  int i;  // the last row whose successor lies after t_now (the table's last two rows at most)
  double t0, t1;
  if (rows <= 64) {
    const int lane = (int)(threadIdx.x & 63);
    const uint64_t later = __builtin_amdgcn_ballot_w64(lane < rows && t_now < times);
    r.zero = !(later >> (rows - 1) & 1);
    if (r.zero) return r;
    const uint64_t inner = later & ((uint64_t(1) << (rows - 1)) - 2);  // rows 1 .. rows - 2
    i = inner ? (int)__builtin_ctzll(inner) - 1 : rows - 2;
    t0 = __shfl(times, i, 64);
    t1 = __shfl(times, i + 1, 64);
  } else {
    r.zero = !(t_now < tab[(int64_t)(rows - 1) * cols]);
    if (r.zero) return r;
    i = wave_first(0, rows - 2, [&](int k) { return t_now < tab[(int64_t)(k + 1) * cols]; });
    t0 = tab[(int64_t)i * cols];
    t1 = tab[(int64_t)(i + 1) * cols];
  }
  r.lo = tab + (int64_t)i * cols + 1;
  r.hi = r.lo + cols;
  r.per = (t_now - t0) / (t1 - t0);
  return r;
}

template <class DP> __device__ inline RainRows wave_rain_rows(DP a, double t_now) {
  return wave_rain_rows(a, t_now, wave_rain_times(a));
}

// Rain rate of a cell whose station index is k.
template <class T> __device__ inline T station_rate(const RainRows& rr, int k, double scale) {
  if (rr.zero || k < 0 || k >= rr.n_st) return T(0);
  const double lo = rr.lo[k], hi = rr.hi[k];
  return T((lo + rr.per * (hi - lo)) * scale);
}

}  // namespace hp
