// The step as a column walk (gfx950): the flux stencil of both step forms
// (flux pass, single-pass step) in both precisions.
//
// A workgroup is one wave64.  Its lanes load 64 consecutive columns
// [x0 - 2, x0 + 62) and walk down rows y0 - 2 .. y0 + R + 1 of the planes,
// finishing rows y0 .. y0 + R - 1 of the 60 columns [x0, x0 + 60) (lanes
// 2 .. 61; the two lanes on either side are the x halo).  Nothing is staged
// in LDS:
//   * a cell's x neighbours come from the lanes beside it through DPP
//     wavefront shifts (one VALU move per value), its y neighbours from the
//     rows the lane already holds (a rolling window of four rows: the row
//     being finished, the next two, and the one being prefetched);
//   * every limited slope (MUSCL: h, qx, qy, z along x and along y; order 1:
//     z) is formed once per cell and serves the cell's two faces on that
//     axis (the reference's per-edge form evaluates it twice; minmod is
//     symmetric and odd, so the faces are the same numbers);
//   * each lane solves the west edge of its cell (the west neighbour's east
//     face arrives by a lane shift) and the south edge between the row being
//     finished and the next (both faces in its registers); the west
//     neighbour's share of the x edge goes back to it by the opposite shift,
//     the next row's share of the y edge stays in the lane for the next row.
// An edge is solved in its own frame (in float on the west / north cell's
// datum), HLLC after the hydrostatic reconstruction, bed terms on both sides;
// a cell sums its E, N, W, S shares in the reference's order and scales the
// sum by dt / dx.
//
// Two paths through a row.  The vector instructions bound this kernel, and a
// good part of them only serve nodata: the selects that replace a nodata
// neighbour by the cell itself, and the ghosts of boundary edges.  Where all
// 64 lanes of the row and of the two below it hold valid cells (a ballot per
// row), the row runs without them, its two edges as one straight block; any
// other row runs the general path.  Both give the same bits, which the edges
// between two units need: each unit may solve them on another path.  The
// listing rule works on the ballots of wet lanes in scalar registers, and the
// edges between two rows (or a row's x edges) are skipped where every lane is
// dry.  (A further path for rows whose lanes are all wet was tried: on terrain
// with a few dry cells in a hundred it is rarely taken.)
//
// A unit alone on its SIMD walks at about 2 us a row, bound by its own
// instruction stream: that, not the rate with all waves in flight, is what a
// small domain and the end of every launch see.  Hence the pointers of the
// planes stay in scalar registers, the update's inputs are asked for a row
// ahead and before the row's stores, no load sits under a condition (where
// paths join, its register would be copied, and waited for), and boundary
// edges share the interior edges' solver call.  Measured on one MI355X, single
// pass, order 2, per step at the chosen unit height, from the two-row-prologue
// walk (double: an LDS tile of 64 x 4 cells per block) to this one: float 64^2
// 14.4 -> 8.3 us, 2048^2 72.7 -> 60.5, 8192^2 with a rain field and mass sums
// 921 -> 810; double 2048^2 216 -> 139, 256^2 17.1 -> 11.8.
//
// Geometry: a unit is (strip bx, row block by); 60 columns x R rows.  Each
// interior x edge is solved once, except the one between two strips (solved
// by both); each interior y edge once, except the one between two row
// blocks.

namespace hp {

constexpr int kWalkLanes = 64;
constexpr int kWalkOwn = 60;

// Lane i receives lane i - 1's value (lane 0 reads 0); all 64 lanes must be
// active.  Lanes 0 and 63 are halo lanes whose results are never used, so
// the out-of-range value does not matter, and without an `old` operand the
// shift is one instruction.
__device__ inline int from_west(int v) { return __builtin_amdgcn_mov_dpp(v, 0x138 /* wave_shr:1 */, 0xf, 0xf, true); }
__device__ inline float from_west(float v) { return __builtin_bit_cast(float, from_west(__builtin_bit_cast(int, v))); }
// Lane i receives lane i + 1's value (lane 63 reads 0).
__device__ inline int from_east(int v) { return __builtin_amdgcn_mov_dpp(v, 0x130 /* wave_shl:1 */, 0xf, 0xf, true); }
__device__ inline float from_east(float v) { return __builtin_bit_cast(float, from_east(__builtin_bit_cast(int, v))); }

// A double shifts as its two words.
__device__ inline double from_west(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)from_west((int)(uint32_t)u), hi = (uint32_t)from_west((int)(uint32_t)(u >> 32));
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}
__device__ inline double from_east(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)from_east((int)(uint32_t)u), hi = (uint32_t)from_east((int)(uint32_t)(u >> 32));
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

template <class T> struct WRow {
  T h, qx, qy, z;
  int ty;  // type slot, 0 for nodata or outside the domain
};

// Limited slopes of one cell along one axis (order 1 uses z only).
template <class T> struct WSlope {
  T h, qx, qy, z;
};

// One edge's two shares: mass, momentum across the edge axis, momentum along
// it with the side's bed term folded in.
template <class T> struct WPart {
  T m, across, along;
};

// The walk holds the pointers of the planes that every row touches in scalar
// registers (WalkPlanes) and reads the rest of the domain descriptor (boundary
// tables, infiltration, flux planes) through a KDesc that is laundered at
// every row, so that those fields are fetched where a row needs them: all of
// the descriptor held across the walk would spill, and all of it fetched again
// in every row put a dozen scalar-load round trips into each.

// Plane access: the row's element offset is the same for the whole wave (the
// base plus the row is scalar arithmetic), the lane's column a 32-bit offset
// from there.  The planes are device memory: the accesses name the global
// address space, so they compile to global loads and stores whatever memory
// the descriptor holding the base came from.
#define HP_GLOBAL __attribute__((address_space(1)))
// base + row as a scalar pointer; the empty asm keeps the row's offset from
// being added to the column's first, which would make every plane's address
// 64-bit vector arithmetic.
template <class V> __device__ inline HP_GLOBAL char* pl_row(const void* base, int64_t row) {
  HP_GLOBAL char* p = (HP_GLOBAL char*)base + row * (int64_t)sizeof(V);
  asm("" : "+s"(p));
  return p;
}
template <class V> __device__ inline V pl_ld(const void* base, int64_t row, uint32_t col) {
  return *(const HP_GLOBAL V*)(pl_row<V>(base, row) + col * (uint32_t)sizeof(V));
}
template <class V> __device__ inline void pl_st(void* base, int64_t row, uint32_t col, V v) {
  *(HP_GLOBAL V*)(pl_row<V>(base, row) + col * (uint32_t)sizeof(V)) = v;
}

// The lane's column, hidden from the compiler: its 64-bit extension is then
// made beside the access, where it folds into the address, instead of once
// for the kernel.  Called in the block that holds the accesses.
__device__ inline uint32_t pl_col(uint32_t cx) {
  asm volatile("" : "+v"(cx));
  return cx;
}

// The same value in every lane, kept in scalar registers.
__device__ inline int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ inline float uniform(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}
__device__ inline double uniform(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)uniform((int)(uint32_t)u), hi = (uint32_t)uniform((int)(uint32_t)(u >> 32));
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

// Values of a unit that are the same for the whole wave (scalar registers).
template <class T> struct WalkEnv {
  T dt_dx;
  T dx, dt;
  T cfl_dx;
  bool t_zero;   // t == 0: every valid cell is listed
  int n_rates;   // station rates in LDS (the table's stations at this t)
  T rate;        // the rate of every cell where no plane tells them apart
  int rain;      // 0 one rate for all, 1 by station, 2 by cell
  int c0y;       // row of compact cell 0, and all lanes but its own
  uint64_t c0_not;
  int rd, rw, rq;  // rows of the boundary series (depth, water level, discharge) at this t
  const T *s_rate, *s_man;  // LDS: station rates, Manning values by class
  int n_classes;
};

// The row of a boundary series in force at t (the first whose time is not
// before t, or the last), searched 64 rows at a time by the whole wave.
template <class T> __device__ inline int wave_series_row(const void* tab, int rows, int w, T t) {
  if (tab == nullptr || rows <= 1) return 0;
  const T* p = (const T*)tab;
  return wave_first(0, rows - 1, [&](int r) { return !(t > p[(int64_t)r * w]); });
}

// The boundary values of a cell with mask code `code`; only the value that
// the type's ghost uses is fetched.
template <class T, class DP> __device__ inline BcValues<T> walk_bc_values(const WalkEnv<T>& env, DP a, int code) {
  BcValues<T> b;
  int id;
  decode_code(code, b.type, id);
  b.gd = b.gwl = b.gqx = b.gqy = T(0);
  if (b.type == 6) b.gd = series_at<T>((const T*)a->given_depth, a->gd_rows, a->gd_w, env.rd, id + 1);
  if (b.type == 8) b.gwl = series_at<T>((const T*)a->given_wl, a->gwl_rows, a->gwl_w, env.rw, id + 1);
  if (b.type == 7) {
    b.gqx = series_at<T>((const T*)a->given_q, a->gq_rows, a->gq_w, env.rq, 1 + 2 * id);
    b.gqy = series_at<T>((const T*)a->given_q, a->gq_rows, a->gq_w, env.rq, 2 + 2 * id);
  }
  return b;
}

// The planes of every row, and the row geometry.
struct WalkPlanes {
  const void *type, *h, *qx, *qy, *z, *landuse, *h_max, *rain;
  void *h_out, *qx_out, *qy_out;
  int64_t pitch;
  int ny;
  template <class DP> __device__ WalkPlanes(DP a)
      : type(a->type_slot), h(a->h), qx(a->qx), qy(a->qy), z(a->z), landuse(a->landuse), h_max(a->h_max),
        rain(a->rain_mode == HP_RAIN_FIELD ? (const void*)a->rain_field : (const void*)a->station), h_out(a->h_out),
        qx_out(a->qx_out), qy_out(a->qy_out), pitch(a->pitch), ny(a->ny) {}
};

// Row gy of the lane's column (cx: the column, clamped into the plane).
// Rows and columns outside the domain get type 0; their other words are those
// of the nearest cell inside, which nothing reads.
template <class T> __device__ inline WRow<T> walk_load(const WalkPlanes& p, uint32_t cx, int gy, bool col_in) {
  WRow<T> w;
  const int y = gy < 0 ? 0 : (gy < p.ny ? gy : p.ny - 1);
  const int64_t row = (int64_t)y * p.pitch;
  cx = pl_col(cx);
  const int ty = pl_ld<uint8_t>(p.type, row, cx);
  w.h = pl_ld<T>(p.h, row, cx);
  w.qx = pl_ld<T>(p.qx, row, cx);
  w.qy = pl_ld<T>(p.qy, row, cx);
  w.z = pl_ld<T>(p.z, row, cx);
  w.ty = col_in && y == gy ? ty : 0;
  return w;
}

// A row's valid lanes and its wet ones (valid, depth above h_small).
struct WMask {
  uint64_t valid, wet;
};
template <class T> __device__ inline WMask walk_mask(const WRow<T>& w) {
  const uint64_t valid = __builtin_amdgcn_ballot_w64(w.ty != 0);
  return WMask{valid, valid & __builtin_amdgcn_ballot_w64(gt_hs(w.h))};
}
// Whether every lane is dry: no wet one, and none that is neither (a NaN).
template <class T> __device__ inline bool walk_dry(const WMask& m, T h) {
  return m.wet == 0 && __builtin_amdgcn_ballot_w64(!lt_hs(h)) == 0;
}
constexpr uint64_t kAllLanes = ~uint64_t(0);
// This lane's bit of a mask that is the same for the whole wave.
__device__ inline bool lane_of(uint64_t m) { return __builtin_amdgcn_inverse_ballot_w64(m); }

// minmod(c - l, r - c) with a nodata neighbour replaced by the cell itself
// (FULL: both neighbours are valid).
template <int ORDER, bool FULL, class T>
__device__ inline WSlope<T> walk_slope(const WRow<T>& c, const WRow<T>& l, const WRow<T>& r) {
  using P = Prec<T>;
  WSlope<T> s;
  const bool lv = either(FULL, l.ty != 0), rv = either(FULL, r.ty != 0);
  s.z = P::limit(c.z - (lv ? l.z : c.z), (rv ? r.z : c.z) - c.z);
  if (ORDER == 2) {
    s.h = P::limit(c.h - (lv ? l.h : c.h), (rv ? r.h : c.h) - c.h);
    s.qx = P::limit(c.qx - (lv ? l.qx : c.qx), (rv ? r.qx : c.qx) - c.qx);
    s.qy = P::limit(c.qy - (lv ? l.qy : c.qy), (rv ? r.qy : c.qy) - c.qy);
  } else {
    s.h = s.qx = s.qy = T(0);
  }
  return s;
}

// The edge between cells A and B (B east of A for D = 0, south for D = 3).
// eL / eR: A's and B's faces toward the edge in the edge frame, with z holding
// the half bed slope (A's face bed is z_A + eL.z, B's z_B - eR.z; order 1
// applies each only where the other side is wet).  Float works on A's datum
// (z_A = 0).  Returns A's and B's shares, zero between two dry cells.
// FULL: both cells are valid in every lane.  Otherwise a lane with one valid
// cell solves a boundary edge where `need` says that an owned cell reads it:
// the valid cell and its ghost (from the cell's mask code: codeA or codeB)
// take the two faces' places, in the frame of the cell's outward normal, and
// the solver runs once for all lanes.
template <int ORDER, int D, bool FULL, class T, class DP>
__device__ inline void walk_edge(const WalkEnv<T>& env, DP a, const WRow<T>& A, const WRow<T>& B, FrameCell<T> eL,
                                 FrameCell<T> eR, int codeA, int codeB, bool need, WPart<T>& pa, WPart<T>& pb) {
  const T g = T(kG);
  constexpr bool local = Prec<T>::local_datum;
  T zA = local ? T(0) : A.z;
  T zB = local ? B.z - A.z : B.z;
  const T zL = local ? eL.z : zA + eL.z, zR = zB - eR.z;
  if (ORDER == 1) {
    // bed faces only where the other side is wet (eL.z / eR.z hold the
    // half slopes on entry)
    eL.z = gt_hs(B.h) ? zL : zA;
    eR.z = gt_hs(A.h) ? zR : zB;
  } else {
    eL.z = zL;
    eR.z = zR;
  }
  T hA = A.h, hB = B.h;
  T etaC = local ? A.h : A.h + zA, etaR = B.h + zB;
  const bool vA = either(FULL, A.ty != 0), vB = either(FULL, B.ty != 0);
  const bool rim = both(need, vA != vB);
  // (order 2: a dry cell's faces carry no momentum; a ghost's and its cell's
  // are taken as they are)
  bool stillA = both(ORDER == 2, lt_hs(A.h)), stillB = both(ORDER == 2, lt_hs(B.h));
  if (!FULL && __builtin_amdgcn_ballot_w64(rim) != 0) {
    if (rim) {
      const int d = vA ? D : (D + 2) & 3;
      const T ch = vA ? A.h : B.h, cz = vA ? A.z : B.z, cqx = vA ? A.qx : B.qx, cqy = vA ? A.qy : B.qy;
      const T qn = D == 0 ? cqx : -cqy, qt = D == 0 ? cqy : cqx;
      const T zref = local ? cz : T(0);
      FrameCell<T> c;
      c.h = ch;
      c.qn = vA ? qn : -qn;
      c.qt = vA ? qt : -qt;
      c.z = local ? T(0) : cz;  // the valid cell's own datum in float
      const BcValues<T> bv = walk_bc_values<T>(env, a, vA ? codeA : codeB);
      const T gwl = bv.gwl - zref;
      const FrameCell<T> gh = bc_ghost<T>(bv.type, c, d, bv.gd, gwl, bv.gqx, bv.gqy);
      etaC = c.h + c.z;
      etaR = ORDER == 1 ? gh.h + gh.z : ghost_wl<T>(bv.type, etaC, gh, gwl);
      eL = c;
      eR = gh;
      hA = c.h;
      hB = gh.h;
      zA = c.z;
      stillA = stillB = false;
    }
  }
  const bool off = both(lt_hs(hA), lt_hs(hB));
  T fh, fn, ft;
  hllc_edge<T, ORDER>(eL, eR, etaC, etaR, fh, fn, ft, off, stillA, stillB);
  // raw fluxes: the cell scales its summed increments by dt / dx once
  const T bA = T(0.5) * g * (eL.h + hA), dzA = local && FULL ? eL.z : eL.z - zA;
  const T bB = T(0.5) * g * (eR.h + hB), dzB = eR.z - zB;
  constexpr T nA = D == 0 ? T(1) : T(-1);
  const T axis = D == 0 ? fn : -fn;
  T alongA = fma(nA * bA, dzA, axis), alongB = fma(nA * bB, dzB, axis), fhB = fh;
  if (!FULL) {
    // a boundary edge's bed term is that of its valid cell, whichever side
    const T rim_along = axis + nA * mul_alone(bA, dzA);
    alongA = rim ? rim_along : alongA;
    alongB = rim ? rim_along : alongB;
    fhB = rim ? -fh : fh;
    const bool on = either(both(vA, vB), rim);
    const bool onA = both(on, vA), onB = both(on, vB);
    pa = WPart<T>{onA ? fh : T(0), onA ? ft : T(0), both(onA, !off) ? alongA : T(0)};
    pb = WPart<T>{onB ? fhB : T(0), onB ? ft : T(0), both(onB, !off) ? alongB : T(0)};
  } else {
    pa = WPart<T>{fh, ft, off ? T(0) : alongA};
    pb = WPart<T>{fh, ft, off ? T(0) : alongB};
  }
}

// The faces of an edge frame from a cell, its slopes and the side (+1: the
// face toward increasing index along the axis, -1 the other).  D = 0: qn =
// qx, qt = qy; D = 3 (south): qn = -qy, qt = qx.  z carries the half slope.
template <int ORDER, int D, class T>
__device__ inline FrameCell<T> walk_face(const WRow<T>& c, const WSlope<T>& s, T side) {
  FrameCell<T> f;
  if (ORDER == 2) {
    f.h = fma(T(0.5) * side, s.h, c.h);
    const T fqx = fma(T(0.5) * side, s.qx, c.qx), fqy = fma(T(0.5) * side, s.qy, c.qy);
    f.qn = D == 0 ? fqx : -fqy;
    f.qt = D == 0 ? fqy : fqx;
  } else {
    f.h = c.h;
    f.qn = D == 0 ? c.qx : -c.qy;
    f.qt = D == 0 ? c.qy : c.qx;
  }
  f.z = T(0.5) * s.z;  // the half slope; walk_edge turns it into the face bed
  return f;
}

// Per-cell inputs of the update for the lane's cell of row gy; lanes that own
// no cell read the clamped column and are not used.  They are asked for a row
// ahead (past the last row, that row again: a load under a condition would be
// copied, and waited for, where the paths join), before the stores of the row
// in hand, so that waiting for them waits for nothing issued later.
template <class T> struct WalkIn {
  T hmax;
  int cls;  // landuse class
  int aux;  // the rain plane's word: a rate in m/s (float bits), or the station pair holding the cell's
};
template <class T>
__device__ inline WalkIn<T> walk_cell_in(const WalkEnv<T>& env, const WalkPlanes& p, uint32_t cx, int gy) {
  WalkIn<T> in;
  const int64_t row = (int64_t)(gy < p.ny ? gy : p.ny - 1) * p.pitch;
  cx = pl_col(cx);
  in.cls = pl_ld<uint8_t>(p.landuse, row, cx);
  in.hmax = pl_ld<T>(p.h_max, row, cx);
  in.aux = 0;
  // (planes are aligned to four elements and rows hold a multiple of four, so
  // the word of a station pair lies in the row)
  if (env.rain == 1) in.aux = *(const HP_GLOBAL int*)(pl_row<int16_t>(p.rain, row) + (cx & ~1u) * 2u);
  else if (env.rain == 2) in.aux = pl_ld<int>(p.rain, row, cx);
  return in;
}
// The rain rate of the cell in column cx from its word.
template <class T, class DP> __device__ inline T walk_rain(const WalkEnv<T>& env, DP a, const WalkIn<T>& in, uint32_t cx) {
  if (env.rain == 0) return env.rate;
  if (env.rain == 2) return T(__builtin_bit_cast(float, in.aux)) * T(a->rain_scale);
  const int st = cx & 1u ? in.aux >> 16 : (int)(int16_t)in.aux;
  return (st >= 0 && st < env.n_rates) ? env.s_rate[st] : T(0);
}

// Walk state carried from one row to the next.
template <class T> struct WalkCarry {
  WSlope<T> sy;          // y slopes of the row being finished
  WPart<T> north;     // its share of the edge with the row above
  WMask up, m, next;  // the row above, the row being finished, the next one
  T mn;               // CFL minimum so far
  double* sums;       // this lane's FP64 volume / flux / rain sums (LDS; with mass sums only)
};

// What a row's edges leave: the flux increments of the lane's cell (zero
// unless the flux rule lists it), and what the next row starts from.
template <class T> struct WalkFlux {
  T h, qx, qy;
  WSlope<T> sy;
  WPart<T> north;
};

template <class T> __device__ inline void walk_west(WRow<T>& w, const WRow<T>& c) {
  w.h = from_west(c.h); w.qx = from_west(c.qx); w.qy = from_west(c.qy); w.z = from_west(c.z);
}
template <class T> __device__ inline void walk_east(WRow<T>& e, const WRow<T>& c) {
  e.h = from_east(c.h); e.qx = from_east(c.qx); e.qy = from_east(c.qy); e.z = from_east(c.z);
}

// The cell's increments from its four shares, in the reference's order: E, N,
// W, S; scaled by dt / dx once (each product on its own, so that the update
// adds the same number whatever path it came by).
template <class T>
__device__ inline void walk_sum(const WalkEnv<T>& env, const WPart<T>& pe, const WPart<T>& pn, const WPart<T>& pw,
                                const WPart<T>& ps, WalkFlux<T>& o) {
  T ah = T(0), aqx = T(0), aqy = T(0);
  ah -= pe.m; aqx -= pe.along; aqy -= pe.across;
  ah += pn.m; aqx += pn.across; aqy += pn.along;
  ah += pw.m; aqx += pw.along; aqy += pw.across;
  ah -= ps.m; aqx -= ps.across; aqy -= ps.along;
  o.h = mul_alone(ah, env.dt_dx);
  o.qx = mul_alone(aqx, env.dt_dx);
  o.qy = mul_alone(aqy, env.dt_dx);
}

// The lanes of row gy that the flux rule lists (fluxMask): t == 0, wet, or a
// wet valid neighbour E, N, W, S that is not compact cell 0
// (fluxMaskGenerator_Kernel.cu:36).
template <class T>
__device__ inline uint64_t walk_listed(const WalkEnv<T>& env, const WMask& up, const WMask& m, const WMask& dn, int gy) {
  const int d = env.c0y - gy;
  const uint64_t n_up = up.wet & (d == -1 ? env.c0_not : kAllLanes), n_m = m.wet & (d == 0 ? env.c0_not : kAllLanes);
  const uint64_t n_dn = dn.wet & (d == 1 ? env.c0_not : kAllLanes);
  const uint64_t on = m.wet | (n_m << 1) | (n_m >> 1) | n_up | n_dn;
  return m.valid & (env.t_zero ? kAllLanes : on);
}

// The edges of row gy: `cur` is row gy, `nxt` gy + 1, `nw` gy + 2 (its mask
// m_nw).  FULL: every lane of the three rows is valid.
template <int ORDER, bool FULL, class T, class DP>
__device__ inline WalkFlux<T> walk_edges(const WalkEnv<T>& env, DP a, const WRow<T>& cur, const WRow<T>& nxt,
                                         const WRow<T>& nw, const WalkCarry<T>& k, uint64_t listed, bool own,
                                         bool need_x) {
  WalkFlux<T> o;
  // mask codes of the two rows, for boundary edges
  const int code = FULL ? 0 : a->slot_code[cur.ty], code_n = FULL ? 0 : a->slot_code[nxt.ty];
  // y slopes of the next row; the edge between this row and the next
  o.sy = walk_slope<ORDER, FULL>(nxt, cur, nw);
  WPart<T> ps{T(0), T(0), T(0)};
  o.north = ps;
  if (!(FULL && walk_dry(k.m, cur.h) && walk_dry(k.next, nxt.h)))
    walk_edge<ORDER, 3, FULL>(env, a, cur, nxt, walk_face<ORDER, 3>(cur, k.sy, T(1)),
                              walk_face<ORDER, 3>(nxt, o.sy, T(-1)), code, code_n, own, ps, o.north);
  WPart<T> pe{T(0), T(0), T(0)}, pw = pe;
  if (!(FULL && walk_dry(k.m, cur.h))) {
    // x neighbours by lane shifts, x slopes, the west edge of every lane
    WRow<T> w, e;
    walk_west(w, cur);
    walk_east(e, cur);
    if (!FULL) {
      w.ty = from_west(cur.ty);
      e.ty = from_east(cur.ty);
    }
    const WSlope<T> sx = walk_slope<ORDER, FULL>(cur, w, e);
    const FrameCell<T> east_face = walk_face<ORDER, 0>(cur, sx, T(1));
    FrameCell<T> eL;  // the west neighbour's east face
    eL.h = from_west(east_face.h);
    eL.qn = from_west(east_face.qn);
    eL.qt = from_west(east_face.qt);
    eL.z = from_west(east_face.z);
    WPart<T> pw_a;  // the west edge's shares: the west neighbour's (pw_a), this cell's (pw)
    walk_edge<ORDER, 0, FULL>(env, a, w, cur, eL, walk_face<ORDER, 0>(cur, sx, T(-1)), FULL ? 0 : from_west(code), code,
                              need_x, pw_a, pw);
    pe.m = from_east(pw_a.m);  // this cell's share of its east edge, solved by the east lane
    pe.across = from_east(pw_a.across);
    pe.along = from_east(pw_a.along);
  }
  walk_sum(env, pe, k.north, pw, ps, o);
  if (!FULL || listed != kAllLanes) {
    const bool on = lane_of(listed);
    o.h = on ? o.h : T(0);
    o.qx = on ? o.qx : T(0);
    o.qy = on ? o.qy : T(0);
  }
  return o;
}

// The time control a unit steps by (the same for the whole wave).
struct WalkClock {
  double t, dt;
  bool stopped, synced;
};
// From the domain's control block, which no launch of this kernel writes:
// constant memory, scalar loads.
__device__ inline WalkClock walk_clock(KCtrl c) {
  return WalkClock{c->t, c->dt, c->t_stop > 0.0 && c->t >= c->t_stop, c->stopped_synced != 0.0};
}
// Folded: the minima of the step before, advanced from its control block; the
// lead unit hands the result on and clears the slots of the next step.
template <class T> __device__ inline WalkClock walk_fold(const WalkFold& f, bool lead) {
  const int lane = (int)threadIdx.x;
  const KCtrl b = (KCtrl)&f.st->ring[(f.k + 1) & 1];
  StepCtrl e = StepCtrl::of(b);
  if (f.k > 0) {
    const uint64_t m = f.st->slots[(f.k + 2) % 3][lane];
    // (the minima of a float step are floats)
    e = next_ctrl_single_pass(e, (double)wave_min(T(__builtin_bit_cast(double, m))));
  }
  if (lead) {
    f.st->slots[(f.k + 1) % 3][lane] = kNoMinimum;
    if (lane == 0) {
      hp_ctrl* to = &f.st->ring[f.k & 1];
      e.put(to);
      to->export_T = e.export_T;
      to->t_stop = e.t_stop;
    }
  }
  return WalkClock{uniform(e.t), uniform(e.dt), uniform((int)e.stopped()) != 0, uniform((int)(e.synced != 0.0)) != 0};
}

// What a unit does besides the step itself (the same for the whole launch).
struct WalkMode {
  bool save_flux;     // also write the flux increments to dh, dqx, dqy
  bool time_control;  // CFL candidates and partial records
  bool sums;          // FP64 mass sums
};

// Finish row gy: `cur` is row gy, `nxt` gy + 1, `nw` gy + 2 (all loaded), wi
// its update inputs; `pre` receives row gy + 3, wi_next the inputs of gy + 1.
template <int ORDER, bool FUSED, class T, class DP>
__device__ __forceinline__ void walk_row(const WalkEnv<T>& env, DP a, const WalkPlanes& p, const WalkMode& mode,
                                         const WRow<T>& cur, const WRow<T>& nxt, const WRow<T>& nw, WRow<T>& pre,
                                         const WalkIn<T>& wi, WalkIn<T>& wi_next, WalkCarry<T>& k, uint32_t cx, int gy,
                                         bool own, bool need_x, bool col_in) {
  a = launder(a);
  if (FUSED) wi_next = walk_cell_in<T>(env, p, cx, gy + 1);
  pre = walk_load<T>(p, cx, gy + 3, col_in);

  const WMask m_nw = walk_mask(nw);
  const uint64_t listed = walk_listed(env, k.up, k.m, k.next, gy);
  WalkFlux<T> f;
  if ((k.m.valid & k.next.valid & m_nw.valid) == kAllLanes)
    f = walk_edges<ORDER, true>(env, a, cur, nxt, nw, k, listed, own, need_x);
  else f = walk_edges<ORDER, false>(env, a, cur, nxt, nw, k, listed, own, need_x);

  if (own) {
    const int64_t row = (int64_t)gy * p.pitch;
    if (!FUSED || mode.save_flux) {
      const uint32_t c = pl_col(cx);
      pl_st<T>(a->dh, row, c, f.h);
      pl_st<T>(a->dqx, row, c, f.qx);
      pl_st<T>(a->dqy, row, c, f.qy);
    }
    if (FUSED) {
      CellIn<T> in{walk_rain<T>(env, a, wi, cx), wi.hmax, env.s_man[min(wi.cls, env.n_classes - 1)], wi.cls,
                   wi.cls != 255};
      T hn = cur.h, qxn = cur.qx, qyn = cur.qy, hm = in.hmax;
      T dF = T(0);
      if (a->infil_ks && lane_of(listed)) {  // infiltration over the flux list (SWE_CUDA.py:439-443)
        const uint32_t c = pl_col(cx);
        const T F = pl_ld<T>(a->infil_F, row, c);
        dF = green_ampt<T>(hn, F, ((const T*)a->infil_ks)[in.cls], ((const T*)a->infil_phi)[in.cls],
                           ((const T*)a->infil_dtheta)[in.cls], env.dt);
        pl_st<T>(a->infil_F, row, c, F + dF);
      }
      T cand, vh, fh, rh;
      update_state<T>(in, hn, qxn, qyn, f.h, f.qx, f.qy, dF, env.dt, env.cfl_dx, hm, cand, vh, fh, rh,
                      mode.time_control);
      k.mn = Prec<T>::min2(k.mn, cand);
      if (mode.sums) {
        k.sums[0] += (double)vh;
        k.sums[kWalkLanes] += (double)fh;
        k.sums[2 * kWalkLanes] += (double)rh;
      }
      const uint32_t c = pl_col(cx);
      pl_st<T>(p.h_out, row, c, hn);
      pl_st<T>(p.qx_out, row, c, qxn);
      pl_st<T>(p.qy_out, row, c, qyn);
      if (hm != in.hmax) pl_st<T>((void*)p.h_max, row, pl_col(cx), hm);
    }
  }
  k.sy = f.sy;
  k.north = f.north;
  k.up = k.m;
  k.m = k.next;
  k.next = m_nw;
}

// The issue priority of a wave that has `left` of its unit's R rows to go.  A
// SIMD issues for the oldest of its waves first, so waves started together
// drift apart, and a launch ends with the youngest of each SIMD walking
// alone, at about 2 us a row where five together take 0.7 us for each.  In the
// units that no later unit will take over from, the waves with the most rows
// left go first, and a SIMD's waves finish together.  Units before those keep
// the top priority: they finish staggered, so that the prologues of the units
// taking over overlap with rows.  Measured per 2048^2 step in float, order 2,
// 15 rows a unit: 71 -> 59 us.
__device__ inline void walk_priority(int left, int R) {
  if (4 * left > 3 * R) __builtin_amdgcn_s_setprio(3);
  else if (2 * left > R) __builtin_amdgcn_s_setprio(2);
  else if (4 * left > R) __builtin_amdgcn_s_setprio(1);
  else __builtin_amdgcn_s_setprio(0);
}

// One unit: strip bx (columns [60 bx, 60 bx + 60)), rows [R by, R by + R).
// FUSED false: write the flux accumulators (flux pass).  FUSED true: finish
// the step into h_out / qx_out / qy_out with one partial record per unit
// (none without time control); save_flux also writes the flux; force_copy
// makes a stopped domain copy its state through even when marked in step.
// (inlined into each kernel: the launder needs the descriptor pointer known
// uniform, which a call shared by two kernels would not let the compiler see)
// fold: where the step's time control comes from and its minimum goes, when
// no launch of its own runs it (lead: the unit that carries the domain's
// control block on).  last: no unit takes over when this one is done.
template <class T, int ORDER, bool FUSED, class DP>
__device__ __forceinline__ void walk_unit(DP a, int bx, int by, int R, const Partials& part, int64_t pidx, bool save_flux,
                                          bool time_control, bool force_copy, const WalkFold& fold, bool lead,
                                          bool last) {
  __builtin_amdgcn_s_setprio(3);
  __shared__ T s_rate[FUSED ? kMaxStations : 1], s_man[FUSED ? 256 : 1];
  __shared__ double s_sums[FUSED ? 3 * kWalkLanes : 1];
  const int lane = (int)threadIdx.x;
  const int gx0 = bx * kWalkOwn - 2, gx = gx0 + lane;
  const bool col_in = gx >= 0 && gx < a->nx;
  const uint32_t cx = (uint32_t)(gx < 0 ? 0 : (gx < a->nx ? gx : a->nx - 1));
  const bool own = lane >= 2 && lane < 2 + kWalkOwn && gx < a->nx;
  // lanes whose west edge an owned cell reads: the owned ones and the lane
  // east of them (the last owned cell's east edge)
  const bool need_x = lane >= 2 && lane <= 2 + kWalkOwn && gx <= a->nx;
  const int y0 = by * R;
  // The unit's first rows y0 - 2 .. y0 + 1 are asked for before anything
  // else: the time control and the tables below take memory round trips of
  // their own meanwhile.
  const WalkPlanes p(a);
  WRow<T> A = walk_load<T>(p, cx, y0 - 2, col_in), B = walk_load<T>(p, cx, y0 - 1, col_in);
  WRow<T> C = walk_load<T>(p, cx, y0, col_in), D = walk_load<T>(p, cx, y0 + 1, col_in);
  // (the rain table's times too)
  const double rain_times = FUSED ? wave_rain_times(a) : 0.0;
  const bool folded = FUSED && fold.st != nullptr;
  const WalkClock clock = folded ? walk_fold<T>(fold, lead) : walk_clock((KCtrl)a->ctrl);
  if (clock.stopped) {
    if (FUSED) {
      if (lane == 0 && !folded) part.put(pidx, INFINITY, 0.0, 0.0, 0.0, a->mass_sums != 0);
      // (once the time control has marked the copy done, both sets of planes
      // hold the state)
      if (clock.synced && !force_copy) return;
      if (own) {
        for (int r = 0; r < R; ++r) {
          const int gy = y0 + r;
          if (gy >= a->ny) break;
          const int64_t row = (int64_t)gy * a->pitch;
          pl_st<T>(a->h_out, row, cx, pl_ld<T>(a->h, row, cx));
          pl_st<T>(a->qx_out, row, cx, pl_ld<T>(a->qx, row, cx));
          pl_st<T>(a->qy_out, row, cx, pl_ld<T>(a->qy, row, cx));
        }
      }
    }
    return;
  }
  const double t_now = clock.t;
  WalkEnv<T> env;
  env.dt = uniform(T(clock.dt));
  env.dx = uniform(T(a->dx));
  env.dt_dx = uniform(env.dt / env.dx);
  env.cfl_dx = uniform(T(a->cfl) * T(a->dx));
  env.t_zero = uniform((int)(T(t_now) == T(0))) != 0;
  env.rain = a->rain_mode == HP_RAIN_FIELD ? 2 : (a->rain_mode == HP_RAIN_STATION && a->station ? 1 : 0);
  const int c0 = a->cell0_x - gx0;
  env.c0y = a->cell0_y;
  env.c0_not = c0 >= 0 && c0 < kWalkLanes ? ~(uint64_t(1) << c0) : kAllLanes;
  WalkIn<T> I{}, J{};
  if (FUSED) I = walk_cell_in<T>(env, p, cx, y0);
  env.rd = wave_series_row<T>(a->given_depth, a->gd_rows, a->gd_w, T(t_now));
  env.rw = wave_series_row<T>(a->given_wl, a->gwl_rows, a->gwl_w, T(t_now));
  env.rq = wave_series_row<T>(a->given_q, a->gq_rows, a->gq_w, T(t_now));
  env.n_rates = 0;
  env.rate = T(0);
  env.n_classes = a->n_classes;
  env.s_rate = s_rate;
  env.s_man = s_man;
  if (FUSED) {
    for (int c = lane; c < env.n_classes; c += kWalkLanes) s_man[c] = ((const T*)a->manning)[c];
    if (a->rain_mode == HP_RAIN_STATION) {
      // the table's station rates at this step's t, in LDS (as many as the
      // table has stations, at most 1024, which the host enforces: a cell
      // naming another station, or any cell once the table has ended, gets
      // no rain, as station_rate gives); without a station plane every cell
      // takes station 0
      const RainRows rr = wave_rain_rows(a, t_now, rain_times);
      if (env.rain == 0) {
        env.rate = uniform(station_rate<T>(rr, 0, a->rain_scale));
      } else {
        env.n_rates = rr.zero ? 0 : min(rr.n_st, kMaxStations);
        for (int st = lane; st < env.n_rates; st += kWalkLanes) s_rate[st] = station_rate<T>(rr, st, a->rain_scale);
      }
    }
    __syncthreads();
  }
  const WalkMode mode{save_flux, time_control, time_control && a->mass_sums != 0};

  // prologue: the edge between rows y0 - 1 and y0
  WalkCarry<T> k;
  {
    const WSlope<T> sy_b = walk_slope<ORDER, false>(B, A, C);
    k.sy = walk_slope<ORDER, false>(C, B, D);
    WPart<T> unused;
    walk_edge<ORDER, 3, false>(env, a, B, C, walk_face<ORDER, 3>(B, sy_b, T(1)), walk_face<ORDER, 3>(C, k.sy, T(-1)),
                               a->slot_code[B.ty], a->slot_code[C.ty], own, unused, k.north);
  }
  k.up = walk_mask(B);
  k.m = walk_mask(C);
  k.next = walk_mask(D);
  k.mn = INFINITY;
  // the FP64 sums live in LDS, one column per lane, so they hold no
  // registers across the walk
  k.sums = s_sums + lane;
  if (FUSED && mode.sums) k.sums[0] = k.sums[kWalkLanes] = k.sums[2 * kWalkLanes] = 0.0;
  A = walk_load<T>(p, cx, y0 + 2, col_in);
  const int y_end = min(y0 + R, p.ny);
  for (int y = y0;; y += 4) {
    if (last) walk_priority(y_end - y, R);
    walk_row<ORDER, FUSED>(env, a, p, mode, C, D, A, B, I, J, k, cx, y, own, need_x, col_in);
    if (y + 1 >= y_end) break;
    if (last) walk_priority(y_end - y - 1, R);
    walk_row<ORDER, FUSED>(env, a, p, mode, D, A, B, C, J, I, k, cx, y + 1, own, need_x, col_in);
    if (y + 2 >= y_end) break;
    if (last) walk_priority(y_end - y - 2, R);
    walk_row<ORDER, FUSED>(env, a, p, mode, A, B, C, D, I, J, k, cx, y + 2, own, need_x, col_in);
    if (y + 3 >= y_end) break;
    if (last) walk_priority(y_end - y - 3, R);
    walk_row<ORDER, FUSED>(env, a, p, mode, B, C, D, A, J, I, k, cx, y + 3, own, need_x, col_in);
    if (y + 4 >= y_end) break;
  }
  if (FUSED && time_control) {
    const bool sums = mode.sums;
    const T mn = wave_min(k.mn);
    double vol = 0.0, fs = 0.0, rs = 0.0;
    if (sums) {
      vol = k.sums[0];
      fs = k.sums[kWalkLanes];
      rs = k.sums[2 * kWalkLanes];
    }
    if (sums) {
      vol = wave_sum(vol);
      fs = wave_sum(fs);
      rs = wave_sum(rs);
    }
    if (lane == 0) {
      if (folded) {
        // (another unit's minimum may land first: order does not matter)
        __hip_atomic_fetch_min(&fold.st->slots[fold.k % 3][pidx % kFoldSlots],
                               (unsigned long long)__builtin_bit_cast(uint64_t, (double)mn), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        if (sums) fold.records[pidx] = Sums{vol, fs, rs, 0.0};
      } else {
        part.put(pidx, (double)mn, vol, fs, rs, sums);
      }
    }
  }
}

// Waves per SIMD asked of the compiler (96 registers in float, 168 in double).
// Six in float (80 registers) spill a few to scratch memory, and each reload
// waits for every load in flight: 73.2 -> 76.5 us per 2048^2 step.
template <class T> constexpr int walk_waves() { return sizeof(T) == 4 ? 5 : 3; }
// Units in flight at once: 256 CUs of four SIMDs.
constexpr int kSimds = 1024;
template <class T> constexpr int walk_slots() { return kSimds * walk_waves<T>(); }

// The descriptor is the kernel's first argument: read it in place.
// flags: 1 also save the step's flux in dh, dqx, dqy; 2 no time-control
// outputs (a frozen schedule); 4 a stopped domain copies its state through
// even when marked in step.
// With fold.st set, the grid may begin with blocks that fold the FP64 sums of
// the step before (n_units: the blocks that walk); without it, with blocks
// that copy the gauge depths of the state the step starts from (a launch of
// its own for those cost a calibration step 3 us).
template <class T, int ORDER, bool FUSED>
__global__ __launch_bounds__(kWalkLanes, walk_waves<T>()) void k_walk(hp_grid_desc a, Divisor strips, int rows,
                                                                       int flags, int n_units, WalkFold fold,
                                                                       const Sums* prev, WalkGauges gauges) {
  const KDesc pa = kernarg_desc();
  const int extra = (int)gridDim.x - n_units;
  if (FUSED && (int)blockIdx.x < extra) {
    if (fold.st == nullptr) {
      const int i = (int)(blockIdx.x * kWalkLanes + threadIdx.x);
      if (i < gauges.n) ((T*)gauges.row)[i] = ((const T*)pa->h)[gauges.off[i]];
      return;
    }
    fold_sums_block(pa->ctrl, fold.st, fold.k, (int)blockIdx.x, prev, n_units, pa->dx);
    return;
  }
  const int unit = xcd_band((int)blockIdx.x - extra, n_units);
  const int by = strips.div(unit);
  walk_unit<T, ORDER, FUSED>(pa, unit - by * strips.n, by, rows, Partials(a.work, n_units), unit, (flags & 1) != 0,
                             (flags & 2) == 0, (flags & 4) != 0, fold, unit == 0,
                             (int)blockIdx.x - extra >= n_units - walk_slots<T>());
}

// Every unit of every domain of an ensemble; map[i] = (domain, unit), domain
// by domain, so a domain's partial records are one contiguous range
// (ranges[domain] = first, count).
// With fold.st set (one state per domain) the time control of every domain is
// folded, as in k_walk, and with prev set the grid begins with the sum blocks
// of every domain.
template <class T, int ORDER, bool FUSED>
__global__ __launch_bounds__(kWalkLanes, walk_waves<T>()) void k_walk_multi(const hp_grid_desc* __restrict__ doms,
                                                           const int2* __restrict__ map, void* parts, int n_total,
                                                           int rows, WalkFold fold, const Sums* prev,
                                                           const int2* __restrict__ ranges) {
  const int extra = (int)gridDim.x - n_total;
  if (FUSED && (int)blockIdx.x < extra) {
    const int d = (int)blockIdx.x / kFoldSumBlocks;
    const hp_grid_desc& g = doms[d];
    if (g.mass_sums)
      fold_sums_block(g.ctrl, fold.st + d, fold.k, (int)blockIdx.x - d * kFoldSumBlocks, prev + ranges[d].x,
                      ranges[d].y, g.dx);
    return;
  }
  const int slot = xcd_band((int)blockIdx.x - extra, n_total);
  // (the map entry is the same for the whole wave)
  const int dom = __builtin_amdgcn_readfirstlane(map[slot].x), unit = __builtin_amdgcn_readfirstlane(map[slot].y);
  // the descriptor array is read-only for the launch: read it as constant
  // memory, by scalar loads, as the single-domain kernel reads its argument
  const KDesc a = (KDesc)(doms + dom);
  const int nstrips = (a->nx + kWalkOwn - 1) / kWalkOwn;
  const int by = uniform(unit / nstrips);
  walk_unit<T, ORDER, FUSED>(a, unit - by * nstrips, by, rows, Partials(parts, n_total), slot, false, true, false,
                             WalkFold{fold.st ? fold.st + dom : nullptr, fold.k, fold.records}, unit == 0,
                             (int)blockIdx.x >= (int)gridDim.x - walk_slots<T>());
}

}  // namespace hp
