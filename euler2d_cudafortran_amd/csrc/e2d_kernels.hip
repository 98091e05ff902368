// gfx950 kernels of the euler2d hot path.
//
// Fused step (implementationVersion 0): one kernel per time step.  Each
// wavefront owns a strip of 64 consecutive columns (60 output columns and a
// 2-column halo each side) and marches upward through a segment of rows.  The
// y-neighbourhood of a cell stays in the lane's registers (rolling rows of
// primitive variables); x-neighbours come from adjacent lanes through
// cross-lane shuffles, so no LDS tile is needed.  Per cell the primitive
// variables, slopes and trace source terms are computed once; per face one
// Riemann problem is solved.  Ghost cells are produced on load from their
// interior source (make_boundaries, serial_ref/m_run.f90:561-648) and written
// back to the input buffer, so buffers end up exactly as the reference leaves
// them.  The update epilogue also folds the CFL rate of the new state into the
// running invDt of the next step (compute_dt, serial_ref/m_run.f90:248-312).
//
// Materialised steps (implementationVersion 1: primitive variables, slopes,
// face states and fluxes in HBM, cuf/m_HydroRun_gpu.cuf:393-418;
// implementationVersion 2: primitive variables and fluxes, :421-446; both with
// serial_ref arithmetic): boundaries (launched by the caller), then one kernel,
// the fused step's march with every stage stored as it is formed.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstdlib>

#include "e2d_adjoint.hpp"
#include "e2d_common.hpp"
#include "e2d_internal.hpp"
#include "e2d_numerics.hpp"

namespace e2d {

// ---------------------------------------------------------------------------
// fused step

// Columns of a wavefront's strip: lane l of strip s holds column
// s kOut + kFirst - kHalo + l, and the strip's own columns are those of the
// lanes kHalo .. 63 - kHalo.  The fused step: 60 columns from the first
// interior one, 2 halo columns each side.  With stages (STAGES != 0): 56
// columns from column 0, so that every row of 8-byte values that is stored
// begins and ends on a 64-byte boundary (of 4-byte ones, 224 bytes, every second
// strip's begins within a piece).  With partial 64-byte pieces at every strip's
// edge, and with stores that the caches keep, the stage arrays wrote at 3 TB/s;
// aligned and non-temporal, at 5 (version 1 in FP64 at 2048^2, per step: 570 us,
// aligned 530, both 385; now, with 2 wavefronts per SIMD, 340, in FP32 285).
template <int STAGES>
struct Strip {
  static constexpr int kHalo = STAGES ? 4 : 2, kOut = 64 - 2 * kHalo, kFirst = STAGES ? 0 : 2;
};
constexpr int kStripOut = Strip<0>::kOut;
// Independent wavefronts per workgroup of the step kernels (their
// wavefronts share nothing).  One per workgroup: measured on MI355X, the FP64
// step takes 196.0-197.2 us at 2048^2 against 197.9-198.6 with four, and
// 680.6-683.4 against 689.5-692.5 at 4096^2, with the same results; the float
// kernels time the same either way, eight is slower.
#ifndef E2D_WAVES_PER_BLOCK
#define E2D_WAVES_PER_BLOCK 1
#endif
constexpr int kWavesPerBlock = E2D_WAVES_PER_BLOCK;

// 1: the fused step takes the update's input rows from an LDS ring (0: loads
// them again from memory); 1: wavefronts that load only interior cells skip
// the boundary map (0: every load goes through it).  Both give the same bits.
#ifndef E2D_FUSED_UOLD_LDS
#define E2D_FUSED_UOLD_LDS 1
#endif
#ifndef E2D_FUSED_PLAIN
#define E2D_FUSED_PLAIN 1
#endif

// optional register cap for the fused kernel (minimum resident waves per SIMD)
#if defined(E2D_FUSED_MIN_WAVES) && E2D_FUSED_MIN_WAVES > 0
#define E2D_FUSED_ATTR __attribute__((amdgpu_waves_per_eu(E2D_FUSED_MIN_WAVES)))
#else
#define E2D_FUSED_ATTR
#endif

// An upper bound of a cell's CFL rate in binary32, to leave out the rates that
// cannot raise the running maximum: the maximum starts from the running invDt
// that the step read, so a cell whose bound lies below that needs no rate, and
// nearly every wavefront is left with none to form (a primitive conversion and
// a sound speed: 4 divisions and a root of the update type).  The bound's terms
// are those of cfl_rate; `slack` covers the cancellation of E / rho against the
// kinetic energy, kRateMargin the roundings (about 20 of 2^-24 in the bound,
// and cfl_rate's own in binary32).  Where the energy is below 2^-60 or the
// density above 2^60, which binary32 may hold as subnormal, zero or infinite,
// the rate is formed; a density below binary32's normal range makes the bound
// infinite or NaN, an infinite or NaN energy or momentum too, the comparison is
// then false, and the rate is formed.  10 steps at 2048^2 FP64 1823 ->
// 1778 us, 6 steps at 4096^2 mixed 2251 -> 2193, 3001 x 1537 fp32_native 641 -> 620
// (with their sums).
struct RateBound {
  float gg1, smallc2, smallr, inv_dx, inv_dy;  // gamma0 (gamma0 - 1), smallc^2
};
constexpr float kRateMargin = 1e-5f, kRateLeast = 0x1p-60f;
__device__ __forceinline__ float rate_limit_of(double invdt) {  // wave-uniform
  const float x = static_cast<float>(invdt) * (1.0f - kRateMargin);
  return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, x)));
}
template <class U>
__device__ __forceinline__ bool rate_below(const RateBound& b, const U u[4], float limit) {
  const float ir = __builtin_amdgcn_rcpf(__builtin_fmaxf(static_cast<float>(static_cast<double>(u[0])), b.smallr));
  const float vx = __builtin_fabsf(static_cast<float>(static_cast<double>(u[2]))) * ir;
  const float vy = __builtin_fabsf(static_cast<float>(static_cast<double>(u[3]))) * ir;
  const float energy = static_cast<float>(static_cast<double>(u[1]));
  const float e = energy * ir;
  const float kin = 0.5f * (vx * vx + vy * vy);
  const float slack = 2e-6f * (__builtin_fabsf(e) + kin);
  const float c = __builtin_amdgcn_sqrtf(b.gg1 * (__builtin_fmaxf(e - kin, 0.0f) + slack) + b.smallc2);
  return (energy >= kRateLeast) & (ir >= kRateLeast) & ((c + vx) * b.inv_dx + (c + vy) * b.inv_dy < limit);
}

template <class P>
struct StepArgs {
  Hydro<typename P::T> hT;
  Hydro<typename P::U> hU;
  Grid g;
  typename P::S* uin;   // read (interior, corners) and ghost write-back
  typename P::S* uout;  // interior written
  double* scal;
  int dt_from_device, slot_cur, track_dt, slot_next;
  double dt_host;
  RateBound rate;
  // Row segments, one per wavefront: items [0, nlong) are nsegs segments of
  // seg_rows rows per strip over rows [2, short_base); items [nlong, nitems)
  // are nshort segments of short_rows rows per strip over [short_base, ny + 2);
  // each range is numbered by tile_item.
  int nsegs, seg_rows, nlong;
  int nshort, short_rows, short_base, nitems;
  int chunk;  // items per chunk dealt to one XCD (see fused_segment)
  int nstrips, tile;  // items are numbered over tiles of `tile` adjacent strips (see tile_item)
  // Packed last strip: when the last strip has at most 12 (28) output columns
  // (8 or 24 with stages, whose halo is wider),
  // its wavefronts are split into groups of pk_w = 16 (32) lanes, each group on
  // its own segment of pk_rows rows, so the strip takes a quarter (half) of the
  // wavefronts.  Items [nlong - npk, nlong) are its wavefronts; segment k of the
  // strip covers rows [2 + k pk_rows, 2 + (k+1) pk_rows), the last one moved
  // back to end at ny + 2 (it overlaps its neighbour, whose rows it then
  // computes again with the same bits).  pk_w == 0: no packing; the last
  // strip's index is nstrips (the regular strips are 0 .. nstrips - 1).
  int pk_w, pk_rows, pk_nseg, npk;
};

// with the stage arrays of implementation versions 1 (all) and 2 (q, fx, fy)
template <class P>
struct StageArgs : StepArgs<P> {
  typename P::T *q, *dqx, *dqy, *qxm, *qxp, *qym, *qyp;
  typename P::U *fx, *fy;
};

// Item k of a tiled numbering of nstrips strips x nper segments each: tiles of
// `tile` adjacent strips (the last one narrower), numbered tile by tile and
// within a tile segment by segment, so that consecutive items are horizontal
// neighbours first.  tile == 1 is the strip-major order.
__device__ __forceinline__ void tile_item(int k, int nper, int nstrips, int tile, int& strip, int& seg) {
  const int span = tile * nper;
  const int tc = k / span;
  const int w = min(tile, nstrips - tc * tile);
  const int in = k - tc * span;
  seg = in / w;
  strip = tc * tile + (in - seg * w);
}

// Segment (strip, rows [j0, j1), below ny + 2 + kMore) of wavefront `wave` of block b; false for a
// wavefront without one.  Blocks go to the 8 XCDs round-robin (b % 8) and
// start in order on each.  The long segments are dealt to the XCDs in chunks
// of `chunk` consecutive items (vertical neighbours, which share rows, meet in
// one L2; every XCD gets a spread of the domain, so a region of costly
// segments does not load one XCD), then the short ones the same way: every XCD
// ends its share on short segments, which shortens the tail where the device
// runs out of wavefronts.
template <int kMore, class P>
__device__ __forceinline__ bool fused_segment(const StepArgs<P>& a, int b, int wave, int lane, int& strip, int& j0,
                                              int& j1, int& group_w) {
  int item;
  bool is_long;
  if (!dealt_item(b, wave, kWavesPerBlock, a.nlong, a.nitems, a.chunk, item, is_long)) return false;
  int seg;
  group_w = 64;
  if (is_long && item >= a.nlong - a.npk) {
    // a wavefront of the packed last strip: group lane / pk_w takes segment
    // (item - first) * (64 / pk_w) + group; a group past the last segment
    // repeats the last one
    group_w = a.pk_w;
    strip = a.nstrips;
    seg = min((item - (a.nlong - a.npk)) * (64 / a.pk_w) + lane / a.pk_w, a.pk_nseg - 1);
    j0 = 2 + seg * a.pk_rows;
    j1 = j0 + a.pk_rows;
    if (j1 > a.g.ny + 2 + kMore) {
      j1 = a.g.ny + 2 + kMore;
      j0 = j1 - a.pk_rows;
    }
    return true;
  }
  if (is_long) {
    tile_item(item, a.nsegs, a.nstrips, a.tile, strip, seg);
    j0 = 2 + seg * a.seg_rows;
    j1 = min(j0 + a.seg_rows, a.short_base);
  } else {
    tile_item(item, a.nshort, a.nstrips, a.tile, strip, seg);
    j0 = a.short_base + seg * a.short_rows;
    j1 = min(j0 + a.short_rows, a.g.ny + 2 + kMore);
  }
  return true;
}

// Loads of cell (ci, r) of the input, taken from its boundary source as
// stored (ghost cells are never read: every ghost maps to an interior cell,
// corners to themselves), so the loads of several rows can be in flight at
// once.  source_cell applies the reflection's sign flip when the values are
// used and writes ghost values back, so that the input buffer ends up as
// make_boundaries leaves it; doing that here, right after the loads, would
// make every load wait for its data.  plain (uniform over the wavefront):
// every cell the wavefront loads is interior, so the boundary map is skipped.
template <class P>
__device__ __forceinline__ void fetch_cell(const StepArgs<P>& a, int ci, int r, bool plain,
                                           typename P::S raw[4]) {
  if (plain) {
#pragma unroll
    for (int v = 0; v < 4; ++v) raw[v] = a.uin[at(a.g, ci, r, v)];
    return;
  }
  const Src s = ghost_source(a.g, ci, r);
#pragma unroll
  for (int v = 0; v < 4; ++v) raw[v] = a.uin[at(a.g, s.i, s.j, v)];
}

template <class P>
__device__ __forceinline__ void source_cell(const StepArgs<P>& a, int ci, bool col_ok, int r, bool plain,
                                            typename P::S raw[4]) {
  if (plain) return;
  const Src s = ghost_source(a.g, ci, r);
#pragma unroll
  for (int v = 0; v < 4; ++v) raw[v] = (v == s.flip) ? -raw[v] : raw[v];
  if (s.ghost && col_ok) {
#pragma unroll
    for (int v = 0; v < 4; ++v) a.uin[at(a.g, ci, r, v)] = raw[v];
  }
}

template <class P>
__device__ __forceinline__ typename P::T prim_of(const Hydro<typename P::T>& h, const typename P::S raw[4],
                                                 typename P::T q[4], typename P::T& irho) {
  using T = typename P::T;
  T u[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) u[v] = static_cast<T>(raw[v]);
  return cons_to_prim<T, typename P::M>(h, u, q, irho);
}
template <class P>
__device__ __forceinline__ typename P::T prim_of(const Hydro<typename P::T>& h, const typename P::S raw[4],
                                                 typename P::T q[4]) {
  typename P::T irho;
  return prim_of<P>(h, raw, q, irho);
}

// nothing in the step reads a stage array again: non-temporal
template <class X>
__device__ __forceinline__ void store_stage(X* a, const Grid& g, int i, int j, const X x[4]) {
#pragma unroll
  for (int v = 0; v < 4; ++v) __builtin_nontemporal_store(x[v], a + at(g, i, j, v));
}

// kMinmod: instantiated for slope_type == 1 (the benchmark's minmod), whose
// limiter has a short form (see cell_slopes) and needs no first-order select.
// STAGES 1, 2: implementation versions 1 and 2, which store their stage arrays
// on the way: q on every cell, slopes and face states on [1, size-2]^2, fx and
// fy on [2, size-2]^2.  The input's ghost cells are filled, so every cell is
// loaded as it is stored, and rows go one further than the update needs (the
// reference's arrays hold the fluxes of row ny+2).
template <class P, int SOLVER, bool kMinmod, int STAGES = 0, class Args>
__device__ __forceinline__ void step_fused_body(const Args& a) {
  using T = typename P::T;
  using U = typename P::U;
  using S = typename P::S;
  using M = typename P::M;

  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const Grid& g = a.g;
  int strip, j0, j1, group_w;
  constexpr int kMore = STAGES != 0 ? 1 : 0;
  if (!fused_segment<kMore, P>(a, blockIdx.x, wave, lane, strip, j0, j1, group_w)) return;  // whole wavefront: no barrier here
  // lanes per column group: 64, or 16 / 32 in the packed last strip, whose
  // groups march different rows (j0, j1 per lane, j1 - j0 the same for all)
  const int col = lane & (group_w - 1);
  using SG = Strip<STAGES>;
  const int ci = strip * SG::kOut + SG::kFirst - SG::kHalo + col;  // column of this lane
  const bool col_ok = ci < g.isize;
  const int cl = col_ok ? (STAGES != 0 ? max(ci, 0) : ci) : g.isize - 1;  // clamped column for loads
  const bool own = col >= SG::kHalo && col < group_w - SG::kHalo;
  const bool out_lane = own && ci <= g.nx + 1 && (STAGES == 0 || ci >= 2);
  // columns strip*60 .. strip*60+63 and rows j0-2 .. j1+1 all interior (never
  // in the packed strip, which holds the last columns)
#if E2D_FUSED_PLAIN
  const bool plain = STAGES != 0 || __builtin_amdgcn_readfirstlane(group_w == 64 && strip * kStripOut >= 2 &&
                                                    strip * kStripOut + 63 <= g.nx + 1 && j0 - 2 >= 2 &&
                                                    j1 + 1 <= g.ny + 1 ? 1 : 0) != 0;
#else
  const bool plain = STAGES != 0;
#endif
  // with stages: the columns whose q, slopes and face states, and fluxes this lane stores
  const bool q_lane = own && ci < g.isize;
  const bool slope_lane = own && ci >= 1 && ci <= g.nx + 2;
  const bool flux_lane = own && ci >= 2 && ci <= g.nx + 2;
  // iterations r = j0 - 1 .. j1 of the row loop, the same number on every lane
  const int n_it = __builtin_amdgcn_readfirstlane(j1 - j0 + 2);

  const Hydro<T>& h = a.hT;
  U rate_max = U(0);

  // the running invDt and the first three rows are all requested before any
  // of them is used, so their round trips overlap
  double invdt_cur = 0.0;
  if (a.dt_from_device) invdt_cur = invdt_part(a.scal, a.slot_cur);
  T qa[4], qb[4], qc[4];
  T irb, irc;  // 1/rho of rows r and r+1 as the primitive conversion forms it, for the trace
  S raw[4], raw_next[4], raw_b[4];
  fetch_cell<P>(a, cl, j0 - 2, plain, raw);
  fetch_cell<P>(a, cl, j0 - 1, plain, raw_b);
  fetch_cell<P>(a, cl, j0, plain, raw_next);
  source_cell<P>(a, cl, col_ok, j0 - 2, plain, raw);
  const T pa = prim_of<P>(h, raw, qa);
  source_cell<P>(a, cl, col_ok, j0 - 1, plain, raw_b);
  const T pb = prim_of<P>(h, raw_b, qb, irb);
  // bits 0, 1, 2: row r+1, r, r-1 holds a cell that takes the limiter's long form
  unsigned long_rows = 0;
  if constexpr (kMinmod) long_rows = (any_long_slope(pa) ? 2 : 0) + (any_long_slope(pb) ? 1 : 0);
  if constexpr (STAGES != 0) {
    if (j0 == 2 && q_lane) {
      store_stage(a.q, g, ci, 0, qa);
      store_stage(a.q, g, ci, 1, qb);
    }
  }

  // dt of this step (serial_ref/m_run.f90:308, 384-385)
  U dt;
  if (a.dt_from_device) {
    invdt_cur = invdt_reduce(invdt_cur);
    dt = a.hU.cfl / static_cast<U>(invdt_cur);
  } else {
    dt = static_cast<U>(a.dt_host);
  }
  const U dtdxU = dt / a.hU.dx;
  const U dtdyU = dt / a.hU.dy;
  const T dtdx = static_cast<T>(dtdxU);
  const T dtdy = static_cast<T>(dtdyU);
  const float rate_limit = rate_limit_of(invdt_cur);

  T ymax_prev[4];
  U fy_prev[4] = {U(0), U(0), U(0), U(0)}, fx_prev[4] = {U(0), U(0), U(0), U(0)};
  U fy_cur[4] = {U(0), U(0), U(0), U(0)}, fx_cur[4] = {U(0), U(0), U(0), U(0)};

#if E2D_FUSED_UOLD_LDS
  // The update of row r-1 adds to that row's input, loaded two iterations
  // earlier: each lane keeps its last three input rows in LDS (slot of row k:
  // k mod 3) instead of loading them again from memory, where the line may
  // have left L2 by then.  A lane reads only what it wrote itself.
  // (raw storage: S may have a constructor, which __shared__ does not allow)
  __shared__ __align__(16) unsigned char rows_in_mem[kWavesPerBlock * 3 * 4 * 64 * sizeof(S)];
  S* const rows_in = reinterpret_cast<S*>(rows_in_mem) + wave * (3 * 4 * 64);  // [slot][v][lane]
  int slot_w = 0;  // slot of row r+1; the next slot (mod 3) holds row r-1, written two iterations back
#endif
  // Variable 0 of row r+2 of the input and of row r-1 of the output in the
  // lane's clamped column cl (ci on every lane that stores), moved one row on
  // per iteration: no row-index product per access.
  const S* in_row = a.uin + at(g, cl, j0 + 1, 0);
  S* out_row = a.uout + at(g, cl, j0 - 2, 0);
  for (int it = 0; it < n_it; ++it, in_row += g.pitch, out_row += g.pitch) {
    const int r = j0 - 1 + it;
    // software pipeline: row r+1 was fetched one iteration ago; fetch row r+2
    // now, so its load is in flight during the Riemann solves
#pragma unroll
    for (int v = 0; v < 4; ++v) raw[v] = raw_next[v];
    if (it < n_it - 1) {  // r + 2 <= j1 + 1
      if constexpr (STAGES != 0) {
        // clamped to the last row there is, past which the results are not used
        fetch_cell<P>(a, cl, min(r + 2, g.jsize - 1), true, raw_next);
      } else if (plain) {
#pragma unroll
        for (int v = 0; v < 4; ++v) raw_next[v] = in_row[v * g.plane];
      } else {
        fetch_cell<P>(a, cl, r + 2, plain, raw_next);
      }
    }
    S uold[4];
    const bool do_update = it >= 2;  // r >= j0 + 1
#if !E2D_FUSED_UOLD_LDS
    if (do_update && out_lane) {
#pragma unroll
      for (int v = 0; v < 4; ++v) uold[v] = a.uin[at(g, ci, r - 1, v)];
    }
#endif
    source_cell<P>(a, cl, col_ok, r + 1, plain, raw);
#if E2D_FUSED_UOLD_LDS
    // row r+1 as stored (interior cells carry no reflection flip)
#pragma unroll
    for (int v = 0; v < 4; ++v) rows_in[(slot_w * 4 + v) * 64 + lane] = raw[v];
#endif
    const T pc = prim_of<P>(h, raw, qc, irc);
    if constexpr (kMinmod) long_rows = (long_rows << 1 | (any_long_slope(pc) ? 1 : 0)) & 7;
    if constexpr (STAGES != 0) {
      // row r+1 in [j0, j1), and the topmost row with the last segment
      if (q_lane && (it < n_it - 2 || (it == n_it - 2 && j1 == g.ny + 2 + kMore))) store_stage(a.q, g, ci, r + 1, qc);
    }

    // slopes and trace sources of row r
    T qxm[4], qxp[4], dqx[4], dqy[4], s[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      qxm[v] = from_left(qb[v]);
      qxp[v] = from_right(qb[v]);
    }
    if (kMinmod && __builtin_expect(long_rows != 0, 0))
      cell_slopes<kMinmod, true>(h, qb, qxp, qxm, qc, qa, dqx, dqy);
    else
      cell_slopes<kMinmod>(h, qb, qxp, qxm, qc, qa, dqx, dqy);
    trace_sources<T, M>(h, qb, dqx, dqy, s, irb);
    if constexpr (STAGES == 1) {
      if (slope_lane && ((it >= 1 && it < n_it - 1) || (it == 0 && j0 == 2))) {
        store_stage(a.dqx, g, ci, r, dqx);
        store_stage(a.dqy, g, ci, r, dqy);
        T f[4];
        face_state(h, qb, dqx, s, dtdx, true, f);
        store_stage(a.qxm, g, ci, r, f);
        face_state(h, qb, dqx, s, dtdx, false, f);
        store_stage(a.qxp, g, ci, r, f);
        face_state(h, qb, dqy, s, dtdy, true, f);
        store_stage(a.qym, g, ci, r, f);
        face_state(h, qb, dqy, s, dtdy, false, f);
        store_stage(a.qyp, g, ci, r, f);
      }
    }

    // y-face between rows r-1 and r
    if (it >= 1) {  // r >= j0
      T ymin[4], f[4];
      face_state(h, qb, dqy, s, dtdy, false, ymin);
      riemann_y<T, M, SOLVER>(h, ymax_prev, ymin, f);
#pragma unroll
      for (int v = 0; v < 4; ++v) fy_cur[v] = static_cast<U>(f[v]) * dtdyU;
      if constexpr (STAGES != 0) {
        if (it < n_it - 1 && flux_lane) store_stage(a.fy, g, ci, r, fy_cur);
      }
    }
    face_state(h, qb, dqy, s, dtdy, true, ymax_prev);

    // x-face between columns ci-1 and ci, row r
    if (it >= 1 && it < n_it - 1) {  // j0 <= r < j1
      T xmin[4], xmax[4], xl[4], gd[4], f[4];
      face_state(h, qb, dqx, s, dtdx, false, xmin);
      face_state(h, qb, dqx, s, dtdx, true, xmax);
#pragma unroll
      for (int v = 0; v < 4; ++v) xl[v] = from_left(xmax[v]);
      riemann<T, M, SOLVER>(h, xl, xmin, gd, f);
#pragma unroll
      for (int v = 0; v < 4; ++v) fx_cur[v] = static_cast<U>(f[v]) * dtdxU;
      if constexpr (STAGES != 0) {
        if (flux_lane) store_stage(a.fx, g, ci, r, fx_cur);
      }
    }

    // conservative update of row r-1 (updateHydro, serial_ref/m_run.f90:504-513)
    if (do_update) {
      U fxr[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) fxr[v] = from_right(fx_prev[v]);
      if (out_lane && (STAGES == 0 || r - 1 <= g.ny + 1)) {
        const int jr = r - 1;
#if E2D_FUSED_UOLD_LDS
        const int slot_r = slot_w == 2 ? 0 : slot_w + 1;  // slot of row r - 1
#pragma unroll
        for (int v = 0; v < 4; ++v) uold[v] = rows_in[(slot_r * 4 + v) * 64 + lane];
#endif
        U un[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const U flux_tot = (fy_prev[v] - fy_cur[v]) + (fx_prev[v] - fxr[v]);
          const S sn = static_cast<S>(static_cast<U>(uold[v]) + flux_tot);
          out_row[v * g.plane] = sn;
          un[v] = static_cast<U>(sn);
        }
        // CFL rate of the new state over the compute_dt window [2, n] (0-based)
        if (a.track_dt && ci <= g.nx && jr <= g.ny && !rate_below(a.rate, un, rate_limit)) {
          const U rate = cfl_rate<U, typename P::MU>(a.hU, un);
          rate_max = rate_max > rate ? rate_max : rate;
        }
      }
    }

#pragma unroll
    for (int v = 0; v < 4; ++v) {
      qa[v] = qb[v];
      qb[v] = qc[v];
      fy_prev[v] = fy_cur[v];
      fx_prev[v] = fx_cur[v];
    }
    irb = irc;
#if E2D_FUSED_UOLD_LDS
    slot_w = slot_w == 2 ? 0 : slot_w + 1;
#endif
  }

  if (a.track_dt) {
    double m = static_cast<double>(rate_max);
    m = m > invdt_cur ? m : invdt_cur;  // running maximum carries over
    m = wave_max(m);
    if (lane == 0) invdt_fold(a.scal, a.slot_next, static_cast<int>(blockIdx.x) * kWavesPerBlock + wave, m);
  }
}

// Resident wavefronts per SIMD the fused step is held at: 3 for FP64
// arithmetic (168 VGPRs), 5 for FP32 (102), 4 for the native-arithmetic
// variants (128), no cap for the tangent's dual numbers.  The packed last
// strip's per-lane rows cost registers the compiler would otherwise take
// (FP64 179, FP32 107: one wavefront fewer); held at these counts neither
// spills.
template <class P>
constexpr int fused_waves() {
  if constexpr (sizeof(typename P::T) > 8) return 1;
  else if constexpr (sizeof(typename P::T) == 8) return 3;
  else if constexpr (!std::is_same<typename P::M, FastMath>::value) return 5;
  else return 4;
}

template <class P, int SOLVER, bool kMinmod = false>
__global__ __launch_bounds__(64 * kWavesPerBlock) __attribute__((amdgpu_waves_per_eu(fused_waves<P>())))
E2D_FUSED_ATTR void k_step_fused(const StepArgs<P> a) {
  step_fused_body<P, SOLVER, kMinmod>(a);
}

// The HLLC step in its own kernel, held at 3 resident wavefronts per SIMD
// (168 VGPRs): left alone the FP64 instantiation takes 172 and drops to 2.
template <class P>
__global__ __launch_bounds__(64 * kWavesPerBlock) __attribute__((amdgpu_waves_per_eu(3))) void k_step_fused_hllc(
    const StepArgs<P> a) {
  step_fused_body<P, 2, false>(a);
}

// ---------------------------------------------------------------------------
// The fused step on tiles, for grids too small to fill the device with marching
// wavefronts (there a step lasts as long as one wavefront's chain of row
// iterations).  A workgroup takes a strip of 64 columns (60 stored) and R rows,
// one row a wavefront and R + 2 wavefronts, and its rows meet in LDS: each
// wavefront forms its row's primitives (the outer two also those of the rows
// beyond), then its slopes, face states and x-face problems, then the y-face
// problems below its row, with the row below's upper face states from LDS, then
// its update, with the y-flux above from LDS.  The chain is one row with two
// Riemann problems whatever R is.  It forms the marching kernel's values by the
// same routines on the same operands, so the bits are the same.
// Each wavefront holds one row only: 80 VGPRs in FP64 (6 wavefronts per SIMD,
// against the march's 3) and about 50 in the float variants.  us per FP64 step,
// march against tiles: 128^2 11.4, 8.4; 250 x 130 11.5, 8.7; 512^2 22.9, 20.5;
// 768^2 40.9, 36.4.  On grids that fill the device (2048^2: 157 against 208)
// the barriers and the rows formed twice cost more than the chain saves.
constexpr int kTileMaxRows = 14;
template <class P>
constexpr int tile_waves() {
  return sizeof(typename P::T) == 8 ? 6 : 8;
}
// rows of LDS (4 variables x 64 lanes of T) of a tile of R rows: primitives and
// the lower states, then fluxes, of the y-faces
constexpr int tile_lds_rows(int rows) { return (rows + 4) + (rows + 1); }

template <class P, bool kMinmod>
__global__ __launch_bounds__(64 * (kTileMaxRows + 2)) __attribute__((amdgpu_waves_per_eu(tile_waves<P>())))
void k_step_tile(const StepArgs<P> a) {
  using T = typename P::T;
  using U = typename P::U;
  using S = typename P::S;
  using M = typename P::M;
  extern __shared__ __align__(16) unsigned char tile_mem[];
  const Grid& g = a.g;
  const Hydro<T>& h = a.hT;
  const int R = a.seg_rows;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int lane = static_cast<int>(threadIdx.x & 63);
  const int lb = xcd_logical_block(blockIdx.x, gridDim.x);
  const int strip = lb / a.nsegs;
  const int j0 = 2 + (lb - strip * a.nsegs) * R;
  const int nr = min(R, g.ny + 2 - j0);  // this tile's rows [j0, j0 + nr)
  const int ci = strip * kStripOut + lane;
  const bool col_ok = ci < g.isize;
  const int cl = col_ok ? ci : g.isize - 1;
  const bool out_lane = lane >= 2 && lane < 62 && ci <= g.nx + 1;
  const int left = lane > 0 ? lane - 1 : 0, right = lane < 63 ? lane + 1 : 63;
  const int r = j0 - 1 + wave;  // the wavefront's row
  const bool has_row = wave < nr + 2, x_row = wave >= 1 && wave <= nr, y_face = wave >= 1 && wave <= nr + 1;
  const bool up_row = wave <= nr;
  const bool plain = strip * kStripOut >= 2 && strip * kStripOut + 63 <= g.nx + 1 && j0 >= 4 && j0 + nr <= g.ny;

  T* const q_lds = reinterpret_cast<T*>(tile_mem);  // row k: grid row j0 - 2 + k
  T* const y_lds = q_lds + (R + 4) * 256;           // y-face k, between rows j0-1+k and j0+k

  double invdt_cur = 0.0;
  if (a.dt_from_device) invdt_cur = invdt_part(a.scal, a.slot_cur);
  T q[4], irho;
  if (has_row) {
    S raw[4], raw2[4];
    const bool ends = wave == 0 || wave == nr + 1;
    const int r2 = wave == 0 ? r - 1 : r + 1;
    fetch_cell<P>(a, cl, r, plain, raw);
    if (ends) fetch_cell<P>(a, cl, r2, plain, raw2);
    source_cell<P>(a, cl, col_ok, r, plain, raw);
    prim_of<P>(h, raw, q, irho);
#pragma unroll
    for (int v = 0; v < 4; ++v) q_lds[((wave + 1) * 4 + v) * 64 + lane] = q[v];
    if (ends) {
      T q2[4];
      source_cell<P>(a, cl, col_ok, r2, plain, raw2);
      prim_of<P>(h, raw2, q2);
#pragma unroll
      for (int v = 0; v < 4; ++v) q_lds[((r2 - j0 + 2) * 4 + v) * 64 + lane] = q2[v];
    }
  }
  U dt;
  if (a.dt_from_device) {
    invdt_cur = invdt_reduce(invdt_cur);
    dt = a.hU.cfl / static_cast<U>(invdt_cur);
  } else {
    dt = static_cast<U>(a.dt_host);
  }
  const U dtdxU = dt / a.hU.dx;
  const U dtdyU = dt / a.hU.dy;
  const T dtdx = static_cast<T>(dtdxU);
  const T dtdy = static_cast<T>(dtdyU);
  __syncthreads();

  T ymin[4], fx[4] = {T(0), T(0), T(0), T(0)};
  S uold[4] = {S(0), S(0), S(0), S(0)};
  if (has_row) {
    T dqx[4], dqy[4], s[4];
    const T* const qr = q_lds + (wave + 1) * 256;
    auto slopes = [&](auto take_long) {
      T xm[4], xp[4], ym[4], yp[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        xm[v] = qr[v * 64 + left];
        xp[v] = qr[v * 64 + right];
        ym[v] = qr[v * 64 + lane - 256];
        yp[v] = qr[v * 64 + lane + 256];
      }
      cell_slopes<kMinmod, decltype(take_long)::value>(h, q, xp, xm, yp, ym, dqx, dqy);
    };
    if (kMinmod && __builtin_expect(any_long_slope(sizes_of_rows(qr + lane)), 0))
      slopes(std::true_type{});
    else
      slopes(std::false_type{});
    trace_sources<T, M>(h, q, dqx, dqy, s, irho);
    if (up_row) {
      T f[4];
      face_state(h, q, dqy, s, dtdy, true, f);
#pragma unroll
      for (int v = 0; v < 4; ++v) y_lds[(wave * 4 + v) * 64 + lane] = f[v];
    }
    face_state(h, q, dqy, s, dtdy, false, ymin);
    if (x_row) {
      T xl[4], xr[4], gd[4];
      face_state(h, q, dqx, s, dtdx, true, xl);
      face_state(h, q, dqx, s, dtdx, false, xr);
#pragma unroll
      for (int v = 0; v < 4; ++v) xl[v] = from_left(xl[v]);
      riemann<T, M, 0>(h, xl, xr, gd, fx);
    }
  }
  __syncthreads();
  T* const fy = y_lds + (wave - 1) * 256;  // y-face below the wavefront's row
  T fyl[4];
  if (y_face) {
    T lo[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) lo[v] = fy[v * 64 + lane];
    if (x_row && out_lane) {
#pragma unroll
      for (int v = 0; v < 4; ++v) uold[v] = a.uin[at(g, ci, r, v)];
    }
    riemann_y<T, M, 0>(h, lo, ymin, fyl);
#pragma unroll
    for (int v = 0; v < 4; ++v) fy[v * 64 + lane] = fyl[v];
  }
  __syncthreads();
  if (x_row) {
    U rate_max = U(0), un[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const U fxs = static_cast<U>(fx[v]) * dtdxU;
      const U flux_tot = (static_cast<U>(fyl[v]) * dtdyU - static_cast<U>(fy[v * 64 + lane + 256]) * dtdyU) +
                         (fxs - from_right(fxs));
      const S sn = static_cast<S>(static_cast<U>(uold[v]) + flux_tot);
      if (out_lane) a.uout[at(g, ci, r, v)] = sn;
      un[v] = static_cast<U>(sn);
    }
    if (a.track_dt) {
      if (out_lane && ci <= g.nx && r <= g.ny && !rate_below(a.rate, un, rate_limit_of(invdt_cur)))
        rate_max = cfl_rate<U, typename P::MU>(a.hU, un);
      double m = static_cast<double>(rate_max);
      m = m > invdt_cur ? m : invdt_cur;  // running maximum carries over
      m = wave_max(m);
      if (lane == 0) invdt_fold(a.scal, a.slot_next, static_cast<int>(blockIdx.x) * R + wave, m);
    }
  }
}

// The materialised versions' step (STAGES 1 and 2) on the same march.  As six
// and four kernels that passed q, slopes, face states and fluxes through HBM,
// version 1 moved 3.5 GB and version 2 1.4 GB per 2048^2 FP64 step, at the rate
// of a copy; here each stage is written once and read by nothing (1.58 GB and
// 0.79 GB): 756 -> 341 us and 356 -> 192 us per step.  Version 1 is bound by its
// writes (4.6 TB/s); in FP64 it is held at 2 wavefronts per SIMD, since at 3 it
// spills 60 B per lane (385 us).  Version 2 is bound by VALU issue, as the fused step.
template <class P, int STAGES>
constexpr int staged_waves() {
  return STAGES == 1 && sizeof(typename P::T) == 8 ? 2 : fused_waves<P>();
}
template <class P, int SOLVER, bool kMinmod, int STAGES>
__global__ __launch_bounds__(64 * kWavesPerBlock) __attribute__((amdgpu_waves_per_eu(staged_waves<P, STAGES>())))
void k_step_staged(const StageArgs<P> a) {
  step_fused_body<P, SOLVER, kMinmod, STAGES>(a);
}

static int env_int(const char* name, int dflt) {
  const char* v = getenv(name);
  return v && *v ? atoi(v) : dflt;
}

// Rows per long segment where the whole-round plan does not apply (small
// grids).  Each segment re-primes its rolling rows (two
// extra row loads and primitive conversions, one extra row of y-faces), so
// long segments are cheaper per row; short ones give more wavefronts to hide
// latency and balance the data-dependent Newton work, and on small grids a
// wavefront's rows are the critical path.  About ny/128 rows at 3 resident
// wavefronts per SIMD (the FP64 kernels), proportionally fewer where more are
// resident, within [1, 32]; E2D_FUSED_SEG_ROWS overrides it.  Measured on
// MI355X with long segments over 75% of the rows: 8 rows at 1024^2 (76 us per
// FP64 step against 86 us for uniform ny/170-row segments), 4 at 512^2 (29.6
// against 35.6).
static int fused_seg_rows(int ny, int waves_per_simd = 3) {
  const int r = env_int("E2D_FUSED_SEG_ROWS", 0);
  if (r >= 1) return r;
  const int d = static_cast<int>(ny / 128.0 * 3.0 / std::max(1, waves_per_simd) + 0.5);
  return d < 1 ? 1 : (d > 32 ? 32 : d);
}

// resident wavefronts per SIMD of a kernel launched with kWavesPerBlock waves per block
static int waves_per_simd(const void* kernel) {
  int blocks_per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks_per_cu, kernel, 64 * kWavesPerBlock, 0) !=
          hipSuccess ||
      blocks_per_cu <= 0)
    return 3;
  return std::max(1, blocks_per_cu * kWavesPerBlock / 4);
}

// Segment plan of a fused launch over ncols columns and ny rows.  Long segments cover
// about 80% (FP64) or 88% (FP32, mixed) of each strip's rows, in as many
// segments per strip as fill k whole rounds of the device's resident
// wavefronts (k the least that keeps them within 40 rows); short ones of a
// quarter of their length cover the rest.
// Every long segment then starts in the first k rounds, and what is left when
// they end is short work, so no long segment runs alone at the end of the
// launch.  Measured on MI355X (us per step, dt on the device): 2048^2 FP64
// 19-row long segments (one round) 213.5 against 223 with 16 rows over 75%
// (which leaves 9% of the long segments for a second round); FP32 12 rows
// 134-136 against 139-140; fp32_native 106.3 against 107.1; 4096^2 FP64 37 rows
// (two rounds) 711 against 716, 74 rows (one round) 719.  Where the rounds
// would give segments of fewer than 8 rows (grids up to about 1300^2 in FP64,
// 1600^2 in FP32) the plan is segments of one length in FP64 (below), and long
// segments of fused_seg_rows rows over 75% of the rows otherwise.
// E2D_FUSED_SEG_ROWS or E2D_FUSED_LONG_PCT select that plan with the given
// values, E2D_FUSED_SHORT_ROWS the short length; the environment is read at
// every launch.  Returns the number of blocks.
template <class SG, class P>
static int plan_segments(StepArgs<P>& a, int ncols, int ny, int wps, int resident) {
  const int nstrips_all = (ncols + SG::kOut - 1) / SG::kOut;
  // the packed last strip (see StepArgs): output columns left for it
  const int last_cols = ncols - SG::kOut * (nstrips_all - 1);
  int pk_w = 0;
  if (nstrips_all >= 2 && env_int("E2D_FUSED_PACK", 1) != 0)
    pk_w = last_cols <= 16 - 2 * SG::kHalo ? 16 : (last_cols <= 32 - 2 * SG::kHalo ? 32 : 0);
  const int nstrips = pk_w ? nstrips_all - 1 : nstrips_all;
  const int groups = pk_w ? 64 / pk_w : 1;  // segments per packed wavefront
  int R = 0, L = 0;
  const bool forced = env_int("E2D_FUSED_SEG_ROWS", 0) >= 1 || env_int("E2D_FUSED_LONG_PCT", -1) >= 0;
  if (!forced && resident >= nstrips) {
    // the long segments' share of the rows: 80% for the FP64 kernels (3
    // resident wavefronts per SIMD), 88% for the float-arithmetic ones (4-5):
    // measured at 2048^2, FP64 210-213 us at 80% against 214-218 at 76, 84 and
    // 88%; FP32 132.5 at 88% against 137 at 80%, fp32_native 104.5 against 107
    const int cover = env_int("E2D_FUSED_COVER_PCT", wps >= 4 ? 88 : 80);
    const double long_rows = std::min(100, std::max(10, cover)) / 100.0 * ny;
    // the packed wavefronts, each as long as a long segment, take their slots
    // out of the rounds first (a second pass once their number is known)
    int npk = 0;
    for (int pass = 0; pass < 2; ++pass) {
      auto per_strip = [&](int k) { return k * ((resident - (npk + k - 1) / k) / nstrips); };
      int k = 1;
      while (per_strip(k) >= 1 && long_rows / per_strip(k) > 40.0) ++k;
      L = per_strip(k);
      if (L < 1) {
        R = 0;
        break;
      }
      R = static_cast<int>(long_rows / L + 0.5);
      if (R < 8) R = 0;  // small grids: the percentage plan below
      while (R > 0 && L * R > ny) --R;
      if (R == 0 || !pk_w) break;
      const int pk = ((ny + R - 1) / R + groups - 1) / groups;
      if (pk == npk) break;
      npk = pk;
    }
  }
  // FP64 grids of about 700^2 (version 0 marches from 830^2) to 1300^2: segments
  // of one length, the least that lets all of them start at once.  us per step
  // against long segments over 75% of the rows: 850^2 42.2 against 50.8, 1024^2
  // 56.2 against 64.4, 1200^2 70.7 against 78.1, 1300^2 82.5 against 87.1 (the float
  // variants gain and lose 2%).  They lose where the other plan's wavefronts all
  // start at once too, on tall grids of about ten strips: 611 x 1294 49.5 against
  // 46.0, 629 x 2240 77.3 against 69.2.
  if (R == 0 && !forced && sizeof(typename P::T) == 8) {
    int rows = 1;
    auto wavefronts = [&](int r) {
      const int segs = (ny + r - 1) / r;
      return nstrips * static_cast<int64_t>(segs) + (pk_w ? (segs + groups - 1) / groups : 0);
    };
    while (rows < 40 && wavefronts(rows) > resident) ++rows;
    if (rows >= 4 && wavefronts(rows) <= resident) {
      R = rows;
      L = (ny + R - 1) / R;
    }
  }
  if (R == 0) {
    R = fused_seg_rows(ny, wps);
    const int pct = std::min(100, std::max(0, env_int("E2D_FUSED_LONG_PCT", 75)));
    L = pct >= 100 ? (ny + R - 1) / R : static_cast<int>(static_cast<int64_t>(ny) * pct / 100 / R);
  }
  const int r = std::max(1, env_int("E2D_FUSED_SHORT_ROWS", R / 4));
  const int covered = std::min(L * R, ny);
  a.seg_rows = R;
  a.nsegs = L;
  a.pk_w = pk_w;
  a.pk_rows = std::min(R, ny);
  a.pk_nseg = pk_w ? (ny + a.pk_rows - 1) / a.pk_rows : 0;
  a.npk = pk_w ? (a.pk_nseg + groups - 1) / groups : 0;
  a.nlong = nstrips * L + a.npk;
  a.short_base = 2 + covered;
  a.short_rows = r;
  a.nshort = covered < ny ? (ny - covered + r - 1) / r : 0;
  a.nitems = a.nlong + nstrips * a.nshort;
  a.chunk = std::max(1, env_int("E2D_FUSED_CHUNK", 16));
  a.nstrips = nstrips;
  a.tile = std::min(std::max(1, env_int("E2D_FUSED_TILE", 1)), std::max(1, nstrips));
  return dealt_blocks(a.nlong, a.nitems, a.chunk, kWavesPerBlock);
}

// Rows per tile, or 0 for the marching kernel.  Tiles up to 2,700 cells per
// compute unit in FP64 and 2,400 in the float variants (about 830^2 and 780^2),
// near which the two cross.  us per step, march against tiles: 640^2 FP64 34.5,
// 28.9; 770^2 42.4, 37.9; 831^2 42.3, 43.4; 850^2 42.2, 43.6; 1000 x 610 41.9, 38.7;
// 770^2 FP32 26.4, 24.7; 800^2 27.4, 27.5; 770^2 fp32_native 23.0, 21.0; 800^2 23.2,
// 24.1.  (Either may be 10% the quicker near the line, as whole rounds of tiles
// and of segments fall: 610 x 727 FP64 31.4, 37.3; 1200 x 520 mixed 25.6, 21.5.)
// Nor more than 100 rows of strips per compute unit: a strip of few columns costs
// a whole one in either kernel, and tall grids of them hold enough rows for the
// march (4 x 50000 FP64 145, 189; 4 x 25000 86, 100, where the march's plan is the
// worse one on most widths).  A step on tiles
// takes about as long as the wavefronts on the busiest compute unit, ceil(tiles
// / compute units) (R + 2), and longer by the root of the residency lost where
// they come in several rounds of tiles of R + 2 wavefronts that do not fill it
// (512^2 FP64: 10 rows 21.0, 6 rows 23.7; 927^2: 6 rows 50.2, 14 rows 53.1).
// The rows with the least of that are taken, among equals the fewest.
// E2D_TILE_ROWS gives the rows (0: march), and any E2D_FUSED_* plan selects the
// march it describes.
static int plan_tile_rows(const Grid& g, int waves_per_cu, int most_cells) {
  const int forced = env_int("E2D_TILE_ROWS", -1);
  if (forced >= 0) return std::min(forced, kTileMaxRows);
  const int cus = device_cus();
  if (static_cast<int64_t>(g.nx) * g.ny > static_cast<int64_t>(most_cells) * cus) return 0;
  for (const char* name : {"E2D_FUSED_SEG_ROWS", "E2D_FUSED_SHORT_ROWS", "E2D_FUSED_LONG_PCT", "E2D_FUSED_COVER_PCT",
                           "E2D_FUSED_CHUNK", "E2D_FUSED_TILE", "E2D_FUSED_PACK"})
    if (getenv(name)) return 0;
  const int64_t strips = (g.nx + kStripOut - 1) / kStripOut;
  if (strips * g.ny > 100 * static_cast<int64_t>(cus)) return 0;
  int best = 0;
  double least = 0.0;
  for (int rows = 1; rows <= kTileMaxRows; ++rows) {
    const int64_t tiles = strips * ((g.ny + rows - 1) / rows);
    const int64_t per_cu = (tiles + cus - 1) / cus;
    const int resident = std::max(1, waves_per_cu / (rows + 2));
    double cost = static_cast<double>(per_cu * (rows + 2)) * (per_cu * (rows + 2));
    if (per_cu > resident) cost *= static_cast<double>(waves_per_cu) / (resident * (rows + 2));
    if (best == 0 || cost < least) {
      best = rows;
      least = cost;
    }
  }
  return best;
}

template <class P, int SOLVER, bool kMinmod, int STAGES = 0, class Args>
static hipError_t launch_fused(Args& a, hipStream_t st) {
  if constexpr (SOLVER == 0 && STAGES == 0 && sizeof(typename P::T) <= 8) {
    const int rows = plan_tile_rows(a.g, 4 * tile_waves<P>(), sizeof(typename P::T) == 8 ? 2700 : 2400);
    if (rows > 0) {
      a.seg_rows = rows;
      a.nsegs = (a.g.ny + rows - 1) / rows;
      const int nstrips = (a.g.nx + kStripOut - 1) / kStripOut;
      hipLaunchKernelGGL((k_step_tile<P, kMinmod>), dim3(nstrips * a.nsegs), dim3(64 * (rows + 2)),
                         tile_lds_rows(rows) * 256 * sizeof(typename P::T), st, a);
      return hipGetLastError();
    }
  }
  void (*kernel)(const Args);
  if constexpr (STAGES != 0)
    kernel = k_step_staged<P, SOLVER, kMinmod, STAGES>;
  else if constexpr (SOLVER == 2)
    kernel = k_step_fused_hllc<P>;
  else
    kernel = k_step_fused<P, SOLVER, kMinmod>;
  thread_local const int wps = waves_per_simd(reinterpret_cast<const void*>(kernel));
  // with stages: every column, and the fluxes of row ny+2
  const int nblocks = plan_segments<Strip<STAGES>, P>(a, STAGES != 0 ? a.g.isize : a.g.nx,
                                                   STAGES != 0 ? a.g.ny + 1 : a.g.ny, wps, 4 * wps * device_cus());
  hipLaunchKernelGGL(kernel, dim3(nblocks), dim3(64 * kWavesPerBlock), 0, st, a);
  return hipGetLastError();
}

template <class P, int STAGES>
static hipError_t fused_step(const e2d_params& p, const DevBuffers& b, const StepCfg& c, hipStream_t st) {
  using T = typename P::T;
  using U = typename P::U;
  std::conditional_t<STAGES != 0, StageArgs<P>, StepArgs<P>> a{};
  a.hT = make_hydro<T>(p);
  a.hU = make_hydro<U>(p);
  a.g = make_grid(p, b);
  a.uin = static_cast<typename P::S*>(b.u[c.buf_in]);
  a.uout = static_cast<typename P::S*>(b.u[c.buf_out]);
  a.scal = b.scal;
  a.dt_from_device = c.dt_from_device ? 1 : 0;
  a.slot_cur = c.slot_cur;
  a.track_dt = c.track_dt ? 1 : 0;
  a.slot_next = c.slot_next;
  a.dt_host = c.dt_host;
  // (smallc^2 at least a normal binary32: the bound may only grow)
  a.rate = {static_cast<float>(p.gamma0 * (p.gamma0 - 1.0)), static_cast<float>(std::max(p.smallc * p.smallc, 1e-37)),
            static_cast<float>(p.smallr), static_cast<float>(p.nx), static_cast<float>(p.ny)};
  if constexpr (STAGES != 0) {
    a.q = static_cast<T*>(b.stage[E2D_STAGE_Q]);
    a.fx = static_cast<U*>(b.stage[E2D_STAGE_FX]);
    a.fy = static_cast<U*>(b.stage[E2D_STAGE_FY]);
    a.dqx = static_cast<T*>(b.stage[E2D_STAGE_DQX]);
    a.dqy = static_cast<T*>(b.stage[E2D_STAGE_DQY]);
    a.qxm = static_cast<T*>(b.stage[E2D_STAGE_QXM]);
    a.qxp = static_cast<T*>(b.stage[E2D_STAGE_QXP]);
    a.qym = static_cast<T*>(b.stage[E2D_STAGE_QYM]);
    a.qyp = static_cast<T*>(b.stage[E2D_STAGE_QYP]);
  }
  const bool hllc = p.riemann_solver == E2D_RIEMANN_HLLC;
  if (hllc) return launch_fused<P, 2, false, STAGES>(a, st);
  if (p.slope_type == 1) return launch_fused<P, 0, true, STAGES>(a, st);
  return launch_fused<P, 0, false, STAGES>(a, st);
}

hipError_t launch_fused_step(const e2d_params& p, const DevBuffers& b, const StepCfg& c, hipStream_t s) {
  return with_arithmetic(p, [&](auto pol) { return fused_step<decltype(pol), 0>(p, b, c, s); });
}

hipError_t launch_materialised_step(const e2d_params& p, const DevBuffers& b, const StepCfg& c, hipStream_t s) {
  // one kernel forms what the reference's three procedures do
  const TraceRange prim("convertToPrimitives");
  const TraceRange flux("computeAndStoreFluxes");
  const TraceRange update("updateHydro");
  return with_arithmetic(p, [&](auto pol) {
    using P = decltype(pol);
    return p.implementation_version == E2D_IMPL_FLUX_STORE ? fused_step<P, 2>(p, b, c, s) : fused_step<P, 1>(p, b, c, s);
  });
}

// ---------------------------------------------------------------------------
// tangent-linear step: the fused kernel on dual numbers (value = the forward
// step's state bit for bit, derivative = the tangent), dt frozen

using PDual = Prec<Dual, Dual, Dual, DualMath<RangedMath>, DualMath<RangedMath>>;

// (U, V) -> dual buffer; V enters on interior cells only (ghost directions
// follow from the interior through the boundary map, corners are constants)
__global__ __launch_bounds__(256) void k_pack_dual(const Grid g, const double* __restrict__ u,
                                                   const double* __restrict__ v, Dual* __restrict__ out) {
  const int i = blockIdx.x * 64 + (threadIdx.x & 63);
  const int j = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (i >= g.isize || j >= g.jsize) return;
  const bool interior = i >= 2 && i <= g.nx + 1 && j >= 2 && j <= g.ny + 1;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int64_t o = at(g, i, j, k);
    out[o] = Dual(u[o], interior ? v[o] : 0.0);
  }
}

__global__ __launch_bounds__(256) void k_unpack_dual(const Grid g, const Dual* __restrict__ in,
                                                     double* __restrict__ v) {
  const int i = blockIdx.x * 64 + (threadIdx.x & 63);
  const int j = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (i >= g.isize || j >= g.jsize) return;
  const bool interior = i >= 2 && i <= g.nx + 1 && j >= 2 && j <= g.ny + 1;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int64_t o = at(g, i, j, k);
    v[o] = interior ? in[o].d : 0.0;
  }
}

hipError_t launch_tangent_step(const e2d_params& p, const DevBuffers& b, int buf, double dt, const double* v_in,
                               double* v_out, void* dual_in, void* dual_out, hipStream_t st) {
  const Grid g = make_grid(p, b);
  const dim3 grid((g.isize + 63) / 64, (g.jsize + 3) / 4);
  hipLaunchKernelGGL(k_pack_dual, grid, dim3(256), 0, st, g, static_cast<const double*>(b.u[buf]), v_in,
                     static_cast<Dual*>(dual_in));
  StepArgs<PDual> a{};
  a.hT = make_hydro<Dual>(p);
  a.hU = a.hT;
  a.g = g;
  a.uin = static_cast<Dual*>(dual_in);
  a.uout = static_cast<Dual*>(dual_out);
  a.scal = b.scal;
  a.dt_from_device = 0;
  a.slot_cur = 0;
  a.track_dt = 0;
  a.slot_next = 1;
  a.dt_host = dt;
  if (hipError_t e = launch_fused<PDual, 0, false>(a, st)) return e;
  hipLaunchKernelGGL(k_unpack_dual, grid, dim3(256), 0, st, g, static_cast<const Dual*>(dual_out), v_out);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// boundaries (make_boundaries): one thread per non-corner ghost cell

template <class S>
__global__ __launch_bounds__(256) void k_boundaries(const Grid g, S* u) {
  const int nxg = 4 * g.ny;  // x-face ghosts: 2 columns each side, interior rows
  const int nyg = 4 * g.nx;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  int i, j;
  if (t < nxg) {
    const int k = t % 4;
    j = 2 + t / 4;
    i = (k < 2) ? k : g.nx + k;  // 0,1 | nx+2, nx+3
  } else if (t < nxg + nyg) {
    const int t2 = t - nxg;
    const int k = t2 % 4;
    i = 2 + t2 / 4;
    j = (k < 2) ? k : g.ny + k;
  } else {
    return;
  }
  const Src s = ghost_source(g, i, j);
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    S x = u[at(g, s.i, s.j, v)];
    if (v == s.flip) x = -x;
    u[at(g, i, j, v)] = x;
  }
}

template <class P>
static hipError_t boundaries(const e2d_params& p, const DevBuffers& b, int buf, hipStream_t st) {
  const Grid g = make_grid(p, b);
  const int n = 4 * (p.nx + p.ny);
  hipLaunchKernelGGL(k_boundaries<typename P::S>, dim3((n + 255) / 256), dim3(256), 0, st, g,
                     static_cast<typename P::S*>(b.u[buf]));
  return hipGetLastError();
}

hipError_t launch_boundaries(const e2d_params& p, const DevBuffers& b, int buf, hipStream_t s) {
  const TraceRange range("make_boundaries");
  return with_precision(p.precision, [&](auto pol) { return boundaries<decltype(pol)>(p, b, buf, s); });
}

// one wavefront: thread t is variable t / 16 of corner cell t % 16
template <class S>
__global__ __launch_bounds__(64) void k_copy_corners(const Grid g, const S* __restrict__ from, S* __restrict__ to) {
  const int t = threadIdx.x;
  const int x = t & 3, y = (t >> 2) & 3;
  const int64_t o = at(g, x < 2 ? x : g.nx + x, y < 2 ? y : g.ny + y, t >> 4);
  to[o] = from[o];
}

hipError_t launch_copy_corners(const e2d_params& p, const DevBuffers& b, hipStream_t s) {
  return with_precision(p.precision, [&](auto pol) {
    using S = typename decltype(pol)::S;
    hipLaunchKernelGGL(k_copy_corners<S>, dim3(1), dim3(64), 0, s, make_grid(p, b), static_cast<const S*>(b.u[0]),
                       static_cast<S*>(b.u[1]));
    return hipGetLastError();
  });
}

// ---------------------------------------------------------------------------
// compute_dt reduction: max CFL rate over [2, nx] x [2, ny] (0-based)

template <class P>
__global__ __launch_bounds__(256) void k_max_invdt(const Hydro<typename P::U> h, const Grid g,
                                                    const typename P::S* __restrict__ u, double* scal, int slot,
                                                    double* per_block) {
  using U = typename P::U;
  __shared__ double red[4];
  const int w = g.nx - 1, hgt = g.ny - 1;  // window extent
  const int64_t n = static_cast<int64_t>(w) * hgt;
  U m = U(0);
  for (int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; t < n;
       t += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int i = 2 + static_cast<int>(t % w);
    const int j = 2 + static_cast<int>(t / w);
    U c[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) c[v] = static_cast<U>(u[at(g, i, j, v)]);
    const U r = cfl_rate<U, typename P::MU>(h, c);
    m = m > r ? m : r;
  }
  double md = wave_max(static_cast<double>(m));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = md;
  __syncthreads();
  if (threadIdx.x == 0) {
    double x = red[0];
    for (int k = 1; k < 4; ++k) x = x > red[k] ? x : red[k];
    if (per_block)
      per_block[blockIdx.x] = x;
    else
      invdt_fold(scal, slot, blockIdx.x, x);
  }
}

template <class P>
static hipError_t max_invdt(const e2d_params& p, const DevBuffers& b, int buf, int slot, double* per_block,
                            int* nblocks, hipStream_t st) {
  const Grid g = make_grid(p, b);
  const int64_t n = static_cast<int64_t>(p.nx - 1) * (p.ny - 1);
  int nb = static_cast<int>((n + 255) / 256);
  if (nb > kMaxInvdtBlocks) nb = kMaxInvdtBlocks;
  if (nb < 1) nb = 1;
  hipLaunchKernelGGL(k_max_invdt<P>, dim3(nb), dim3(256), 0, st, make_hydro<typename P::U>(p), g,
                     static_cast<const typename P::S*>(b.u[buf]), b.scal, slot, per_block);
  if (nblocks) *nblocks = nb;
  return hipGetLastError();
}

hipError_t launch_max_invdt(const e2d_params& p, const DevBuffers& b, int buf, int slot, hipStream_t s) {
  return with_arithmetic(p,
                         [&](auto pol) { return max_invdt<decltype(pol)>(p, b, buf, slot, nullptr, nullptr, s); });
}

hipError_t launch_block_invdt(const e2d_params& p, const DevBuffers& b, int buf, double* out, int* nblocks,
                              hipStream_t s) {
  return with_arithmetic(p, [&](auto pol) { return max_invdt<decltype(pol)>(p, b, buf, 0, out, nblocks, s); });
}

__global__ void k_fill(double* dst, int n, double v) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) dst[t] = v;
}

hipError_t launch_fill(double* dst, int n, double v, hipStream_t s) {
  hipLaunchKernelGGL(k_fill, dim3((n + 63) / 64), dim3(64), 0, s, dst, n, v);
  return hipGetLastError();
}

__global__ void k_start_slots(double* scal, const double* src, double v) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < kInvdtSlot) scal[t] = src ? *src : v;
  else if (t < 2 * kInvdtSlot) scal[t] = 0.0;
}

hipError_t launch_start_slots(double* scal, const double* src, double v, hipStream_t s) {
  hipLaunchKernelGGL(k_start_slots, dim3(2 * kInvdtSlot / 256), dim3(256), 0, s, scal, src, v);
  return hipGetLastError();
}

// one wavefront: *dst = the value of the running-invDt slot at `slot` (the maximum of its parts)
__global__ __launch_bounds__(64) void k_slot_value(const double* slot, double* dst) {
  const double v = invdt_read_wave(slot, 0);
  if (threadIdx.x == 0) *dst = v;
}

hipError_t launch_slot_value(const double* slot, double* dst, hipStream_t s) {
  hipLaunchKernelGGL(k_slot_value, dim3(1), dim3(64), 0, s, slot, dst);
  return hipGetLastError();
}

// *flag = 1 when two device arrays of n 64-bit words differ in any bit
__global__ void k_words_differ(const unsigned long long* a, const unsigned long long* b, int64_t n, double* flag) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; t < n; t += stride)
    if (a[t] != b[t]) *flag = 1.0;
}

hipError_t launch_words_differ(const void* a, const void* b, size_t bytes, double* flag, hipStream_t s) {
  hipError_t e = launch_fill(flag, 1, 0.0, s);
  if (e != hipSuccess) return e;
  const int64_t n = static_cast<int64_t>(bytes / sizeof(unsigned long long));
  const int64_t blocks = (n + 255) / 256;
  hipLaunchKernelGGL(k_words_differ, dim3(static_cast<unsigned>(blocks < 4096 ? (blocks > 0 ? blocks : 1) : 4096)),
                     dim3(256), 0, s, static_cast<const unsigned long long*>(a),
                     static_cast<const unsigned long long*>(b), n, flag);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// initial conditions (init_implode, serial_ref/m_run.f90:524-555; diag; bumps)

struct Bumps {
  double v[16 * 5];  // cx, cy, amp_rho, amp_p, sigma
};

template <class P>
__global__ __launch_bounds__(256) void k_init(const Grid g, typename P::S* u, typename P::S* u2,
                                              int problem, typename P::U gamma0, Bumps bumps) {
  using U = typename P::U;
  using S = typename P::S;
  const int i = blockIdx.x * 64 + (threadIdx.x & 63);
  const int j = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (i >= g.isize || j >= g.jsize) return;
  U rho, e;
  if (problem == E2D_PROBLEM_IMPLODE) {
    // tmp in default real (FP32) whatever the run's precision
    const float tmp = 1.0f * static_cast<float>(i - 2) / static_cast<float>(g.nx) +
                      1.0f * static_cast<float>(j - 2) / static_cast<float>(g.ny);
    if (static_cast<U>(tmp) > U(0.5)) {
      rho = U(1.0);
      e = U(1.0) / (gamma0 - U(1.0));
    } else {
      rho = U(0.125);
      e = static_cast<U>(0.14f) / (gamma0 - U(1.0));
    }
  } else {
    const U x = static_cast<U>(i - 2) / static_cast<U>(g.nx);
    const U y = static_cast<U>(j - 2) / static_cast<U>(g.ny);
    U pr;
    if (x + y < U(1)) {
      rho = U(1);
      pr = U(1);
    } else {
      rho = U(0.125);
      pr = U(0.1);
    }
    if (problem == E2D_PROBLEM_BUMPS) {
      const double xc = (static_cast<double>(i - 2) + 0.5) / g.nx;
      const double yc = (static_cast<double>(j - 2) + 0.5) / g.ny;
      double dr = 0.0, dp = 0.0;
      for (int k = 0; k < 16; ++k) {
        const double* bk = bumps.v + 5 * k;
        const double ddx = xc - bk[0], ddy = yc - bk[1], sg = bk[4];
        const double w = exp(-(ddx * ddx + ddy * ddy) / (2.0 * sg * sg));
        dr += bk[2] * w;
        dp += bk[3] * w;
      }
      rho = rho + static_cast<U>(dr);
      pr = pr + static_cast<U>(dp);
    }
    e = pr / (gamma0 - U(1));
  }
  const S vals[4] = {static_cast<S>(rho), static_cast<S>(e), S(0), S(0)};
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    u[at(g, i, j, v)] = vals[v];
    u2[at(g, i, j, v)] = S(0);
  }
}

template <class P>
static hipError_t init_problem(const e2d_params& p, const DevBuffers& b, int problem, const double* bumps,
                               hipStream_t st) {
  const Grid g = make_grid(p, b);
  Bumps bb{};
  if (bumps)
    for (int k = 0; k < 16 * 5; ++k) bb.v[k] = bumps[k];
  hipLaunchKernelGGL(k_init<P>, dim3((g.isize + 63) / 64, (g.jsize + 3) / 4), dim3(256), 0, st, g,
                     static_cast<typename P::S*>(b.u[0]), static_cast<typename P::S*>(b.u[1]), problem,
                     static_cast<typename P::U>(p.gamma0), bb);
  return hipGetLastError();
}

hipError_t launch_init_problem(const e2d_params& p, const DevBuffers& b, int problem, const double* bumps,
                               hipStream_t s) {
  return with_precision(p.precision,
                        [&](auto pol) { return init_problem<decltype(pol)>(p, b, problem, bumps, s); });
}

template <class S>
__global__ __launch_bounds__(256) void k_zero(const Grid g, S* u) {
  const int i = blockIdx.x * 64 + (threadIdx.x & 63);
  const int j = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (i >= g.isize || j >= g.jsize) return;
#pragma unroll
  for (int v = 0; v < 4; ++v) u[at(g, i, j, v)] = S(0);
}

hipError_t launch_zero_state(const e2d_params& p, const DevBuffers& b, int buf, hipStream_t s) {
  const Grid g = make_grid(p, b);
  const dim3 grid((g.isize + 63) / 64, (g.jsize + 3) / 4);
  if (state_elem_bytes(p.precision) == 8)
    hipLaunchKernelGGL(k_zero<double>, grid, dim3(256), 0, s, g, static_cast<double*>(b.u[buf]));
  else
    hipLaunchKernelGGL(k_zero<float>, grid, dim3(256), 0, s, g, static_cast<float*>(b.u[buf]));
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// deterministic FP64 sums over the interior: block k reduces rows k, k+B, ...
// in a fixed order, then one block adds the partials in block order.  Bound by
// the memory's latency: a thread adds its values one by one, so it loads
// kSumAhead of them (times 4 variables) before it adds the first, of one row or
// of several (960 wavefronts with 4 loads in flight each read 134 MB in 34 us and
// 537 MB in 186; with 32 in flight, 22 and 119), and the partials pass through
// LDS (added from memory one by one they took 30 us, now 4).  The order of the
// additions is the same.
constexpr int kSumAhead = 8;

template <class S>
__global__ __launch_bounds__(256) void k_sums_partial(const Grid g, const S* __restrict__ u, double* partial) {
  __shared__ double red[4][256];
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  const int tid = static_cast<int>(threadIdx.x);
  int j = 2 + static_cast<int>(blockIdx.x), i0 = 0;  // the row and the column (from the first interior one) of thread 0
  while (j <= g.ny + 1) {
    S x[kSumAhead][4];
#pragma unroll
    for (int k = 0; k < kSumAhead; ++k) {
#pragma unroll
      for (int v = 0; v < 4; ++v) x[k][v] = S(0);
      if (j <= g.ny + 1) {  // uniform, as the address of the row
        const S* const row = u + static_cast<int64_t>(j) * g.pitch + (2 + i0);
        if (i0 + tid < g.nx) {
#pragma unroll
          for (int v = 0; v < 4; ++v) x[k][v] = row[v * g.plane + tid];
        }
        i0 += 256;
        if (i0 >= g.nx) {
          i0 = 0;
          j += static_cast<int>(gridDim.x);
        }
      }
    }
    // a zero in the place of a column past the last leaves a sum as it is (no sum is -0)
#pragma unroll
    for (int k = 0; k < kSumAhead; ++k)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[v] += static_cast<double>(x[k][v]);
  }
#pragma unroll
  for (int v = 0; v < 4; ++v) red[v][threadIdx.x] = acc[v];
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w)
#pragma unroll
      for (int v = 0; v < 4; ++v) red[v][threadIdx.x] += red[v][threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x < 4) partial[blockIdx.x * 4 + threadIdx.x] = red[threadIdx.x][0];
}

__global__ __launch_bounds__(256) void k_sums_final(const double* partial, double* out) {
  __shared__ double p[kSumBlocks * 4];
  for (int t = threadIdx.x; t < kSumBlocks * 4; t += 256) p[t] = partial[t];
  __syncthreads();
  if (threadIdx.x < 4) {
    double s = 0.0;
#pragma unroll 16
    for (int k = 0; k < kSumBlocks; ++k) s += p[k * 4 + threadIdx.x];
    out[threadIdx.x] = s;
  }
}

hipError_t launch_sums(const e2d_params& p, const DevBuffers& b, int buf, double* out4, hipStream_t s) {
  const Grid g = make_grid(p, b);
  if (state_elem_bytes(p.precision) == 8)
    hipLaunchKernelGGL(k_sums_partial<double>, dim3(kSumBlocks), dim3(256), 0, s, g,
                       static_cast<const double*>(b.u[buf]), b.partial);
  else
    hipLaunchKernelGGL(k_sums_partial<float>, dim3(kSumBlocks), dim3(256), 0, s, g,
                       static_cast<const float*>(b.u[buf]), b.partial);
  hipLaunchKernelGGL(k_sums_final, dim3(1), dim3(256), 0, s, b.partial, out4);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// host layout <-> pitched device layout

template <class S>
__global__ __launch_bounds__(256) void k_pack(const Grid g, const double* __restrict__ src, S* dst) {
  const int i = blockIdx.x * 64 + (threadIdx.x & 63);
  const int j = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (i >= g.isize || j >= g.jsize) return;
  const int64_t hp = static_cast<int64_t>(g.isize) * g.jsize;
#pragma unroll
  for (int v = 0; v < 4; ++v)
    dst[at(g, i, j, v)] = static_cast<S>(src[v * hp + static_cast<int64_t>(j) * g.isize + i]);
}

template <class S>
__global__ __launch_bounds__(256) void k_unpack(const Grid g, const S* __restrict__ src, double* dst) {
  const int i = blockIdx.x * 64 + (threadIdx.x & 63);
  const int j = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (i >= g.isize || j >= g.jsize) return;
  const int64_t hp = static_cast<int64_t>(g.isize) * g.jsize;
#pragma unroll
  for (int v = 0; v < 4; ++v)
    dst[v * hp + static_cast<int64_t>(j) * g.isize + i] = static_cast<double>(src[at(g, i, j, v)]);
}

hipError_t launch_pack(const e2d_params& p, const DevBuffers& b, int buf, const double* d_src, hipStream_t s) {
  const Grid g = make_grid(p, b);
  const dim3 grid((g.isize + 63) / 64, (g.jsize + 3) / 4);
  if (state_elem_bytes(p.precision) == 8)
    hipLaunchKernelGGL(k_pack<double>, grid, dim3(256), 0, s, g, d_src, static_cast<double*>(b.u[buf]));
  else
    hipLaunchKernelGGL(k_pack<float>, grid, dim3(256), 0, s, g, d_src, static_cast<float*>(b.u[buf]));
  return hipGetLastError();
}

hipError_t launch_unpack(const e2d_params& p, const DevBuffers& b, const void* d_state, int elem_bytes,
                         double* d_dst, hipStream_t s) {
  const Grid g = make_grid(p, b);
  const dim3 grid((g.isize + 63) / 64, (g.jsize + 3) / 4);
  if (elem_bytes == 8)
    hipLaunchKernelGGL(k_unpack<double>, grid, dim3(256), 0, s, g, static_cast<const double*>(d_state), d_dst);
  else
    hipLaunchKernelGGL(k_unpack<float>, grid, dim3(256), 0, s, g, static_cast<const float*>(d_state), d_dst);
  return hipGetLastError();
}

hipError_t launch_pack_field(const e2d_params& p, const DevBuffers& b, const double* d_src, double* d_field,
                             hipStream_t s) {
  const Grid g = make_grid(p, b);
  hipLaunchKernelGGL(k_pack<double>, dim3((g.isize + 63) / 64, (g.jsize + 3) / 4), dim3(256), 0, s, g, d_src,
                     d_field);
  return hipGetLastError();
}

size_t state_elem_bytes(int precision) {
  return with_precision(precision, [](auto pol) { return sizeof(typename decltype(pol)::S); });
}

// q, slopes and face states in the flux arithmetic type, fx and fy in the update type
size_t stage_elem_bytes(int precision, int stage) {
  return with_precision(precision, [&](auto pol) {
    using P = decltype(pol);
    return (stage == E2D_STAGE_FX || stage == E2D_STAGE_FY) ? sizeof(typename P::U) : sizeof(typename P::T);
  });
}

// ---------------------------------------------------------------------------
// pointwise numerics (known-answer tests of the device routines)

template <class P>
__global__ __launch_bounds__(256) void k_pointwise(const Hydro<typename P::T> h, int func, int n,
                                                    const double* __restrict__ x, double* __restrict__ y) {
  using T = typename P::T;
  using M = typename P::M;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  T a[20], o[8], g[4];
  switch (func) {
    case E2D_FN_PRIM: {
      for (int m = 0; m < 4; ++m) a[m] = static_cast<T>(x[4 * k + m]);
      cons_to_prim<T, M>(h, a, o);
      const T c = sound_speed<T, M>(h, o);
      for (int m = 0; m < 4; ++m) y[5 * k + m] = o[m];
      y[5 * k + 4] = c;
    } break;
    case E2D_FN_SLOPE: {
      for (int m = 0; m < 20; ++m) a[m] = static_cast<T>(x[20 * k + m]);
      cell_slopes(h, a, a + 4, a + 8, a + 12, a + 16, o, o + 4);
      for (int m = 0; m < 8; ++m) y[8 * k + m] = o[m];
    } break;
    case E2D_FN_TRACE: {
      for (int m = 0; m < 14; ++m) a[m] = static_cast<T>(x[15 * k + m]);
      const int face = static_cast<int>(x[15 * k + 14]);
      T s[4];
      trace_sources<T, M>(h, a, a + 4, a + 8, s);
      const bool xdir = face < 2;
      face_state(h, a, xdir ? a + 4 : a + 8, s, xdir ? a[12] : a[13], (face & 1) == 1, o);
      for (int m = 0; m < 4; ++m) y[4 * k + m] = o[m];
    } break;
    case E2D_FN_RIEMANN:
    case E2D_FN_HLLC: {
      for (int m = 0; m < 8; ++m) a[m] = static_cast<T>(x[8 * k + m]);
      if (func == E2D_FN_RIEMANN)
        riemann_two_shock<T, M>(h, a, a + 4, g, o);
      else
        riemann_hllc<T, ExactMath>(h, a, a + 4, g, o);
      for (int m = 0; m < 4; ++m) y[8 * k + m] = g[m];
      for (int m = 0; m < 4; ++m) y[8 * k + 4 + m] = o[m];
    } break;
    case E2D_FN_CMPFLX: {
      for (int m = 0; m < 4; ++m) a[m] = static_cast<T>(x[4 * k + m]);
      godunov_flux(h, a, o);
      for (int m = 0; m < 4; ++m) y[4 * k + m] = o[m];
    } break;
    case E2D_FN_EOS: {
      const T rho = static_cast<T>(x[2 * k]), eint = static_cast<T>(x[2 * k + 1]);
      const T p = fmax2((h.gamma0 - T(1)) * rho * eint, rho * h.smallp);
      const T c = M::sqrt(M::div(h.gamma0 * p, rho));
      y[2 * k] = p;
      y[2 * k + 1] = c;
    } break;
    case E2D_FN_DIV:
      y[k] = M::div(static_cast<T>(x[2 * k]), static_cast<T>(x[2 * k + 1]));
      break;
    case E2D_FN_SQRT:
      y[k] = M::sqrt(static_cast<T>(x[k]));
      break;
    case E2D_FN_DIV_ROOT: {
      T inv;
      const T s = M::sqrt_pos_inv(static_cast<T>(x[2 * k + 1]), inv);
      y[2 * k] = M::div_inv(static_cast<T>(x[2 * k]), s, inv);
      y[2 * k + 1] = s;
    } break;
    case E2D_FN_DIV_NEAR: {
      const T b = static_cast<T>(x[3 * k + 1]);
      y[k] = M::div_inv(static_cast<T>(x[3 * k]), b, M::recip_near(b, static_cast<T>(x[3 * k + 2])));
    } break;
    case E2D_FN_CONV_GT:
      y[k] = M::quot_gt(static_cast<T>(x[2 * k]), static_cast<T>(x[2 * k + 1]), h.conv_tol, h.conv_half_ulp) ? 1.0 : 0.0;
      break;
    default: break;
  }
}

hipError_t launch_pointwise(const e2d_params& p, int func, int n, const double* d_x, double* d_y, hipStream_t s) {
  const dim3 grid((n + 255) / 256);
  with_arithmetic(p, [&](auto pol) {
    using P = decltype(pol);
    hipLaunchKernelGGL(k_pointwise<P>, grid, dim3(256), 0, s, make_hydro<typename P::T>(p), func, n, d_x, d_y);
    return 0;
  });
  return hipGetLastError();
}

}  // namespace e2d
