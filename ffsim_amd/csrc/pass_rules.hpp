// Which kernel runs a pass and on what tiles: rules on sizes alone.  Plain host
// code without HIP, so that tests evaluate them on the CPU; the library passes
// the device's limits.
#pragma once

#include <algorithm>
#include <cstdlib>

#include "../../include/ffsim_amd.h"
#include "host_core.hpp"

namespace ffsim_amd {

struct PassLimits {
  size_t lds_max;  // bytes of a workgroup
  long n_cu;
};

constexpr size_t align16(size_t x) { return (x + 15) & ~size_t(15); }

// LDS of a fused store's per-tile tables: for every 4-orbital nibble t of the
// window and every occupation pattern p of it, the product of the batch
// columns' factors over p; then one factor per column for the batch term and
// the fiber's orbitals outside the window (the same for every tile string).
// An entry is one complex double (kFactorBytes).
constexpr size_t kFactorBytes = 16;
constexpr int fuse_nibble_entries(int win, int W) { return (((win + 3) >> 2) * 16 + 1) * W; }

// ------------------------------------------------- geometry of pipelined tiles
constexpr int kPipeCompute = 8;  // compute waves
constexpr int kPipeMemory = 4;   // memory waves
constexpr int kPipeThreads = 64 * (kPipeCompute + kPipeMemory);
constexpr int kPipeSlots = 3;    // fibers whose rows are in LDS at once
constexpr int kPipeMaxLo = 11;   // sub-window starts of a 16-orbital window

// Geometry of a tile with `units` 16-byte units per string: 8 for windows of
// part of the orbitals (128-byte segments), and fewer where that lets a tile
// hold every string of a sector, whose rotation is then a single pass.
// A sweep is one 16-byte access of every memory lane.
constexpr int pipe_step(int units) { return 64 * kPipeMemory / units; }  // strings per sweep
constexpr int pipe_sweeps(int units) { return units == 8 ? 29 : units == 1 ? 26 : 27; }
constexpr int pipe_max_rows(int units, int sweeps) { return pipe_step(units) * sweeps; }
constexpr int pipe_max_rows(int units) { return pipe_max_rows(units, pipe_sweeps(units)); }
constexpr int pipe_width(int units, size_t elem) { return units * 16 / (int)elem; }
// Columns that a compute lane rotates together: complex64 passes with several
// tiles per CU take both columns of a 16-byte unit, which halves the LDS
// instructions, address and coefficient work of a rotation (norb 16 1.19 ->
// 1.12 ms a launch, norb 15 0.79 -> 0.65, norb 14 0.197 -> 0.174).  A launch of
// one tile per CU waits for one chunk's chain of instructions, which that doubles
// (norb 12 39 -> 48 us, norb 13 69 -> 71): one column there, and for sectors of
// at most 256 strings (64 states of norb 10: 58 us against 69).
constexpr int pipe_cols(int units, size_t elem) { return units == 4 ? 1 : 16 / (int)elem; }

// Variants of the pipelined kernel.
enum { PIPE_PLAIN = 0, PIPE_PHASES = 1, PIPE_TRANSPOSE = 2, PIPE_TRANSPOSE_PHASES = 3, PIPE_FUSED = 4,
       PIPE_SMALL_ROWS = 5, PIPE_SMALL_COLS = 6, PIPE_VARIANTS = 7 };

// ------------------------------------------------------------- tiles and windows
inline size_t elem_bytes(int dtype) { return dtype == FFSIM_C64 ? 8 : 16; }

// LDS kept free for the staged program of a pass (sub-passes + steps).
constexpr size_t kProgramLdsReserve = 20480;
// LDS kept free beside the tile, row indices and row strings of a window pass.
constexpr size_t kGroupLdsReserve = 16384;

inline int tile_width(int dtype) {
  static int env_w = [] {
    const char* e = std::getenv("FFSIM_AMD_TILE_W");
    return e ? std::atoi(e) : 0;
  }();
  if (env_w == 4 || env_w == 8 || env_w == 16) return env_w;
  // c128: 8 columns (128-byte row segments, one tile per CU).  c64: 4 columns,
  // so that several independent tiles share a CU and one tile's barrier waits
  // overlap another's work (measured 8% faster than 8 columns, 20% than 16).
  return dtype == FFSIM_C64 ? 4 : 8;
}

inline int window_cap() {
  static int cap = [] {
    const char* e = std::getenv("FFSIM_AMD_MAX_WINDOW");
    const int v = e ? std::atoi(e) : 0;
    return (v >= 2 && v <= 16) ? v : 12;
  }();
  return cap;
}

// The beta rotation runs in place with strings on columns when a whole beta
// vector fits one tile and its window (all norb orbitals) is no wider than
// the row-mode window cap, whose group tables the LDS reserve is sized for.
inline bool beta_in_columns(int norb, long dim_b, int dtype, const PassLimits& lim) {
  return norb <= window_cap() &&
         (size_t)dim_b * (tile_width(dtype) + 1) * elem_bytes(dtype) + kProgramLdsReserve <=
             lim.lds_max &&
         dim_b < 65536;
}

// Largest fiber of a window of width w for nocc electrons on norb orbitals.
inline int max_fiber(int norb, int nocc, int w) {
  int lo_k = std::max(0, nocc - (norb - w)), hi_k = std::min(nocc, w);
  uint64_t m = 0;
  for (int kp = lo_k; kp <= hi_k; ++kp) m = std::max(m, binom(w, kp));
  return (int)m;
}

// Largest window (up to the cap) whose fiber tiles fit in LDS.
inline int choose_window(const PassLimits& lim, int norb, int nocc, int dtype) {
  const int W = tile_width(dtype);
  // tile row + row index + row string (phase passes); the reserve holds the group
  // tables, wave schedule and orbital phases
  const size_t per_row = (size_t)(W + 1) * elem_bytes(dtype) + 4 + (norb <= 32 ? 4 : 8);
  int best = std::min(norb, 2);
  for (int w = std::min(norb, window_cap()); w >= 2; --w) {
    if ((size_t)max_fiber(norb, nocc, w) * per_row + kGroupLdsReserve <= lim.lds_max) {
      best = w;
      break;
    }
  }
  if (norb <= 1) best = std::max(norb, 1);
  return best;
}

// How the passes of a sector with strings on rows run: the window width, and
// the 16-byte units per string of a pipelined tile (0: plain passes).
//
// Up to norb 16, a sector whose strings all fit one tile at some tile width
// runs as one pass over all orbitals instead of three over 12-orbital windows:
// a third of the traffic and of the launches, and 8 to 10 register sub-passes
// instead of 10 to 12, for narrower segments in memory (64, 32 or 16 bytes of
// a row; neighbouring tiles run on one XCD and share its L2).  Measured per
// sector rotation, LUCJ: norb=13 (1716 strings, 4 complex128 columns) 160 ->
// 107 us, norb=14 (3432, 2 columns) 449 -> 281 us, norb=15 (6435, 1 column)
// 1614 -> 945 us; complex64 153 -> 81, 324 -> 220 and 1080 -> 810 us.
struct SectorGeom {
  int w = 0, units = 0, sweeps = 0;
  int cols = 1;        // columns of a compute lane
  bool whole = false;  // a tile holds every string of the sector (one pass)
  bool small = false;  // in place, several states (norb <= 12)
};

// LDS of a pipelined launch, following the kernel's layout.
inline size_t pipe_lds_bytes(const SectorGeom& g, size_t elem, int image_dwords, int variant,
                             int n_fac, int win) {
  const int units = g.units;
  const bool small = variant >= PIPE_SMALL_ROWS;
  const bool whole = small || units < 8;
  const bool tstore = variant == PIPE_TRANSPOSE || variant == PIPE_TRANSPOSE_PHASES ||
                      variant == PIPE_FUSED;
  const bool dg = variant == PIPE_PHASES || variant == PIPE_TRANSPOSE_PHASES || small;
  const size_t R = pipe_max_rows(units, g.sweeps), W = pipe_width(units, elem);
  const size_t slots = whole ? 1 : kPipeSlots;
  size_t b = (size_t)(g.sweeps + 1) * 4096 + (tstore || whole ? 0 : slots * R * 4) +
             align16((size_t)image_dwords * 4);
  if (dg || variant == PIPE_FUSED) b += slots * R * 2;
  if (dg) b += 68 * kFactorBytes;
  if (variant == PIPE_FUSED || small) b += 16;
  if (variant == PIPE_FUSED)
    b += (W * n_fac + (size_t)fuse_nibble_entries(win, (int)W)) * kFactorBytes;
  return b;
}

// Geometry of the in-place whole-sector passes of norb 6 to 12 (units 0: none),
// from the tiles that hold the sector's strings.  A tile's time is the chain of
// its sub-passes, one chunk each of 6-orbital groups, which a wider tile makes
// longer; a launch takes rounds of one tile per CU.  So the form is the one whose
// rounds take the least time.  SmallForm::first and ::more are the microseconds of
// a launch's first round and of each further one, measured at the largest sectors
// of each class (924 and 792, 495, 462, 252 strings; 1 to 64 states), where the
// least sum is the fastest form for every count, or within 5% of it.  Examples,
// us a launch, narrow against wide rows: norb 12 (6, 6) complex128 one state 42
// and 50, two states 65 and 54; complex64 two states 42 and 61, three 68 and 64,
// five 91 and 99, eight 118 and 102; norb 11 (5, 5) complex64 four states 32 and 37
// (and 53 for 256-byte rows), ten 74, 60 and 57, 24 135, 88 and 91.
// A lane takes both complex64 columns of a unit where that is the faster form of a
// wide tile: 32 states of norb 12 (6, 6) 313 against 366 us, (4, 4) 159 against 141.
// A single column (the other sector empty or full) runs with strings on columns
// (small_in_columns).
struct SmallForm {
  int units, sweeps, cols;
  double first, more;
};
inline SectorGeom small_geom(const PassLimits& lim, int dtype, int norb, int nocc, long n_batch,
                             int n_states) {
  SectorGeom g;
  g.w = norb;
  const size_t elem = elem_bytes(dtype);
  if (norb < kMaxSubWindow || norb > std::min(window_cap(), 12) || n_batch > (1l << 30) ||
      tile_width(dtype) != (dtype == FFSIM_C64 ? 4 : 8))
    return g;
  const long rows = (long)binom(norb, nocc);
  if (rows == 0 || rows > pipe_max_rows(8, 29)) return g;
  static constexpr SmallForm kForms[2][4][3] = {
      {{{8, 8, 1, 25, 19}, {16, 16, 1, 31, 21}},
       {{4, 15, 1, 31, 21}, {8, 15, 1, 36, 25}, {16, 29, 1, 49, 33}},
       {{4, 15, 1, 41, 23}, {8, 29, 1, 42, 26}},
       {{4, 15, 1, 41, 23}, {8, 29, 1, 52, 31}}},
      {{{8, 8, 1, 25, 19}, {16, 16, 1, 31, 21}},
       {{4, 15, 1, 31, 21}, {8, 15, 1, 36, 25}, {16, 29, 2, 52, 35}},
       {{4, 15, 1, 41, 25}, {8, 29, 1, 47, 32}},
       {{4, 15, 1, 41, 25}, {8, 29, 2, 61, 37}}}};
  const int cls = rows <= pipe_max_rows(16, 16)   ? 0
                  : rows <= pipe_max_rows(16, 29) ? 1
                  : rows <= 512                   ? 2
                                                  : 3;
  g.whole = g.small = true;
  double best = 0.0;
  for (const SmallForm& f : kForms[dtype == FFSIM_C64][cls]) {
    if (f.units == 0) break;
    const long w = pipe_width(f.units, elem), tiles = (n_batch + w - 1) / w * n_states;
    const double t = f.first + f.more * (double)((tiles + lim.n_cu - 1) / lim.n_cu - 1);
    if (g.units && t >= best) continue;
    best = t;
    g.units = f.units;
    g.sweeps = f.sweeps;
    g.cols = f.cols;
  }
  return g;
}

// Whether an in-place whole-sector pass takes its strings to be on columns.  One
// column is contiguous either way; with strings on rows a unit of two complex64
// columns would reach past it.
inline bool small_in_columns(int dtype, bool strings_on_columns, long n_batch) {
  return strings_on_columns || n_batch < (long)(16 / elem_bytes(dtype));
}

inline SectorGeom sector_geom(const PassLimits& lim, int dtype, int norb, int nocc, long n_batch) {
  SectorGeom g;
  g.w = choose_window(lim, norb, nocc, dtype);
  const size_t elem = elem_bytes(dtype);
  if (n_batch > (1l << 30) || tile_width(dtype) != (dtype == FFSIM_C64 ? 4 : 8)) return g;
  const long rows = (long)binom(norb, nocc);
  // (a single string has nothing to rotate: windows skip all but the last pass,
  // whose plain tiles are one row; norb 16 with (8, 0) electrons 116 against 138 us)
  if (norb > window_cap() && norb >= kMaxSubWindow && norb <= 16 && rows > 1)
    for (int units : {8, 4, 2, 1})
      if (rows <= pipe_max_rows(units) &&
          n_batch >= pipe_width(units, elem)) {
        g.w = norb;
        g.units = units;
        g.sweeps = pipe_sweeps(units);
        g.cols = pipe_cols(units, elem);
        g.whole = true;
        return g;
      }
  if (g.w >= kMaxSubWindow && g.w <= 16 && n_batch >= pipe_width(8, elem)) {
    g.units = 8;
    g.sweeps = pipe_sweeps(8);
    g.cols = pipe_cols(8, elem);
  }
  return g;
}

// Whether a row pass over n_f fibers of up to `rows` strings runs pipelined
// (fiber_pipe_kernel).
// Whole-sector tiles always do.  For the others, both kernels walk their tiles
// in rounds over the CUs, one pipelined tile per CU against one plain
// complex128 tile or three plain complex64 tiles of a quarter of the columns.
// Measured on the 12-orbital passes of norb 13 to 16: a round takes about 17.6
// / 21 us (complex128) and 24 / 21.5 us (complex64), and a pipelined launch
// 16 us more to fill and drain, so it wins from 5 rounds on in complex128 (25
// rounds: 482 against 538 us per launch; 2 rounds: 58 against 53).  Fibers
// whose plain tiles leave room for a second workgroup per CU gain nothing from
// it in complex128 (norb=16 (4,4) in 12-orbital windows, 495 strings: 180
// against 126 us).
inline bool pipe_applies(const PassLimits& lim, int dtype, const SectorGeom& g, int rows, long n_f,
                         long n_batch) {
  if (g.units == 0) return false;
  if (g.whole) return true;
  if (rows > pipe_max_rows(8)) return false;
  const bool c128 = dtype == FFSIM_C128;
  if (c128 ? 2 * (size_t)rows * 128 <= lim.lds_max : rows < 400) return false;
  auto rounds = [&](int width, long per_cu) {
    const long tiles = (n_batch + width - 1) / width * n_f;
    return (double)((tiles + per_cu * lim.n_cu - 1) / (per_cu * lim.n_cu));
  };
  return (c128 ? 17.6 : 24.0) * rounds(pipe_width(8, elem_bytes(dtype)), 1) + 16.0 <
         (c128 ? 21.0 * rounds(8, 1) : 21.5 * rounds(4, 3));
}

// -------------------------------------------------------- transition RDM
// How the beta sector of a transition RDM reads lam and psi (da x db, its
// strings on columns): as they lie where one dimension is 1 (a row or a column
// is its own transpose); in transposed slabs of rows, whose strings then index
// rows as the alpha sector's do, all rows if their transposes take no more than
// kTrdmSlabBytes (norb 13), else as many as fit, their sums added up (norb 14:
// 4.3 ms along columns, 1.1 in 4 slabs); or along the columns in place, where a
// slab would have fewer rows than a wave has lanes: few rows of many columns,
// for each of which all slabs would be gone through.  Columns against slabs,
// complex128: norb 24 with (1, 8) electrons 32 and 153 ms (slabs of 4 rows), (1, 12)
// 178 and 3591 (1 row), norb 20 (2, 9) 18 and 43 (18 of 190 rows), (2, 7) 7.6 and
// 9.0 (40); the other way round norb 18 (3, 9) 24.7 and 18.3 (64 of 816).
struct TrdmBeta {
  enum Form { kNone, kAsRows, kSlabs, kColumns } form = kNone;
  long slab = 0;
};
constexpr long kTrdmSlabBytes = 96l << 20;
constexpr long kTrdmMinSlab = 64;
inline TrdmBeta trdm_beta_layout(int dtype, long da, long db, int n_beta) {
  TrdmBeta r;
  if (n_beta == 0 || da == 0 || db == 0) return r;
  if (da == 1 || db == 1) {
    r.form = TrdmBeta::kAsRows;
    return r;
  }
  r.slab = std::min<long>(da, kTrdmSlabBytes / (2 * db * (long)elem_bytes(dtype)));
  if (r.slab < da && r.slab < kTrdmMinSlab) {
    r.form = TrdmBeta::kColumns;
    return r;
  }
  // (grid.y of the transposition: 32 rows each)
  r.slab = std::min(r.slab, 32l * 65535);
  if (r.slab < da && r.slab > 64) r.slab -= r.slab % 64;
  r.form = TrdmBeta::kSlabs;
  return r;
}

}  // namespace ffsim_amd
