// The library's rules on pass geometry, for tests on the CPU (MI355X limits).
#include "../../ffsim_amd/csrc/pass_rules.hpp"

using namespace ffsim_amd;

static const PassLimits kLim{163840, 256};

// 0 none, 1 as rows, 2 slabs, 3 columns; *slab: rows of a slab
extern "C" int trdm_layout(int dtype, long da, long db, int n_beta, long* slab) {
  const TrdmBeta r = trdm_beta_layout(dtype, da, db, n_beta);
  *slab = r.slab;
  return (int)r.form;
}

// In-place whole-sector passes: 16-byte units per string (0: no such pass), strings
// taken to be on columns or not, sweeps, columns a lane.
extern "C" void small_pass(int dtype, int norb, int nocc, long n_batch, int n_states,
                           int on_columns, int* out) {
  const SectorGeom g = small_geom(kLim, dtype, norb, nocc, n_batch, n_states);
  out[0] = g.small ? g.units : 0;
  out[1] = small_in_columns(dtype, on_columns != 0, n_batch);
  out[2] = g.sweeps;
  out[3] = g.cols;
}

// Passes of a sector with strings on rows: window, units of a pipelined tile,
// whether a tile holds the whole sector; returns whether a pass over all fibers
// of the window [0, w) runs pipelined.
extern "C" int sector_pass(int dtype, int norb, int nocc, long n_batch, int* out) {
  const SectorGeom g = sector_geom(kLim, dtype, norb, nocc, n_batch);
  out[0] = g.w;
  out[1] = g.units;
  out[2] = g.whole;
  long n_f = 0;
  for (int kp = std::max(0, nocc - (norb - g.w)); kp <= std::min(nocc, g.w); ++kp)
    n_f += (long)binom(norb - g.w, nocc - kp);
  return pipe_applies(kLim, dtype, g, max_fiber(norb, nocc, g.w), n_f, n_batch);
}
