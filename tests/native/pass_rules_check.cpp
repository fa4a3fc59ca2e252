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
