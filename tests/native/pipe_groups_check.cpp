// Compares the register groups of the pipelined passes (base rank plus shared
// member offsets) with a direct enumeration of the window's strings.
#include <algorithm>
#include <cstdio>
#include <map>
#include <set>

#include "../../ffsim_amd/csrc/host_core.hpp"

using namespace ffsim_amd;

// 0: equal; otherwise the number of the check that failed.
extern "C" int check_pipe_groups(int w, int kp, int merge, int units, int per_chunk) {
  const int W2 = kMaxSubWindow, NW = 8;
  const PipeGroups T = make_pipe_groups(w, kp, kp, merge != 0, units, NW, per_chunk);
  std::map<uint64_t, uint32_t> rank;
  const std::vector<uint64_t> strs = make_strings(w, kp);
  for (size_t i = 0; i < strs.size(); ++i) rank[strs[i]] = (uint32_t)i;
  for (int lo2 = 0; lo2 < T.n_lo2; ++lo2) {
    const uint64_t sub = ((1ull << W2) - 1) << lo2;
    // every outside pattern with 0 < k2 < W2 electrons inside, and its members
    std::multiset<std::vector<uint32_t>> want, got;
    std::set<uint64_t> outs;
    for (uint64_t s : strs) outs.insert(s & ~sub);
    for (uint64_t o : outs) {
      const int k2 = kp - __builtin_popcountll(o);
      if (k2 <= 0 || k2 >= W2) continue;
      const bool flip = merge && 2 * k2 > W2;
      std::vector<uint32_t> v{(uint32_t)(flip ? W2 - k2 : k2), (uint32_t)flip};
      for (uint64_t x : make_strings(W2, flip ? W2 - k2 : k2)) {
        const uint64_t bits = flip ? (~x & ((1ull << W2) - 1)) : x;
        v.push_back(rank.at(o | (bits << lo2)));
      }
      want.insert(v);
    }
    const size_t set = (size_t)kp * T.n_lo2 + lo2;
    const int d0 = T.index[2 * set], nd = T.index[2 * set + 1];
    int last_size = 1 << 30, last_cls = -1;
    for (int g = 0; g < nd; ++g) {
      const uint32_t d = T.desc[d0 + g];
      const int cls = d & 7;
      const uint32_t toff = ((d >> 4) & 0xfff) * 4;
      const int n = (int)binom(W2, cls);
      if ((int)(toff + n) > T.offs_index[2 * lo2 + 1]) return 1;
      std::vector<uint32_t> v{(uint32_t)cls, (d >> 3) & 1};
      for (int m = 0; m < n; ++m) {
        const uint32_t b = T.offs[T.offs_index[2 * lo2] + toff + m];
        if (b % (16 * units)) return 2;
        v.push_back((d >> 16) + b / (16 * units));
      }
      got.insert(v);
      // classes are contiguous, larger groups first
      if (n > last_size || (n == last_size && cls < last_cls)) return 3;
      last_size = n;
      last_cls = cls;
    }
    if (want != got) return 4;
    // the wave schedule covers every group once, one class per chunk
    std::vector<int> seen(nd, 0);
    for (int wv = 0; wv < NW; ++wv) {
      const int32_t* wi = T.wave_index.data() + (set * NW + wv) * 2;
      for (int c = 0; c < wi[1]; ++c) {
        const uint32_t ch = T.chunks[wi[0] + c];
        const int g0 = ch >> 8, ng = ch & 0xff;
        if (ng > per_chunk || g0 + ng > nd) return 5;
        for (int g = g0; g < g0 + ng; ++g) {
          ++seen[g];
          if ((T.desc[d0 + g] & 7) != (T.desc[d0 + g0] & 7)) return 6;
        }
      }
    }
    for (int s : seen)
      if (s != 1) return 7;
    // consecutive waves' chunks are contiguous (the kernel stages them in one copy)
    for (int wv = 0; wv + 1 < NW; ++wv) {
      const int32_t* wi = T.wave_index.data() + (set * NW + wv) * 2;
      if (wi[2] != wi[0] + wi[1]) return 8;
    }
  }
  return 0;
}
