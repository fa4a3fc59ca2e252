// fiber_pipe_kernel: a window pass of Givens rotations (strings on rows) whose
// memory traffic runs on waves of its own.
//
// fiber_kernel's waves load, rotate and store a tile in turn, so the memory
// instructions (issuing the next tile's loads behind the last tile's stores,
// draining the stores, staging the loaded tile) take 31% of a tile's time
// while the VALU idles, and the prefetched tile holds 64 registers of every
// wave.  One 118 KB complex128 tile fills a CU's LDS, so no second workgroup
// hides that.  Here a workgroup has 8 compute waves, which only run register
// sub-passes on the tile in LDS, and 4 memory waves, which hold a whole tile
// in registers (29 16-byte units a lane): during the sub-passes they store the
// previous tile from them and load the next one into them, and between two
// tiles they exchange registers and LDS.  Both kinds meet at the sub-passes'
// barriers, so the traffic is spread evenly over the sub-passes (all of it
// before the first barrier instead: 2.27 ms per launch).
//
// Rows of 128 bytes for both types: 8 complex128 or 16 complex64 columns.  16
// columns fill the complex64 chunks (4 groups x 16 columns: 20 groups of the
// largest class are exactly 5 chunks), 23% fewer wave instructions than the 4
// columns of fiber_kernel.
//
// Measured at norb=16 (12870 x 12870, LUCJ n_reps=4, average launch): complex128
// 2.28 -> 1.77 ms (3.0 TB/s algorithmic), complex64 1.49 -> 1.29 ms.  What bounds it: without
// the memory waves' traffic and exchange a launch takes 1.47 / 1.13 ms, without the
// rotations 1.38 / 0.83 ms; the VALU is busy 49% / 60% of the time, the rest of
// a sub-pass goes to its LDS reads and writes and the barrier.
#pragma once

#include "kernels.hpp"

namespace ffsim_amd {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// a 16-byte access to memory that is only 8-byte aligned (complex64 rows)
typedef u32x4 u32x4_a8 __attribute__((aligned(8)));

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
constexpr int pipe_max_rows(int units) { return pipe_step(units) * pipe_sweeps(units); }
constexpr int pipe_width(int units, size_t elem) { return units * 16 / (int)elem; }

// Tables of a pipelined pass (PipeGroups in device memory) and the distinct
// sub-window starts that its sub-passes use.
struct PipeTables {
  const uint32_t* desc;
  const int32_t* index;
  const uint32_t* offs;
  const int32_t* offs_index;
  const uint32_t* chunks;
  const int32_t* wave_index;
  int n_lo2;
  int n_slots;
  int lo2[kPipeMaxLo];
};
struct PipeSlot {
  int d_off;  // first group of this sub-window start in LDS
  int o_off;  // first member offset
};

// Applies the layer pairs of one sub-pass to one register group (one batch
// column): p is the group's base address in the tile, off its members' offsets.
template <typename T, int W2, int K2>
__device__ __forceinline__ void pipe_group_apply(unsigned char* p, const uint32_t* __restrict__ off,
                                                 const LayerPair* lp, int n_lp, bool flip) {
  constexpr int N = binom_const(W2, K2);
  Cx<T> v[N];
  Cx<T>* at[N];
#pragma unroll
  for (int m = 0; m < N; ++m) at[m] = reinterpret_cast<Cx<T>*>(p + off[m]);
#pragma unroll
  for (int m = 0; m < N; ++m) v[m] = *at[m];
  apply_layers<T, W2, K2>(v, lp, n_lp, flip);
#pragma unroll
  for (int m = 0; m < N; ++m) *at[m] = v[m];
}

// A diagonal Coulomb evolution fused into the store of a transposing pass,
// without its factor of the tile's strings alone (that one commutes with
// everything up to the next rotation of their sector, and the pass after
// this one applies it to whole columns, see cfac).
struct PipeFuse {
  const Cx<double>* bfac;  // [n_batch][n_fac]: per orbital q < norb, then the batch term
  int n_fac;               // norb + 1
};

// UNITS: 16-byte units per string.  TST: store the transposed state (rows of a
// window [0, w), contiguous).  DG: multiply by the orbital phases (and cfac, a
// factor per column).  FUSE: multiply by a diagonal evolution, transposing.
// Tiles of fewer than 8 units hold a whole sector (contiguous rows, one fiber).
template <typename T, int UNITS, bool TST, bool DG, bool FUSE>
__global__ void __launch_bounds__(kPipeThreads)
    fiber_pipe_kernel(const Cx<T>* src, Cx<T>* dst, long ld_src, long ld_dst, int n_batch,
                      const Fiber* __restrict__ fibers, int n_fibers,
                      const int32_t* __restrict__ row_table, PipeTables tb,
                      const SubPass* __restrict__ subs_g, int n_sub,
                      const LayerPair* __restrict__ layers_g, int n_layers,
                      const double* __restrict__ diag, const uint64_t* __restrict__ strings,
                      int win_lo, int win_w, int gd_cap, int go_cap, int gc_cap,
                      const Cx<double>* __restrict__ cfac, PipeFuse fz) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  constexpr int W2 = kMaxSubWindow;
  constexpr int W = pipe_width(UNITS, sizeof(Cx<T>));
  constexpr int EU = W / UNITS;  // elements of a unit
  constexpr int NW = kPipeCompute;
  constexpr int STEP = pipe_step(UNITS), SWEEPS = pipe_sweeps(UNITS);
  constexpr int R = STEP * SWEEPS;
  constexpr bool CONTIG = TST || UNITS < 8;  // rows row0, row0 + 1, ...
  constexpr int SLOTS = UNITS < 8 ? 1 : kPipeSlots;
  size_t off = 0;
  u32x4* tile4 = reinterpret_cast<u32x4*>(smem_raw);
  off += (size_t)(SWEEPS + 1) * 4096;
  int32_t* rslot = reinterpret_cast<int32_t*>(smem_raw + off);
  if (!CONTIG) off += (size_t)SLOTS * R * sizeof(int32_t);
  PipeSlot* gslot = reinterpret_cast<PipeSlot*>(smem_raw + off);
  off += align16((size_t)kPipeMaxLo * sizeof(PipeSlot));
  uint32_t* goff = reinterpret_cast<uint32_t*>(smem_raw + off);
  off += align16((size_t)go_cap * sizeof(uint32_t));
  uint32_t* gdesc = reinterpret_cast<uint32_t*>(smem_raw + off);
  off += align16((size_t)gd_cap * sizeof(uint32_t));
  int32_t* wsched = reinterpret_cast<int32_t*>(smem_raw + off);
  off += (size_t)kPipeMaxLo * NW * 2 * sizeof(int32_t);
  uint32_t* wchunks = reinterpret_cast<uint32_t*>(smem_raw + off);
  off += align16((size_t)gc_cap * sizeof(uint32_t));
  // launches that multiply by orbital phases or a fused diagonal
  uint16_t* lbits = reinterpret_cast<uint16_t*>(smem_raw + off);
  if (DG || FUSE) off += (size_t)SLOTS * R * sizeof(uint16_t);
  Cx<double>* ptab = reinterpret_cast<Cx<double>*>(smem_raw + off);  // phases per nibble pattern
  if (DG) off += 64 * sizeof(Cx<double>);
  Cx<double>* pout = reinterpret_cast<Cx<double>*>(smem_raw + off);  // phase outside the window
  if (DG) off += 4 * sizeof(Cx<double>);
  uint32_t* arrived = reinterpret_cast<uint32_t*>(smem_raw + off);
  if (FUSE) off += 16;
  Cx<double>* ffac = reinterpret_cast<Cx<double>*>(smem_raw + off);
  if (FUSE) off += (size_t)W * fz.n_fac * sizeof(Cx<double>);
  Cx<double>* ntab = reinterpret_cast<Cx<double>*>(smem_raw + off);

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n_bt = (n_batch + W - 1) / W;
  const long n_tiles = (long)n_bt * n_fibers;
  const int G = gridDim.x;
  const int bid = (G & 7) == 0 ? (int)(blockIdx.x & 7) * (G >> 3) + (int)(blockIdx.x >> 3)
                               : (int)blockIdx.x;
  long t = bid;
  if (t >= n_tiles) return;

  if (wave < kPipeCompute) {
    // ------------------------------------------------------ compute waves
    const int lane = tid & 63;
    constexpr int NTC = 64 * kPipeCompute;
    auto stage_tables = [&](int kp) {
      int d_base = 0, c_base = 0, o_base = 0;
      for (int u = 0; u < tb.n_slots; ++u) {
        const int set = kp * tb.n_lo2 + tb.lo2[u];
        const int d0 = tb.index[2 * set], nd = tb.index[2 * set + 1];
        if (tid == 0) gslot[u] = PipeSlot{d_base, o_base};
        for (int k = tid; k < nd; k += NTC) gdesc[d_base + k] = tb.desc[d0 + k];
        const int32_t* wi = tb.wave_index + (long)set * NW * 2;
        const int first = wi[0];
        const int total = wi[2 * (NW - 1)] + wi[2 * (NW - 1) + 1] - first;
        if (tid < NW) {
          wsched[(u * NW + tid) * 2] = c_base + (wi[2 * tid] - first);
          wsched[(u * NW + tid) * 2 + 1] = wi[2 * tid + 1];
        }
        for (int k = tid; k < total; k += NTC) wchunks[c_base + k] = tb.chunks[first + k];
        d_base += nd;
        c_base += total;
        o_base += tb.offs_index[2 * tb.lo2[u] + 1];
      }
    };
    int kp = fibers[(int)(t / n_bt)].kp;
    if (n_sub > 0) {
      stage_tables(kp);
      int o_base = 0;
      for (int u = 0; u < tb.n_slots; ++u) {
        const int o0 = tb.offs_index[2 * tb.lo2[u]], no = tb.offs_index[2 * tb.lo2[u] + 1];
        for (int k = tid; k < no; k += NTC) goff[o_base + k] = tb.offs[o0 + k];
        o_base += no;
      }
    }
    if (FUSE && tid == 0) *arrived = 0;
    __syncthreads();
    bool odd = true;  // where the tile lies (see exchange)
    while (true) {
      unsigned char* cur = smem_raw + (odd ? 4096 : 0);
      odd = !odd;
      for (int sp = 0; sp < n_sub; ++sp) {
        const SubPass P = subs_g[sp];
        const PipeSlot gs = gslot[P.slot];
        const LayerPair* lp = layers_g + P.lp0;
        const int c0 = wsched[(P.slot * NW + wave) * 2];
        const int nc = wsched[(P.slot * NW + wave) * 2 + 1];
        for (int c = 0; c < nc; ++c) {
          const uint32_t ch = wchunks[c0 + c];
          const int gl = lane / W, j = lane % W;
          if (gl < (int)(ch & 0xff)) {
            const uint32_t d = gdesc[gs.d_off + (int)(ch >> 8) + gl];
            unsigned char* p = cur + (d >> 16) * (16 * UNITS) + j * (int)sizeof(Cx<T>);
            const uint32_t* mo = goff + gs.o_off + ((d >> 4) & 0xfff) * 4;
            const bool flip = (d >> 3) & 1;
            switch (d & 7) {
              case 1: pipe_group_apply<T, W2, 1>(p, mo, lp, P.n_lp, flip); break;
              case 2: pipe_group_apply<T, W2, 2>(p, mo, lp, P.n_lp, flip); break;
              case 3: pipe_group_apply<T, W2, 3>(p, mo, lp, P.n_lp, flip); break;
              // complex64 groups of 4 and 5 electrons are complemented ones of 2 and 1
              case 4: if constexpr (sizeof(T) == 8) pipe_group_apply<T, W2, 4>(p, mo, lp, P.n_lp, flip); break;
              case 5: if constexpr (sizeof(T) == 8) pipe_group_apply<T, W2, 5>(p, mo, lp, P.n_lp, flip); break;
              default: break;
            }
          }
        }
        __syncthreads();
      }
      // the memory waves exchange the tile; meanwhile the next fiber's tables
      const long tn = t + G;
      if (tn < n_tiles && n_sub > 0) {
        const int kpn = fibers[(int)(tn / n_bt)].kp;
        if (kpn != kp) stage_tables(kpn);
        kp = kpn;
      }
      __syncthreads();
      t = tn;
      if (t >= n_tiles) break;
    }
    return;
  }

  // --------------------------------------------------------- memory waves
  const int m = tid - 64 * kPipeCompute;
  const int u = m & (UNITS - 1), i0 = m / UNITS;
  const int nt = (win_w + 3) >> 2;
  auto cmul = [](const Cx<double>& x, const Cx<double>& y) {
    return Cx<double>{x.re * y.re - x.im * y.im, x.re * y.im + x.im * y.re};
  };
  const uint64_t win_mask = ((1ull << win_w) - 1) << win_lo;
  if constexpr (DG) {
    if (m < 16 * nt) {
      const int t4 = 4 * (m >> 4), pat = m & 15;
      Cx<double> P{1.0, 0.0};
      for (int b = 0; b < 4; ++b)
        if (((pat >> b) & 1) && t4 + b < win_w)
          P = cmul(P, Cx<double>{diag[2 * (win_lo + t4 + b)], diag[2 * (win_lo + t4 + b) + 1]});
      ptab[m] = P;
    }
  }
  // what this thread needs of a fiber's strings (i = i0 + 32 k): their rows, and
  // their bits inside the window for the phases
  auto stage_rows = [&](const Fiber& fd, int slot) {
    if constexpr (!CONTIG || DG || FUSE) {
#pragma unroll 1
      for (int k = 0; k < SWEEPS; ++k) {
        const int i = i0 + k * STEP;
        const int r = row_table[fd.row_off + min(i, fd.n_rows - 1)];
        if constexpr (!CONTIG) rslot[slot * R + i] = r;
        if constexpr (DG || FUSE)
          lbits[slot * R + i] = (uint16_t)((strings[r] & win_mask) >> win_lo);
      }
    }
    if constexpr (DG) {
      if (m == 0) {
        uint64_t bits = strings[row_table[fd.row_off]] & ~win_mask;
        Cx<double> P{1.0, 0.0};
        while (bits) {
          const int q = __builtin_ctzll(bits);
          bits &= bits - 1;
          P = cmul(P, Cx<double>{diag[2 * q], diag[2 * q + 1]});
        }
        pout[slot] = P;
      }
    }
    asm volatile("" ::: "memory");
  };
  // Fused diagonal: the batch columns' factors of a tile go to LDS before the
  // tile leaves it, and are multiplied out over the nibble patterns before its
  // stores.
  Cx<double> bf[FUSE ? 2 : 1];
  auto load_bfac = [&](int b0) {
    if constexpr (FUSE) {
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int e = min(m + 256 * k, W * fz.n_fac - 1);
        const int cs = e / fz.n_fac, q = e - cs * fz.n_fac;
        const int col = min(b0 + cs / EU * EU, n_batch - EU) + cs % EU;
        bf[k] = fz.bfac[(long)col * fz.n_fac + q];
      }
    }
  };
  auto write_ffac = [&]() {
    if constexpr (FUSE) {
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int e = m + 256 * k;
        if (e < W * fz.n_fac) {
          const int q = e % fz.n_fac;
          Cx<double> v = bf[k];
          if (diag && q < fz.n_fac - 1) v = cmul(v, Cx<double>{diag[2 * q], diag[2 * q + 1]});
          ffac[e] = v;
        }
      }
    }
  };
  auto build_ntab = [&](uint64_t fixed) {
    if constexpr (FUSE) {
      for (int e = m; e < (nt * 16 + 1) * W; e += 256) {
        const int j = e % W, k = e / W;
        const Cx<double>* F = ffac + j * fz.n_fac;
        Cx<double> P{1.0, 0.0};
        if (k < nt * 16) {
          const int t4 = 4 * (k >> 4), pat = k & 15;
#pragma unroll 1
          for (int b = 0; b < 4; ++b)
            if (((pat >> b) & 1) && t4 + b < win_w) P = cmul(P, F[t4 + b]);
        } else {
          P = F[fz.n_fac - 1];
          uint64_t bits = fixed;
          while (bits) {
            const int q = __builtin_ctzll(bits);
            bits &= bits - 1;
            P = cmul(P, F[q]);
          }
        }
        ntab[e] = P;
      }
    }
  };
  // the memory waves wait for each other (all four get here once per tile)
  uint32_t target = 0;
  auto meet = [&]() {
    if constexpr (FUSE) {
      target += kPipeMemory;
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      if ((m & 63) == 0)
        __hip_atomic_fetch_add(arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      while (__hip_atomic_load(arrived, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < target)
        __builtin_amdgcn_s_sleep(1);
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    }
  };
  // memory instructions ahead of the compute waves' arithmetic
  __builtin_amdgcn_s_setprio(3);
  u32x4 buf[SWEEPS];
  // first column of this thread's unit in the tile at column b0 (units that
  // reach past the last column are moved back: they then hold columns that
  // another unit stores, and the store skips those)
  auto unit_col = [&](int b0) { return min(b0 + u * EU, n_batch - EU); };
  // register k holds sweep k of its tile, or sweep 28 - k (see exchange): string
  // first + k step.  Transposing passes work on contiguous rows (window [0, w)).
  auto load = [&](auto k0c, auto k1c, int first, int step, int slot, int nr, int row0, int b0) {
    constexpr int K0 = decltype(k0c)::value, K1 = decltype(k1c)::value;
    const Cx<T>* p = src + unit_col(b0);
    __builtin_amdgcn_sched_barrier(0);
    uint32_t row[K1 - K0];
#pragma unroll
    for (int k = K0; k < K1; ++k)
      row[k - K0] = CONTIG ? (uint32_t)(row0 + min(first + k * step, nr - 1))
                        : (uint32_t)rslot[slot * R + first + k * step];
#pragma unroll
    for (int k = K0; k < K1; ++k)
      buf[k] = *reinterpret_cast<const u32x4_a8*>(p + (uint64_t)row[k - K0] * (uint32_t)ld_src);
    __builtin_amdgcn_sched_barrier(0);
  };
  Cx<double> po[EU];  // the stored tile's factor shared by all its strings
  auto store = [&](auto k0c, auto k1c, int first, int step, int nr, int slot, int row0, int b0) {
    constexpr int K0 = decltype(k0c)::value, K1 = decltype(k1c)::value;
    const bool full = b0 + W <= n_batch;
    const int c0 = unit_col(b0), skip = b0 + u * EU - c0;
#pragma unroll
    for (int k = K0; k < K1; ++k) {
      const int i = first + k * step;
      if (i < nr) {
        const uint32_t row =
            CONTIG ? (uint32_t)(row0 + i) : (uint32_t)rslot[slot * R + i];
        u32x4 q = buf[k];
        Cx<T> e[EU];
        __builtin_memcpy(e, &q, 16);
        if constexpr (DG || FUSE) {
          const uint32_t bits = lbits[slot * R + i];
          Cx<double> Q{1.0, 0.0};
          if constexpr (!FUSE) {
            Q = ptab[bits & 15];
#pragma unroll 1
            for (int x = 1; x < nt; ++x) Q = cmul(Q, ptab[x * 16 + ((bits >> (4 * x)) & 15)]);
          }
#pragma unroll
          for (int z = 0; z < EU; ++z) {
            Cx<double> P;
            if constexpr (FUSE) {
              const Cx<double>* f = ntab + u * EU + z;
              P = f[nt * 16 * W];
#pragma unroll 1
              for (int x = 0; x < nt; ++x)
                P = cmul(P, f[(x * 16 + ((bits >> (4 * x)) & 15)) * W]);
            } else {
              P = cmul(Q, po[z]);
            }
            const T pr = (T)P.re, pi = (T)P.im;
            const T a = e[z].re * pr - e[z].im * pi;
            e[z].im = e[z].re * pi + e[z].im * pr;
            e[z].re = a;
          }
          __builtin_memcpy(&q, e, 16);
        }
        if constexpr (TST) {
#pragma unroll
          for (int z = 0; z < EU; ++z)
            if (full || z >= skip) dst[(uint64_t)(uint32_t)(c0 + z) * (uint32_t)ld_dst + row] = e[z];
        } else {
          Cx<T>* p = dst + c0 + (uint64_t)row * (uint32_t)ld_dst;
          if (full || skip == 0) {
            *reinterpret_cast<u32x4_a8*>(p) = q;
          } else {
#pragma unroll
            for (int z = 0; z < EU; ++z)
              if (z >= skip) p[z] = e[z];
          }
        }
      }
      // one unit's factor at a time: the registers are the buffer's
      if constexpr (DG || FUSE) __builtin_amdgcn_sched_barrier(0);
    }
  };
  // Exchanges the tile in LDS with the registers.  The tile moves by one sweep
  // each time (it lies at sweep 0 or 1 of a region one sweep longer), so that
  // every new unit goes where the previous unit was just read: a unit's old
  // value lands in the register that its new value left.  Moving up, the
  // sweeps run from the last to the first.
  auto exchange = [&](uint32_t wr, uint32_t rd, int step) {
#pragma unroll
    for (int k = 0; k < SWEEPS; ++k) {
      tile4[wr + k * step] = buf[k];
      asm volatile("" ::: "memory");
      buf[k] = tile4[rd + k * step];
      asm volatile("" ::: "memory");
    }
  };
#define KC(x) std::integral_constant<int, x>{}
  // Iteration q stores tile q - 2 from the registers, loads tile q into them
  // and exchanges them with tile q - 1 in LDS once the compute waves are done.
  int p_nr = 0, p_b0 = 0, p_slot = 0, p_row0 = 0;            // tile q - 2
  int c_nr = 0, c_b0 = 0, c_slot = 0, c_row0 = 0, c_f = -1;  // tile q - 1
  uint64_t p_fixed = 0, c_fixed = 0;  // electrons outside the window
  int bars_per_tile = 0;
  bool up = true;  // the first tile goes to sweep 1
  auto tile_factor = [&]() {
    if constexpr (DG && !FUSE) {
      // the phase of the fiber's electrons outside the window, and the column
      // factor that the previous gate left to this pass
#pragma unroll
      for (int z = 0; z < EU; ++z) {
        po[z] = pout[p_slot];
        if (cfac) po[z] = cmul(po[z], cfac[unit_col(p_b0) + z]);
      }
    }
    if constexpr (FUSE) {
      build_ntab(p_fixed);
      meet();
    }
  };
  while (true) {
    const bool more = t < n_tiles;  // after the last tile the loads repeat its addresses
    const int f = more ? (int)(t / n_bt) : c_f;
    const int n_b0 = more ? (int)(t % n_bt) * W : c_b0;
    const Fiber fn = fibers[f];
    int step = up ? -STEP : STEP, mv = m;
    // (opaque: the compiler would otherwise keep the loop-invariant addresses
    // of every sweep in registers)
    asm volatile("" : "+s"(step), "+v"(mv));
    const int first = mv / UNITS + (up ? R - STEP : 0);
    const int p_first = mv / UNITS + (up ? 0 : R - STEP);
    int n_slot = c_slot, n_row0 = c_row0;
    uint64_t n_fixed = c_fixed;
    if (f != c_f) {
      n_slot = c_slot + 1 >= SLOTS ? 0 : c_slot + 1;
      stage_rows(fn, n_slot);
      n_row0 = row_table[fn.row_off];
      if (FUSE) n_fixed = strings[n_row0] & ~win_mask;
    }
    if (p_nr > 0) tile_factor();
    int bars = 0;
    auto upto = [&](int n) {
#pragma unroll 1
      for (; bars < n; ++bars) __syncthreads();
    };
    // the stores and loads of a tile are spread evenly over its sub-passes
#define FFSIM_PORTION(A, B, N)                                     \
  store(KC(A), KC(B), p_first, -step, p_nr, p_slot, p_row0, p_b0); \
  load(KC(A), KC(B), first, step, n_slot, fn.n_rows, n_row0, n_b0); \
  upto((bars_per_tile * N + 5) / 9);
    FFSIM_PORTION(0, 4, 1)
    FFSIM_PORTION(4, 8, 2)
    FFSIM_PORTION(8, 12, 3)
    FFSIM_PORTION(12, 16, 4)
    FFSIM_PORTION(16, 19, 5)
    FFSIM_PORTION(19, 22, 6)
    FFSIM_PORTION(22, 25, 7)
    FFSIM_PORTION(25, SWEEPS, 8)
#undef FFSIM_PORTION
    load_bfac(c_b0);
    upto(bars_per_tile);
    write_ffac();
    exchange(mv + (up ? SWEEPS * 256 : 0), mv + (up ? (SWEEPS - 1) * 256 : 256), up ? -256 : 256);
    up = !up;
    __syncthreads();
    p_nr = c_nr;
    p_b0 = c_b0;
    p_slot = c_slot;
    p_row0 = c_row0;
    p_fixed = c_fixed;
    c_nr = fn.n_rows;
    c_f = f;
    c_b0 = n_b0;
    c_slot = n_slot;
    c_row0 = n_row0;
    c_fixed = n_fixed;
    t += G;
    bars_per_tile = n_sub;
    if (!more) break;
  }
  const int step = up ? -STEP : STEP;
  const int p_first = i0 + (up ? 0 : R - STEP);
  tile_factor();
  store(KC(0), KC(8), p_first, -step, p_nr, p_slot, p_row0, p_b0);
  store(KC(8), KC(16), p_first, -step, p_nr, p_slot, p_row0, p_b0);
  store(KC(16), KC(22), p_first, -step, p_nr, p_slot, p_row0, p_b0);
  store(KC(22), KC(SWEEPS), p_first, -step, p_nr, p_slot, p_row0, p_b0);
#undef KC
}

// Kernel of a tile geometry and variant (the launching code and the
// instantiations of each type are compiled apart).
enum { PIPE_PLAIN = 0, PIPE_PHASES = 1, PIPE_TRANSPOSE = 2, PIPE_TRANSPOSE_PHASES = 3, PIPE_FUSED = 4,
       PIPE_VARIANTS = 5 };
template <typename T, int UNITS>
const void* pipe_kernel_units(int variant) {
  switch (variant) {
    case PIPE_PLAIN: return (const void*)fiber_pipe_kernel<T, UNITS, false, false, false>;
    case PIPE_PHASES: return (const void*)fiber_pipe_kernel<T, UNITS, false, true, false>;
    case PIPE_TRANSPOSE: return (const void*)fiber_pipe_kernel<T, UNITS, true, false, false>;
    case PIPE_TRANSPOSE_PHASES: return (const void*)fiber_pipe_kernel<T, UNITS, true, true, false>;
    default: return (const void*)fiber_pipe_kernel<T, UNITS, true, false, true>;
  }
}
template <typename T>
const void* pipe_kernel(int units, int variant) {
  switch (units) {
    case 8: return pipe_kernel_units<T, 8>(variant);
    case 4: return pipe_kernel_units<T, 4>(variant);
    case 2: return pipe_kernel_units<T, 2>(variant);
    default: return pipe_kernel_units<T, 1>(variant);
  }
}
const void* pipe_kernel_c128(int units, int variant);
const void* pipe_kernel_c64(int units, int variant);

}  // namespace ffsim_amd
