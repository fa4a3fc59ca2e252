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
// Rows of 128 bytes for both types: 8 complex128 or 16 complex64 columns, one
// 16-byte unit to a compute lane (see pipe_cols).
//
// Measured at norb=16 (12870 x 12870, LUCJ n_reps=4, average launch): complex128
// 2.28 -> 1.72 ms (3.1 TB/s algorithmic), complex64 1.49 -> 1.12 ms.  What bounds
// it: without the memory waves' traffic and exchange a complex128 launch takes
// 1.47 ms, without the rotations 1.38; the VALU is busy 49% of the time, the rest
// of a sub-pass goes to its LDS reads and writes and the barrier.
//
// SMALL launches rotate whole sectors in place (norb 6 to 12, one or several
// states, strings on rows or on columns).  One tile per CU or few, so what
// bounds them is a tile's chain of sub-passes: at norb 12 about 730 clocks of
// program and schedule reads, 450 of LDS reads, 280 per layer pair's scalar
// loads, the rotations of one chunk at 4.5 clocks an instruction, 560 of LDS
// writes.  Against fiber_kernel, whose workgroups held 8 columns (complex128)
// and staged tables by dependent reads: norb 12 complex128 50 -> 42 us and complex64
// 48 -> 41, 32 states of norb 12 601 -> 511 and 381 -> 368, 32 states of norb
// 10 61 -> 51 and 67 -> 33.
#pragma once

#include "kernels.hpp"
#include "pass_rules.hpp"

namespace ffsim_amd {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// a 16-byte access to memory that is only 8-byte aligned (complex64 rows)
typedef u32x4 u32x4_a8 __attribute__((aligned(8)));

// Tables of a pipelined pass: one image per electron count kp of the window,
// laid out as the workgroup keeps it in LDS (dword offsets): PipeSlot per
// sub-window start, member offsets (from kPipeImageOffs), group words, (offset,
// count) of chunks per (start, compute wave), chunks.  One copy stages it,
// with no dependent reads.
struct PipeTables {
  const uint32_t* image;
  int dwords;
  int kp_lo;  // kp of the first image
  int desc, sched, chunks;
};
struct PipeSlot {
  int d_off;  // first group of this sub-window start
  int o_off;  // first member offset
};
constexpr int kPipeImageOffs = (2 * kPipeMaxLo + 3) / 4 * 4;

// The states of an in-place whole-sector launch, each with its own layer pairs
// and phases at the given strides (states null: one state, the src argument).
struct PipeStates {
  void* const* states;
  int n_states;
  long layer_stride;  // LayerPairs
  long diag_stride;   // doubles
};

// Applies the layer pairs of one sub-pass to one register group (NC batch
// columns): p is the group's base address in the tile, off its members' offsets.
template <typename T, int W2, int K2, int NC>
__device__ __forceinline__ void pipe_group_apply(unsigned char* p, const uint32_t* __restrict__ off,
                                                 const LayerPair* lp, int n_lp, bool flip) {
  constexpr int N = binom_const(W2, K2);
  struct alignas(NC * sizeof(Cx<T>)) Unit { Cx<T> c[NC]; };
  Cx<T> v[NC * N];  // column-major
  Unit* at[N];
#pragma unroll
  for (int m = 0; m < N; ++m) at[m] = reinterpret_cast<Unit*>(p + off[m]);
#pragma unroll
  for (int m = 0; m < N; ++m) {
    const Unit x = *at[m];
#pragma unroll
    for (int k = 0; k < NC; ++k) v[k * N + m] = x.c[k];
  }
  apply_layers<T, W2, K2, NC>(v, lp, n_lp, flip);
#pragma unroll
  for (int m = 0; m < N; ++m) {
    Unit x;
#pragma unroll
    for (int k = 0; k < NC; ++k) x.c[k] = v[k * N + m];
    *at[m] = x;
  }
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
// SMALL: in place on whole sectors of several states (norb <= 12), strings on
// rows or (COLS) on columns, with phases if diag is given.  Tiles of fewer
// than 8 units and SMALL ones hold a whole sector (rows 0, 1, ..., one fiber
// of whole_rows strings with whole_kp electrons).
template <typename T, int UNITS, int SWEEPS, int NC, bool TST, bool DG, bool FUSE, bool SMALL, bool COLS>
__global__ void __launch_bounds__(kPipeThreads)
    fiber_pipe_kernel(const Cx<T>* src, Cx<T>* dst, long ld_src, long ld_dst, int n_batch,
                      const Fiber* __restrict__ fibers, int n_fibers,
                      const int32_t* __restrict__ row_table, PipeTables tb,
                      const SubPass* __restrict__ subs_g, int n_sub,
                      const LayerPair* __restrict__ layers_g, int n_layers,
                      const double* __restrict__ diag, const uint64_t* __restrict__ strings,
                      int win_lo, int win_w, int whole_rows, int whole_kp,
                      const Cx<double>* __restrict__ cfac, PipeFuse fz, PipeStates ms) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  constexpr int W2 = kMaxSubWindow;
  constexpr int W = pipe_width(UNITS, sizeof(Cx<T>));
  constexpr int EU = W / UNITS;  // elements of a unit
  constexpr int NW = kPipeCompute;
  constexpr int STEP = pipe_step(UNITS), LANES = 64 * kPipeMemory;
  constexpr int R = STEP * SWEEPS;
  constexpr bool WHOLE = SMALL || UNITS < 8;
  constexpr bool CONTIG = TST || WHOLE;  // rows row0, row0 + 1, ...
  constexpr int SLOTS = WHOLE ? 1 : kPipeSlots;
  static_assert(!SMALL || (DG && !TST && !FUSE), "small passes: in place, with phases");
  static_assert(!COLS || SMALL, "strings on columns: in place only");
  size_t off = 0;
  u32x4* tile4 = reinterpret_cast<u32x4*>(smem_raw);
  off += (size_t)(SWEEPS + 1) * LANES * 16;
  int32_t* rslot = reinterpret_cast<int32_t*>(smem_raw + off);
  if (!CONTIG) off += (size_t)SLOTS * R * sizeof(int32_t);
  uint32_t* img = reinterpret_cast<uint32_t*>(smem_raw + off);
  off += align16((size_t)tb.dwords * sizeof(uint32_t));
  const PipeSlot* gslot = reinterpret_cast<const PipeSlot*>(img);
  const uint32_t* goff = img + kPipeImageOffs;
  const uint32_t* gdesc = img + tb.desc;
  const uint32_t* wsched = img + tb.sched;
  const uint32_t* wchunks = img + tb.chunks;
  // launches that multiply by orbital phases or a fused diagonal
  uint16_t* lbits = reinterpret_cast<uint16_t*>(smem_raw + off);
  if (DG || FUSE) off += (size_t)SLOTS * R * sizeof(uint16_t);
  Cx<double>* ptab = reinterpret_cast<Cx<double>*>(smem_raw + off);  // phases per nibble pattern
  if (DG) off += 64 * sizeof(Cx<double>);
  Cx<double>* pout = reinterpret_cast<Cx<double>*>(smem_raw + off);  // phase outside the window
  if (DG) off += 4 * sizeof(Cx<double>);
  uint32_t* arrived = reinterpret_cast<uint32_t*>(smem_raw + off);
  if (FUSE || SMALL) off += 16;
  Cx<double>* ffac = reinterpret_cast<Cx<double>*>(smem_raw + off);
  if (FUSE) off += (size_t)W * fz.n_fac * sizeof(Cx<double>);
  Cx<double>* ntab = reinterpret_cast<Cx<double>*>(smem_raw + off);

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n_bt = (n_batch + W - 1) / W;
  // SMALL: tile t is batch tile t % n_bt of state t / n_bt
  const long n_tiles = (long)n_bt * (SMALL ? ms.n_states : WHOLE ? 1 : n_fibers);
  const int G = gridDim.x;
  const int bid = (G & 7) == 0 ? (int)(blockIdx.x & 7) * (G >> 3) + (int)(blockIdx.x >> 3)
                               : (int)blockIdx.x;
  long t = bid;
  if (t >= n_tiles) return;

  if (wave < NW) {
    // ------------------------------------------------------ compute waves
    const int lane = tid & 63;
    constexpr int NTC = 64 * NW;
    auto stage_tables = [&](int kp) {
      const uint32_t* im = tb.image + (long)(kp - tb.kp_lo) * tb.dwords;
      for (int k = tid; k < tb.dwords; k += NTC) img[k] = im[k];
    };
    // Touches the lines of the pass program, so that a sub-pass's scalar loads
    // find them in the scalar cache: the program was just copied to device
    // memory, and a launch that gives a workgroup one tile would wait for
    // memory once per layer pair (norb 12: 22 of them).
    auto warm = [&](const LayerPair* L) {
      const uint32_t* q = reinterpret_cast<const uint32_t*>(L);
      const int n = 2 * n_layers;
      uint32_t a = 0;
      for (int l = 8 * wave; l < n; l += 8 * NW) {
#pragma unroll
        for (int k = 0; k < 8; ++k) a |= q[16 * min(l + k, n - 1)];
      }
      asm volatile("" ::"s"(a));
    };
    const LayerPair* layers = layers_g;
    int st = 0;
    if constexpr (SMALL) {
      st = (int)(t / n_bt);
      layers += st * ms.layer_stride;
    }
    int kp = WHOLE ? whole_kp : fibers[(int)(t / n_bt)].kp;
    if (n_sub > 0) {
      stage_tables(kp);
      warm(layers);
      asm volatile("" ::"s"(reinterpret_cast<const uint32_t*>(subs_g)[4 * min(wave, n_sub - 1)]));
    }
    if ((FUSE || SMALL) && tid == 0) *arrived = 0;
    __syncthreads();
    bool odd = true;  // where the tile lies (see exchange)
    while (true) {
      unsigned char* cur = smem_raw + (odd ? LANES * 16 : 0);
      odd = !odd;
      for (int sp = 0; sp < n_sub; ++sp) {
        const SubPass P = subs_g[sp];
        const PipeSlot gs = gslot[P.slot];
        const LayerPair* lp = layers + P.lp0;
        const int c0 = (int)wsched[(P.slot * NW + wave) * 2];
        const int nc = (int)wsched[(P.slot * NW + wave) * 2 + 1];
        for (int c = 0; c < nc; ++c) {
          const uint32_t ch = wchunks[c0 + c];
          const int gl = lane / (W / NC), j = lane % (W / NC);
          if (gl < (int)(ch & 0xff)) {
            const uint32_t d = gdesc[gs.d_off + (int)(ch >> 8) + gl];
            unsigned char* p = cur + (d >> 16) * (16 * UNITS) + j * (int)(NC * sizeof(Cx<T>));
            const uint32_t* mo = goff + gs.o_off + ((d >> 4) & 0xfff) * 4;
            const bool flip = (d >> 3) & 1;
            switch (d & 7) {
              case 1: pipe_group_apply<T, W2, 1, NC>(p, mo, lp, P.n_lp, flip); break;
              case 2: pipe_group_apply<T, W2, 2, NC>(p, mo, lp, P.n_lp, flip); break;
              case 3: pipe_group_apply<T, W2, 3, NC>(p, mo, lp, P.n_lp, flip); break;
              // complex64 groups of 4 and 5 electrons are complemented ones of 2 and 1
              case 4: if constexpr (sizeof(T) == 8) pipe_group_apply<T, W2, 4, NC>(p, mo, lp, P.n_lp, flip); break;
              case 5: if constexpr (sizeof(T) == 8) pipe_group_apply<T, W2, 5, NC>(p, mo, lp, P.n_lp, flip); break;
              default: break;
            }
          }
        }
        __syncthreads();
      }
      // the memory waves exchange the tile; meanwhile the next fiber's tables or
      // the next state's program
      const long tn = t + G;
      if (tn < n_tiles && n_sub > 0) {
        if constexpr (SMALL) {
          const int sn = (int)(tn / n_bt);
          if (sn != st) {
            st = sn;
            layers = layers_g + st * ms.layer_stride;
            warm(layers);
          }
        } else if constexpr (!WHOLE) {
          const int kpn = fibers[(int)(tn / n_bt)].kp;
          if (kpn != kp) stage_tables(kpn);
          kp = kpn;
        }
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
  // products of the phases over each nibble's patterns
  auto build_ptab = [&](const double* d) {
    if (m < 16 * nt) {
      const int t4 = 4 * (m >> 4), pat = m & 15;
      Cx<double> P{1.0, 0.0};
#pragma unroll 1
      for (int b = 0; b < 4; ++b)
        if (((pat >> b) & 1) && t4 + b < win_w)
          P = cmul(P, Cx<double>{d[2 * (win_lo + t4 + b)], d[2 * (win_lo + t4 + b) + 1]});
      ptab[m] = P;
    }
  };
  if constexpr (DG && !SMALL) build_ptab(diag);
  // what this thread needs of a fiber's strings (i = i0 + STEP k): their rows, and
  // their bits inside the window for the phases
  auto stage_rows = [&](const Fiber& fd, int slot) {
    if constexpr (!CONTIG || DG || FUSE) {
#pragma unroll 1
      for (int k = 0; k < SWEEPS; ++k) {
        const int i = i0 + k * STEP;
        const int r = WHOLE ? min(i, fd.n_rows - 1) : row_table[fd.row_off + min(i, fd.n_rows - 1)];
        if constexpr (!CONTIG) rslot[slot * R + i] = r;
        if constexpr (DG || FUSE)
          lbits[slot * R + i] = (uint16_t)((strings[r] & win_mask) >> win_lo);
      }
    }
    if constexpr (DG && !WHOLE) {
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
        const int e = min(m + LANES * k, W * fz.n_fac - 1);
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
        const int e = m + LANES * k;
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
      for (int e = m; e < (nt * 16 + 1) * W; e += LANES) {
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
    if constexpr (FUSE || SMALL) {
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
  // (a single complex64 column: strings on columns, both halves of a unit hold it)
  auto unit_col = [&](int b0) {
    const int c = min(b0 + u * EU, n_batch - EU);
    return COLS && EU > 1 ? max(c, 0) : c;
  };
  // register k holds sweep k of its tile, or sweep SWEEPS - 1 - k (see exchange): string
  // first + k step.  Transposing passes work on contiguous rows (window [0, w)).
  auto load = [&](auto k0c, auto k1c, const Cx<T>* base, int first, int step, int slot, int nr,
                  int row0, int b0) {
    constexpr int K0 = decltype(k0c)::value, K1 = decltype(k1c)::value;
    __builtin_amdgcn_sched_barrier(0);
    uint32_t row[K1 - K0];
#pragma unroll
    for (int k = K0; k < K1; ++k)
      row[k - K0] = CONTIG ? (uint32_t)(row0 + min(first + k * step, nr - 1))
                           : (uint32_t)rslot[slot * R + first + k * step];
    if constexpr (COLS) {
      const Cx<T>* p = base + (uint64_t)(uint32_t)unit_col(b0) * (uint32_t)ld_src;
      const uint32_t ldz = n_batch < EU ? 0 : (uint32_t)ld_src;
#pragma unroll
      for (int k = K0; k < K1; ++k) {
        Cx<T> e[EU];
#pragma unroll
        for (int z = 0; z < EU; ++z) e[z] = p[(uint64_t)z * ldz + row[k - K0]];
        __builtin_memcpy(&buf[k], e, 16);
      }
    } else {
      const Cx<T>* p = base + unit_col(b0);
#pragma unroll
      for (int k = K0; k < K1; ++k)
        buf[k] = *reinterpret_cast<const u32x4_a8*>(p + (uint64_t)row[k - K0] * (uint32_t)ld_src);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  Cx<double> po[EU];  // the stored tile's factor shared by all its strings
  auto store = [&](auto k0c, auto k1c, Cx<T>* base, int first, int step, int nr, int slot, int row0,
                   int b0) {
    constexpr int K0 = decltype(k0c)::value, K1 = decltype(k1c)::value;
    const bool full = b0 + W <= n_batch;
    const int c0 = unit_col(b0), skip = b0 + u * EU - c0;
    const bool single = COLS && n_batch < EU;
#pragma unroll
    for (int k = K0; k < K1; ++k) {
      const int i = first + k * step;
      if (i < nr) {
        const uint32_t row =
            CONTIG ? (uint32_t)(row0 + i) : (uint32_t)rslot[slot * R + i];
        u32x4 q = buf[k];
        Cx<T> e[EU];
        __builtin_memcpy(e, &q, 16);
        if ((DG || FUSE) && (!SMALL || diag)) {
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
              P = SMALL ? Q : cmul(Q, po[z]);
            }
            const T pr = (T)P.re, pi = (T)P.im;
            const T a = e[z].re * pr - e[z].im * pi;
            e[z].im = e[z].re * pi + e[z].im * pr;
            e[z].re = a;
          }
          __builtin_memcpy(&q, e, 16);
        }
        if constexpr (TST || COLS) {
#pragma unroll
          for (int z = 0; z < EU; ++z)
            if (full || (z >= skip && (z == 0 || !single)))
              base[(uint64_t)(uint32_t)(c0 + z) * (uint32_t)ld_dst + row] = e[z];
        } else {
          Cx<T>* p = base + c0 + (uint64_t)row * (uint32_t)ld_dst;
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
  int p_nr = 0, p_b0 = 0, p_slot = 0, p_row0 = 0, p_st = 0;            // tile q - 2
  int c_nr = 0, c_b0 = 0, c_slot = 0, c_row0 = 0, c_st = 0, c_f = -1;  // tile q - 1
  uint64_t p_fixed = 0, c_fixed = 0;  // electrons outside the window
  int built = -1;                     // the state whose phases ptab holds
  int bars_per_tile = 0;
  bool up = true;  // the first tile goes to sweep 1
  auto state_ptr = [&](int st) -> Cx<T>* {
    if constexpr (SMALL) {
      if (ms.states) return reinterpret_cast<Cx<T>*>(ms.states[st]);
    }
    return dst;
  };
  auto tile_factor = [&]() {
    if constexpr (SMALL) {
      if (diag && p_st != built) {
        // (between two tiles' stores: the exchange's barriers lie between them)
        built = p_st;
        build_ptab(diag + p_st * ms.diag_stride);
        meet();
      }
    } else if constexpr (DG) {
      // the phase of the fiber's electrons outside the window, and the column
      // factor that the previous gate left to this pass
#pragma unroll
      for (int z = 0; z < EU; ++z) {
        po[z] = WHOLE ? Cx<double>{1.0, 0.0} : pout[p_slot];
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
    const int f = WHOLE ? 0 : more ? (int)(t / n_bt) : c_f;
    const int n_st = SMALL && more ? (int)(t / n_bt) : c_st;
    const int n_b0 = more ? (int)(t % n_bt) * W : c_b0;
    const Fiber fn = WHOLE ? Fiber{0, whole_rows, whole_kp, 0} : fibers[f];
    int step = up ? -STEP : STEP, mv = m;
    // (opaque: the compiler would otherwise keep the loop-invariant addresses
    // of every sweep in registers)
    asm volatile("" : "+s"(step), "+v"(mv));
    const int first = mv / UNITS + (up ? R - STEP : 0);
    const int p_first = mv / UNITS + (up ? 0 : R - STEP);
    int n_slot = c_slot, n_row0 = c_row0;
    uint64_t n_fixed = c_fixed;
    const bool new_fiber = f != c_f;
    if (new_fiber) {
      n_slot = c_slot + 1 >= SLOTS ? 0 : c_slot + 1;
      if constexpr (!CONTIG) stage_rows(fn, n_slot);
      if constexpr (!WHOLE) {
        n_row0 = row_table[fn.row_off];
        if (FUSE) n_fixed = strings[n_row0] & ~win_mask;
      }
    }
    if (p_nr > 0) tile_factor();
    const Cx<T>* n_src = SMALL ? state_ptr(n_st) : src;
    Cx<T>* p_dst = state_ptr(p_st);
    int bars = 0;
    auto upto = [&](int n) {
#pragma unroll 1
      for (; bars < n; ++bars) __syncthreads();
    };
    // the stores and loads of a tile are spread evenly over its sub-passes
#define FFSIM_PORTION(N)                                                                  \
  store(KC((N - 1) * SWEEPS / 8), KC(N * SWEEPS / 8), p_dst, p_first, -step, p_nr, p_slot, \
        p_row0, p_b0);                                                                    \
  load(KC((N - 1) * SWEEPS / 8), KC(N * SWEEPS / 8), n_src, first, step, n_slot, fn.n_rows, \
       n_row0, n_b0);                                                                     \
  upto((bars_per_tile * N + 5) / 9);
    FFSIM_PORTION(1)
    FFSIM_PORTION(2)
    FFSIM_PORTION(3)
    FFSIM_PORTION(4)
    FFSIM_PORTION(5)
    FFSIM_PORTION(6)
    FFSIM_PORTION(7)
    FFSIM_PORTION(8)
#undef FFSIM_PORTION
    // (read by the stores of this tile, after the exchange)
    if constexpr (CONTIG) {
      if (new_fiber) stage_rows(fn, n_slot);
    }
    load_bfac(c_b0);
    upto(bars_per_tile);
    write_ffac();
    exchange(mv + (up ? SWEEPS * LANES : 0), mv + (up ? (SWEEPS - 1) * LANES : LANES),
             up ? -LANES : LANES);
    up = !up;
    __syncthreads();
    p_nr = c_nr;
    p_b0 = c_b0;
    p_slot = c_slot;
    p_row0 = c_row0;
    p_st = c_st;
    p_fixed = c_fixed;
    c_nr = fn.n_rows;
    c_f = f;
    c_b0 = n_b0;
    c_slot = n_slot;
    c_row0 = n_row0;
    c_st = n_st;
    c_fixed = n_fixed;
    t += G;
    bars_per_tile = n_sub;
    if (!more) break;
  }
  const int step = up ? -STEP : STEP;
  const int p_first = i0 + (up ? 0 : R - STEP);
  tile_factor();
  Cx<T>* p_dst = state_ptr(p_st);
  store(KC(0), KC(SWEEPS / 4), p_dst, p_first, -step, p_nr, p_slot, p_row0, p_b0);
  store(KC(SWEEPS / 4), KC(SWEEPS / 2), p_dst, p_first, -step, p_nr, p_slot, p_row0, p_b0);
  store(KC(SWEEPS / 2), KC(SWEEPS), p_dst, p_first, -step, p_nr, p_slot, p_row0, p_b0);
#undef KC
}

// Kernel of a tile geometry and variant (the launching code and the
// instantiations of each type are compiled apart).
template <typename T, int UNITS, int NC>
const void* pipe_kernel_units(int variant) {
  constexpr int S = pipe_sweeps(UNITS);
  switch (variant) {
    case PIPE_PLAIN:
      return (const void*)fiber_pipe_kernel<T, UNITS, S, NC, false, false, false, false, false>;
    case PIPE_PHASES:
      return (const void*)fiber_pipe_kernel<T, UNITS, S, NC, false, true, false, false, false>;
    case PIPE_TRANSPOSE:
      return (const void*)fiber_pipe_kernel<T, UNITS, S, NC, true, false, false, false, false>;
    case PIPE_TRANSPOSE_PHASES:
      return (const void*)fiber_pipe_kernel<T, UNITS, S, NC, true, true, false, false, false>;
    default: return (const void*)fiber_pipe_kernel<T, UNITS, S, NC, true, false, true, false, false>;
  }
}
template <typename T, int UNITS, int SWEEPS, int NC>
const void* pipe_kernel_small(int variant) {
  return variant == PIPE_SMALL_ROWS
             ? (const void*)fiber_pipe_kernel<T, UNITS, SWEEPS, NC, false, true, false, true, false>
             : (const void*)fiber_pipe_kernel<T, UNITS, SWEEPS, NC, false, true, false, true, true>;
}
template <typename T>
const void* pipe_kernel(int units, int sweeps, int cols, int variant) {
  constexpr int EU = 16 / (int)sizeof(Cx<T>);  // columns of a unit
  if (cols != 1 && cols != EU) return nullptr;
  if (variant >= PIPE_SMALL_ROWS) {
    if (cols == 1) {
      if (units == 4 && sweeps == 15) return pipe_kernel_small<T, 4, 15, 1>(variant);
      if (units == 8 && sweeps == 8) return pipe_kernel_small<T, 8, 8, 1>(variant);
      if (units == 8 && sweeps == 15) return pipe_kernel_small<T, 8, 15, 1>(variant);
      if (units == 16 && sweeps == 16) return pipe_kernel_small<T, 16, 16, 1>(variant);
    }
    if (units == 8 && sweeps == 29)
      return cols == 1 ? pipe_kernel_small<T, 8, 29, 1>(variant)
                       : pipe_kernel_small<T, 8, 29, EU>(variant);
    if (units == 16 && sweeps == 29)
      return cols == 1 ? pipe_kernel_small<T, 16, 29, 1>(variant)
                       : pipe_kernel_small<T, 16, 29, EU>(variant);
    return nullptr;
  }
  if (sweeps != pipe_sweeps(units) || cols != pipe_cols(units, sizeof(Cx<T>))) return nullptr;
  switch (units) {
    case 8: return pipe_kernel_units<T, 8, EU>(variant);
    case 4: return pipe_kernel_units<T, 4, 1>(variant);
    case 2: return pipe_kernel_units<T, 2, EU>(variant);
    case 1: return pipe_kernel_units<T, 1, EU>(variant);
    default: return nullptr;
  }
}
const void* pipe_kernel_c128(int units, int sweeps, int cols, int variant);
const void* pipe_kernel_c64(int units, int sweeps, int cols, int variant);

}  // namespace ffsim_amd
