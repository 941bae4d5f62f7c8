// wt_colseg.h -- region geometry and memory access shared by the temporally
// blocked column-segment kernels (wt_colseg.hip in float, wt_f64_blocked.hip in
// double; the thread mapping is described in wt_colseg.hip).  Not part of the
// public ABI.
#pragma once

#include <utility>

#include "wt_internal.h"

namespace wt {

// Largest number of steps one launch of these kernels may take (the input
// samples of a launch are staged in LDS).
constexpr int CS_MAX_TBLOCK = 256;
// Largest number of special pixels / probe taps one tile may hold.
constexpr int CS_MAX_TABLE = 256;
// Static LDS of the float kernels next to the launch's dynamic LDS, at most.
constexpr int CS_STATIC_LDS = 7424;
// Probe-seed table: at most this many probe pixels per region.
constexpr int CS_MAX_SEEDS = 16;

struct CsGeom {
  int R0, RH, C0, RW;     // region
  int or0, or1, oc0, oc1; // output rows / cols (domain)
  int k, c;               // segment, column of this thread
  int RWm;                // thread-mapping width: t = k * RWm + c
  bool active;            // thread owns cells
  int CS;                 // LDS column stride (odd)
  int base;               // LDS index of this thread's first cell
};

// LAYOUT: take the thread-mapping width and LDS column stride the host chose
// (cs_layout, descriptor words 12 and 13; the plain mapping unless they fit
// this launch's rows per thread and threads) -- the forward kernels, whose
// LDS allocation holds the padded stride.  Otherwise (the adjoints, which
// wait little on LDS) the plain mapping t -> (t / RW, t % RW).
template <int R, bool LAYOUT = false>
__device__ __forceinline__ CsGeom cs_geom(const int32_t *td, int tid) {
  CsGeom g;
  g.R0 = td[0]; g.RH = td[1]; g.C0 = td[2]; g.RW = td[3];
  g.or0 = td[4]; g.or1 = td[5]; g.oc0 = td[6]; g.oc1 = td[7];
  const int nseg = (g.RH + R - 1) / R;
  if constexpr (LAYOUT) {
    int RWm = td[12], CS = td[13];
    if (RWm < g.RW || CS < nseg * R + 2 || CS > ((nseg * R + 2) | 1) + cs_lds_slack(R) ||
        RWm * nseg > (int)blockDim.x) {
      RWm = g.RW;
      CS = (nseg * R + 2) | 1;
    }
    g.CS = CS;
    g.RWm = RWm;
    g.k = tid / RWm;
    g.c = tid - g.k * RWm;
    g.active = g.k < nseg && g.c < g.RW;
  } else {
    g.RWm = g.RW;
    g.k = tid / g.RW;
    g.c = tid - g.k * g.RW;
    g.active = g.k < nseg;
    g.CS = (nseg * R + 2) | 1;
  }
  g.base = (g.c + 1) * g.CS + g.k * R + 1;
  return g;
}

// Steps of a launch of n in which this thread's rows still influence the
// output rows: the halo shrinks by a row a step, so they are its first ones
// (0 for a thread without cells).
template <int R>
__device__ __forceinline__ int cs_live_steps(const CsGeom &g, int row0, int n) {
  const int olo = g.or0 - g.R0, ohi = g.or1 - g.R0;
  int q = 0;  // steps that must be left
  if (ohi < g.RH) q = max(q, row0 - ohi + 1);
  if (olo > 0) q = max(q, olo - row0 - R + 1);
  return g.active ? n - q : 0;
}

// Owner of the region cell (x, y): thread k * RWm + c, its row r in [0, R);
// -1 outside the region.
template <int R>
__device__ __forceinline__ int cs_owner(const CsGeom &g, int x, int y, int &r) {
  const int rr = x - g.R0, cc = y - g.C0;
  if (rr < 0 || rr >= g.RH || cc < 0 || cc >= g.RW) return -1;
  const int k = rr / R;
  r = rr - k * R;
  return k * g.RWm + cc;
}

// Special pixels of a region for the adjoints.  The table's entries find
// their owners (a scan of the whole table in every thread, and in one thread
// for the probe pixels, took about half of a launch with a line source of 100
// pixels): entry kk lowers own[owner] and raises own[n + owner] (n =
// blockDim.x; at most two entries per thread, so the two extremes are both of
// them), and its probe-seed slot is its rank among the probe pixels, which
// the host stored as a prefix count (word 6).  Phases, a barrier between each:
// cs_special_load, then cs_special_stage, cs_special_scatter, cs_special_read.
constexpr int CS_SP_W = 7;
struct CsSpecials {
  int sr0 = -1, sr1 = -1, sd0 = -1, sd1 = -1, sl0 = -1, sl1 = -1;  // row, seed slot, source slot
};
// This thread's entry of the table (loads only: they travel with the set-up's
// other loads), then table and owners' extremes in LDS.
__device__ __forceinline__ void cs_special_load(const int32_t *spx, int lo, int nsp,
                                                int (&e)[CS_SP_W]) {
#pragma unroll
  for (int j = 0; j < CS_SP_W; ++j) e[j] = 0;
  if ((int)threadIdx.x < nsp) {
    const int32_t *p = spx + (lo + threadIdx.x) * SPX_W;
#pragma unroll
    for (int j = 0; j < CS_SP_W; ++j) e[j] = p[j];
  }
}
__device__ __forceinline__ void cs_special_stage(const int32_t *spx, int lo, int nsp,
                                                 const int (&e)[CS_SP_W], int *tb_sp, int *own) {
  own[threadIdx.x] = 0x7fffffff;
  own[blockDim.x + threadIdx.x] = -1;
  if ((int)threadIdx.x < nsp) {
#pragma unroll
    for (int j = 0; j < CS_SP_W; ++j) tb_sp[CS_SP_W * threadIdx.x + j] = e[j];
  }
  for (int i = threadIdx.x + blockDim.x; i < nsp; i += blockDim.x)  // more entries than threads
    for (int j = 0; j < CS_SP_W; ++j) tb_sp[CS_SP_W * i + j] = spx[(lo + i) * SPX_W + j];
}
template <int R>
__device__ __forceinline__ void cs_special_scatter(const CsGeom &g, int nsp, const int *tb_sp,
                                                   int *own, int *seed_px, int *nseeds) {
  for (int kk = threadIdx.x; kk < nsp; kk += blockDim.x) {
    const int *e = tb_sp + CS_SP_W * kk;
    int r;
    const int t = cs_owner<R>(g, e[0], e[1], r);
    if (t >= 0) {
      atomicMin(&own[t], kk);
      atomicMax(&own[blockDim.x + t], kk);
    }
    const int slot = e[6] - tb_sp[6];
    const bool has_tap = e[5] > e[4];
    if (has_tap && slot < CS_MAX_SEEDS) seed_px[slot] = kk;
    if (kk == nsp - 1) *nseeds = min(slot + (has_tap ? 1 : 0), CS_MAX_SEEDS);
  }
  if (nsp == 0 && threadIdx.x == 0) *nseeds = 0;
}
__device__ __forceinline__ CsSpecials cs_special_read(const CsGeom &g, int row0, const int *tb_sp,
                                                      const int *own) {
  CsSpecials sp;
  const int k0 = own[threadIdx.x], k1 = own[blockDim.x + threadIdx.x];
  if (k1 >= 0) {
    const int *e = tb_sp + CS_SP_W * k0;
    sp.sr0 = e[0] - g.R0 - row0;
    sp.sd0 = e[5] > e[4] ? e[6] - tb_sp[6] : -1;
    sp.sl0 = e[2] > 0 ? e[3] : -1;
    if (k1 > k0) {
      e = tb_sp + CS_SP_W * k1;
      sp.sr1 = e[0] - g.R0 - row0;
      sp.sd1 = e[5] > e[4] ? e[6] - tb_sp[6] : -1;
      sp.sl1 = e[2] > 0 ? e[3] : -1;
    }
  }
  return sp;
}

// Probe tap handled by this thread (taps in the output region): LDS index of
// its cell, kind and output column, or pidx = -1.  Thread t takes tap t;
// blocks of fewer threads than the tile's row range has taps count the ones
// in its columns.  `e`: this thread's row of the table, loaded with the
// set-up's other loads (cs_tap_load).
struct CsTap {
  int pidx = -1, pkind = 0, pcol = 0;
};
__device__ __forceinline__ void cs_tap_load(const int32_t *taps, int lo, int ntp,
                                            int (&e)[TAP_W]) {
#pragma unroll
  for (int j = 0; j < TAP_W; ++j) e[j] = 0;
  if ((int)threadIdx.x < ntp) {
    const int32_t *p = taps + (lo + threadIdx.x) * TAP_W;
#pragma unroll
    for (int j = 0; j < TAP_W; ++j) e[j] = p[j];
  }
}
__device__ __forceinline__ CsTap cs_tap(const CsGeom &g, const int32_t *taps, int lo, int ntp,
                                        int (&e)[TAP_W]) {
  CsTap p;
  bool mine = (int)threadIdx.x < ntp && e[1] >= g.oc0 && e[1] < g.oc1;
  if (ntp > (int)blockDim.x) {
    mine = false;
    for (int t = 0, kk = 0; t < ntp; ++t) {
      const int32_t *q = taps + (lo + t) * TAP_W;
      if (q[1] < g.oc0 || q[1] >= g.oc1) continue;
      if (kk++ == (int)threadIdx.x) {
        mine = true;
        for (int j = 0; j < TAP_W; ++j) e[j] = q[j];
      }
    }
  }
  if (mine) {
    p.pidx = (e[1] - g.C0 + 1) * g.CS + (e[0] - g.R0) + 1;
    p.pkind = e[2];
    p.pcol = e[3];
  }
  return p;
}

// Special rows after a step's rows are done: one code path computes every
// row, and the waves that hold a special pixel then pick its row with selects,
// change it and put it back (registers and LDS), instead of carrying the
// addition through every row of every wave.
// (Written out by expansion: of a loop over r == row the compiler makes an
// indexed access, which moves the rows from registers to scratch memory.)
template <int R, typename T, int... I>
__device__ __forceinline__ T cs_pick_(const T (&v)[R], int row,
                                      std::integer_sequence<int, I...>) {
  T x = v[0];
  ((x = (I == row) ? v[I] : x), ...);
  return x;
}
template <int R, typename T>
__device__ __forceinline__ T cs_pick(const T (&v)[R], int row) {
  return cs_pick_<R>(v, row, std::make_integer_sequence<int, R>{});
}
template <int R, typename T, int... I>
__device__ __forceinline__ void cs_put_(T (&v)[R], int row, T x,
                                        std::integer_sequence<int, I...>) {
  ((v[I] = (I == row) ? x : v[I]), ...);
}
template <int R, typename T>
__device__ __forceinline__ void cs_put(T (&v)[R], int row, T x) {
  cs_put_<R>(v, row, x, std::make_integer_sequence<int, R>{});
}
// Adds x_n to the rows in the mask `srows` (bit r: row r is a source pixel):
// `one`: no lane of the wave holds more than one.
template <int R, typename T>
__device__ __forceinline__ void cs_add_source(T (&v)[R], T *Q, int srows, bool one, T xv) {
  if (one) {
    const int row = __ffs(srows) - 1;
    const T x = cs_pick<R>(v, row) + xv;
    cs_put<R>(v, row, x);
    if (row >= 0) Q[row] = x;
  } else {
#pragma unroll
    for (int r = 0; r < R; ++r)
      if ((srows >> r) & 1) {
        v[r] = v[r] + xv;
        Q[r] = v[r];
      }
  }
}

// A special pixel of this thread in a reverse step: seed `gs` added to its
// row (LDS too, as w * lambda), and lambda_m stored for dJ/dx where the pixel
// is a source of the output rows (`gx`, else null).
template <int R, typename T>
__device__ __forceinline__ void cs_adj_special(T (&Ln)[R], T *Q, int row, T kw, T gs, T *gx) {
  const T v = cs_pick<R>(Ln, row) + gs;
  cs_put<R>(Ln, row, v);
  if (row >= 0) Q[row] = kw * v;
  if (gx) *gx = v;
}

// Raw buffer access with hardware range checking (gfx9 descriptor word 3 =
// 0x00020000): a load outside [0, num_records) bytes returns 0 and a store
// there is dropped.  The slices below put the buffer base at the first
// output row of the tile, so rows above the output rows give negative byte
// offsets (huge as unsigned) and rows below give offsets >= num_records:
// both fall outside the range without any per-row predicate.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t cs_rsrc(const void *p, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void *)p, (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ float cs_bload(__amdgpu_buffer_rsrc_t rs, uint32_t off) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, (int)off, 0, 0));
}
__device__ __forceinline__ void cs_bstore(__amdgpu_buffer_rsrc_t rs, uint32_t off, float v) {
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), rs, (int)off, 0, 0);
}
// Byte offset of this thread's first cell relative to the first output row
// of its tile (column C0 + c); an out-of-range marker if the thread's column
// is outside the tile's output columns.
template <typename T>
__device__ __forceinline__ uint32_t cs_out_voff(const CsGeom &g, int row0, int Ny) {
  const int gc = g.C0 + g.c;
  if (!g.active || gc < g.oc0 || gc >= g.oc1) return 0x80000000u;
  return (uint32_t)(((g.R0 + row0 - g.or0) * Ny + gc) * (int)sizeof(T));
}

// Zeroes LDS buffer b1 and, of b0, only the cells that the workgroup's fill
// of b0 (every cell of every segment of the region's columns) leaves alone:
// the ring columns 0 and RW+1 and, in the region's columns, the ring row 0
// and the rows past the last segment (CS - nrows cells per column).
template <typename T>
__device__ __forceinline__ void cs_zero_lds(T *b0, T *b1, const CsGeom &g, int nrows,
                                            int NBUF) {
  for (int i = threadIdx.x; i < NBUF; i += blockDim.x) b1[i] = T(0);
  const int tail = g.CS - nrows;
  const int nring = 2 * g.CS + g.RW * tail;
  for (int i = threadIdx.x; i < nring; i += blockDim.x) {
    int idx;
    if (i < g.CS) {
      idx = i;
    } else if (i < 2 * g.CS) {
      idx = (g.RW + 1) * g.CS + (i - g.CS);
    } else {
      const int j = i - 2 * g.CS, col = j / tail, r = j - col * tail;
      idx = (col + 1) * g.CS + (r == 0 ? 0 : nrows + r);
    }
    b0[idx] = T(0);
  }
}

// Resident sweeps: one launch walks all T steps in chunks,
// each workgroup with its own tile, whose cells and coefficients stay in its
// registers.  Between two chunks only the halo is read again, from the state
// that the neighbours stored: that exchange takes about 3 us (the stores'
// and the flag's way to the memory side, a poll, the halo loads), a launch
// and its set-up 6 to 10 us.
//
// Word w of `prog` (CS_WALK_W ints apart, zero at the start) holds 1 + the
// chunks that work item w's owner has done, 0 while it has no owner.  Chunk n
// starts when every tile whose output reaches into this region has n chunks
// done; tiles reach into each other mutually, so these are then also past
// reading the state that chunk n overwrites (two pairs of fields alternate).
// A workgroup raises its word when all of its stores have completed.
//
// The device holds all workgroups of such a launch at once, but nothing
// relies on it (another stream's work may hold compute units): a workgroup
// that waits for a tile without an owner takes the tile over after
// CS_WALK_US, and an owner of several works on the one with the fewest
// chunks.  So the least advanced of all tiles has an owner that works on it,
// or a neighbour that will take it, or none that waits for it while its own
// workgroup is still to start; every wait ends.
constexpr int CS_WALK_US = 50;

// A value the compiler knows nothing about: what is derived from it per row
// is formed where it is used.  (Of loop-invariant row predicates and offsets
// it keeps one pair of scalar registers each, and spills 100 of them.)
template <typename T>
__device__ __forceinline__ T cs_opaque(T v) {
  asm volatile("" : "+v"(v));
  return v;
}

// State shared between the workgroups of one launch: accessed at device
// scope, the eight dies' L2 caches are not coherent for ordinary accesses.
template <typename T>
__device__ __forceinline__ T cs_dev_load(const T *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void cs_dev_store(T *p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// First wave: waits until the tiles of sample b in `nbr` (bit q of lane l:
// tile l + 64 q) have n chunks done.  -1: they have; -2: given up after about
// a minute (HOOK: at once where `give_up` says so); else the work item without
// an owner that was taken over.
template <bool HOOK>
__device__ __forceinline__ int cs_walk_wait(int *prog, int ntiles, int b, int nbr, int n,
                                            int give_up) {
  if (HOOK && give_up) return -2;
  const int lane = cs_opaque((int)threadIdx.x);
  nbr = cs_opaque(nbr);
  const uint64_t t0 = wall_clock64();
  for (int polls = 0; polls < (1 << 26); ++polls) {
    bool ok = true;
    int unowned = -1;
#pragma unroll
    for (int q = 0; q < CS_WALK_MAX / 64; ++q)
      if ((nbr >> q) & 1) {
        const int j = b * ntiles + lane + 64 * q;
        const int v = __hip_atomic_load(prog + j * CS_WALK_W, __ATOMIC_RELAXED,
                                        __HIP_MEMORY_SCOPE_AGENT);
        if (v < n + 1) ok = false;
        if (v == 0) unowned = j;
      }
    if (__ballot(!ok) == 0) return -1;
    const uint64_t cand = __ballot(unowned >= 0);
    if (cand && wall_clock64() - t0 > 100 * CS_WALK_US) {  // the clock runs at 100 MHz
      const int first = __ffsll((unsigned long long)cand) - 1;
      int got = -1;
      if (lane == first && atomicCAS(prog + unowned * CS_WALK_W, 0, 1) == 0) got = unowned;
      got = __shfl(got, first);
      if (got >= 0) return got;
    }
    __builtin_amdgcn_s_sleep(1);
  }
  return -2;
}

// First wave: the tiles whose output rows and columns reach into tile ti's
// region, as cs_walk_wait takes them.
__device__ __forceinline__ int cs_walk_neighbours(const int32_t *tiles, int ntiles, int ti) {
  const int32_t *td = tiles + ti * TILE_W;
  int nbr = 0;
#pragma unroll
  for (int q = 0; q < CS_WALK_MAX / 64; ++q) {
    const int j = threadIdx.x + 64 * q;
    if (j < ntiles && j != ti) {
      const int32_t *o = tiles + j * TILE_W;
      if (o[4] < td[0] + td[1] && o[5] > td[0] && o[6] < td[2] + td[3] && o[7] > td[2])
        nbr |= 1 << q;
    }
  }
  return nbr;
}

// A wait of a sweep was given up with steps n0 and later of sample b to do:
// NaN to all of their probe values and field snapshots.  (A neighbour's later
// store can only be a value that it could still compute.)
template <typename Args, typename T>
__device__ __forceinline__ void cs_walk_failed(const Args &a, int b, int n0, T nan) {
  auto mark = [&](T *p, int64_t per, int64_t lo, int64_t hi) {
    if (p)
      for (int64_t i = lo * per + threadIdx.x; i < hi * per; i += blockDim.x)
        p[b * hi * per + i] = nan;
  };
  mark(a.y, a.ntap, n0, a.T);
  mark(a.yraw, a.ntap, n0, a.T);
  mark(a.fields, (int64_t)a.Nx * a.Ny, n0 / a.fstride, a.T / a.fstride);
}

// After a chunk's state is stored: when every wave's stores have completed,
// the work item's word.
__device__ __forceinline__ void cs_walk_raise(int *prog, int w, int chunk) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0)
    __hip_atomic_store(prog + w * CS_WALK_W, 2 + chunk, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace wt
