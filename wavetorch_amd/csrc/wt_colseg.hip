// wt_colseg.hip -- column-segment, temporally blocked WaveRNN kernels (gfx950).
//
// Same contract as the flat kernels of wt_tiled.hip (one workgroup advances
// one region = tile + halo of one sample by `nsteps` steps), with a thread
// mapping that keeps vertical neighbours in registers.  A launch's workgroups
// do not wait for each other, but for the resident sweeps (k_fwd_cs_walk,
// k_adj_cs_walk; the scheme stands in wt_colseg.h).
//
//   thread t -> column c = t % RW, segment k = t / RW; it owns the R cells
//   (rows k*R .. k*R+R-1, column c) of the region.  u_n and u_{n-1} of those
//   cells, and their coefficients, live in VGPRs; up/down neighbours are the
//   thread's own registers except at the segment ends.
//
//   LDS holds the field column-major: cell (row, col) at (col+1)*CS + row+1,
//   CS odd (consecutive lanes = consecutive columns hit distinct banks), with
//   a zero column on each side and a zero row above/below.  Per cell and step
//   one LDS write (the new value) and two reads (left, right neighbours);
//   every LDS address is a per-thread base plus an immediate offset.
//
//   Halo cone: rows whose value can no longer reach the output rows before
//   the end of the launch are not computed (whole segments are skipped).
//
// Forward per cell, in the reference's operation order (cell.py:12-17):
//     s = up + lf;  s = fma(-4, ctr, s)  (== s + (-4*ctr): the product is
//     exact);  s = s + rt;  lap = s + dn
//     v = A*(((s2*ctr) - (Bm*u_prev)) + (C2*lap))   then + x_n at sources.
// Adjoint per cell (linear cell, row strips):
//     lam_m = a1*lam_{m+1} + L(w*lam_{m+1}) - a2*lam_{m+2} (+ probe seed)
//     gacc += lap(u_{m-1}) * lam_m
// Cells with a source pixel or a probe tap take a slower code path that only
// the waves containing them execute (wave-uniform branch).
#include "wt_colseg.h"

namespace wt {

// The segment record (lap u, u) is written once by the recompute and read
// once by the adjoint.  Cache policies of those accesses (the buffer
// instructions' cache-policy operand: 2 = nt, 16 = sc1).  Measured on MI355X
// for the training step: nt writes double the recompute's time (the record
// rows are narrower than a cache line); nt reads with default writes slow
// the adjoint by 8%; the default policy on both is fastest overall.
#ifndef WT_RECORD_LOAD_CPOL
#define WT_RECORD_LOAD_CPOL 0
#endif
#ifndef WT_RECORD_STORE_CPOL
#define WT_RECORD_STORE_CPOL 0
#endif
__device__ __forceinline__ float cs_rec_load(__amdgpu_buffer_rsrc_t rs, uint32_t off) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_raw_buffer_load_b32(rs, (int)off, 0, WT_RECORD_LOAD_CPOL));
}
__device__ __forceinline__ void cs_rec_store(__amdgpu_buffer_rsrc_t rs, uint32_t off, float v) {
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), rs, (int)off, 0,
                                        WT_RECORD_STORE_CPOL);
}

// ------------------------------------------------------------------ forward

// Correctly rounded quotients of the nonlinear forward in 3 to 6 operations
// instead of the 11 of the general division (scaling and special cases):
// a quotient from a reciprocal and one residual correction, Markstein's
// method ("IA-64 and Elementary Functions", 2000): q = a y, r = a - b q,
// q + r y, with y = 1/b to the last bit.  Checked on MI355X against the
// general division for all 2^23 mantissas of the variable operand at 141
// exponents and 1032 pairs of constants: not one differs.  Configurations whose
// operands would leave the normal range run other kernels (quotients_hold in
// wt_runtime.hip).
// a / b for a wave-uniform b with rb = 1/b (rounded to nearest)
__device__ __forceinline__ float nl_div_by(float a, float b, float rb) {
  const float q = a * rb;
  return __builtin_fmaf(__builtin_fmaf(-b, q, a), rb, q);
}
// a / b
__device__ __forceinline__ float nl_div(float a, float b) {
  float y = __builtin_amdgcn_rcpf(b);
  y = __builtin_fmaf(__builtin_fmaf(-b, y, 1.0f), y, y);
  const float q = a * y;
  return __builtin_fmaf(__builtin_fmaf(-b, q, a), y, q);
}
// 1 / b
__device__ __forceinline__ float nl_rcp(float b) {
  float y = __builtin_amdgcn_rcpf(b);
  y = __builtin_fmaf(__builtin_fmaf(-b, y, 1.0f), y, y);
  return __builtin_fmaf(__builtin_fmaf(-b, y, 1.0f), y, y);
}

// One forward step of this thread's segment; REC records lap(u_n) (and u_n
// for the nonlinear cell) of the output rows through range-checked buffers.
// UH: grid step 1, where each product with t1 = h^-2 is the value itself and
// -4*ctr is exact.  Otherwise the five products are formed and added in
// conv2d's order, one v_mul per neighbour (the centre's is the product the
// rows above and below use): 15 VALU operations per row instead of 11.
template <int R, int NL, bool REC, bool UH>
__device__ __forceinline__ void cs_fwd_rows(const FwdArgs &a, const float *__restrict__ P,
                                            float *__restrict__ Q,
                                            float (&Uc)[R], float (&Up)[R], const float (&KA)[R],
                                            const float (&KB)[R], const float (&KC)[R],
                                            const float (&KD)[R], int base, int CS,
                                            float ruth, __amdgpu_buffer_rsrc_t rsl, __amdgpu_buffer_rsrc_t rsu,
                                            uint32_t voff, int Ny) {
  const int lfb = base - CS, rtb = base + CS;
  // the row above and, for UH = false, this row times t1
  float upv = UH ? P[base - 1] : a.t1 * P[base - 1];
  float ctv = UH ? 0.0f : a.t1 * Uc[0];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const float ct = Uc[r];
    const float dn = (r < R - 1) ? Uc[r + 1] : P[base + R];
    const float lf = P[lfb + r], rt = P[rtb + r];
    float lap;
    if (UH) {
      float sacc = upv + lf;
      sacc = __builtin_fmaf(-4.0f, ct, sacc);
      sacc = sacc + rt;
      lap = sacc + dn;
      upv = ct;
    } else {
      const float dnv = a.t1 * dn;
      float sacc = upv + a.t1 * lf;
      sacc = sacc + a.t4 * ct;
      sacc = sacc + a.t1 * rt;
      lap = sacc + dnv;
      upv = ctv;
      ctv = dnv;
    }
    float A, Bm, C2;
    if (NL == 0) {
      A = KA[r]; Bm = KB[r]; C2 = KC[r];
    } else {
      float bb = KA[r], cc = KB[r];
      if (a.nlf & 1) {
        // b0 / (1 + |u/uth|^2).  1 + q^2 stops at 2^120 (also where u/uth
        // overflows): b0 over it adds nothing to dt^-2
        const float q = nl_div_by(ct, a.sat_uth, ruth);
        const float d = fminf(q * q + 1.0f, 0x1p120f);
        bb = bb + KC[r] * nl_div(a.sat_b0, d);
      }
      if (a.nlf & 2) cc = cc + KD[r] * (ct * ct);
      if (a.nlf & 4) cc = fminf(fmaxf(cc, a.cmin), a.cmax);
      const float bd = bb * a.dtm1;
      A = nl_rcp(a.dtm2 + bd);
      Bm = a.dtm2 - bd;
      C2 = cc * cc;
    }
    const float p1 = a.s2 * ct;
    const float p2 = Bm * Up[r];
    const float p3 = C2 * lap;
    const float v = A * ((p1 - p2) + p3);
    Up[r] = v;
    Q[base + r] = v;
    if (REC) {
      const uint32_t o = voff + (uint32_t)(r * Ny * 4);
      cs_rec_store(rsl, o, lap);
      if (NL) cs_rec_store(rsu, o, ct);
    }
  }
}

#ifdef WT_PHASE_TIMING
__device__ unsigned long long *wt_phase_ts = nullptr;
#endif

// A forward workgroup's tile: its geometry, special pixels and cells.
template <int R>
struct CsFwd {
  CsGeom g;
  CsTap tap;
  int b, row0, srows;   // sample, region row of cell 0, source rows (bit mask)
  uint32_t vmask, voff; // cells inside the region; cs_out_voff
  bool wave_src, one_src, wave_part;
  float *buf0, *buf1, *xs;
  float U0[R], U1[R];                    // u_n, u_{n-1}
  float KA[R], KB[R], KC[R], KD[R];
};

// Loads tile ti of sample b (state from in1, in2; DEV: shared with other
// workgroups of this launch) and the input samples n0 .. n0 + nsteps - 1,
// and fills buf0.  Ends with a barrier.
template <int R, int NL, bool DEV>
__device__ __forceinline__ void fwd_cs_setup(const FwdArgs &a, CsFwd<R> &S, int b, int ti,
                                             const float *in1, const float *in2, int n0,
                                             int nsteps) {
  extern __shared__ float smem[];
  const int tid = threadIdx.x;
  const int32_t *td = a.tiles + ti * TILE_W;
  S.b = b;
  S.g = cs_geom<R, true>(td, tid);
  const CsGeom &g = S.g;
  const int NBUF = (g.RW + 2) * g.CS;
  S.buf0 = smem;
  S.buf1 = smem + NBUF;
  S.xs = smem + 2 * NBUF;  // the input samples of this launch
  const int Ny = a.Ny;
  const int64_t F = (int64_t)a.Nx * Ny;
  const int64_t boff = (int64_t)b * F;

  // source rows of each thread as a bit mask, filled by the table's entries
  // (behind the input samples, in the space sized for the adjoint's seeds)
  int *own = (int *)(S.xs + CS_MAX_TBLOCK);
  const int nsp = min(td[9] - td[8], CS_MAX_TABLE), ntp = min(td[11] - td[10], CS_MAX_TABLE);

  const int row0 = S.row0 = g.k * R;
  S.vmask = 0;
  // 1) all global loads first (one round trip for the whole set-up)
#pragma unroll
  for (int r = 0; r < R; ++r) {
    float u1 = 0.f, u2 = 0.f, v0 = 0.f, v1 = 0.f, v2 = 0.f, v3 = 0.f;
    if (g.active && row0 + r < g.RH) {
      S.vmask |= 1u << r;
      const int64_t q = (int64_t)(g.R0 + row0 + r) * Ny + (g.C0 + g.c);
      if (NL == 0) {
        v0 = a.A[q]; v1 = a.Bm[q]; v2 = a.C2[q + (int64_t)b * a.c2_bstride];
      } else {
        v0 = a.bgeom[q]; v1 = a.clin[q]; v2 = a.rho[q]; v3 = a.rhoc[q];
      }
      u1 = DEV ? cs_dev_load(in1 + boff + q) : in1[boff + q];
      u2 = DEV ? cs_dev_load(in2 + boff + q) : in2[boff + q];
    }
    S.U0[r] = u1; S.U1[r] = u2;
    S.KA[r] = v0; S.KB[r] = v1; S.KC[r] = v2; S.KD[r] = v3;
  }
  float xsv = 0.0f;
  if (tid < nsteps) xsv = a.x[(int64_t)b * a.T + n0 + tid];
  int spv0 = 0, spv1 = 0, spv2 = 0;
  if (tid < nsp) {
    const int32_t *e = a.spx + (td[8] + tid) * SPX_W;
    spv0 = e[0]; spv1 = e[1]; spv2 = e[2];
  }
  int te[TAP_W];
  cs_tap_load(a.taps, td[10], ntp, te);
  // 2) LDS (buf0's region cells are filled from U0 below)
  cs_zero_lds<float>(S.buf0, S.buf1, g, ((g.RH + R - 1) / R) * R, NBUF);
  own[tid] = 0;
  WT_TS(4);
  if (tid < nsteps) S.xs[tid] = xsv;
  // blocks of fewer threads than steps (small grids)
  for (int i = tid + blockDim.x; i < nsteps; i += blockDim.x)
    S.xs[i] = a.x[(int64_t)b * a.T + n0 + i];
  __syncthreads();
  WT_TS(5);
  if (g.active) {
#pragma unroll
    for (int r = 0; r < R; ++r) S.buf0[g.base + r] = S.U0[r];
  }
  // source pixels (multiplicity 1; the host routes pixels shared by several
  // sources to the other kernels) mark the rows of their owners
  for (int kk = tid; kk < nsp; kk += blockDim.x) {
    if (kk != tid) {  // more entries than threads
      const int32_t *e = a.spx + (td[8] + kk) * SPX_W;
      spv0 = e[0]; spv1 = e[1]; spv2 = e[2];
    }
    int rr;
    const int t = spv2 > 0 ? cs_owner<R>(g, spv0, spv1, rr) : -1;
    if (t >= 0) atomicOr(&own[t], 1 << rr);
  }
  __syncthreads();
  WT_TS(6);
  S.tap = cs_tap(g, a.taps, td[10], ntp, te);
  S.srows = own[tid];
  S.wave_src = __ballot(S.srows != 0) != 0;
  S.one_src = __ballot((S.srows & (S.srows - 1)) != 0) == 0;
  S.wave_part = __ballot(g.active && S.vmask != (1u << R) - 1u) != 0;
  S.voff = cs_out_voff<float>(g, row0, Ny);
}

// Steps n0 .. n0 + nsteps - 1 of the tile: after an even number of them u_n is
// in U0 and buf0, u_{n-1} in U1, after an odd number the other way round.
template <int R, int NL, bool REC, bool BATCH, bool UH>
__device__ __forceinline__ void fwd_cs_steps(const FwdArgs &a, CsFwd<R> &S, int n0, int nsteps) {
  const CsGeom &g = S.g;
  const CsTap &tap = S.tap;
  const int b = S.b, Ny = a.Ny;
  const int64_t F = (int64_t)a.Nx * Ny;
  const uint32_t voff = S.voff;
  const float ruth = NL ? 1.0f / a.sat_uth : 0.0f;
  const int64_t out_bytes = (int64_t)(g.or1 - g.or0) * Ny * 4;
  // record slots of this sample; steps at or past its length are not
  // recorded (empty slice: the stores are dropped)
  const int64_t rslot0 =
      (BATCH && a.rec_soff) ? (int64_t)a.rec_soff[b] : (int64_t)b * a.rec_K;
  const int Lb = (BATCH && a.Tlim) ? a.Tlim[b] : 0x7fffffff;

  // What a step needs beyond its rows is a pointer that moves: the per-step
  // address arithmetic of every wave is on the path between two barriers.
  const int live = cs_live_steps<R>(g, S.row0, nsteps);
  const float *recl = REC ? a.rec_lap + (rslot0 + (n0 - a.rec_n0)) * F + (int64_t)g.or0 * Ny
                          : a.in1;
  const float *recu = (REC && NL) ? a.rec_u + (rslot0 + (n0 - a.rec_n0)) * F +
                                        (int64_t)g.or0 * Ny
                                  : a.in1;
  const int64_t yo = ((int64_t)b * a.T + n0) * a.ntap + tap.pcol;
  float *yp = a.y ? a.y + yo : nullptr, *yrp = a.yraw ? a.yraw + yo : nullptr;
  // next snapshot: at step `snap`, written by the threads from their registers
  int snap = a.fields ? a.fstride - 1 - n0 % a.fstride : -1;
  const float *fp = a.fields ? a.fields +
                                   ((int64_t)b * (a.T / a.fstride) + n0 / a.fstride) * F +
                                   (int64_t)g.or0 * Ny
                             : a.in1;

  auto step = [&](const float *P, float *Q, float(&Uc)[R], float(&Up)[R], int s) {
    // the (sample, step) slice of the record, based at the first output row;
    // steps at or past the sample's length: an empty slice
    const int64_t rbytes = (!BATCH || n0 + s < Lb) ? out_bytes : 0;
    const __amdgpu_buffer_rsrc_t rsl = cs_rsrc(recl, REC ? rbytes : 0);
    const __amdgpu_buffer_rsrc_t rsu = cs_rsrc(recu, (REC && NL) ? rbytes : 0);
    if (s < live) {
      cs_fwd_rows<R, NL, REC, UH>(a, P, Q, Uc, Up, S.KA, S.KB, S.KC, S.KD, g.base, g.CS, ruth,
                                  rsl, rsu, voff, Ny);
      // rows past the region stay zero (the linear cell has A = 0 there)
      if (NL && S.wave_part) {
#pragma unroll
        for (int r = 0; r < R; ++r)
          if (!((S.vmask >> r) & 1u)) {
            Up[r] = 0.0f;
            Q[g.base + r] = 0.0f;
          }
      }
      // v + x_n at the source pixels (source.py:22)
      if (S.wave_src) cs_add_source<R>(Up, Q + g.base, S.srows, S.one_src, S.xs[s]);
      if (s == snap) {
        const __amdgpu_buffer_rsrc_t rf = cs_rsrc(fp, out_bytes);
#pragma unroll
        for (int r = 0; r < R; ++r) cs_bstore(rf, voff + (uint32_t)(r * Ny * 4), Up[r]);
      }
    }
    if (s == snap) {
      snap += a.fstride;
      fp += F;
    }
    if (REC) recl += F;
    if (REC && NL) recu += F;
    __syncthreads();
    if (tap.pidx >= 0) {
      const float v = Q[tap.pidx];
      if (yp) {
        *yp = tap.pkind ? v * v : v;
        yp += a.ntap;
      }
      if (yrp) {
        *yrp = v;
        yrp += a.ntap;
      }
    }
  };

  WT_TS(1);
  int s = 0;
  for (; s + 1 < nsteps; s += 2) {
    step(S.buf0, S.buf1, S.U0, S.U1, s);
    step(S.buf1, S.buf0, S.U1, S.U0, s + 1);
  }
  if (s < nsteps) step(S.buf0, S.buf1, S.U0, S.U1, s);
  WT_TS(2);
}

// Work item w (sample w / ntiles, tile w % ntiles) of the forward launch
// described by `a`; shared by the single-configuration kernel and the
// batched kernel (one launch over several configurations; BATCH compiles in
// the per-sample lengths and record slots).
template <int NT, int R, int NL, bool REC, bool BATCH, bool UH>
__device__ __forceinline__ void fwd_cs_body(const FwdArgs &a, const int w) {
  WT_TS(0);
  const int b = w / a.ntiles, ti = w - (w / a.ntiles) * a.ntiles;
  // a sample whose own length ends before this launch has nothing to do (a
  // recording launch too: the adjoint reads no record of a step at or past
  // the sample's length)
  if (BATCH && a.Tlim && a.n0 >= a.Tlim[b]) return;
  CsFwd<R> S;
  fwd_cs_setup<R, NL, false>(a, S, b, ti, a.in1, a.in2, a.n0, a.nsteps);
  fwd_cs_steps<R, NL, REC, BATCH, UH>(a, S, a.n0, a.nsteps);
  const CsGeom &g = S.g;
  const bool odd = (a.nsteps & 1) != 0;
  if (g.active) {
    const int gc = g.C0 + g.c;
    if (gc >= g.oc0 && gc < g.oc1) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int gr = g.R0 + S.row0 + r;
        if (S.row0 + r < g.RH && gr >= g.or0 && gr < g.or1) {
          const int64_t q = (int64_t)b * a.Nx * a.Ny + (int64_t)gr * a.Ny + gc;
          a.out1[q] = odd ? S.U1[r] : S.U0[r];
          a.out2[q] = odd ? S.U0[r] : S.U1[r];
        }
      }
    }
  }
  WT_TS(3);
}

template <int NT, int R, int NL, bool REC, bool UH = true>
__global__ __launch_bounds__(NT) void k_fwd_cs(FwdArgs a) {
  fwd_cs_body<NT, R, NL, REC, false, UH>(a, xcd_remap(blockIdx.x, gridDim.x));
}

// The resident forward (the scheme stands in wt_colseg.h): 1024 x 1024, one
// sample, 18-step chunks of 256 tiles: 5016 us per 4000 steps with a launch
// per chunk, 3968 us resident; 141 x 141, 24 samples, 1501 steps: 1064 to
// 880 us.
// This thread's output rows of the tile, and its first cell.
template <int R>
__device__ __forceinline__ uint32_t cs_walk_out(const FwdArgs &a, const CsFwd<R> &S, int64_t &q0) {
  const CsGeom &g = S.g;
  uint32_t m = 0;
  if (S.voff != 0x80000000u) {
    const int lo = max(g.or0 - g.R0 - S.row0, 0), hi = min(g.or1 - g.R0 - S.row0, R);
    if (hi > lo) m = ((1u << hi) - 1u) & ~((1u << lo) - 1u) & S.vmask;
  }
  q0 = ((int64_t)S.b * a.Nx + g.R0 + S.row0) * a.Ny + g.C0 + g.c;
  return m;
}

// After chunk `chunk` (of nsteps steps): the later state to V0, and the output
// rows to the state pair that the next chunk reads; then the work item's word.
template <int R, typename Args>
__device__ __forceinline__ void cs_walk_store(const Args &a, float (&V0)[R], float (&V1)[R], int w,
                                              int chunk, int nsteps, uint32_t omask, int64_t q0) {
  if (nsteps & 1) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const float u = V0[r];
      V0[r] = V1[r];
      V1[r] = u;
    }
  }
  const int64_t BF = (int64_t)a.B * a.Nx * a.Ny;
  float *o1 = a.out1 + (chunk & 1) * 2 * BF, *o2 = o1 + BF;
  const uint32_t out = cs_opaque(omask);
  int64_t q = cs_opaque(q0);
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if ((out >> r) & 1u) {
      cs_dev_store(o1 + q, V0[r]);
      cs_dev_store(o2 + q, V1[r]);
    }
    q += a.Ny;
  }
  cs_walk_raise(a.prog, w, chunk);
}

template <int NT, int R, int NL, bool REC, bool UH, bool HOOK = false>
__global__ __launch_bounds__(NT) void k_fwd_cs_walk(FwdArgs a) {
  const int tid = threadIdx.x;
  const int64_t BF = (int64_t)a.B * a.Nx * a.Ny;
  const int nchunks = (a.T + a.nsteps - 1) / a.nsteps;
  __shared__ int msg;
  int w = xcd_remap(blockIdx.x, gridDim.x) * (HOOK ? a.walk.every : 1);
  if (tid == 0) msg = atomicCAS(a.prog + w * CS_WALK_W, 0, 1);
  __syncthreads();
  if (msg != 0) return;  // a neighbour took it over
  CsFwd<R> S;
  int64_t q0;
  int chunk = 0, got;
  {
    const int b = w / a.ntiles, ti = w - b * a.ntiles;
    const int nbr = tid < 64 ? cs_walk_neighbours(a.tiles, a.ntiles, ti) : 0;
    fwd_cs_setup<R, NL, true>(a, S, b, ti, a.in1, a.in2, 0, min(a.nsteps, a.T));
    const uint32_t omask = cs_walk_out<R>(a, S, q0);
    while (true) {
      const int n0 = chunk * a.nsteps, nsteps = min(a.nsteps, a.T - n0);
      fwd_cs_steps<R, NL, REC, false, UH>(a, S, n0, nsteps);
      if (chunk + 1 == nchunks) return;
      cs_walk_store<R>(a, S.U0, S.U1, w, chunk, nsteps, omask, q0);
      ++chunk;
      const int n1 = n0 + nsteps;
      for (int i = tid; i < min(a.nsteps, a.T - n1); i += blockDim.x)
        S.xs[i] = a.x[(int64_t)b * a.T + n1 + i];
      if (tid < 64) {
        const int r = cs_walk_wait<HOOK>(a.prog, a.ntiles, b, nbr, chunk, a.walk.give_up);
        if (tid == 0) msg = r;
      }
      __syncthreads();
      got = msg;
      if (got != -1) break;
      const float *in1 = a.out1 + ((chunk - 1) & 1) * 2 * BF, *in2 = in1 + BF;
      const uint32_t halo = cs_opaque(S.vmask & ~omask);
      int64_t q = cs_opaque(q0);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if ((halo >> r) & 1u) {
          S.U0[r] = cs_dev_load(in1 + q);
          S.U1[r] = cs_dev_load(in2 + q);
        }
        q += a.Ny;
      }
      if (S.g.active) {
#pragma unroll
        for (int r = 0; r < R; ++r) S.buf0[S.g.base + r] = S.U0[r];
      }
      __syncthreads();
    }
  }
  // Work items taken over: from here on every chunk of this workgroup starts
  // with a whole set-up.
  __shared__ int own_w[CS_WALK_MAX], own_n[CS_WALK_MAX];
  int nown = 1, at = 0;
  while (true) {
    // -1: run the chunk that was waited for; >= 0: one more work item
    if (got == -2) {
      cs_walk_failed(a, w / a.ntiles, chunk * a.nsteps, __builtin_nanf(""));
      return;
    }
    if (got >= 0) {
      if (tid == 0) {
        own_w[at] = w;
        own_n[at] = chunk;
        own_w[nown] = got;
        own_n[nown] = 0;
      }
      ++nown;
    } else {
      const int n0 = chunk * a.nsteps, nsteps = min(a.nsteps, a.T - n0);
      const float *in1 = chunk ? a.out1 + ((chunk - 1) & 1) * 2 * BF : a.in1;
      fwd_cs_setup<R, NL, true>(a, S, w / a.ntiles, w % a.ntiles, in1, in1 + BF, n0, nsteps);
      const uint32_t omask = cs_walk_out<R>(a, S, q0);
      fwd_cs_steps<R, NL, REC, false, UH>(a, S, n0, nsteps);
      cs_walk_store<R>(a, S.U0, S.U1, w, chunk, nsteps, omask, q0);
      ++chunk;
      if (chunk == nchunks && --nown == 0) return;
      if (tid == 0) {
        own_n[at] = chunk;
        if (chunk == nchunks) {
          own_w[at] = own_w[nown];
          own_n[at] = own_n[nown];
        }
      }
    }
    __syncthreads();
    at = 0;  // the least advanced one next
    for (int i = 1; i < nown; ++i)
      if (own_n[i] < own_n[at]) at = i;
    w = own_w[at];
    chunk = own_n[at];
    if (tid < 64) {
      const int ti = w % a.ntiles;
      const int r = chunk > 0 ? cs_walk_wait<HOOK>(
                                    a.prog, a.ntiles, w / a.ntiles,
                                    cs_walk_neighbours(a.tiles, a.ntiles, ti), chunk,
                                    a.walk.give_up)
                              : -1;
      if (tid == 0) msg = r;
    }
    __syncthreads();
    got = msg;
  }
}

// Group of a batched launch that work item w belongs to.
__device__ __forceinline__ int batch_group(const int32_t (&start)[WT_MAX_GROUPS + 1], int ngrp,
                                           int w) {
  int gi = 0;
  while (gi + 1 < ngrp && w >= start[gi + 1]) ++gi;
  return gi;
}

template <int NT, int R, int NL, bool REC>
__global__ __launch_bounds__(NT) void k_fwd_cs_batch(BatchFwd bl) {
  const int w = xcd_remap(blockIdx.x, gridDim.x);
  const int gi = batch_group(bl.start, bl.ngrp, w);
  fwd_cs_body<NT, R, NL, REC, true, true>(bl.grp[gi], w - bl.start[gi]);
}

// ------------------------------------------------------------------ adjoint

// One reverse step of this thread's segment, without probe seeds.  a2 = A*Bm
// is formed as a1 - 1 (with a1 = A*s2 = 2/(1+b*dt), a2 = (1-b*dt)/(1+b*dt)).
// The thread's own w*lambda values (up/centre/down neighbours) are re-formed
// as KW*Lc -- the same fp32 product the previous step stored to LDS --
// instead of being kept in R more registers.
template <int R>
__device__ __forceinline__ void cs_adj_rows(const float *__restrict__ P, float *__restrict__ Q,
                                            float (&Lc)[R], float (&Ln)[R],
                                            const float (&KA1)[R], const float (&KW)[R],
                                            int base, int CS) {
  const int lfb = base - CS, rtb = base + CS;
  float upv = P[base - 1];
  float ct = KW[0] * Lc[0];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const float dn = (r < R - 1) ? KW[r + 1] * Lc[r + 1] : P[base + R];
    const float lf = P[lfb + r], rt = P[rtb + r];
    float lapw = upv + lf;
    lapw = __builtin_fmaf(-4.0f, ct, lapw);
    lapw = lapw + rt;
    lapw = lapw + dn;
    // a1*L1 + lapw - (a1-1)*L2 = a1*(L1 - L2) + (lapw + L2)
    const float lam = __builtin_fmaf(KA1[r], Lc[r] - Ln[r], lapw + Ln[r]);
    upv = ct;
    ct = dn;
    Ln[r] = lam;
    Q[base + r] = KW[r] * lam;
  }
}

// An adjoint workgroup's tile.
template <int R>
struct CsAdj {
  CsGeom g;
  CsSpecials sp;        // this thread's special pixels
  int b, row0, Lb;      // sample, region row of cell 0, the sample's length (batches)
  uint32_t omask, voff; // output rows of this thread; cs_out_voff
  bool wave_sp, wave_sp2;
  float kw0, kw1;       // w of the special rows
  float *buf0, *buf1, *seeds;
  float L1[R], L2[R];   // lambda_{m+1}, lambda_{m+2}
  float KA1[R], KW[R];
  float G[R];           // gradient sum of this launch or chunk
  float SG0[R], SG1[R]; // lap(u) of its even and odd steps
};

// Loads tile ti of sample b; DEV: the state is shared with other workgroups of
// this launch.  `tb_sp`, `seed_px`, `nseeds`: the tile's special pixels in LDS.
// Ends before the barrier that must follow adj_cs_start.
template <int R, bool DEV>
__device__ __forceinline__ void adj_cs_setup(const AdjArgs &a, CsAdj<R> &S, int b, int ti,
                                             const float *in1, const float *in2, int *tb_sp,
                                             int *seed_px, int *nseeds) {
  extern __shared__ float smem[];
  const int32_t *td = a.tiles + ti * TILE_W;
  S.b = b;
  S.g = cs_geom<R>(td, threadIdx.x);
  const CsGeom &g = S.g;
  const int NBUF = (g.RW + 2) * g.CS;
  S.buf0 = smem;
  S.buf1 = smem + NBUF;
  S.seeds = smem + 2 * NBUF;  // (CS_MAX_SEEDS, nsteps) probe seeds
  const int Ny = a.Ny;
  const int64_t boff = (int64_t)b * a.Nx * Ny;
  const float s2 = a.s2;

  const int nsp = min(td[9] - td[8], CS_MAX_TABLE);
  const int row0 = S.row0 = g.k * R;
  // 1) all global loads first
  float KC2[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    float A = 0.f, C2 = 0.f, u1 = 0.f, u2 = 0.f;
    if (g.active && row0 + r < g.RH) {
      const int64_t q = (int64_t)(g.R0 + row0 + r) * Ny + (g.C0 + g.c);
      A = a.A[q]; C2 = a.C2[q + (int64_t)b * a.c2_bstride];
      u1 = DEV ? cs_dev_load(in1 + boff + q) : in1[boff + q];
      u2 = DEV ? cs_dev_load(in2 + boff + q) : in2[boff + q];
    }
    S.KA1[r] = A; KC2[r] = C2;
    S.L1[r] = u1; S.L2[r] = u2;
  }
  // (the owners' table lies behind the seeds, or under them in launches of
  // more than 128 steps, with a barrier more)
  int *own = (int *)(S.seeds + (a.nsteps > 128 ? 0 : 128 * CS_MAX_SEEDS));
  int spe[CS_SP_W];
  cs_special_load(a.spx, td[8], nsp, spe);
  // 2) LDS (buf0's region cells are filled from the lambda pair below)
  cs_zero_lds<float>(S.buf0, S.buf1, g, ((g.RH + R - 1) / R) * R, NBUF);
  cs_special_stage(a.spx, td[8], nsp, spe, tb_sp, own);
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const float A = S.KA1[r];
    // w carries the Laplacian's h^-2 (exactly 1 at h = 1): no step pays for it
    S.KA1[r] = A * s2; S.KW[r] = (A * KC2[r]) * a.t1;
  }
  __syncthreads();
  cs_special_scatter<R>(g, nsp, tb_sp, own, seed_px, nseeds);
  if (g.active) {
#pragma unroll
    for (int r = 0; r < R; ++r) S.buf0[g.base + r] = S.KW[r] * S.L1[r];
  }
  __syncthreads();
  // special rows of this thread: probe taps (seed slot) / source pixels (slot)
  S.sp = cs_special_read(g, row0, tb_sp, own);
  if (a.nsteps > 128) __syncthreads();
  // waves with special pixels, with two in a thread
  S.wave_sp = __ballot(S.sp.sr0 >= 0) != 0;
  S.wave_sp2 = __ballot(S.sp.sr1 >= 0) != 0;
  S.kw0 = cs_pick<R>(S.KW, S.sp.sr0);
  S.kw1 = cs_pick<R>(S.KW, S.sp.sr1);
  // output cells of this thread (gradient write-back, dJ/dx)
  S.omask = 0;
  if (g.active && g.C0 + g.c >= g.oc0 && g.C0 + g.c < g.oc1) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int gr = g.R0 + row0 + r;
      if (row0 + r < g.RH && gr >= g.or0 && gr < g.or1) S.omask |= 1u << r;
    }
  }
  S.voff = cs_out_voff<float>(g, row0, Ny);
}

// Record of step j (read at reverse step m = j + 1): a sample's steps at or
// past its length are not recorded, and lambda_m is exactly 0 there, so
// those reads are sent out of range (they return 0).
template <int R, bool BATCH>
__device__ __forceinline__ uint32_t adj_cs_rec_off(const CsAdj<R> &S, uint32_t voff, int j) {
  return (!BATCH || j < S.Lb) ? voff : 0x80000000u;
}
// Slice of the record read at reverse step m (the steps below it lie F values
// before each other).
template <int R, bool BATCH>
__device__ __forceinline__ const float *adj_cs_rec(const AdjArgs &a, const CsAdj<R> &S, int m) {
  const int64_t sslot0 =
      (BATCH && a.seg_soff) ? (int64_t)a.seg_soff[S.b] : (int64_t)S.b * a.seg_K;
  return a.seg_lap + (sslot0 + (m - 1 - a.seg_n0)) * ((int64_t)a.Nx * a.Ny) +
         (int64_t)S.g.or0 * a.Ny;
}

// What the reverse steps m_hi .. m_hi - nsteps + 1 read besides the state:
// probe seeds (a barrier must follow) and the record of the first two.
template <int R, bool BATCH>
__device__ __forceinline__ void adj_cs_start(const AdjArgs &a, CsAdj<R> &S, int m_hi, int nsteps,
                                             const int *tb_sp, const int *seed_px, int nseeds) {
  const int b = S.b, Ny = a.Ny;
  // seeds[k][s] = sum over taps of pixel k of dy/du * ybar at step m = m_hi - s
  for (int i = cs_opaque((int)threadIdx.x); i < nseeds * nsteps; i += blockDim.x) {
    const int k = i / nsteps, s = i - (i / nsteps) * nsteps;
    const int m = m_hi - s;
    const int *e = tb_sp + CS_SP_W * seed_px[k];
    float gs = 0.0f;
    if (a.ybar && (!a.Tlim || m - 1 < a.Tlim[b])) {
      for (int t = e[4]; t < e[5]; ++t) {
        const int32_t *tp = a.taps + t * TAP_W;
        const int64_t o = ((int64_t)b * a.T + (m - 1)) * a.ntap + tp[3];
        const float gy = a.ybar[o];
        gs += tp[2] ? 2.0f * a.yraw[o] * gy : gy;
      }
    }
    S.seeds[i] = gs;
  }
  const int64_t F = (int64_t)a.Nx * Ny, out_bytes = (int64_t)(S.g.or1 - S.g.or0) * Ny * 4;
  const float *rec0 = adj_cs_rec<R, BATCH>(a, S, m_hi);
  const uint32_t voff = cs_opaque(S.voff);
  // lap(u_{m-1}) of the first two steps (SG0: even steps, SG1: odd steps)
  const __amdgpu_buffer_rsrc_t rs0 = cs_rsrc(rec0, out_bytes);
  const uint32_t voff0 = adj_cs_rec_off<R, BATCH>(S, voff, m_hi - 1);
#pragma unroll
  for (int r = 0; r < R; ++r) S.SG0[r] = cs_rec_load(rs0, voff0 + (uint32_t)(r * Ny * 4));
  // issued even for a one-step launch (out of range, reads nothing) so
  // that the loop's wait counts need not cover a path without them
  const bool two = nsteps > 1;
  const __amdgpu_buffer_rsrc_t rs1 = cs_rsrc(two ? rec0 - F : rec0, out_bytes);
  const uint32_t voff1 = two ? adj_cs_rec_off<R, BATCH>(S, voff, m_hi - 2) : 0x80000000u;
#pragma unroll
  for (int r = 0; r < R; ++r) S.SG1[r] = cs_rec_load(rs1, voff1 + (uint32_t)(r * Ny * 4));
#pragma unroll
  for (int r = 0; r < R; ++r) S.G[r] = 0.0f;
}

// Reverse steps m_hi .. m_hi - nsteps + 1: after an even number of them the
// pair (lambda_{m_lo}, lambda_{m_lo + 1}) is (L1, L2), after an odd (L2, L1).
template <int R, bool BATCH>
__device__ __forceinline__ void adj_cs_steps(const AdjArgs &a, CsAdj<R> &S, int m_hi, int nsteps) {
  const CsGeom &g = S.g;
  const int Ny = a.Ny;
  const int64_t F = (int64_t)a.Nx * Ny, out_bytes = (int64_t)(g.or1 - g.or0) * Ny * 4;
  const int live = cs_live_steps<R>(g, S.row0, nsteps);
  const uint32_t voff = cs_opaque(S.voff);
  // the step after next
  const float *recp = adj_cs_rec<R, BATCH>(a, S, m_hi) - 2 * F;
  const bool gx0 = S.sp.sl0 >= 0 && S.sp.sr0 >= 0 && ((S.omask >> S.sp.sr0) & 1u);
  const bool gx1 = S.sp.sl1 >= 0 && S.sp.sr1 >= 0 && ((S.omask >> S.sp.sr1) & 1u);
  float *gsrc_row = a.gsrc + ((int64_t)S.b * a.T + (m_hi - 1)) * a.nsrcslot;

  const float *sd0p = S.seeds + (S.sp.sd0 >= 0 ? S.sp.sd0 * nsteps : 0);
  const float *sd1p = S.seeds + (S.sp.sd1 >= 0 ? S.sp.sd1 * nsteps : 0);

  auto step = [&](const float *P, float *Q, float(&Lc)[R], float(&Ln)[R], float(&SG)[R],
                  int s) {
    // record index m-3-seg_n0 >= 0: m-2 >= m_hi-nsteps+1 >= seg_n0+1
    const bool prefetch = s + 2 < nsteps;
    const __amdgpu_buffer_rsrc_t rsn = cs_rsrc(recp, out_bytes);
    const uint32_t pvoff =
        prefetch ? adj_cs_rec_off<R, BATCH>(S, voff, m_hi - s - 3) : 0x80000000u;
    if (s < live) {
      cs_adj_rows<R>(P, Q, Lc, Ln, S.KA1, S.KW, g.base, g.CS);
      if (S.wave_sp) {
        cs_adj_special<R>(Ln, Q + g.base, S.sp.sr0, S.kw0, S.sp.sd0 >= 0 ? sd0p[s] : 0.0f,
                          gx0 ? gsrc_row + S.sp.sl0 : nullptr);
        if (S.wave_sp2)
          cs_adj_special<R>(Ln, Q + g.base, S.sp.sr1, S.kw1, S.sp.sd1 >= 0 ? sd1p[s] : 0.0f,
                            gx1 ? gsrc_row + S.sp.sl1 : nullptr);
      }
    }
    // gradient sum, then refill SG with lap(u) of step m-2 (the record is
    // read through a range-checked buffer based at the tile's first output
    // row, zero outside the output rows): one issue point
    // outside the branches, so the loads stay in flight across two steps.
    // Threads whose segment left the cone (or own no cells) accumulate
    // stale values into rows that are not output rows and never written.
    // The loads are always issued (pvoff is out of range when there is no
    // step m-2 in this launch) so that the wait counts stay exact.
    // The empty asm keeps each sum in this step: deferred into the next
    // step, the old and the refilled SG would both be live and the loop
    // would copy the fresh loads (waiting for them) at its back edge.
#pragma unroll
    for (int r = 0; r < R; ++r) {
      S.G[r] = __builtin_fmaf(SG[r], Ln[r], S.G[r]);
      asm volatile("" : "+v"(S.G[r]));
      SG[r] = cs_rec_load(rsn, pvoff + (uint32_t)(r * Ny * 4));
    }
    recp -= F;
    gsrc_row -= a.nsrcslot;
    __syncthreads();
  };

  WT_TS(1);
  int s = 0;
  for (; s + 1 < nsteps; s += 2) {
    step(S.buf0, S.buf1, S.L1, S.L2, S.SG0, s);   // lambda_m -> L2
    step(S.buf1, S.buf0, S.L2, S.L1, S.SG1, s + 1);
  }
  if (s < nsteps) step(S.buf0, S.buf1, S.L1, S.L2, S.SG0, s);
  WT_TS(2);
}

// Linear cell.  LDS holds w*lambda.  Work item w of the launch `a` (BATCH:
// the batched kernel, with per-sample lengths and record slots).
template <int NT, int R, bool BATCH>
__device__ __forceinline__ void adj_cs_body(const AdjArgs &a, const int w) {
  WT_TS(0);
  const int b = w / a.ntiles, ti = w - (w / a.ntiles) * a.ntiles;
  // lambda_m = 0 for every m of this launch when the sample ends before it
  if (BATCH && a.Tlim && a.m_hi - a.nsteps + 1 > a.Tlim[b]) return;
  __shared__ int tb_sp[CS_MAX_TABLE * CS_SP_W];
  __shared__ int seed_px[CS_MAX_SEEDS];
  __shared__ int nseeds;
  CsAdj<R> S;
  S.Lb = (BATCH && a.Tlim) ? a.Tlim[b] : 0x7fffffff;
  adj_cs_setup<R, false>(a, S, b, ti, a.in1, a.in2, tb_sp, seed_px, &nseeds);
  adj_cs_start<R, BATCH>(a, S, a.m_hi, a.nsteps, tb_sp, seed_px, nseeds);
  __syncthreads();
  adj_cs_steps<R, BATCH>(a, S, a.m_hi, a.nsteps);
  const CsGeom &g = S.g;
  const bool odd = (a.nsteps & 1) != 0;
  if (g.active) {
    // running gradient sums: all loads first, then the stores
    const int64_t q0 =
        ((int64_t)b * a.Nx + (g.R0 + S.row0)) * a.Ny + (g.C0 + g.c);
    float gold[R];
#pragma unroll
    for (int r = 0; r < R; ++r)
      gold[r] = ((S.omask >> r) & 1u) ? a.gacc[q0 + (int64_t)r * a.Ny] : 0.0f;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if ((S.omask >> r) & 1u) {
        const int64_t q = q0 + (int64_t)r * a.Ny;
        a.out1[q] = odd ? S.L2[r] : S.L1[r];
        a.out2[q] = odd ? S.L1[r] : S.L2[r];
        a.gacc[q] = gold[r] + S.G[r];
      }
    }
  }
  WT_TS(3);
}

template <int NT, int R>
__global__ __launch_bounds__(NT) void k_adj_cs(AdjArgs a) {
  adj_cs_body<NT, R, false>(a, xcd_remap(blockIdx.x, gridDim.x));
}

// Reverse steps of the chunk that starts at m: chunks end at multiples of
// a.group steps, so that the gradient is summed over the same spans whatever
// the record's segments are.
__device__ __forceinline__ int adj_walk_steps(const AdjArgs &a, int m) {
  const int lo = a.group > 0 ? (m - 1) / a.group * a.group : 0;
  return min(a.nsteps, m - lo);
}

// Adds a chunk's gradient sums to the running ones (the output rows have one
// owner from the first chunk to the last).
template <int R>
__device__ __forceinline__ void adj_walk_sum(const AdjArgs &a, const float (&G)[R],
                                             uint32_t omask, int64_t q0) {
  const uint32_t out = cs_opaque(omask);
  const int64_t q = cs_opaque(q0);
  float gold[R];
#pragma unroll
  for (int r = 0; r < R; ++r)
    gold[r] = ((out >> r) & 1u) ? a.gacc[q + (int64_t)r * a.Ny] : 0.0f;
#pragma unroll
  for (int r = 0; r < R; ++r)
    if ((out >> r) & 1u) a.gacc[q + (int64_t)r * a.Ny] = gold[r] + G[r];
}

// The resident adjoint: k_fwd_cs_walk's scheme for the reverse sweep.  The
// record of a chunk's first steps and its probe seeds are read before the
// wait for the neighbours.  The gradient is summed chunk by chunk, as the
// launches of the other path do, in registers where there is room (KEEP).
// (us of a training step, a launch per chunk and resident: 150 x 150, 64
// samples, 3000 steps 9876 and 8729; 100 x 100, 4 samples, 1000 steps 1259
// and 1126; 500 x 380, one sample, 800 steps 1210 and 1063.)
template <int NT, int R, bool HOOK = false>
__global__ __launch_bounds__(NT) void k_adj_cs_walk(AdjArgs a) {
  const int tid = threadIdx.x;
  const int64_t BF = (int64_t)a.B * a.Nx * a.Ny;
  __shared__ int tb_sp[CS_MAX_TABLE * CS_SP_W];
  __shared__ int seed_px[CS_MAX_SEEDS];
  __shared__ int nseeds;
  __shared__ int msg;
  int w = xcd_remap(blockIdx.x, gridDim.x) * (HOOK ? a.walk.every : 1);
  if (tid == 0) msg = atomicCAS(a.prog + w * CS_WALK_W, 0, 1);
  __syncthreads();
  if (msg != 0) return;  // a neighbour took it over
  constexpr bool KEEP = R <= 6;
  CsAdj<R> S;
  float GT[R];
  int64_t q0;
  int chunk = 0, m = a.T, got;
  {
    const int b = w / a.ntiles, ti = w - b * a.ntiles;
    const int nbr = tid < 64 ? cs_walk_neighbours(a.tiles, a.ntiles, ti) : 0;
    adj_cs_setup<R, true>(a, S, b, ti, a.in1, a.in2, tb_sp, seed_px, &nseeds);
    const CsGeom &g = S.g;
    q0 = ((int64_t)b * a.Nx + (g.R0 + S.row0)) * a.Ny + (g.C0 + g.c);
    uint32_t halo = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      GT[r] = 0.0f;
      if (g.active && S.row0 + r < g.RH && !((S.omask >> r) & 1u)) halo |= 1u << r;
    }
    int nsteps = adj_walk_steps(a, m);
    adj_cs_start<R, false>(a, S, m, nsteps, tb_sp, seed_px, nseeds);
    __syncthreads();
    while (true) {
      adj_cs_steps<R, false>(a, S, m, nsteps);
      m -= nsteps;
      if (KEEP) {
#pragma unroll
        for (int r = 0; r < R; ++r) GT[r] = GT[r] + S.G[r];
      }
      if (m > 0) cs_walk_store<R>(a, S.L1, S.L2, w, chunk, nsteps, S.omask, q0);
      if (!KEEP) adj_walk_sum<R>(a, S.G, S.omask, q0);
      if (m == 0) break;
      ++chunk;
      nsteps = adj_walk_steps(a, m);
      adj_cs_start<R, false>(a, S, m, nsteps, tb_sp, seed_px, nseeds);
      if (tid < 64) {
        const int r = cs_walk_wait<HOOK>(a.prog, a.ntiles, b, nbr, chunk, a.walk.give_up);
        if (tid == 0) msg = r;
      }
      __syncthreads();
      got = msg;
      if (got != -1) break;
      const float *in1 = a.out1 + ((chunk - 1) & 1) * 2 * BF, *in2 = in1 + BF;
      const uint32_t hm = cs_opaque(halo);
      int64_t q = cs_opaque(q0);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if ((hm >> r) & 1u) {
          S.L1[r] = cs_dev_load(in1 + q);
          S.L2[r] = cs_dev_load(in2 + q);
        }
        q += a.Ny;
      }
      if (g.active) {
#pragma unroll
        for (int r = 0; r < R; ++r) S.buf0[g.base + r] = S.KW[r] * S.L1[r];
      }
      __syncthreads();
    }
    if (KEEP) adj_walk_sum<R>(a, GT, S.omask, q0);
    if (m == 0) return;
  }
  // Work items taken over: from here on every chunk of this workgroup starts
  // with a whole set-up (of a work item that nobody else touches any more).
  __shared__ int own_w[CS_WALK_MAX], own_n[CS_WALK_MAX];
  int nown = 1, at = 0;
  while (true) {
    if (got == -2) {
      // given up: NaN to the gradient's first cell of the tile (after the sums
      // above) and to lambda at the source pixels for the steps left
      const int32_t *td = a.tiles + w % a.ntiles * TILE_W;
      const int b = w / a.ntiles;
      m = a.T;
      for (int i = 0; i < chunk; ++i) m -= adj_walk_steps(a, m);
      __syncthreads();
      if (tid == 0) a.gacc[((int64_t)b * a.Nx + td[4]) * a.Ny + td[6]] = __builtin_nanf("");
      for (int64_t i = tid; i < (int64_t)m * a.nsrcslot; i += blockDim.x)
        a.gsrc[(int64_t)b * a.T * a.nsrcslot + i] = __builtin_nanf("");
      return;
    }
    if (got >= 0) {
      if (tid == 0) {
        own_w[at] = w;
        own_n[at] = chunk;
        own_w[nown] = got;
        own_n[nown] = 0;
      }
      ++nown;
    } else {
      const float *in1 = chunk ? a.out1 + ((chunk - 1) & 1) * 2 * BF : a.in1;
      m = a.T;
      for (int i = 0; i < chunk; ++i) m -= adj_walk_steps(a, m);
      const int nsteps = adj_walk_steps(a, m);
      adj_cs_setup<R, true>(a, S, w / a.ntiles, w % a.ntiles, in1, in1 + BF, tb_sp, seed_px,
                            &nseeds);
      adj_cs_start<R, false>(a, S, m, nsteps, tb_sp, seed_px, nseeds);
      __syncthreads();
      adj_cs_steps<R, false>(a, S, m, nsteps);
      q0 = ((int64_t)S.b * a.Nx + (S.g.R0 + S.row0)) * a.Ny + (S.g.C0 + S.g.c);
      adj_walk_sum<R>(a, S.G, S.omask, q0);
      cs_walk_store<R>(a, S.L1, S.L2, w, chunk, nsteps, S.omask, q0);
      ++chunk;
      const bool done = m == nsteps;
      if (done && --nown == 0) return;
      if (tid == 0) {
        own_n[at] = chunk;
        if (done) {
          own_w[at] = own_w[nown];
          own_n[at] = own_n[nown];
        }
      }
    }
    __syncthreads();
    at = 0;  // the least advanced one next
    for (int i = 1; i < nown; ++i)
      if (own_n[i] < own_n[at]) at = i;
    w = own_w[at];
    chunk = own_n[at];
    if (tid < 64) {
      const int r =
          chunk > 0 ? cs_walk_wait<HOOK>(a.prog, a.ntiles, w / a.ntiles,
                                         cs_walk_neighbours(a.tiles, a.ntiles, w % a.ntiles),
                                         chunk, a.walk.give_up)
                    : -1;
      if (tid == 0) msg = r;
    }
    __syncthreads();
    got = msg;
  }
}

template <int NT, int R>
__global__ __launch_bounds__(NT) void k_adj_cs_batch(BatchAdj bl) {
  const int w = xcd_remap(blockIdx.x, gridDim.x);
  const int gi = batch_group(bl.start, bl.ngrp, w);
  adj_cs_body<NT, R, true>(bl.grp[gi], w - bl.start[gi]);
}

// ------------------------------------------------------------------ nonlinear adjoint
//
// Temporally blocked adjoint of the nonlinear cell (cell.py:94-102 inside
// cell.py:12-17; the per-step form is k_loop_adj_nl_plain in wt_plain.hip,
// whose formulas this follows term by term).  The step's b and c depend on
// u, so
//   lambda_m = P_m lambda_{m+1} + L(w_m lambda_{m+1}) - a2_{m+1} lambda_{m+2} + g_m
// with w_m = A_m c_m^2, a2_m = A_m Bm_m and P_m the pointwise factor.  Each
// iteration m forms lambda_m, then the coefficients of step m-1 from
// u_{m-1}, u_{m-2} and lap(u_{m-1}) (segment record), accumulates that step's
// parameter gradients and carries w_{m-1}, P_{m-1}, a2_{m-1} in registers to
// the next iterations.  Between launches the carried coefficients travel
// through global memory with the two lambdas (NlCarry), so a launch may start
// at any step.  The halo cells also need the record (their coefficients
// drive lambda inside the cone), so the record is read over the whole region.
template <int NT, int R, bool GB>
__global__ __launch_bounds__(NT) void k_adj_cs_nl(AdjArgs a, NlCarry cy) {
  extern __shared__ float smem[];
  const int tid = threadIdx.x;
  const int w = xcd_remap(blockIdx.x, gridDim.x);
  const int b = w / a.ntiles, ti = w - (w / a.ntiles) * a.ntiles;
  const int32_t *td = a.tiles + ti * TILE_W;
  const CsGeom g = cs_geom<R>(td, tid);
  const int NBUF = (g.RW + 2) * g.CS;
  float *buf0 = smem, *buf1 = smem + NBUF;
  float *seeds = smem + 2 * NBUF;
  // material (b_geom, c_linear, rho, 0) of every region cell, LDS index as
  // the field buffers, one 16-byte read per cell and step
  float4 *mat = (float4 *)(smem + ((2 * NBUF + CS_MAX_SEEDS * CS_MAX_TBLOCK + 3) & ~3));
  __shared__ int seed_px[CS_MAX_SEEDS];
  __shared__ int nseeds;
  __shared__ int tb_sp[CS_MAX_TABLE * CS_SP_W];
  const int Ny = a.Ny;
  const int64_t F = (int64_t)a.Nx * Ny;
  const int64_t boff = (int64_t)b * F;
  const int nsp = min(td[9] - td[8], CS_MAX_TABLE);
  const int row0 = g.k * R;
  const int col = g.C0 + g.c;

  float Lc[R], Ln[R], Wm[R], Pm[R], A2a[R], A2b[R], U1[R], Gc[R], Gr[R], Gb[R];
  uint32_t vmask = 0;
  // byte offset of this thread's first cell within one (Nx,Ny) field
  const uint32_t voff = (uint32_t)(((g.R0 + row0) * Ny + col) * 4);
  // 1) global loads: lambdas, carried coefficients, u_{m_hi - 1}, material
  {
    const __amdgpu_buffer_rsrc_t ru = cs_rsrc(
        a.seg_u + ((int64_t)b * a.seg_K + (a.m_hi - 1 - a.seg_n0)) * F, F * 4);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      float l1 = 0.f, l2 = 0.f, wv = 0.f, pv = 0.f, xa = 0.f, xb = 0.f, uu = 0.f;
      float4 mt = make_float4(0.f, 0.f, 0.f, 0.f);
      if (g.active && row0 + r < g.RH) {
        vmask |= 1u << r;
        const int64_t q = (int64_t)(g.R0 + row0 + r) * Ny + col;
        l1 = a.in1[boff + q]; l2 = a.in2[boff + q];
        wv = cy.w_in[boff + q]; pv = cy.p_in[boff + q];
        xa = cy.a2a_in[boff + q]; xb = cy.a2b_in[boff + q];
        uu = cs_bload(ru, voff + (uint32_t)(r * Ny * 4));
        mt = make_float4(a.bgeom[q], a.clin[q], a.rho[q], 0.f);
      }
      Lc[r] = l1; Ln[r] = l2; Wm[r] = wv; Pm[r] = pv; A2a[r] = xa; A2b[r] = xb; U1[r] = uu;
      Gc[r] = 0.f; Gr[r] = 0.f; Gb[r] = 0.f;
      if (g.active) mat[g.base + r] = mt;
    }
  }
  // (the owners' table lies behind the seeds, or under them in launches of
  // more than 128 steps, with a barrier more)
  int *own = (int *)(seeds + (a.nsteps > 128 ? 0 : 128 * CS_MAX_SEEDS));
  int spe[CS_SP_W];
  cs_special_load(a.spx, td[8], nsp, spe);
  // 2) LDS: w_m * lambda_{m+1} of the region, tables, probe seeds
  for (int i = tid; i < 2 * NBUF; i += blockDim.x) smem[i] = 0.0f;
  cs_special_stage(a.spx, td[8], nsp, spe, tb_sp, own);
  __syncthreads();
  cs_special_scatter<R>(g, nsp, tb_sp, own, seed_px, &nseeds);
  if (g.active) {
#pragma unroll
    for (int r = 0; r < R; ++r) buf0[g.base + r] = Wm[r] * Lc[r];
  }
  __syncthreads();
  // special rows of this thread: probe taps (seed slot) / source pixels (slot)
  const CsSpecials sp = cs_special_read(g, row0, tb_sp, own);
  const int sr0 = sp.sr0, sr1 = sp.sr1, sd0 = sp.sd0, sd1 = sp.sd1, sl0 = sp.sl0, sl1 = sp.sl1;
  if (a.nsteps > 128) __syncthreads();
  for (int i = tid; i < nseeds * a.nsteps; i += blockDim.x) {
    const int k = i / a.nsteps, s = i - (i / a.nsteps) * a.nsteps;
    const int m = a.m_hi - s;
    const int *e = tb_sp + CS_SP_W * seed_px[k];
    float gs = 0.0f;
    if (a.ybar) {
      for (int t = e[4]; t < e[5]; ++t) {
        const int32_t *tp = a.taps + t * TAP_W;
        const int64_t o = ((int64_t)b * a.T + (m - 1)) * a.ntap + tp[3];
        const float gy = a.ybar[o];
        gs += tp[2] ? 2.0f * a.yraw[o] * gy : gy;
      }
    }
    seeds[i] = gs;
  }
  uint32_t omask = 0;
  if (g.active && col >= g.oc0 && col < g.oc1) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int gr = g.R0 + row0 + r;
      if (row0 + r < g.RH && gr >= g.or0 && gr < g.or1) omask |= 1u << r;
    }
  }
  __syncthreads();

  const float s2 = a.s2, dtm1 = a.dtm1, dtm2 = a.dtm2;
  const float uth = a.sat_uth, b0 = a.sat_b0, cnl = a.c_nl;
  const int nlf = a.nlf;
  // Record values of the step being formed: LL = lap(u_{m-1}) and UL =
  // u_{m-2} (from the checkpoint's u_{n0-1} when m-2 precedes the segment).
  // Each step loads those of the next step at its end, outside every branch
  // and always issued (out of range, reading nothing, past the launch's last
  // step or outside the region: vmask), so that they travel during the
  // barrier and the next step's lambda pass.
  float LL[R], UL[R];
  auto load_record = [&](int m, bool valid) {
    const __amdgpu_buffer_rsrc_t rl =
        cs_rsrc(a.seg_lap + ((int64_t)b * a.seg_K + (valid ? m - 1 - a.seg_n0 : 0)) * F, F * 4);
    const __amdgpu_buffer_rsrc_t ru =
        (!valid || (m - 2) < a.seg_n0)
            ? cs_rsrc(cy.uprev0 + boff, F * 4)
            : cs_rsrc(a.seg_u + ((int64_t)b * a.seg_K + (m - 2 - a.seg_n0)) * F, F * 4);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const uint32_t o =
          (valid && ((vmask >> r) & 1u)) ? voff + (uint32_t)(r * Ny * 4) : 0x80000000u;
      LL[r] = cs_rec_load(rl, o);
      UL[r] = cs_rec_load(ru, o);
    }
  };
  load_record(a.m_hi, true);
  const int live = cs_live_steps<R>(g, row0, a.nsteps);
  float *gsrc0 = a.gsrc + ((int64_t)b * a.T + (a.m_hi - 1)) * a.nsrcslot;
  auto step = [&](const float *P, float *Q, float(&Lx)[R], float(&Ly)[R], int s) {
    // Lx = lambda_{m+1}, Ly = lambda_{m+2} on entry, lambda_m on exit
    const int m = a.m_hi - s;
    if (s < live) {
      const float gs0 = sd0 >= 0 ? seeds[sd0 * a.nsteps + s] : 0.0f;
      const float gs1 = sd1 >= 0 ? seeds[sd1 * a.nsteps + s] : 0.0f;
      const int lfb = g.base - g.CS, rtb = g.base + g.CS;
      // 1) lambda_m of every row (needs only this step's coefficients)
      float upv = P[g.base - 1];
      float ct = Wm[0] * Lx[0];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const float dn = (r < R - 1) ? Wm[r + 1] * Lx[r + 1] : P[g.base + R];
        const float lf = P[lfb + r], rt = P[rtb + r];
        float lapw = upv + lf;
        lapw = __builtin_fmaf(-4.0f, ct, lapw);
        lapw = lapw + rt;
        lapw = lapw + dn;
        float lam = (Pm[r] * Lx[r] + lapw) - A2a[r] * Ly[r];
        if (r == sr0) lam += gs0;
        if (r == sr1) lam += gs1;
        upv = ct;
        ct = dn;
        Ly[r] = lam;
      }
      // 2) coefficients of step m-1 at each cell (u = u_{m-1}, up = u_{m-2}),
      // that step's parameter gradients, w_{m-1} * lambda_m to LDS
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const float lam = Ly[r];
        const float4 mt = mat[g.base + r];
        const float u = U1[r], up = UL[r], lapu = LL[r], rho = mt.z;
        float bb = mt.x, cc = mt.y, sd = 0.0f, c2raw = 0.0f, dbdu = 0.0f, dcdu = 0.0f;
        if (nlf & 1) {
          const float q = adj_div(u, uth), d = 1.0f + q * q;
          sd = adj_div(b0, d);
          bb += rho * sd;
          dbdu = adj_div(rho * b0 * adj_div(-2.0f * q, uth), d * d);
        }
        if (nlf & 2) {
          c2raw = cnl * (u * u);
          cc += rho * c2raw;
          dcdu = 2.0f * rho * cnl * u;
        }
        bool clamped = false;
        if (nlf & 4) {
          if (cc < a.cmin) { cc = a.cmin; clamped = true; }
          if (cc > a.cmax) { cc = a.cmax; clamped = true; }
        }
        const float bd = bb * dtm1;
        const float A = adj_div(1.0f, dtm2 + bd);
        const float Bm = dtm2 - bd;
        const float v = A * ((s2 * u - Bm * up) + (cc * cc) * lapu);
        const float dvdb = A * dtm1 * (up - v);
        const float dvdc = clamped ? 0.0f : 2.0f * A * cc * lapu;
        Gc[r] = __builtin_fmaf(dvdc, lam, Gc[r]);
        if (GB) Gb[r] = __builtin_fmaf(dvdb, lam, Gb[r]);
        Gr[r] = __builtin_fmaf(dvdb * sd + dvdc * c2raw, lam, Gr[r]);
        const float wn = (A * (cc * cc)) * a.t1;  // with the Laplacian's h^-2
        Wm[r] = wn;
        Pm[r] = s2 * A + dvdb * dbdu + dvdc * dcdu;
        A2a[r] = A2b[r];
        A2b[r] = A * Bm;
        U1[r] = up;
        Q[g.base + r] = wn * lam;
      }
      if (sr0 >= 0) {
        // lambda_m at source pixels of the output rows -> dJ/dx[b, m-1]:
        // picked with selects, at most two stores
        float *gsrc_row = gsrc0 - (int64_t)s * a.nsrcslot;
        float v0 = Ly[0], v1 = Ly[0];
#pragma unroll
        for (int r = 1; r < R; ++r) {
          v0 = (r == sr0) ? Ly[r] : v0;
          v1 = (r == sr1) ? Ly[r] : v1;
        }
        if (sl0 >= 0 && ((omask >> sr0) & 1u)) gsrc_row[sl0] = v0;
        if (sl1 >= 0 && sr1 >= 0 && ((omask >> sr1) & 1u)) gsrc_row[sl1] = v1;
      }
    }
    load_record(m - 1, s + 1 < a.nsteps);
    __syncthreads();
  };

  int s = 0;
  for (; s + 1 < a.nsteps; s += 2) {
    step(buf0, buf1, Lc, Ln, s);      // lambda_m -> Ln
    step(buf1, buf0, Ln, Lc, s + 1);  // lambda_{m-1} -> Lc
  }
  if (s < a.nsteps) step(buf0, buf1, Lc, Ln, s);
  const bool odd = (a.nsteps & 1) != 0;
  if (g.active) {
    const int64_t q0 = boff + (int64_t)(g.R0 + row0) * Ny + col;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if ((omask >> r) & 1u) {
        const int64_t q = q0 + (int64_t)r * Ny;
        a.out1[q] = odd ? Ln[r] : Lc[r];
        a.out2[q] = odd ? Lc[r] : Ln[r];
        cy.w_out[q] = Wm[r];
        cy.p_out[q] = Pm[r];
        cy.a2a_out[q] = A2a[r];
        cy.a2b_out[q] = A2b[r];
        a.gacc[q] += Gc[r];
        a.gacc_rho[q] += Gr[r];
        if (GB) a.gacc_b[q] += Gb[r];
      }
    }
  }
}

// ------------------------------------------------------------------ launchers

static int cs_max_dyn_lds() { return max_dyn_lds_dev(); }

#define WT_CS_VARIANTS(X) \
  X(1024, 4)              \
  X(1024, 6)              \
  X(1024, 8)              \
  X(1024, 10)             \
  X(1024, 12)             \
  X(512, 16)              \
  X(512, 20)              \
  X(512, 24)

#ifdef WT_PHASE_TIMING
extern "C" int wt_debug_phase_buffer(unsigned long long *p) {
  return hipMemcpyToSymbol(HIP_SYMBOL(wt_phase_ts), &p, sizeof(p)) == hipSuccess ? 0 : -3;
}
#endif

bool cs_variant_exists(int nt, int r) {
#define X(A, B) if (nt == A && r == B) return true;
  WT_CS_VARIANTS(X)
#undef X
  return false;
}

// Largest LDS column stride of a region of at most RH rows; `padded`:
// with cs_layout's slack (forward tiles, whose descriptors carry a layout),
// so that every tile of the launch fits the allocation.
static int cs_stride_alloc(int R, int RH, bool padded) {
  int nseg = (RH + R - 1) / R;
  return ((nseg * R + 2) | 1) + (padded ? cs_lds_slack(R) : 0);
}

// LDS bytes of a region with RH rows and RW columns for rows-per-thread R.
size_t cs_shmem_bytes(int R, int RH, int RW, bool padded) {
  int CS = cs_stride_alloc(R, RH, padded);
  // field double buffer + staged inputs (forward) or probe seeds (adjoint)
  return ((size_t)2 * (RW + 2) * CS + (size_t)CS_MAX_SEEDS * CS_MAX_TBLOCK) * sizeof(float);
}

// Threads of a launch whose largest region is RH x RW: whole waves for the
// plain mapping.  cs_layout pads columns only within these waves: an extra
// wave costs a VALU-bound block more than the bank conflicts it removes
// (measured: 12 -> 13 waves made the nonlinear forward 13% slower).
int cs_threads(int R, int RH, int RW) {
  int nseg = (RH + R - 1) / R;
  int t = nseg * RW;
  return (t + 63) / 64 * 64;
}

template <int NT, int R>
static hipError_t cs_fwd_dispatch(bool unit_h, int nl, bool rec, const FwdArgs &a, int nblocks,
                                  int nthreads, size_t shmem, hipStream_t s) {
  constexpr bool hooks = NT == 1024 && R == 4;
  const bool hook = a.prog && a.walk.hook();
  if (hook && !hooks) return hipErrorNotSupported;
#define FT(NL, REC, UH)                                                               \
  do {                                                                                \
    auto kfn = a.prog ? k_fwd_cs_walk<NT, R, NL, REC, UH> : k_fwd_cs<NT, R, NL, REC, UH>; \
    if (hook) kfn = k_fwd_cs_walk<NT, R, NL, REC, UH, hooks>;                         \
    static std::atomic<uint64_t> done[3];                                             \
    hipError_t e = allow_dyn_lds((const void *)kfn, done[hook ? 2 : a.prog != nullptr]); \
    if (e != hipSuccess) return e;                                                    \
    hipLaunchKernelGGL(kfn, dim3(nblocks), dim3(nthreads), shmem, s, a);              \
  } while (0)
  if (nl == 0) {
    if (unit_h) {
      if (rec) FT(0, true, true); else FT(0, false, true);
    } else {
      if (rec) FT(0, true, false); else FT(0, false, false);
    }
  } else if (unit_h) {
    if (rec) FT(8, true, true); else FT(8, false, true);
  } else {
    if (rec) FT(8, true, false); else FT(8, false, false);
  }
#undef FT
  return hipGetLastError();
}

template <int NT, int R>
static hipError_t cs_adj_dispatch(const AdjArgs &a, int nblocks, int nthreads, size_t shmem,
                                  hipStream_t s) {
  constexpr bool hooks = NT == 1024 && (R == 4 || R == 8);  // sums in registers or not
  const bool hook = a.prog && a.walk.hook();
  if (hook && !hooks) return hipErrorNotSupported;
#define AT(...)                                                                       \
  do {                                                                                \
    auto kfn = __VA_ARGS__;                                                           \
    static std::atomic<uint64_t> done{0};                                             \
    hipError_t e = allow_dyn_lds((const void *)kfn, done);                            \
    if (e != hipSuccess) return e;                                                    \
    hipLaunchKernelGGL(kfn, dim3(nblocks), dim3(nthreads), shmem, s, a);              \
  } while (0)
  if (hook) AT(k_adj_cs_walk<NT, R, hooks>);
  else if (a.prog) AT(k_adj_cs_walk<NT, R>);
  else AT(k_adj_cs<NT, R>);
#undef AT
  return hipGetLastError();
}

// The region geometry (RH, RW) of the largest tile decides the block size
// and LDS of the launch; smaller tiles leave threads idle.
hipError_t launch_fwd_cs(int nt, int R, bool unit_h, int nl, bool rec, const FwdArgs &a,
                         int RHmax, int RWmax, hipStream_t s) {
  const int items = a.B * a.ntiles;
  const int nblocks = a.prog ? walk_blocks(items, a.walk) : items;
  size_t shmem = cs_shmem_bytes(R, RHmax, RWmax, true);
  int nthreads = cs_threads(R, RHmax, RWmax);
  if (shmem + CS_STATIC_LDS > (size_t)cs_max_dyn_lds() || nthreads > nt ||
      (a.prog && items > CS_WALK_MAX))
    return hipErrorInvalidConfiguration;
#define X(A, B) \
  if (nt == A && R == B)                                                                \
    return cs_fwd_dispatch<A, B>(unit_h, nl, rec, a, nblocks, nthreads, shmem, s);
  WT_CS_VARIANTS(X)
#undef X
  return hipErrorInvalidValue;
}

hipError_t launch_adj_cs(int nt, int R, const AdjArgs &a, int RHmax, int RWmax, hipStream_t s) {
  const int items = a.B * a.ntiles;
  const int nblocks = a.prog ? walk_blocks(items, a.walk) : items;
  size_t shmem = cs_shmem_bytes(R, RHmax, RWmax, false);
  int nthreads = cs_threads(R, RHmax, RWmax);
  if (shmem + CS_STATIC_LDS + (a.prog ? CS_WALK_LDS : 0) > (size_t)cs_max_dyn_lds() ||
      nthreads > nt || (a.prog && items > CS_WALK_MAX))
    return hipErrorInvalidConfiguration;
#define X(A, B) if (nt == A && R == B) return cs_adj_dispatch<A, B>(a, nblocks, nthreads, shmem, s);
  WT_CS_VARIANTS(X)
#undef X
  return hipErrorInvalidValue;
}

// Nonlinear adjoint: 4 rows per thread at 1024 threads (the carried
// coefficients fill the register file; 6 rows spill).
bool cs_nl_variant_exists(int nt, int r) { return nt == 1024 && r == 4; }

size_t cs_nl_shmem_bytes(int R, int RH, int RW) {
  int CS = cs_stride_alloc(R, RH, false);
  return cs_shmem_bytes(R, RH, RW, false) + 16 + (size_t)(RW + 2) * CS * 16;
}

hipError_t launch_adj_cs_nl(int nt, int R, bool gb, const AdjArgs &a, const NlCarry &cy,
                            int RHmax, int RWmax, hipStream_t s) {
  int nblocks = a.B * a.ntiles;
  size_t shmem = cs_nl_shmem_bytes(R, RHmax, RWmax);
  int nthreads = cs_threads(R, RHmax, RWmax);
  if (shmem + CS_STATIC_LDS > (size_t)cs_max_dyn_lds() || nthreads > nt || !cs_nl_variant_exists(nt, R))
    return hipErrorInvalidConfiguration;
#define NLK(RR, G)                                                                     \
  do {                                                                                 \
    auto kfn = k_adj_cs_nl<1024, RR, G>;                                               \
    static std::atomic<uint64_t> done{0};                                              \
    hipError_t e = allow_dyn_lds((const void *)kfn, done);                             \
    if (e != hipSuccess) return e;                                                     \
    hipLaunchKernelGGL(kfn, dim3(nblocks), dim3(nthreads), shmem, s, a, cy);           \
  } while (0)
  if (gb) NLK(4, true); else NLK(4, false);
#undef NLK
  return hipGetLastError();
}

// Batched launches (linear cell): one launch over the work items of every
// configuration in `bl`; RHmax/RWmax are the largest region over all of them.
template <int NT, int R>
static hipError_t cs_fwd_batch_dispatch(bool rec, const BatchFwd &bl, int nblocks, int nthreads,
                                        size_t shmem, hipStream_t s) {
#define FB(REC)                                                                       \
  do {                                                                                \
    auto kfn = k_fwd_cs_batch<NT, R, 0, REC>;                                         \
    static std::atomic<uint64_t> done{0};                                             \
    hipError_t e = allow_dyn_lds((const void *)kfn, done);                            \
    if (e != hipSuccess) return e;                                                    \
    hipLaunchKernelGGL(kfn, dim3(nblocks), dim3(nthreads), shmem, s, bl);             \
  } while (0)
  if (rec) FB(true); else FB(false);
#undef FB
  return hipGetLastError();
}

template <int NT, int R>
static hipError_t cs_adj_batch_dispatch(const BatchAdj &bl, int nblocks, int nthreads,
                                        size_t shmem, hipStream_t s) {
  auto kfn = k_adj_cs_batch<NT, R>;
  static std::atomic<uint64_t> done{0};
  hipError_t e = allow_dyn_lds((const void *)kfn, done);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kfn, dim3(nblocks), dim3(nthreads), shmem, s, bl);
  return hipGetLastError();
}

hipError_t launch_fwd_cs_batch(int nt, int R, bool rec, const BatchFwd &bl, int RHmax,
                               int RWmax, hipStream_t s) {
  int nblocks = bl.start[bl.ngrp];
  if (nblocks <= 0) return hipSuccess;
  size_t shmem = cs_shmem_bytes(R, RHmax, RWmax, true);
  int nthreads = cs_threads(R, RHmax, RWmax);
  if (shmem + CS_STATIC_LDS > (size_t)cs_max_dyn_lds() || nthreads > nt) return hipErrorInvalidConfiguration;
#define X(A, B) \
  if (nt == A && R == B) return cs_fwd_batch_dispatch<A, B>(rec, bl, nblocks, nthreads, shmem, s);
  WT_CS_VARIANTS(X)
#undef X
  return hipErrorInvalidValue;
}

hipError_t launch_adj_cs_batch(int nt, int R, const BatchAdj &bl, int RHmax, int RWmax,
                               hipStream_t s) {
  int nblocks = bl.start[bl.ngrp];
  if (nblocks <= 0) return hipSuccess;
  size_t shmem = cs_shmem_bytes(R, RHmax, RWmax, false);
  int nthreads = cs_threads(R, RHmax, RWmax);
  if (shmem + CS_STATIC_LDS > (size_t)cs_max_dyn_lds() || nthreads > nt) return hipErrorInvalidConfiguration;
#define X(A, B) \
  if (nt == A && R == B) return cs_adj_batch_dispatch<A, B>(bl, nblocks, nthreads, shmem, s);
  WT_CS_VARIANTS(X)
#undef X
  return hipErrorInvalidValue;
}

}  // namespace wt
