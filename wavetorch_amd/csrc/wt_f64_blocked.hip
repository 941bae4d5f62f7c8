// wt_f64_blocked.hip -- the linear WaveRNN loop in double precision,
// temporally blocked (gfx950).
//
// The thread mapping and the launches are those of the float kernels
// (wt_colseg.hip): one workgroup advances one tile of one sample plus a halo
// by `nsteps` steps, a thread's R rows of one column in registers and the
// field in LDS.  Double vector instructions issue at the rate of the
// non-packed float ones on this chip, so a step costs what it costs in
// float; registers and LDS hold half the cells.
//
// The forward with gradients records lap(u_n) of every step (the tape's size:
// T x B x Nx x Ny doubles), which is all of the field that the adjoint of the
// linear cell reads:
//   lambda_m = a1 lambda_{m+1} + L(w lambda_{m+1}) - a2 lambda_{m+2} + seeds
//   dJ/dc    = 2 A c sum_m lap(u_{m-1}) lambda_m
// so nothing is recomputed, and each step of the adjoint reads 8 bytes per
// cell instead of the fields u_{m+1} .. u_{m-2}, both lambdas and the
// gradient sum (the per-step kernels of wt_f64.hip, which stay for the
// nonlinear cell, for dJ/db and for field seeds).  The forward follows the
// reference's operation order (cell.py:12-17, operators.py:5-11), bitwise
// equal to the per-step kernel's.
#include <algorithm>

#include "wt_colseg.h"

namespace wt {

struct F64Blk {
  int B, Nx, Ny, T, ntiles, ntap, nslot;
  const int32_t *tiles, *spx, *taps;
  const double *A, *Bm, *C2;
  double s2, t1, t4;
  const double *in1, *in2;  // null: zero fields
  double *out1, *out2;
  int n0, nsteps;           // forward: first step of the launch
  const double *x;
  double *y, *yraw, *fields, *rec;
  int fstride;
  int *prog;                // resident forward: progress words, else null
  WalkStart walk;
  const double *ybar;       // adjoint: reverse steps m_hi .. m_hi - nsteps + 1
  double *gacc, *gsrc;
  int m_hi;
  int first;                // adjoint: gacc holds nothing yet
};

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ double b64_load(__amdgpu_buffer_rsrc_t rs, uint32_t off) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rs, (int)off, 0, 0));
}
__device__ __forceinline__ void b64_store(__amdgpu_buffer_rsrc_t rs, uint32_t off, double v) {
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), rs, (int)off, 0, 0);
}

// Output rows (bit mask) of a thread whose cells inside the region are vmask.
template <int R>
__device__ __forceinline__ uint32_t cs64_out_rows(const CsGeom &g, int row0, uint32_t voff,
                                                  uint32_t vmask) {
  uint32_t m = 0;
  if (voff != 0x80000000u) {
    const int lo = max(g.or0 - g.R0 - row0, 0), hi = min(g.or1 - g.R0 - row0, R);
    if (hi > lo) m = ((1u << hi) - 1u) & ~((1u << lo) - 1u) & vmask;
  }
  return m;
}

// State after nsteps steps to (o1, o2); DEV: the later one to V0 first.
template <int R, bool DEV>
__device__ __forceinline__ void cs64_store(const F64Blk &a, const CsGeom &g, double (&V0)[R],
                                           double (&V1)[R], int nsteps, uint32_t voff,
                                           uint32_t omask, int64_t q0, int b, double *o1,
                                           double *o2) {
  const bool odd = (nsteps & 1) != 0;
  if (DEV) {
    if (odd) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const double u = V0[r];
        V0[r] = V1[r];
        V1[r] = u;
      }
    }
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
  } else {
    const int64_t at = ((int64_t)b * a.Nx + g.or0) * a.Ny;
    const int64_t out_bytes = (int64_t)(g.or1 - g.or0) * a.Ny * 8;
    const __amdgpu_buffer_rsrc_t r1 = cs_rsrc(o1 + at, out_bytes), r2 = cs_rsrc(o2 + at, out_bytes);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      b64_store(r1, voff + (uint32_t)(r * a.Ny * 8), odd ? V1[r] : V0[r]);
      b64_store(r2, voff + (uint32_t)(r * a.Ny * 8), odd ? V0[r] : V1[r]);
    }
  }
}

template <int R>
__device__ __forceinline__ void cs64_halo(const F64Blk &a, double (&V0)[R], double (&V1)[R],
                                          uint32_t halo, int64_t q0, const double *in1,
                                          const double *in2) {
  const uint32_t hm = cs_opaque(halo);
  int64_t q = cs_opaque(q0);
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if ((hm >> r) & 1u) {
      V0[r] = cs_dev_load(in1 + q);
      V1[r] = cs_dev_load(in2 + q);
    }
    q += a.Ny;
  }
}

// A forward workgroup's tile and its sweeps: set-up, the steps n0 .. n0 +
// nsteps - 1 (after an even number u_n is in U0, else in U1) and write-back.
// DEV: the state is shared with the other workgroups of the launch.
template <int R, bool REC, bool UH, bool DEV>
struct Fwd64 {
  CsGeom g;
  CsTap tap;
  int b, row0, srows;
  uint32_t voff, vmask, omask;  // cs_out_voff; cells of the region; output rows
  int64_t q0;                   // first cell
  bool wave_src, one_src;
  double *buf0, *buf1, *xs;
  double U0[R], U1[R], KA[R], KB[R], KC[R];

  __device__ __forceinline__ void setup(const F64Blk &a, int w, const double *in1,
                                        const double *in2) {
    extern __shared__ double smem64[];
    __shared__ int own[1024];  // source rows of each thread, a bit mask
    const int tid = threadIdx.x;
    b = w / a.ntiles;
    const int32_t *td = a.tiles + (w - b * a.ntiles) * TILE_W;
    g = cs_geom<R>(td, tid);
    const int NBUF = (g.RW + 2) * g.CS;
    buf0 = smem64;
    buf1 = smem64 + NBUF;
    xs = smem64 + 2 * NBUF;
    const int nsp = min(td[9] - td[8], CS_MAX_TABLE), ntp = min(td[11] - td[10], CS_MAX_TABLE);
    row0 = g.k * R;
    q0 = ((int64_t)b * a.Nx + g.R0 + row0) * a.Ny + g.C0 + g.c;
    vmask = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      double u1 = 0., u2 = 0., v0 = 0., v1 = 0., v2 = 0.;
      if (g.active && row0 + r < g.RH) {
        vmask |= 1u << r;
        const int64_t q = (int64_t)(g.R0 + row0 + r) * a.Ny + (g.C0 + g.c);
        v0 = a.A[q]; v1 = a.Bm[q]; v2 = a.C2[q];
        if (in1) {
          const int64_t o = q0 + (int64_t)r * a.Ny;
          u1 = DEV ? cs_dev_load(in1 + o) : in1[o];
          u2 = DEV ? cs_dev_load(in2 + o) : in2[o];
        }
      }
      U0[r] = u1; U1[r] = u2; KA[r] = v0; KB[r] = v1; KC[r] = v2;
    }
    int spx0 = 0, spx1 = 0, spx2 = 0, te[TAP_W];
    if (tid < nsp) {
      const int32_t *e = a.spx + (td[8] + tid) * SPX_W;
      spx0 = e[0]; spx1 = e[1]; spx2 = e[2];
    }
    cs_tap_load(a.taps, td[10], ntp, te);
    own[tid] = 0;
    cs_zero_lds<double>(buf0, buf1, g, ((g.RH + R - 1) / R) * R, NBUF);
    __syncthreads();
    fill();
    // source pixels mark the rows of their owners
    for (int kk = tid; kk < nsp; kk += blockDim.x) {
      if (kk != tid) {  // more entries than threads
        const int32_t *e = a.spx + (td[8] + kk) * SPX_W;
        spx0 = e[0]; spx1 = e[1]; spx2 = e[2];
      }
      int rr;
      const int t = spx2 > 0 ? cs_owner<R>(g, spx0, spx1, rr) : -1;
      if (t >= 0) atomicOr(&own[t], 1 << rr);
    }
    __syncthreads();
    tap = cs_tap(g, a.taps, td[10], ntp, te);
    srows = own[tid];
    wave_src = __ballot(srows != 0) != 0;
    one_src = __ballot((srows & (srows - 1)) != 0) == 0;
    voff = cs_out_voff<double>(g, row0, a.Ny);
    omask = cs64_out_rows<R>(g, row0, voff, vmask);
  }
  __device__ __forceinline__ void fill() {
    if (g.active) {
#pragma unroll
      for (int r = 0; r < R; ++r) buf0[g.base + r] = U0[r];
    }
  }
  // the input samples of a chunk (a barrier must follow)
  __device__ __forceinline__ void prepare(const F64Blk &a, int n0, int nsteps) {
    for (int i = cs_opaque((int)threadIdx.x); i < nsteps; i += blockDim.x)
      xs[i] = a.x[(int64_t)b * a.T + n0 + i];
  }
  __device__ __forceinline__ void run(const F64Blk &a, int n0, int nsteps) {
    const int Ny = a.Ny;
    const int64_t F = (int64_t)a.Nx * Ny;
    const int64_t out_bytes = (int64_t)(g.or1 - g.or0) * Ny * 8;
    const uint32_t voff = cs_opaque(this->voff);
    const int live = cs_live_steps<R>(g, row0, nsteps);
    const double *recp = REC ? a.rec + ((int64_t)b * a.T + n0) * F + (int64_t)g.or0 * Ny : a.A;
    const int64_t yo = ((int64_t)b * a.T + n0) * a.ntap + tap.pcol;
    double *yp = a.y ? a.y + yo : nullptr, *yrp = a.yraw ? a.yraw + yo : nullptr;
    // next snapshot: at step `snap`
    int snap = a.fields ? a.fstride - 1 - n0 % a.fstride : -1;
    const double *fp = a.fields ? a.fields +
                                      ((int64_t)b * (a.T / a.fstride) + n0 / a.fstride) * F +
                                      (int64_t)g.or0 * Ny
                                : a.A;

    auto step = [&](const double *P, double *Q, double(&Uc)[R], double(&Up)[R], int s) {
      if (s < live) {
        const __amdgpu_buffer_rsrc_t rsl = cs_rsrc(recp, REC ? out_bytes : 0);
        const int lfb = g.base - g.CS, rtb = g.base + g.CS;
        double upv = UH ? P[g.base - 1] : a.t1 * P[g.base - 1];
        double ctv = UH ? 0.0 : a.t1 * Uc[0];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const double ct = Uc[r];
          const double dn = (r < R - 1) ? Uc[r + 1] : P[g.base + R];
          const double lf = P[lfb + r], rt = P[rtb + r];
          double lap;
          if (UH) {  // products with t1 = 1 and t4 = -4 are exact
            double s0 = upv + lf;
            s0 = __builtin_fma(-4.0, ct, s0);
            s0 = s0 + rt;
            lap = s0 + dn;
            upv = ct;
          } else {
            const double dnv = a.t1 * dn;
            double s0 = upv + a.t1 * lf;
            s0 = s0 + a.t4 * ct;
            s0 = s0 + a.t1 * rt;
            lap = s0 + dnv;
            upv = ctv;
            ctv = dnv;
          }
          const double p1 = a.s2 * ct;
          const double p2 = KB[r] * Up[r];
          const double p3 = KC[r] * lap;
          const double v = KA[r] * ((p1 - p2) + p3);
          Up[r] = v;
          Q[g.base + r] = v;
          if (REC) b64_store(rsl, voff + (uint32_t)(r * Ny * 8), lap);
        }
        if (wave_src) cs_add_source<R>(Up, Q + g.base, srows, one_src, xs[s]);
        if (s == snap) {  // the thread's own rows: consecutive lanes, consecutive columns
          const __amdgpu_buffer_rsrc_t rf = cs_rsrc(fp, out_bytes);
#pragma unroll
          for (int r = 0; r < R; ++r) b64_store(rf, voff + (uint32_t)(r * Ny * 8), Up[r]);
        }
      }
      if (s == snap) {
        snap += a.fstride;
        fp += F;
      }
      if (REC) recp += F;
      __syncthreads();
      if (tap.pidx >= 0) {
        const double v = Q[tap.pidx];
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
    int s = 0;
    for (; s + 1 < nsteps; s += 2) {
      step(buf0, buf1, U0, U1, s);
      step(buf1, buf0, U1, U0, s + 1);
    }
    if (s < nsteps) step(buf0, buf1, U0, U1, s);
  }
  // u_n to U0 (DEV), and the output rows to (o1, o2)
  __device__ __forceinline__ void store(const F64Blk &a, int nsteps, double *o1, double *o2) {
    cs64_store<R, DEV>(a, g, U0, U1, nsteps, voff, omask, q0, b, o1, o2);
  }
  // the halo of the next chunk
  __device__ __forceinline__ void refill(const F64Blk &a, const double *in1, const double *in2) {
    cs64_halo<R>(a, U0, U1, vmask & ~omask, q0, in1, in2);
    fill();
  }
};

// One launch of nsteps steps.
template <int NT, int R, bool REC, bool UH>
__global__ __launch_bounds__(NT) void k64_fwd_cs(F64Blk a) {
  Fwd64<R, REC, UH, false> S;
  S.setup(a, xcd_remap(blockIdx.x, gridDim.x), a.in1, a.in2);
  S.prepare(a, a.n0, a.nsteps);
  __syncthreads();
  S.run(a, a.n0, a.nsteps);
  S.store(a, a.nsteps, a.out1, a.out2);
}

// The whole forward in one resident launch, in chunks of nsteps steps (the
// scheme stands in wt_colseg.h); out1: two alternating state pairs.  (150 x
// 140, 16 samples, 1200 steps: 75 launches of 24.0 us, resident 1377 us.  The
// adjoint gained nothing from it: its registers spill in the walk, 1784 us
// against 75 launches of 23.3 us.)
template <int NT, int R, bool REC, bool UH, bool HOOK = false>
__global__ __launch_bounds__(NT) void k64_fwd_walk(F64Blk a) {
  const int tid = threadIdx.x;
  const int64_t BF = (int64_t)a.B * a.Nx * a.Ny;
  const int nchunks = (a.T + a.nsteps - 1) / a.nsteps;
  auto pair = [&](int chunk) { return a.out1 + (chunk & 1) * 2 * BF; };
  auto steps = [&](int chunk) { return min(a.nsteps, a.T - chunk * a.nsteps); };
  auto start = [&](int chunk) { return chunk * a.nsteps; };
  __shared__ int own_w[CS_WALK_MAX], own_n[CS_WALK_MAX];
  __shared__ int msg;
  int w = xcd_remap(blockIdx.x, gridDim.x) * (HOOK ? a.walk.every : 1);
  if (tid == 0) msg = atomicCAS(a.prog + w * CS_WALK_W, 0, 1);
  __syncthreads();
  if (msg != 0) return;  // a neighbour took it over
  Fwd64<R, REC, UH, true> S;
  int chunk = 0, got;
  {
    const int b = w / a.ntiles;
    const int nbr = tid < 64 ? cs_walk_neighbours(a.tiles, a.ntiles, w - b * a.ntiles) : 0;
    S.setup(a, w, nullptr, nullptr);
    S.prepare(a, start(0), steps(0));
    __syncthreads();
    while (true) {
      S.run(a, start(chunk), steps(chunk));
      if (chunk + 1 == nchunks) return;
      S.store(a, steps(chunk), pair(chunk), pair(chunk) + BF);
      cs_walk_raise(a.prog, w, chunk);
      ++chunk;
      S.prepare(a, start(chunk), steps(chunk));
      if (tid < 64) {
        const int r = cs_walk_wait<HOOK>(a.prog, a.ntiles, b, nbr, chunk, a.walk.give_up);
        if (tid == 0) msg = r;
      }
      __syncthreads();
      got = msg;
      if (got != -1) break;
      S.refill(a, pair(chunk - 1), pair(chunk - 1) + BF);
      __syncthreads();
    }
  }
  // Work items taken over: from here on every chunk of this workgroup starts
  // with a whole set-up.
  int nown = 1, at = 0;
  while (true) {
    if (got == -2) {
      cs_walk_failed(a, w / a.ntiles, start(chunk), __builtin_nan(""));
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
      const double *in1 = chunk ? pair(chunk - 1) : nullptr;
      S.setup(a, w, in1, in1 + BF);
      S.prepare(a, start(chunk), steps(chunk));
      __syncthreads();
      S.run(a, start(chunk), steps(chunk));
      S.store(a, steps(chunk), pair(chunk), pair(chunk) + BF);
      cs_walk_raise(a.prog, w, chunk);
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

// LDS holds w * lambda (w with the Laplacian's h^-2); the gradient sum and
// the record values of the next two steps live in registers, the record read
// two steps ahead at one issue point (as in the float kernel).
template <int NT, int R>
__global__ __launch_bounds__(NT) void k64_adj_cs(F64Blk a) {
  extern __shared__ double smem64[];
  __shared__ int tb_sp[CS_MAX_TABLE * CS_SP_W];
  __shared__ int own[2 * NT];
  __shared__ int seed_px[CS_MAX_SEEDS];
  __shared__ int nseeds;
  const int tid = threadIdx.x;
  const int w = xcd_remap(blockIdx.x, gridDim.x);
  const int b = w / a.ntiles, ti = w - (w / a.ntiles) * a.ntiles;
  const int32_t *td = a.tiles + ti * TILE_W;
  const CsGeom g = cs_geom<R>(td, tid);
  const int NBUF = (g.RW + 2) * g.CS;
  double *buf0 = smem64, *buf1 = smem64 + NBUF, *seeds = smem64 + 2 * NBUF;
  const int Ny = a.Ny;
  const int64_t F = (int64_t)a.Nx * Ny, boff = (int64_t)b * F;
  const int nsp = min(td[9] - td[8], CS_MAX_TABLE);
  const int row0 = g.k * R;
  double L1[R], L2[R], KA1[R], KW[R], G[R], SG0[R], SG1[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    double A = 0., C2 = 0., u1 = 0., u2 = 0.;
    if (g.active && row0 + r < g.RH) {
      const int64_t q = (int64_t)(g.R0 + row0 + r) * Ny + (g.C0 + g.c);
      A = a.A[q]; C2 = a.C2[q];
      if (a.in1) { u1 = a.in1[boff + q]; u2 = a.in2[boff + q]; }
    }
    KA1[r] = A * a.s2; KW[r] = (A * C2) * a.t1;
    L1[r] = u1; L2[r] = u2;
    G[r] = 0.0; SG1[r] = 0.0;
  }
  int spe[CS_SP_W];
  cs_special_load(a.spx, td[8], nsp, spe);
  cs_zero_lds<double>(buf0, buf1, g, ((g.RH + R - 1) / R) * R, NBUF);
  cs_special_stage(a.spx, td[8], nsp, spe, tb_sp, own);
  __syncthreads();
  cs_special_scatter<R>(g, nsp, tb_sp, own, seed_px, &nseeds);
  if (g.active) {
#pragma unroll
    for (int r = 0; r < R; ++r) buf0[g.base + r] = KW[r] * L1[r];
  }
  __syncthreads();
  for (int i = tid; i < nseeds * a.nsteps; i += blockDim.x) {
    const int k = i / a.nsteps, s = i - k * a.nsteps, m = a.m_hi - s;
    const int *e = tb_sp + CS_SP_W * seed_px[k];
    double gs = 0.0;
    if (a.ybar)
      for (int t = e[4]; t < e[5]; ++t) {
        const int32_t *tp = a.taps + t * TAP_W;
        const int64_t o = ((int64_t)b * a.T + (m - 1)) * a.ntap + tp[3];
        gs += tp[2] ? 2.0 * a.yraw[o] * a.ybar[o] : a.ybar[o];
      }
    seeds[i] = gs;
  }
  // special rows of this thread (at most two): seed slot, source slot
  const CsSpecials sp = cs_special_read(g, row0, tb_sp, own);
  const int sr0 = sp.sr0, sr1 = sp.sr1, sd0 = sp.sd0, sd1 = sp.sd1, sl0 = sp.sl0, sl1 = sp.sl1;
  const bool wave_sp = __ballot(sr0 >= 0) != 0;
  const uint32_t voff = cs_out_voff<double>(g, row0, Ny);
  const int64_t out_bytes = (int64_t)(g.or1 - g.or0) * Ny * 8;
  const bool wave_sp2 = __ballot(sr1 >= 0) != 0;
  const int olo = g.or0 - g.R0 - row0, ohi = g.or1 - g.R0 - row0;  // output rows, thread's count
  const bool out_col = voff != 0x80000000u;
  const bool gx0 = sl0 >= 0 && out_col && sr0 >= olo && sr0 < ohi;
  const bool gx1 = sl1 >= 0 && out_col && sr1 >= olo && sr1 < ohi;
  const double kw0 = cs_pick<R>(KW, sr0), kw1 = cs_pick<R>(KW, sr1);
  __syncthreads();
  // slice of the record read at reverse step m_hi
  const double *rec0 = a.rec + ((int64_t)b * a.T + (a.m_hi - 1)) * F + (int64_t)g.or0 * Ny;
  {
    const __amdgpu_buffer_rsrc_t rs0 = cs_rsrc(rec0, out_bytes);
#pragma unroll
    for (int r = 0; r < R; ++r) SG0[r] = b64_load(rs0, voff + (uint32_t)(r * Ny * 8));
    const bool two = a.nsteps > 1;
    const __amdgpu_buffer_rsrc_t rs1 = cs_rsrc(two ? rec0 - F : rec0, out_bytes);
    const uint32_t v1 = two ? voff : 0x80000000u;
#pragma unroll
    for (int r = 0; r < R; ++r) SG1[r] = b64_load(rs1, v1 + (uint32_t)(r * Ny * 8));
  }
  const int live = cs_live_steps<R>(g, row0, a.nsteps);
  const double *recp = rec0 - 2 * F;  // the step after next
  double *gsrc_row = a.gsrc + ((int64_t)b * a.T + (a.m_hi - 1)) * a.nslot;
  auto step = [&](const double *P, double *Q, double(&Lc)[R], double(&Ln)[R], double(&SG)[R],
                  int s) {
    const bool prefetch = s + 2 < a.nsteps;
    const __amdgpu_buffer_rsrc_t rsn = cs_rsrc(recp, out_bytes);
    const uint32_t pvoff = prefetch ? voff : 0x80000000u;
    if (s < live) {
      const int lfb = g.base - g.CS, rtb = g.base + g.CS;
      double upv = P[g.base - 1];
      double ct = KW[0] * Lc[0];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const double dn = (r < R - 1) ? KW[r + 1] * Lc[r + 1] : P[g.base + R];
        const double lf = P[lfb + r], rt = P[rtb + r];
        double lapw = upv + lf;
        lapw = __builtin_fma(-4.0, ct, lapw);
        lapw = lapw + rt;
        lapw = lapw + dn;
        // a1 L1 + lapw - a2 L2 with a2 = a1 - 1
        const double lam = __builtin_fma(KA1[r], Lc[r] - Ln[r], lapw + Ln[r]);
        upv = ct;
        ct = dn;
        Ln[r] = lam;
        Q[g.base + r] = KW[r] * lam;
      }
      if (wave_sp) {
        cs_adj_special<R>(Ln, Q + g.base, sr0, kw0, sd0 >= 0 ? seeds[sd0 * a.nsteps + s] : 0.0,
                          gx0 ? gsrc_row + sl0 : nullptr);
        if (wave_sp2)
          cs_adj_special<R>(Ln, Q + g.base, sr1, kw1, sd1 >= 0 ? seeds[sd1 * a.nsteps + s] : 0.0,
                            gx1 ? gsrc_row + sl1 : nullptr);
      }
    }
    // gradient sum, then the record of two steps later into the same
    // registers: one issue point outside the branches, always issued (see
    // the float kernel in wt_colseg.hip)
#pragma unroll
    for (int r = 0; r < R; ++r) {
      G[r] = __builtin_fma(SG[r], Ln[r], G[r]);
      asm volatile("" : "+v"(G[r]));
      SG[r] = b64_load(rsn, pvoff + (uint32_t)(r * Ny * 8));
    }
    recp -= F;
    gsrc_row -= a.nslot;
    __syncthreads();
  };
  int s = 0;
  for (; s + 1 < a.nsteps; s += 2) {
    step(buf0, buf1, L1, L2, SG0, s);
    step(buf1, buf0, L2, L1, SG1, s + 1);
  }
  if (s < a.nsteps) step(buf0, buf1, L1, L2, SG0, s);
  const bool odd = (a.nsteps & 1) != 0;
  const __amdgpu_buffer_rsrc_t r1 = cs_rsrc(a.out1 + boff + (int64_t)g.or0 * Ny, out_bytes);
  const __amdgpu_buffer_rsrc_t r2 = cs_rsrc(a.out2 + boff + (int64_t)g.or0 * Ny, out_bytes);
  const __amdgpu_buffer_rsrc_t rg = cs_rsrc(a.gacc + boff + (int64_t)g.or0 * Ny, out_bytes);
  if (!a.first) {
    double gold[R];
#pragma unroll
    for (int r = 0; r < R; ++r) gold[r] = b64_load(rg, voff + (uint32_t)(r * Ny * 8));
#pragma unroll
    for (int r = 0; r < R; ++r) G[r] = gold[r] + G[r];
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    b64_store(r1, voff + (uint32_t)(r * Ny * 8), odd ? L2[r] : L1[r]);
    b64_store(r2, voff + (uint32_t)(r * Ny * 8), odd ? L1[r] : L2[r]);
    b64_store(rg, voff + (uint32_t)(r * Ny * 8), G[r]);
  }
}

// A = 1/(dt^-2 + b dt^-1), Bm = dt^-2 - b dt^-1, C2 = c^2 of the clamped c
__global__ void k64_coef(const double *__restrict__ b, const double *__restrict__ c, int64_t n,
                         double dtm1, double dtm2, int clamp, double cmin, double cmax,
                         double *__restrict__ A, double *__restrict__ Bm,
                         double *__restrict__ C2) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double bd = b[i] * dtm1;
  double cc = c[i];
  if (clamp) {
    if (cc < cmin) cc = cmin;
    if (cc > cmax) cc = cmax;
  }
  A[i] = 1.0 / (dtm2 + bd);
  Bm[i] = dtm2 - bd;
  C2[i] = cc * cc;
}

// dJ/dc = 2 A c sum_b gacc, zero where the clamp holds c
__global__ void k64_finalize_gc(const double *__restrict__ gacc, int B, int64_t F,
                                const double *__restrict__ c, const double *__restrict__ A,
                                int clamp, double cmin, double cmax, double *__restrict__ gc) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= F) return;
  double s = 0.0;
  for (int b = 0; b < B; ++b) s += gacc[(int64_t)b * F + q];
  const double cc = c[q];
  const bool held = clamp && (cc < cmin || cc > cmax);
  gc[q] = held ? 0.0 : A[q] * 2.0 * cc * s;
}

size_t cs64_shmem_bytes(int R, int RH, int RW, int tb) {
  const int nseg = (RH + R - 1) / R;
  // field double buffer + staged inputs (forward) or probe seeds (adjoint)
  return ((size_t)2 * (RW + 2) * ((nseg * R + 2) | 1) + (size_t)CS_MAX_SEEDS * tb) *
         sizeof(double);
}

bool cs64_variant_exists(int R, bool fwd) { return R == 4 || (fwd ? R == 6 || R == 8 : R == 5); }

template <typename K>
static hipError_t launch64(K kfn, std::atomic<uint64_t> &done, const F64Blk &a, int nthreads,
                           size_t shmem, hipStream_t s) {
  hipError_t e = allow_dyn_lds((const void *)kfn, done);
  if (e != hipSuccess) return e;
  const int items = a.B * a.ntiles;
  const int nblocks = a.prog ? walk_blocks(items, a.walk) : items;
  hipLaunchKernelGGL(kfn, dim3(nblocks), dim3(nthreads), shmem, s, a);
  return hipGetLastError();
}

template <int R, bool REC, bool UH>
static hipError_t launch64_fwd(const F64Blk &a, int nthreads, size_t shmem, hipStream_t s) {
  static std::atomic<uint64_t> done[3];
  if (a.prog && a.walk.hook()) {
    if constexpr (R == 4)
      return launch64(k64_fwd_walk<1024, R, REC, UH, true>, done[2], a, nthreads, shmem, s);
    return hipErrorNotSupported;
  }
  if constexpr (R <= 6) {
    if (a.prog)
      return launch64(k64_fwd_walk<1024, R, REC, UH>, done[1], a, nthreads, shmem, s);
  }
  return launch64(k64_fwd_cs<1024, R, REC, UH>, done[0], a, nthreads, shmem, s);
}

template <int R>
static hipError_t launch64_fwd(bool rec, bool uh, const F64Blk &a, int nthreads, size_t shmem,
                               hipStream_t s) {
  if (uh)
    return rec ? launch64_fwd<R, true, true>(a, nthreads, shmem, s)
               : launch64_fwd<R, false, true>(a, nthreads, shmem, s);
  return rec ? launch64_fwd<R, true, false>(a, nthreads, shmem, s)
             : launch64_fwd<R, false, false>(a, nthreads, shmem, s);
}

template <int R>
static hipError_t launch64_adj(const F64Blk &a, int nthreads, size_t shmem, hipStream_t s) {
  static std::atomic<uint64_t> done{0};
  return launch64(k64_adj_cs<1024, R>, done, a, nthreads, shmem, s);
}

// Whether the forward over these tiles runs as one resident launch: more than
// one chunk, a workgroup for each CU at most, and at most 6 rows per thread
// (8 spill 41 registers in the walk).
static bool walks64(const PlanView &v, const TileView &t) {
  return v.T > t.tb && (int64_t)v.B * t.ntiles <= std::min(CS_WALK_MAX, device_cus()) && t.R <= 6;
}

// Workspace layout in doubles.  saved: A, Bm, C2, the probe amplitudes and
// lap(u_n) of every step; temp: two state pairs and, forward without
// gradients, the coefficients, then a resident launch's progress words, or,
// adjoint, the gradient sum and lambda at the source slots.
struct Blk64 {
  static constexpr int64_t words = CS_WALK_MAX * CS_WALK_W / 2;
  int64_t F, BF, yraw, rec, gsrc;
  int64_t saved() const { return 3 * F + yraw + rec; }
  int64_t fwd_temp() const { return 4 * BF + 3 * F + words; }
  int64_t adj_temp() const { return 5 * BF + gsrc; }
};
static Blk64 blk64(const PlanView &v) {
  Blk64 w;
  w.F = (int64_t)v.Nx * v.Ny;
  w.BF = v.B * w.F;
  w.yraw = (int64_t)v.B * v.T * std::max(v.ntap, 1);
  w.rec = (int64_t)v.T * w.BF;
  w.gsrc = (int64_t)v.B * v.T * std::max(v.nslot, 1);
  return w;
}

static F64Blk args64(const PlanView &v, const wt_scalars_f64 &sc, const TileView &t) {
  F64Blk a{};
  a.B = v.B; a.Nx = v.Nx; a.Ny = v.Ny; a.T = v.T; a.ntap = v.ntap;
  a.nslot = std::max(v.nslot, 1);
  a.ntiles = t.ntiles; a.tiles = t.tiles; a.spx = v.spx; a.taps = v.taps;
  a.s2 = 2.0 * (1.0 / (sc.dt * sc.dt));
  a.t1 = 1.0 / (sc.h * sc.h);
  a.t4 = -4.0 * a.t1;
  a.fstride = 1;
  return a;
}

}  // namespace wt

using namespace wt;

// Common argument checks: a plan whose linear cell runs blocked in double
// precision.
static int check64(const char *what, void *plan, const wt_scalars_f64 *sc, PlanView *v) {
  const int rc = plan ? plan_use_f64(plan) : WT_EINVAL;
  if (plan && rc) return rc;
  if (!plan || plan_view(plan, v) != WT_OK || (sc && (!(sc->dt > 0) || !(sc->h > 0)))) {
    set_error("%s: invalid argument", what);
    return WT_EINVAL;
  }
  if (v->f64.R == 0) {
    set_error("%s: the plan does not run blocked in double precision", what);
    return WT_EUNSUPPORTED;
  }
  return WT_OK;
}

extern "C" int wt_workspace_bytes_rec_f64(void *plan, int32_t with_grad, int64_t *saved,
                                          int64_t *temp) {
  PlanView v;
  if (!saved || !temp) {
    set_error("wt_workspace_bytes_rec_f64: invalid argument");
    return WT_EINVAL;
  }
  const int rc = check64("wt_workspace_bytes_rec_f64", plan, nullptr, &v);
  if (rc) return rc;
  const Blk64 w = blk64(v);
  *saved = with_grad ? w.saved() * 8 : 0;
  *temp = (with_grad ? std::max(w.fwd_temp(), w.adj_temp()) : w.fwd_temp()) * 8;
  return WT_OK;
}

extern "C" int wt_loop_fwd_rec_f64(void *plan, const wt_scalars_f64 *sc, const double *b,
                                   const double *c, const double *x, double *y, double *fields,
                                   int32_t field_stride, int32_t with_grad, void *saved,
                                   void *temp, void *stream) {
  PlanView v;
  if (!sc || !b || !c || !x || !temp || (with_grad && !saved)) {
    set_error("wt_loop_fwd_rec_f64: invalid argument");
    return WT_EINVAL;
  }
  const int rc = check64("wt_loop_fwd_rec_f64", plan, sc, &v);
  if (rc) return rc;
  if (field_stride < 1 || (fields && v.T % field_stride != 0)) {
    set_error("wt_loop_fwd_rec_f64: field_stride %d must divide T = %d", field_stride, v.T);
    return WT_EINVAL;
  }
  hipStream_t s = (hipStream_t)stream;
  const Blk64 w = blk64(v);
  const TileView &t = v.f64;
  F64Blk a = args64(v, *sc, t);
  double *st = (double *)temp;
  double *coef = with_grad ? (double *)saved : st + 4 * w.BF;
  a.A = coef; a.Bm = coef + w.F; a.C2 = coef + 2 * w.F;
  hipLaunchKernelGGL(k64_coef, dim3((unsigned)((w.F + 255) / 256)), dim3(256), 0, s, b, c, w.F,
                     1.0 / sc->dt, 1.0 / (sc->dt * sc->dt), (v.nlf & 4) != 0, sc->c_min,
                     sc->c_max, coef, coef + w.F, coef + 2 * w.F);
  WT_HIP(hipGetLastError());
  a.x = x; a.y = y; a.fields = fields; a.fstride = field_stride;
  if (with_grad) {
    a.yraw = coef + 3 * w.F;
    a.rec = a.yraw + w.yraw;
  }
  const size_t shmem = cs64_shmem_bytes(t.R, t.RHmax, t.RWmax, t.tb);
  const bool walk = walks64(v, t);
  if (walk) {
    a.prog = (int *)(st + w.fwd_temp() - w.words);
    a.walk = v.walk;
    a.walk.every = std::min(a.walk.every, t.ntiles);
    WT_HIP(launch_fill64(st + w.fwd_temp() - w.words, w.words, 0.0, s));
  }
  int pp = 0;
  for (int n = 0; n < v.T; n += t.tb, pp ^= 1) {
    a.n0 = n;
    a.nsteps = walk ? t.tb : std::min(t.tb, v.T - n);
    a.out1 = st + 2 * pp * w.BF;
    a.out2 = a.out1 + w.BF;
    hipError_t e = t.R == 4   ? launch64_fwd<4>(with_grad, sc->h == 1.0, a, t.nthreads, shmem, s)
                   : t.R == 6 ? launch64_fwd<6>(with_grad, sc->h == 1.0, a, t.nthreads, shmem, s)
                              : launch64_fwd<8>(with_grad, sc->h == 1.0, a, t.nthreads, shmem, s);
    WT_HIP(e);
    if (walk) break;
    a.in1 = a.out1;
    a.in2 = a.out2;
  }
  return WT_OK;
}

extern "C" int wt_loop_adj_rec_f64(void *plan, const wt_scalars_f64 *sc, const double *c,
                                   const double *ybar, void *saved, void *temp, double *grad_c,
                                   double *grad_x, void *stream) {
  PlanView v;
  if (!sc || !c || !saved || !temp) {
    set_error("wt_loop_adj_rec_f64: invalid argument");
    return WT_EINVAL;
  }
  const int rc = check64("wt_loop_adj_rec_f64", plan, sc, &v);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  const Blk64 w = blk64(v);
  const TileView &t = v.f64_a;
  F64Blk a = args64(v, *sc, t);
  double *coef = (double *)saved, *st = (double *)temp;
  a.A = coef; a.Bm = coef + w.F; a.C2 = coef + 2 * w.F;
  a.yraw = coef + 3 * w.F;
  a.rec = a.yraw + w.yraw;
  a.ybar = ybar;
  a.gacc = st + 4 * w.BF;
  a.gsrc = st + 5 * w.BF;
  a.first = 1;
  const size_t shmem = cs64_shmem_bytes(t.R, t.RHmax, t.RWmax, t.tb);
  int pp = 0;
  for (int m = v.T; m > 0; m -= t.tb, pp ^= 1) {
    a.m_hi = m;
    a.nsteps = std::min(t.tb, m);
    a.out1 = st + 2 * pp * w.BF;
    a.out2 = a.out1 + w.BF;
    WT_HIP(t.R == 4 ? launch64_adj<4>(a, t.nthreads, shmem, s)
                    : launch64_adj<5>(a, t.nthreads, shmem, s));
    a.in1 = a.out1;
    a.in2 = a.out2;
    a.first = 0;
  }
  if (grad_c) {
    hipLaunchKernelGGL(k64_finalize_gc, dim3((unsigned)((w.F + 255) / 256)), dim3(256), 0, s,
                       a.gacc, v.B, w.F, c, coef, (v.nlf & 4) != 0, sc->c_min, sc->c_max,
                       grad_c);
    WT_HIP(hipGetLastError());
  }
  if (grad_x)
    WT_HIP(v.nslot > 0 ? launch_finalize_gx64(a.gsrc, v.B, v.T, v.nslot, v.mult, grad_x, s)
                       : launch_fill64(grad_x, (int64_t)v.B * v.T, 0.0, s));
  return WT_OK;
}
