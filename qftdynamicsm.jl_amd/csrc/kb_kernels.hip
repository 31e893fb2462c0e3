// kb_kernels.hip -- gfx950 kernels of the 2PI Kadanoff-Baym step.
//
//   hartree        Hartree mass^2 reduction (TwoPIScalar_Initialization.jl:
//                  207-218)
//   memint_step    memory integrals + leapfrog + diagonal of one KB step,
//                  one workgroup per mode block, history read once
//                  (TwoPIScalar_Evolution.jl:766-782, 846-854, 890-915,
//                  951-974)
//   measure        equal-time observables and energies
//                  (TwoPIScalar_Measurement.jl:31-99, 135-174)
// plus small gather/scatter kernels for the host API.
#include "kb_kernels.h"

#include <math.h>

namespace qftkb {

// ---------------------------------------------------------------------------
// Hartree mass: m2 = Mass2 + H ivol sum_p F(t-1,t-1;p)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(1024) void hartree_kernel(const double* __restrict__ H, long NP, int V, long pair,
                                                       double hfac, double Mass2, const double* __restrict__ wgt,
                                                       double* __restrict__ out) {
  __shared__ double red[1024];
  double acc = 0.0;
  for (int p = threadIdx.x; p < V; p += blockDim.x)
    acc += (wgt ? wgt[p] : 1.0) * H[hoff(p / MB, pair, p % MB, NP)];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int w = blockDim.x / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    double h = red[0];
    h *= hfac;
    h += Mass2;
    out[0] = h;
  }
}

// A step's first kernel: its Hartree mass, and its window state, which every
// workgroup works out from the stored one and the last workgroup stores.  (A
// launch of its own for the state took 4 us of a step.)
//
// Bound by latency, HARTREE_LOADS loads in flight per thread; past some 2^18
// sites by the counter, some 35 ns per workgroup, hence at most HARTREE_GROUPS
// of them (112^3: 686 took 25 us).  Each workgroup writes its
// partial sum; the last one to finish (an agent-scope counter: the workgroups
// sit on different XCDs) adds the partials in workgroup order, so the result
// does not depend on which one that is, and resets the counter.
// An ensemble's runs share one launch, like memint_step_runs.
__global__ __launch_bounds__(HARTREE_THREADS) void hartree_step_kernel(HartreeArgs one,
                                                                       const HartreeArgs* __restrict__ runs,
                                                                       int nruns) {
  __shared__ double red[HARTREE_THREADS / 64];
  __shared__ int is_last;
  HartreeArgs a = one;
  int group = blockIdx.x;
  if (nruns > 1) {
    int run = 0;
    while (group >= hartree_groups(runs[run].V)) group -= hartree_groups(runs[run++].V);
    a = runs[run];
  }
  const int N = a.N, V = a.V, G = hartree_groups(V);
  StepState s = a.t ? state_of_step(a.t, N) : *a.st;
  if (!a.t) advance_state(s, N);
  const long pair = pair_off(s.s_tm1, s.s_tm1, N);  // F(t-1,t-1), Evolution.jl:945
  double* part = a.part;
  double acc = 0.0;
  for (int base = group * HARTREE_SITES; base < V; base += G * HARTREE_SITES) {
    double v[HARTREE_LOADS];
#pragma unroll
    for (int u = 0; u < HARTREE_LOADS; ++u) {
      const int p = base + u * HARTREE_THREADS + threadIdx.x;
      v[u] = p < V ? (a.wgt ? a.wgt[p] : 1.0) * a.H[hoff(p / MB, pair, p % MB, a.NP)] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < HARTREE_LOADS; ++u) acc += v[u];
  }
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (G > 1) {
    unsigned* count = reinterpret_cast<unsigned*>(part + G);
    if (threadIdx.x == 0) {
      double b = 0.0;
      for (int w = 0; w < HARTREE_THREADS / 64; ++w) b += red[w];
      part[group] = b;
      is_last = __hip_atomic_fetch_add(count, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)G - 1;
      if (is_last) __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!is_last) return;
    // the partials in a fixed order
    double h = (int)threadIdx.x < G ? part[threadIdx.x] : 0.0;
    for (int o = 32; o > 0; o >>= 1) h += __shfl_xor(h, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = h;
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    double tot = 0.0;
    for (int w = 0; w < HARTREE_THREADS / 64; ++w) tot += red[w];
    a.out[0] = tot * a.hfac + a.Mass2;
    if (a.sum_out) a.sum_out[0] = tot;
    *a.st = s;
  }
}

// ---------------------------------------------------------------------------
// Memory integrals + leapfrog + diagonal, one workgroup per mode block.
//
// With rho antisymmetric and F symmetric, the reference's
//   R_r(t') = -sum_{z=t'+1}^{t-2} Sr(z) r(z,t')                    (Evolution.jl:846-854)
//   R_F(t') = -sum_{z=tmin}^{t-2} w_z Sr(z) F(z,t')
//             +sum_{z=tmin}^{t'-1} w_z SF(z) r(z,t')                (Evolution.jl:766-782)
// (w = 1/2 at tmin, 1 otherwise; S(z) = Sigma(t-1,z)) make every stored
// entry (a,b), a>b, feed two output rows: with u = m w Sr, v = w SF,
// ms = m Sr (m = 0 at z = t-1):
//   R_F(a) += -u(b) F - v(b) r,  R_F(b) += -u(a) F,  R_r(b) += -ms(a) r,
// and the diagonal (a,a) feeds R_F(a) += -u(a) F.  The kernel walks the
// slot triangle once: every 8-lane worker streams chunks of rows of one
// 4-column block (contiguous in HBM) with two row batches in flight,
// keeps the 4 column sums in registers and adds row and column sums into
// per-slot LDS accumulators with ds_add_f64.
// In slot space, pair (hi, lo) has time(hi) < time(lo) exactly when
// lo < s_min <= hi; those pairs swap the roles of a and b.
// ---------------------------------------------------------------------------
// Tile shape (template parameters, picked per lattice and window by the
// autotuner): ROWS slot rows per work item (one chunk of a column block),
// B rows per batch, two batches in flight.

__device__ __forceinline__ void slot_weights(int x, int smin, int N, int L, double& w, double& m) {
  const int rel = window_pos(x, smin, N);
  w = rel == 0 ? 0.5 : 1.0;
  m = rel == L - 1 ? 0.0 : 1.0;
}

// History lines are streamed once per step: load them non-temporally so
// they do not evict the self-energy lines that are re-read from L2.
#ifndef KB_NT_LOADS
#define KB_NT_LOADS 1
#endif
// Loads go through global-address-space pointers: the pointers come from the
// argument struct, so plain dereferences compile to flat loads, whose waits
// also drain the LDS queue and every load in flight (s_waitcnt vmcnt(0)
// lgkmcnt(0)); global loads let a batch wait only for its own lines.
typedef double kb_d2v __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(1))) const kb_d2v kb_gd2v;
__device__ __forceinline__ double2 ld_stream(const double* p) {
#if KB_NT_LOADS
  const kb_d2v v = __builtin_nontemporal_load((kb_gd2v*)(p));
#else
  const kb_d2v v = *(kb_gd2v*)(p);
#endif
  return make_double2(v.x, v.y);
}
__device__ __forceinline__ double2 ld_global(const void* p) {
  const kb_d2v v = *(kb_gd2v*)(p);
  return make_double2(v.x, v.y);
}

template <int B>
struct RowBatch {
  double2 e[B][CB];  // (F, r) of slots (row, c0 + jc)
  double2 fs[B];     // (SigF, Sigr) of the row slot
};

// rows r .. r+MI_B-1 of the column block starting at storage slot cbase;
// rows past rlast are clamped to rlast (re-read, not used)
template <int B>
__device__ __forceinline__ void load_batch(RowBatch<B>& b, const double* __restrict__ Hb,
                                           const double2* __restrict__ Sb, long cbase, int c0, int r, int rlast) {
#pragma unroll
  for (int h = 0; h < B; ++h) {
    const int rr = min(r + h, rlast);
    const long pb = cbase + (long)(rr - c0) * CB;
#pragma unroll
    for (int jc = 0; jc < CB; ++jc) b.e[h][jc] = ld_stream(Hb + (size_t)(pb + jc) * MB * 2);
    b.fs[h] = ld_global(Sb + (size_t)rr * MB);
  }
}

struct ColState {
  double u[CB], v[CB], ms[CB], cF[CB], cR[CB];
  unsigned phi;  // bit jc: column slot lies before s_min (its time is after the wrap)
};

// Pair (r, c), r > c in slot space.  Time order is reversed (time(r) <
// time(c)) exactly when r >= s_min > c; `neg` carries that per column.
__device__ __forceinline__ void pair_update(double Fv, double Pv, bool n, double uc, double vc, double msc,
                                            double ur, double vr, double msr, double& rowF, double& rowR,
                                            double& cF, double& cR) {
  rowF -= uc * Fv + (n ? 0.0 : vc) * Pv;
  rowR += (n ? msc : 0.0) * Pv;
  cF += (n ? vr : 0.0) * Pv - ur * Fv;
  cR -= (n ? 0.0 : msr) * Pv;
}

template <int B>
__device__ __forceinline__ void process_batch(const RowBatch<B>& b, int r, int r1, int dead, int smin, int N, int L,
                                              ColState& cs, double* accF, double* accR, int lane) {
#pragma unroll
  for (int h = 0; h < B; ++h) {
    const int rr = r + h;
    if (rr < r1) {
      const bool okr = rr != dead;
      double w, m;
      slot_weights(rr, smin, N, L, w, m);
      const double ur = okr ? m * w * b.fs[h].y : 0.0;
      const double vr = okr ? w * b.fs[h].x : 0.0;
      const double msr = okr ? m * b.fs[h].y : 0.0;
      const unsigned neg = rr >= smin ? cs.phi : 0u;
      double rowF = 0.0, rowR = 0.0;
#pragma unroll
      for (int jc = 0; jc < CB; ++jc)
        pair_update(b.e[h][jc].x, b.e[h][jc].y, (neg >> jc) & 1u, cs.u[jc], cs.v[jc], cs.ms[jc], ur, vr, msr, rowF,
                    rowR, cs.cF[jc], cs.cR[jc]);
      atomicAdd(&accF[rr * MB + lane], rowF);
      atomicAdd(&accR[rr * MB + lane], rowR);
    }
  }
}

// Sweep of work items [ibeg, iend) of one site block: memory-integral row
// and column sums into the LDS accumulators (see above).  Workers start at
// ibeg + worker and take further items from the LDS counter *next_item.
template <int ROWS, int B>
__device__ __forceinline__ void memint_sweep(const MemintArgs& a, const StepState& ss, int mb, double* accF,
                                             double* accR, int* next_item, int ibeg, int iend) {
  const int N = a.N;
  const int tid = threadIdx.x;
  const int lane = tid & (MB - 1);
  const int worker = tid >> 3;
  const int Rmax = ss.Rmax;
  const int dead = ss.dead;
  const int smin = ss.s_min;
  const int L = ss.L;
  const double* __restrict__ Hb = a.H + hoff(mb, 0, 0, a.NP) + lane * 2;
  // self-energies of this block: (SigF, Sigr) per slot for this lane
  const double2* __restrict__ Sb = reinterpret_cast<const double2*>(a.S + soff(mb, 0, lane, N));
  // work items: (column block J, chunk of MI_ROWS rows), in storage order;
  // the first item of each worker is static, later ones are taken from an
  // LDS counter, so workers that finish early take more
  int item = ibeg + worker;
  while (item < iend) {
    const int2 jk = a.items[item];
    const int J = jk.x;
    const int c0 = J * CB;
    const int r0 = c0 + jk.y * ROWS;
    const int r1 = min(r0 + ROWS, Rmax);
    if (c0 < Rmax && r0 < r1) {
      const long cbase = colblock_offset(J, N);
      ColState cs;
      cs.phi = 0;
#pragma unroll
      for (int jc = 0; jc < CB; ++jc) {
        const int c = c0 + jc;
        const bool ok = c < Rmax && c != dead;
        const double2 fs = ld_global(Sb + (size_t)min(c, N - 1) * MB);
        double w, m;
        slot_weights(c, smin, N, L, w, m);
        cs.u[jc] = ok ? m * w * fs.y : 0.0;
        cs.v[jc] = ok ? w * fs.x : 0.0;
        cs.ms[jc] = ok ? m * fs.y : 0.0;
        cs.cF[jc] = cs.cR[jc] = 0.0;
        cs.phi |= (c < smin ? 1u : 0u) << jc;
      }
      int r = r0;
      // rows crossing the diagonal of the block: columns c0 .. r only
      for (; r < r1 && r < c0 + CB; ++r) {
        const bool okr = r != dead;
        const double2 fs = ld_global(Sb + (size_t)r * MB);
        double w, m;
        slot_weights(r, smin, N, L, w, m);
        const double ur = okr ? m * w * fs.y : 0.0;
        const double vr = okr ? w * fs.x : 0.0;
        const double msr = okr ? m * fs.y : 0.0;
        const unsigned neg = r >= smin ? cs.phi : 0u;
        const long pb = cbase + (long)(r - c0) * CB;
        double rowF = 0.0, rowR = 0.0;
        for (int jc = 0; jc < CB; ++jc) {
          const int c = c0 + jc;
          if (c > r) break;
          const double2 e = ld_global(Hb + (size_t)(pb + jc) * MB * 2);
          if (c == r)
            rowF -= ur * e.x;
          else
            pair_update(e.x, e.y, (neg >> jc) & 1u, cs.u[jc], cs.v[jc], cs.ms[jc], ur, vr, msr, rowF, rowR,
                        cs.cF[jc], cs.cR[jc]);
        }
        atomicAdd(&accF[r * MB + lane], rowF);
        atomicAdd(&accR[r * MB + lane], rowR);
      }
      // full rows: two batches of MI_B rows in flight
      if (r < r1) {
        const int rlast = r1 - 1;
        RowBatch<B> X, Y;
        load_batch(X, Hb, Sb, cbase, c0, r, rlast);
        while (true) {
          load_batch(Y, Hb, Sb, cbase, c0, r + B, rlast);
          process_batch(X, r, r1, dead, smin, N, L, cs, accF, accR, lane);
          r += B;
          if (r >= r1) break;
          load_batch(X, Hb, Sb, cbase, c0, r + B, rlast);
          process_batch(Y, r, r1, dead, smin, N, L, cs, accF, accR, lane);
          r += B;
          if (r >= r1) break;
        }
      }
#pragma unroll
      for (int jc = 0; jc < CB; ++jc) {
        const int c = c0 + jc;
        if (c < Rmax && c != dead) {
          atomicAdd(&accF[c * MB + lane], cs.cF[jc]);
          atomicAdd(&accR[c * MB + lane], cs.cR[jc]);
        }
      }
    }
    // next item: one LDS atomic per worker
    int nxt = 0;
    if (lane == 0) nxt = atomicAdd(next_item, 1);
    item = __shfl(nxt, tid & ~(MB - 1) & 63);
  }
}

// Leapfrog of row t and the diagonal from the accumulated memory integrals
// of one site block; red holds blockDim.x / 64 rows of MB doubles.
__device__ __forceinline__ void memint_leapfrog(const MemintArgs& a, const StepState& ss, int mb,
                                                const double* accF, const double* accR, double (*red)[MB],
                                                double (*diagF)[MB]) {
  const int N = a.N;
  const int tid = threadIdx.x;
  const int lane = tid & (MB - 1);
  const int worker = tid >> 3;
  const int nworkers = blockDim.x >> 3;
  const int Rmax = ss.Rmax;
  const int dead = ss.dead;
  const int smin = ss.s_min;
  const int L = ss.L;
  const double2* __restrict__ Sb = reinterpret_cast<const double2*>(a.S + soff(mb, 0, lane, N));
  // ---- leapfrog of row t (evolve_r!, evolve_F!: Evolution.jl:890-915) ----
  const int p = mb * MB + lane;
  const bool real_site = p < a.V;
  const double m2 = a.m2[0];
  const double dt = a.dt;
  const double dt2 = dt * dt, dt3 = dt * dt * dt;
  const double Om = (a.kL2[p] + m2) * dt2;  // setomega2values!, Evolution.jl:918-921
  double dsum = 0.0;
  double* __restrict__ Hw = a.H + hoff(mb, 0, 0, a.NP);
  constexpr int LU = 4;  // slots per worker in flight
  for (int x0 = worker * LU; x0 < Rmax; x0 += nworkers * LU) {
    double2 e1[LU], e2[LU], fsx[LU];
#pragma unroll
    for (int u = 0; u < LU; ++u) {
      const int x = min(x0 + u, Rmax - 1);
      e1[u] = ld_global(Hw + ((size_t)pair_off(ss.s_tm1, x, N) * MB + lane) * 2);
      e2[u] = ld_global(Hw + ((size_t)pair_off(ss.s_tm2, x, N) * MB + lane) * 2);
      fsx[u] = ld_global(Sb + (size_t)x * MB);
    }
#pragma unroll
    for (int u = 0; u < LU; ++u) {
      const int x = x0 + u;
      if (x >= Rmax || x == dead) continue;
      const int rel = window_pos(x, smin, N);
      const int tx = ss.tmin + rel;
      const double r1 = e1[u].y * (ss.s_tm1 >= x ? 1.0 : -1.0);
      const double r2 = e2[u].y * (ss.s_tm2 >= x ? 1.0 : -1.0);
      const double RHSF = accF[x * MB + lane] * dt3;
      const double Fn = (2.0 - Om) * e1[u].x - e2[u].x + RHSF;
      double rn;
      if (tx == ss.t - 1) {
        rn = dt;
      } else {
        const double RHSr = accR[x * MB + lane] * dt3;
        rn = (2.0 - Om) * r1 - r2 + RHSr;
      }
      if (real_site) {
        double2 o = make_double2(Fn, rn * (ss.s_t >= x ? 1.0 : -1.0));
        *reinterpret_cast<double2*>(Hw + ((size_t)pair_off(ss.s_t, x, N) * MB + lane) * 2) = o;
      }
      // terms of getRHS_F!(t,t) (Evolution.jl:973) over the fresh row
      if (a.integral) {
        const double w = rel == 0 ? 0.5 : 1.0;
        const double m = rel == L - 1 ? 0.0 : 1.0;
        dsum += -(m * w * fsx[u].y) * Fn - (w * fsx[u].x) * rn;
      }
      if (tx == ss.t - 1) diagF[0][lane] = Fn;
      if (tx == ss.t - 2) diagF[1][lane] = Fn;
    }
  }
  // reduce over the 8 workers of the wave (lane bits 3..5), then over waves
  dsum += __shfl_xor(dsum, 8);
  dsum += __shfl_xor(dsum, 16);
  dsum += __shfl_xor(dsum, 32);
  if ((tid & 63) < MB) red[tid >> 6][lane] = dsum;
  __syncthreads();
  if (tid < MB) {
    double RF = 0.0;
    for (int wv = 0; wv < (int)(blockDim.x >> 6); ++wv) RF += red[wv][tid];
    const double Ftt = (2.0 - Om) * diagF[0][tid] - diagF[1][tid] + RF * dt3;
    if (real_site) {
      *reinterpret_cast<double2*>(Hw + ((size_t)pair_off(ss.s_t, ss.s_t, N) * MB + tid) * 2) =
          make_double2(Ftt, 0.0);
    }
  }
}

template <int ROWS, int B, int TPB>
__global__ __launch_bounds__(TPB, 512 / TPB) void memint_step(const MemintArgs* __restrict__ runs,
                                                                 const int* __restrict__ wg_start, int nruns) {
  extern __shared__ double smem[];
  // which run this workgroup belongs to (runs are few; wg_start is uniform)
  int run = 0;
  while (run + 1 < nruns && (int)blockIdx.x >= wg_start[run + 1]) ++run;
  const MemintArgs a = runs[run];
  const StepState ss = *a.st;
  const int N = a.N;
  double* accF = smem;           // R_F per slot, lane
  double* accR = accF + N * MB;  // R_r
  __shared__ double red[TPB / 64][MB];
  __shared__ double diagF[2][MB];
  __shared__ int next_item;
  const int mb = blockIdx.x - wg_start[run];
  const int tid = threadIdx.x;
  for (int i = tid; i < N * MB; i += blockDim.x) {
    accF[i] = 0.0;
    accR[i] = 0.0;
  }
  if (tid == 0) next_item = blockDim.x >> 3;
  __syncthreads();
  if (a.integral) memint_sweep<ROWS, B>(a, ss, mb, accF, accR, &next_item, 0, a.nitems);
  __syncthreads();
  memint_leapfrog(a, ss, mb, accF, accR, red, diagF);
}

// Split form for windows with few site blocks (cubic-orbit storage): each
// site block's work items are cut into nsplit contiguous ranges, one
// workgroup each; memint_partial writes its accumulators to part, and
// memint_finish sums them and runs the leapfrog.
template <int ROWS, int B, int TPB>
__global__ __launch_bounds__(TPB, 512 / TPB) void memint_partial(const MemintArgs* __restrict__ runs, int nsplit,
                                                                    double* __restrict__ part) {
  extern __shared__ double smem[];
  const MemintArgs a = runs[0];
  const StepState ss = *a.st;
  const int N = a.N;
  double* accF = smem;
  double* accR = accF + N * MB;
  __shared__ int next_item;
  const int mb = blockIdx.x / nsplit;
  const int sp = blockIdx.x - mb * nsplit;
  const int ibeg = (int)((long)a.nitems * sp / nsplit);
  const int iend = (int)((long)a.nitems * (sp + 1) / nsplit);
  const int tid = threadIdx.x;
  for (int i = tid; i < N * MB; i += blockDim.x) {
    accF[i] = 0.0;
    accR[i] = 0.0;
  }
  if (tid == 0) next_item = ibeg + (blockDim.x >> 3);
  __syncthreads();
  if (a.integral) memint_sweep<ROWS, B>(a, ss, mb, accF, accR, &next_item, ibeg, iend);
  __syncthreads();
  double* out = part + (size_t)blockIdx.x * 2 * N * MB;
  for (int i = tid; i < 2 * N * MB; i += blockDim.x) out[i] = smem[i];
}

// (1024 threads, four partials in flight: the sum over the splits' partials
// is latency-bound)
__global__ __launch_bounds__(MEMINT_FINISH_THREADS) void memint_finish(MemintArgs a, int nsplit,
                                                                       const double* __restrict__ part) {
  extern __shared__ double smem[];
  const StepState ss = *a.st;
  const int N = a.N;
  double* accF = smem;
  double* accR = accF + N * MB;
  __shared__ double red[MEMINT_FINISH_THREADS / 64][MB];
  __shared__ double diagF[2][MB];
  const int mb = blockIdx.x;
  const size_t stride = (size_t)2 * N * MB;
  const double* in = part + (size_t)mb * nsplit * stride;
  for (int i = threadIdx.x; i < ss.Rmax * MB; i += blockDim.x) {
    double f = 0.0, r = 0.0;
    for (int k0 = 0; k0 < nsplit; k0 += 4) {
      double x[4], y[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const double* q = in + min(k0 + u, nsplit - 1) * stride + i;
        x[u] = q[0];
        y[u] = q[N * MB];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        f += k0 + u < nsplit ? x[u] : 0.0;
        r += k0 + u < nsplit ? y[u] : 0.0;
      }
    }
    accF[i] = f;
    accR[i] = r;
  }
  __syncthreads();
  memint_leapfrog(a, ss, mb, accF, accR, red, diagF);
}

// ---------------------------------------------------------------------------
// The default shape in short windows, and wherever site blocks are few: the
// same integrals with the triangle cut into equal runs.  The rows of the slot
// triangle in use (4 slots each, in memory order: column block after column
// block) are numbered, and every 8-lane worker of a site block takes one
// contiguous run of them, crossing column blocks on the way.
// Bound: HBM latency, not bandwidth -- a short window is a few KB to some 100
// KB per site block.  The 64-row items gave 4 of 32 workers work at
// N_mem = 16 and left a 64-row worker running alone at 96; runs of equal
// length end together.  Small workgroups (one wave per site block up to
// N_mem = 32, where rows t-1 and t-2 are also kept in LDS for the leapfrog)
// put up to 16 site blocks on a CU, so one block's set-up and leapfrog hide
// behind the others' loads.  The coefficients of a block are staged in LDS
// while its first rows are on their way; one row (4 lines) is in flight per
// worker: 2 or 3 need more than 128 registers, and fewer waves cost more
// than the deeper pipeline gives.
// Measured (64-row items -> runs): 112^3 N_mem = 16 4868 -> 946 us (0.63 ->
// 3.2 TB/s), 64^3 N_mem = 32 1267 -> 544 us, 48^3 N_mem = 48 742 -> 466 us,
// 42^3 N_mem = 96 1146 -> 1085 us (5.1 TB/s), 32^3 N_mem = 150 1111 -> 1043
// us (5.7 TB/s), 16^3 N_mem = 64 37.6 -> 30.6 us, 16^2 N_mem = 24 13.3 -> 6.4
// us.  Past N_mem = 208 the staged items are as fast (32^3 N_mem = 300: 3840
// against 3842-3988 us) and keep the call.
// ---------------------------------------------------------------------------
__host__ __device__ inline int run_base(int J, int R) { return J * R - CB / 2 * J * (J - 1); }
__host__ __device__ inline int run_rows(int R) { return run_base((R + CB - 1) / CB, R); }

// column block of row number g < run_rows(R): the largest J with
// run_base(J, R) <= g (a root in float, corrected by at most one)
__device__ __forceinline__ int run_block(int g, int R) {
  const float h = (float)(R + CB / 2);
  int J = (int)((h - sqrtf(fmaxf(h * h - 2.0f * CB * (float)g, 0.0f))) * (1.0f / CB));
  J = max(0, min(J, (R - 1) / CB));
  while (J > 0 && run_base(J, R) > g) --J;
  while (CB * (J + 1) < R && run_base(J + 1, R) <= g) ++J;
  return J;
}

// offset in doubles of slot pair (a, b) from the site block's first pair
__device__ __forceinline__ int pair_rel(int a, int b, int N) {
  const int hi = max(a, b), lo = min(a, b);
  const int J = lo / CB;
  return (CB * (N * J - CB / 2 * J * (J - 1)) + (hi - J * CB) * CB + (lo - J * CB)) * (2 * MB);
}

// Sweep of one site block by worker w of nw: cf (v, ms per slot and lane) and
// the accumulators are staged by the whole workgroup, the first rows are on
// their way meanwhile.
template <int D, bool STASH>
__device__ __forceinline__ void memint_runs(const MemintArgs& a, const StepState& ss, int mb, double2* cf,
                                            double* accF, double* accR, double2* rows, int w, int nw) {
  const int N = a.N, R = ss.Rmax, smin = ss.s_min;
  const int tid = threadIdx.x, lane = tid & (MB - 1);
  const int T = a.integral ? run_rows(R) : 0;
  const int g0 = T * w / nw, n = T * (w + 1) / nw - g0;
  int J = 0, r = 0;
  double2 e[D][CB];
  const double* p = a.H + hoff(mb, 0, lane, a.NP);
  const int gap = (N - R) * (CB * 2 * MB);  // rows not in use at the end of a column block
  int rp = 0, cp = 0, k = 0;  // next row to fetch, its column block's first slot
  auto fetch = [&](double2 (&b)[CB]) {
#pragma unroll
    for (int jc = 0; jc < CB; ++jc) b[jc] = ld_stream(p + jc * 2 * MB);
    if (++k < n) {  // past the last row of the run: read it again
      p += CB * 2 * MB;
      if (++rp == R) {
        cp += CB;
        rp = cp;
        p += gap;
      }
    }
  };
  if (n > 0) {
    J = run_block(g0, R);
    r = CB * J + g0 - run_base(J, R);
    rp = r;
    cp = CB * J;
    p += (CB * (N * J - CB / 2 * J * (J - 1)) + (r - CB * J) * CB) * (2 * MB);
#pragma unroll
    for (int d = 0; d < D; ++d) fetch(e[d]);
  }
  for (int x = tid >> 3; x < R; x += blockDim.x >> 3) {
    const double2 fs = ld_global(a.S + soff(mb, x, lane, N));
    double wt, m;
    slot_weights(x, smin, N, ss.L, wt, m);
    cf[x * MB + lane] = x == ss.dead ? make_double2(0.0, 0.0) : make_double2(wt * fs.x, m * fs.y);
    accF[x * MB + lane] = 0.0;
    accR[x * MB + lane] = 0.0;
  }
  __syncthreads();
  if (n > 0) {
    // column slots c0 .. c0 + 3: u, v and the sums.  ms is only needed where
    // time order is reversed (c < smin), and there u = ms.
    double uc[CB], vc[CB], cF[CB], cR[CB];
    unsigned phi = 0;  // bit jc: column slot lies before smin
    auto columns = [&](int c0) {
      phi = 0;
#pragma unroll
      for (int jc = 0; jc < CB; ++jc) {
        const int c = c0 + jc;
        const double2 q = c < R ? cf[c * MB + lane] : make_double2(0.0, 0.0);
        vc[jc] = q.x;
        uc[jc] = c == smin ? 0.5 * q.y : q.y;
        cF[jc] = cR[jc] = 0.0;
        phi |= (c < smin ? 1u : 0u) << jc;
      }
    };
    auto flush = [&](int c0) {
#pragma unroll
      for (int jc = 0; jc < CB; ++jc)
        if (c0 + jc < R) {
          atomicAdd(&accF[(c0 + jc) * MB + lane], cF[jc]);
          atomicAdd(&accR[(c0 + jc) * MB + lane], cR[jc]);
        }
    };
    int c0 = CB * J;
    columns(c0);
    int left = n;
    auto use = [&](double2 (&b)[CB]) {
      const double2 q = cf[r * MB + lane];
      const double ur = r == smin ? 0.5 * q.y : q.y;
      const unsigned neg = r >= smin ? phi : 0u;
      double rowF = 0.0, rowR = 0.0;
      if constexpr (STASH) {
        // rows t-1 and t-2 for the leapfrog: slot pairs with s_tm1 or s_tm2
        const int d1 = ss.s_tm1 - c0, d2 = ss.s_tm2 - c0;
        if (r == ss.s_tm1 || r == ss.s_tm2) {
          double2* o = rows + (r == ss.s_tm1 ? 0 : N * MB) + c0 * MB + lane;
#pragma unroll
          for (int jc = 0; jc < CB; ++jc)
            if (c0 + jc <= r) o[jc * MB] = b[jc];
        }
#pragma unroll
        for (int jc = 0; jc < CB; ++jc) {
          if (d1 == jc && c0 + jc <= r) rows[r * MB + lane] = b[jc];
          if (d2 == jc && c0 + jc <= r) rows[(N + r) * MB + lane] = b[jc];
        }
      }
      if (__any(r < c0 + CB)) {
        // a worker is on its block's diagonal, which feeds its row once; the
        // slots above it are padding
#pragma unroll
        for (int jc = 0; jc < CB; ++jc) {
          if (c0 + jc == r) rowF -= ur * b[jc].x;
          if (c0 + jc >= r) b[jc] = make_double2(0.0, 0.0);
        }
      }
#pragma unroll
      for (int jc = 0; jc < CB; ++jc) {
        const bool nf = (neg >> jc) & 1u;
        rowF -= uc[jc] * b[jc].x + (nf ? 0.0 : vc[jc]) * b[jc].y;
        rowR += (nf ? uc[jc] : 0.0) * b[jc].y;
        cF[jc] += (nf ? q.x : 0.0) * b[jc].y - ur * b[jc].x;
        cR[jc] -= (nf ? 0.0 : q.y) * b[jc].y;
      }
      atomicAdd(&accF[r * MB + lane], rowF);
      atomicAdd(&accR[r * MB + lane], rowR);
      if (++r == R) {
        flush(c0);
        c0 += CB;
        r = c0;
        if (c0 < R) columns(c0);
      }
    };
    bool more = true;
    while (more) {
#pragma unroll
      for (int d = 0; d < D; ++d)
        if (more) {
          use(e[d]);
          more = --left > 0;
          fetch(e[d]);
        }
    }
    if (c0 < R) flush(c0);
  }
  __syncthreads();
}

// memint_leapfrog with the coefficients in LDS; red: a row of MB doubles per wave
template <int TPB, bool STASH>
__device__ __forceinline__ void leapfrog_runs(const MemintArgs& a, const StepState& ss, int mb, const double2* cf,
                                              const double* accF, const double* accR, const double2* rows,
                                              double (*red)[MB], double (*diagF)[MB]) {
  constexpr int NW = TPB / MB;
  constexpr int LU = 4;  // slots per worker in flight
  const int N = a.N, R = ss.Rmax, smin = ss.s_min;
  const int tid = threadIdx.x, lane = tid & (MB - 1), worker = tid >> 3;
  const int p = mb * MB + lane;
  const bool real_site = p < a.V;
  const double dt = a.dt, dt2 = dt * dt, dt3 = dt * dt * dt;
  const double Om = (a.kL2[p] + a.m2[0]) * dt2;  // setomega2values!, Evolution.jl:918-921
  double dsum = 0.0;
  double* __restrict__ Hw = a.H + hoff(mb, 0, lane, a.NP);
  for (int x0 = worker; x0 < R; x0 += NW * LU) {
    double2 e1[LU], e2[LU];
#pragma unroll
    for (int u = 0; u < LU; ++u) {
      const int x = min(x0 + u * NW, R - 1);
      if (STASH && a.integral) {
        e1[u] = rows[x * MB + lane];
        e2[u] = rows[(N + x) * MB + lane];
      } else {
        e1[u] = ld_global(Hw + pair_rel(ss.s_tm1, x, N));
        e2[u] = ld_global(Hw + pair_rel(ss.s_tm2, x, N));
      }
    }
#pragma unroll
    for (int u = 0; u < LU; ++u) {
      const int x = x0 + u * NW;
      if (x >= R || x == ss.dead) continue;
      const int tx = ss.tmin + window_pos(x, smin, N);
      const double r1 = e1[u].y * (ss.s_tm1 >= x ? 1.0 : -1.0);
      const double r2 = e2[u].y * (ss.s_tm2 >= x ? 1.0 : -1.0);
      const double Fn = (2.0 - Om) * e1[u].x - e2[u].x + accF[x * MB + lane] * dt3;
      const double rn = tx == ss.t - 1 ? dt : (2.0 - Om) * r1 - r2 + accR[x * MB + lane] * dt3;
      if (real_site)
        *reinterpret_cast<double2*>(Hw + pair_rel(ss.s_t, x, N)) = make_double2(Fn, rn * (ss.s_t >= x ? 1.0 : -1.0));
      // terms of getRHS_F!(t,t) (Evolution.jl:973) over the fresh row
      if (a.integral) {
        const double2 q = cf[x * MB + lane];
        dsum += -(x == smin ? 0.5 * q.y : q.y) * Fn - q.x * rn;
      }
      if (tx == ss.t - 1) diagF[0][lane] = Fn;
      if (tx == ss.t - 2) diagF[1][lane] = Fn;
    }
  }
  dsum += __shfl_xor(dsum, 8);
  dsum += __shfl_xor(dsum, 16);
  dsum += __shfl_xor(dsum, 32);
  if ((tid & 63) < MB) red[tid >> 6][lane] = dsum;
  __syncthreads();
  if (tid < MB) {
    double RF = 0.0;
#pragma unroll
    for (int wv = 0; wv < TPB / 64; ++wv) RF += red[wv][tid];
    const double Ftt = (2.0 - Om) * diagF[0][tid] - diagF[1][tid] + RF * dt3;
    if (real_site)
      *reinterpret_cast<double2*>(Hw + pair_rel(ss.s_t, ss.s_t, N)) = make_double2(Ftt, 0.0);
  }
}

// One workgroup per site block; a single run's arguments come by value (no
// chain of loads before the first row), those of several runs from a table.
template <int D, int TPB, bool STASH>
__global__ __launch_bounds__(TPB, D > 1 ? 3 : 4) void memint_step_runs(MemintArgs one,
                                                                       const MemintArgs* __restrict__ runs,
                                                                       const int* __restrict__ wg_start, int nruns) {
  extern __shared__ double smem[];
  MemintArgs a = one;
  int mb = blockIdx.x;
  if (nruns > 1) {
    int run = 0;
    while (run + 1 < nruns && (int)blockIdx.x >= wg_start[run + 1]) ++run;
    a = runs[run];
    mb -= wg_start[run];
  }
  const StepState ss = *a.st;
  double2* cf = reinterpret_cast<double2*>(smem);
  double* accF = smem + 2 * a.N * MB;
  double* accR = accF + a.N * MB;
  double2* rows = reinterpret_cast<double2*>(accR + a.N * MB);  // STASH: rows t-1, t-2
  __shared__ double red[TPB / 64][MB];
  __shared__ double diagF[2][MB];
  memint_runs<D, STASH>(a, ss, mb, cf, accF, accR, rows, threadIdx.x >> 3, TPB / MB);
  leapfrog_runs<TPB, STASH>(a, ss, mb, cf, accF, accR, rows, red, diagF);
}

// Split form: the runs of a site block over the workers of nsplit
// workgroups, whose accumulators go to part; memint_finish does the rest.
template <int D, int TPB>
__global__ __launch_bounds__(TPB, D > 1 ? 3 : 4) void memint_partial_runs(MemintArgs a, int nsplit,
                                                                          double* __restrict__ part) {
  extern __shared__ double smem[];
  const StepState ss = *a.st;
  const int N = a.N, R = ss.Rmax;
  const int mb = blockIdx.x / nsplit, sp = blockIdx.x - mb * nsplit;
  double2* cf = reinterpret_cast<double2*>(smem);
  double* accF = smem + 2 * N * MB;
  double* accR = accF + N * MB;
  memint_runs<D, false>(a, ss, mb, cf, accF, accR, nullptr, sp * (TPB / MB) + ((int)threadIdx.x >> 3),
                        nsplit * (TPB / MB));
  double* out = part + (size_t)blockIdx.x * 2 * N * MB;
  for (int i = threadIdx.x; i < R * MB; i += TPB) {
    out[i] = accF[i];
    out[N * MB + i] = accR[i];
  }
}

constexpr int RUNS_MAX_N = 208;       // longest window of the whole-block form
constexpr int LDS_PER_CU = 160 * 1024;
constexpr int RUNS_FOUR_MAX_N = 152;  // longest of which four workgroups fit a CU (256 bytes of LDS per slot)
// Shorter windows: the second launch costs more than the split gives.  A step of
// 8^3 whole and split: N_mem 40 19.8 and 21.3 us, 48 20.7 and 22.4, 56 24.4 and
// 23.0, 64 28.2 and 23.5, 100 50.5 and 28.9 (the two are level at some 52).
constexpr int RUNS_SPLIT_MIN_N = 48;
constexpr int RUNS_SPLIT_MAX_N = 600; // 256 bytes of LDS per slot
constexpr int RUNS_SPLIT_THREADS = 512;

// the share of the chip's slots that `blocks` workgroups use over their rounds,
// in percent
inline unsigned rounds_full(unsigned blocks, unsigned slots) {
  const unsigned rounds = (blocks + slots - 1) / slots;
  return rounds <= 1 ? 100 : 100ull * blocks / ((unsigned long long)rounds * slots);
}

// Three workgroups to a CU are enough to be faster than the items (six to a CU)
// unless the blocks' last round leaves most of the slots empty: 1000 blocks on
// 768 slots took 427 us at N_mem = 192 against 408, 729 blocks (all at once)
// 285 against 311, 1331 and more 0.89 to 1.02 of the items' time (160 to 208).
// With four they are faster whatever the number of blocks.
bool memint_runs_whole(int tile, int N, unsigned blocks, int cus) {
  return tile == 0 && N <= RUNS_MAX_N && (N <= RUNS_FOUR_MAX_N || rounds_full(blocks, 3 * cus) >= 70);
}

// Workgroups per site block: one per CU in all.  16^2 and 1D lattices, and
// orbit storage, have fewer site blocks than CUs: 128 sites in 1D at
// N_mem = 400 took 298 us on 16 CUs and take 54 us on 256; 122 blocks
// (32^3 in orbits) 247 us as 6 parts of 256 threads and 215 us as 2 of 512.
int memint_runs_split(int tile, int N, int NB, int cus) {
  if (tile != 0 || N < RUNS_SPLIT_MIN_N || N > RUNS_SPLIT_MAX_N) return 1;
  return max(1, min(16, cus / NB));
}

hipError_t memint_runs_prepare() {
  return hipFuncSetAttribute((const void*)memint_partial_runs<3, RUNS_SPLIT_THREADS>,
                             hipFuncAttributeMaxDynamicSharedMemorySize, RUNS_SPLIT_MAX_N * 32 * MB);
}

// Threads per site block: a wave up to N_mem = 32 and two up to 152, if the
// blocks fill the CUs that way (2048 of them), two only if their rounds on the
// chip are at least 80% full (65% up to N_mem = 64; a CU holds eight such
// workgroups or what its LDS takes); four otherwise, and eight for long windows
// on fewer than two blocks per CU (256 blocks, N_mem = 200: 149 us at 256
// threads, 121 at 512).  In parts of the items' time, two waves and four: 40^3
// N_mem = 48 0.58 and 0.61, 100 0.91 and 0.93, 160 (three to a CU) 1.04 and
// 0.96; 26^3 112 (86% full) 0.87 and 0.91, 140 (72%) 1.05 and 0.95; 128^2 100
// (67%) 1.04 and 0.94, 128 (100%) 0.89 and 0.91; 28^3 112 (71%) 0.95 and 0.88,
// 128 (89%) both 0.89; 160^2 48 (78%) 0.61 and 0.64, 128 (78%) 0.94 and 0.91.
hipError_t launch_memint_runs(const MemintArgs& one, const MemintArgs* runs, const int* wg_start, int nruns,
                              unsigned grid, int N, int cus, hipStream_t s) {
  const size_t lds = sizeof(double) * 4 * (size_t)N * MB;
  if (grid >= 2048 && N <= 32)
    hipLaunchKernelGGL((memint_step_runs<1, 64, true>), dim3(grid), dim3(64), 2 * lds, s, one, runs, wg_start, nruns);
  else if (grid >= 2048 && N <= RUNS_FOUR_MAX_N &&
           rounds_full(grid, cus * min(8, LDS_PER_CU / (int)(lds + 256))) >= (N <= 64 ? 65 : 80))
    hipLaunchKernelGGL((memint_step_runs<1, 128, false>), dim3(grid), dim3(128), lds, s, one, runs, wg_start, nruns);
  else if (grid >= 512 || N < 128)
    hipLaunchKernelGGL((memint_step_runs<1, 256, false>), dim3(grid), dim3(256), lds, s, one, runs, wg_start, nruns);
  else
    hipLaunchKernelGGL((memint_step_runs<3, 512, false>), dim3(grid), dim3(512), lds, s, one, runs, wg_start, nruns);
  return hipGetLastError();
}

hipError_t launch_memint_runs_split(const MemintArgs& a, int NB, int nsplit, double* part, hipStream_t s) {
  hipLaunchKernelGGL((memint_partial_runs<3, RUNS_SPLIT_THREADS>), dim3(NB * nsplit), dim3(RUNS_SPLIT_THREADS),
                     sizeof(double) * 4 * (size_t)a.N * MB, s, a, nsplit, part);
  return hipGetLastError();
}

// the tile shapes the autotuner chooses from, as the whole-block kernel and
// the split form's partial kernel (the item table in MemintArgs follows the
// context's shape); entry 0 is the default
#define KB_MEMINT_SHAPE(R, B, T) \
  { R, B, T, (const void*)memint_step<R, B, T>, (const void*)memint_partial<R, B, T> }
const MemintVariant kMemintVariants[NMEMINT_VARIANTS] = {
    KB_MEMINT_SHAPE(64, 2, 256), KB_MEMINT_SHAPE(32, 4, 256),  KB_MEMINT_SHAPE(128, 4, 256),
    KB_MEMINT_SHAPE(64, 4, 256), KB_MEMINT_SHAPE(128, 2, 256), KB_MEMINT_SHAPE(32, 2, 256),
    KB_MEMINT_SHAPE(64, 4, 512), KB_MEMINT_SHAPE(128, 2, 512), KB_MEMINT_SHAPE(32, 4, 512),
    KB_MEMINT_SHAPE(128, 1, 512), KB_MEMINT_SHAPE(64, 1, 512),  KB_MEMINT_SHAPE(128, 1, 256),
    KB_MEMINT_SHAPE(64, 1, 256),
};
#undef KB_MEMINT_SHAPE

// ---------------------------------------------------------------------------
// Measurement (createMeasurement / getE_kin / getE_pot / getE_mem)
// sums over the sites: [0] ddF/2, [1] F, [2] kL2 F, [3] E_mem boundary
// integrand, [4] E_mem interior integrand, [5] n_unstable
// The E_mem integrand walks row t-1 of the history, one line per time, so one
// thread per site was a chain of N_mem dependent rounds (252 us at 32^3,
// N_mem = 400, on 128 workgroups).  meas_workers(N) 8-lane workers share a
// site block's times instead, four times in flight each, on up to
// MEAS_GROUPS workgroups; measure_finish adds their sums in workgroup order
// into host memory.  (A last-workgroup counter instead of the second kernel
// costs some 35 ns per workgroup: 75 us with 2048 of them.)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(MEAS_THREADS) void measure_kernel(MeasArgs a) {
  __shared__ double red[MEAS_THREADS / 64][6];
  const int tid = threadIdx.x, lane = tid & (MB - 1), worker = tid >> 3;
  const int wpb = a.workers;
  const int w = worker & (wpb - 1);
  const int per = MEAS_THREADS / MB / wpb;  // site blocks per round
  double v[6] = {0, 0, 0, 0, 0, 0};
  for (int mb = blockIdx.x * per + worker / wpb; mb * MB + lane < a.V; mb += gridDim.x * per) {
    const int p = mb * MB + lane;
    const double dt = a.dt;
    const double* Hb = a.H + hoff(mb, 0, lane, a.NP);
    const double g = a.wgt ? a.wgt[p] : 1.0;
    if (w == 0) {
      const double Ftt = Hb[pair_rel(a.s_t, a.s_t, a.N)];
      const double Fmt = Hb[pair_rel(a.s_tm1, a.s_t, a.N)];
      const double2 emm = ld_global(Hb + pair_rel(a.s_tm1, a.s_tm1, a.N));
      const double Fmm = emm.x;
      const double ddF = (Ftt - 2.0 * Fmt + Fmm) / (dt * dt);
      const double om = (ddF / Fmm) > 0 ? sqrt(ddF / Fmm) : 0.0;
      double c;
      int bad = 0;
      if (0.25 * (dt * dt) * (om * om) < 1.0) {
        c = sqrt(1.0 - 0.25 * (dt * dt) * (om * om));
      } else {
        c = 1.0;
        bad = 1;
      }
      const double nn = (ddF * Fmm > 0) ? (c * sqrt(ddF * Fmm)) - 0.5 : 0.0;
      if (a.outF) {
        a.outF[p] = Fmm;
        a.outddF[p] = ddF;
        a.outr[p] = emm.y;
        a.outn[p] = nn;
        a.outom[p] = om;
        a.outc[p] = c;
      }
      v[0] += g * 0.5 * ddF;
      v[1] += g * Fmm;
      v[2] += g * a.kL2[p] * Fmm;
      v[5] += g * bad;
    }
    if (a.t != 2 && a.integral) {
      // E_mem integrand over t' in [tmin, t-2] against F(t',t-1), rho(t',t-1)
      const int smin = (a.tmin - 1) % a.N;
      const int n = a.t - 1 - a.tmin;
      const double* Sb = a.S + soff(mb, 0, lane, a.N);
      constexpr int U = 4;
      for (int q0 = w; q0 < n; q0 += wpb * U) {
        double2 e[U], sg[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int q = min(q0 + u * wpb, n - 1);
          const int x = smin + q < a.N ? smin + q : smin + q - a.N;
          e[u] = ld_global(Hb + pair_rel(x, a.s_tm1, a.N));
          sg[u] = ld_global(Sb + x * (2 * MB));
          if (x < a.s_tm1) e[u].y = -e[u].y;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int q = q0 + u * wpb;
          const double term = g * (sg[u].y * e[u].x - sg[u].x * e[u].y);
          if (q == 0)
            v[3] += term;
          else if (q < n)
            v[4] += term;
        }
      }
    }
  }
#pragma unroll
  for (int k = 0; k < 6; ++k)
    for (int o = 32; o > 0; o >>= 1) v[k] += __shfl_xor(v[k], o);
  if ((tid & 63) == 0)
    for (int k = 0; k < 6; ++k) red[tid >> 6][k] = v[k];
  __syncthreads();
  if (tid < 6) {
    double t = 0.0;
    for (int q = 0; q < MEAS_THREADS / 64; ++q) t += red[q][tid];
    a.partial[(size_t)blockIdx.x * 6 + tid] = t;
  }
}

__global__ __launch_bounds__(MEAS_THREADS) void measure_finish(MeasArgs a, int G) {
  __shared__ double red[MEAS_THREADS / 64][6];
  const int tid = threadIdx.x;
  double v[6] = {0, 0, 0, 0, 0, 0};
  for (int b = tid; b < G; b += MEAS_THREADS)
#pragma unroll
    for (int k = 0; k < 6; ++k) v[k] += a.partial[(size_t)b * 6 + k];
#pragma unroll
  for (int k = 0; k < 6; ++k)
    for (int o = 32; o > 0; o >>= 1) v[k] += __shfl_xor(v[k], o);
  if ((tid & 63) == 0)
    for (int k = 0; k < 6; ++k) red[tid >> 6][k] = v[k];
  __syncthreads();
  if (tid < 6) {
    double t = 0.0;
    for (int q = 0; q < MEAS_THREADS / 64; ++q) t += red[q][tid];
    a.sums[tid] = t;
  }
  if (tid == 6) a.sums[6] = a.m2[0];
}

// site-1 history (Measurement.jl:90-96); q = 0 .. t-tmin-1
__global__ void history_kernel(const double* __restrict__ H, const double* __restrict__ S, long NP, int N,
                               int tmin, int t, double* __restrict__ out) {
  const int L = t - tmin;
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= L) return;
  // SigF / Sigr for tp = t-1 down to tmin
  const int tpS = t - 1 - q;
  const int xS = (tpS - 1) % N;
  out[q] = S[soff(0, xS, 0, N)];
  out[L + q] = S[soff(0, xS, 0, N) + 1];
  // F(tmin,tp), rho(tmin,tp) for tp = tmin + q
  const int xm = (tmin - 1) % N;
  const int x = (tmin + q - 1) % N;
  const double* e = H + hoff(0, pair_off(xm, x, N), 0, NP);
  out[2 * L + q] = e[0];
  out[3 * L + q] = e[1] * (xm >= x ? 1.0 : -1.0);
}

// ---------------------------------------------------------------------------
// host-API helpers
// ---------------------------------------------------------------------------
// out[p] = comp(pair)[p] * sign for p < V
__global__ void gather_pair(const double* __restrict__ H, long NP, int V, long pair, int comp, double sign,
                            double* __restrict__ out) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < V) out[p] = H[hoff(p / MB, pair, p % MB, NP) + comp] * sign;
}

__global__ void scatter_pair(double* __restrict__ H, long NP, int V, long pair, int comp, double sign,
                             const double* __restrict__ in) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < V) H[hoff(p / MB, pair, p % MB, NP) + comp] = in[p] * sign;
}

// Streaming-read probe (benchmark support): each thread reads U 16-byte
// vectors per iteration, non-temporally, and the block writes one sum.
__global__ __launch_bounds__(256) void read_probe_kernel(const double* __restrict__ x, size_t n2,
                                                          double* __restrict__ out) {
  typedef double rp_d2 __attribute__((ext_vector_type(2)));
  constexpr int U = 8;
  const rp_d2* v = reinterpret_cast<const rp_d2*>(x);
  double acc = 0.0;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (; i + (U - 1) * stride < n2; i += U * stride) {
    rp_d2 a[U];
#pragma unroll
    for (int u = 0; u < U; ++u) a[u] = __builtin_nontemporal_load(v + i + u * stride);
#pragma unroll
    for (int u = 0; u < U; ++u) acc += a[u].x + a[u].y;
  }
  for (; i < n2; i += stride) acc += v[i].x + v[i].y;
  __shared__ double red[256];
  red[threadIdx.x] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double sum = 0.0;
    for (int k = 0; k < (int)blockDim.x; ++k) sum += red[k];
    out[blockIdx.x] = sum;
  }
}

__global__ void gather_tri(const double* __restrict__ P, long PNP, int V, long pp, double sign,
                           double* __restrict__ out) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < V) out[p] = P[poff(p / MB, pp, p % MB, PNP)] * sign;
}

__global__ void gather_sigma(const double* __restrict__ S, int N, int V, int slot, int comp,
                             double* __restrict__ out) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < V) out[p] = S[soff(p / MB, slot, p % MB, N) + comp];
}

// initSimData! rows (Initialization.jl:8-29): F(1,1)=F(2,1)=(n+1/2)/w,
// F(2,2)=w(n+1/2)dt^2+(n+1/2)/w, rho(2,1)=dt, diagonal rho = 0
__global__ void init_rows_kernel(double* __restrict__ H, long NP, int V, int N, const double* __restrict__ F11,
                                 const double* __restrict__ F21, const double* __restrict__ F22, double dt) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= V) return;
  const int mb = p / MB, lane = p % MB;
  const int s1 = 0, s2 = 1 % N;
  double* e11 = H + hoff(mb, pair_off(s1, s1, N), lane, NP);
  double* e21 = H + hoff(mb, pair_off(s2, s1, N), lane, NP);
  double* e22 = H + hoff(mb, pair_off(s2, s2, N), lane, NP);
  e11[0] = F11[p];
  e11[1] = 0.0;
  e21[0] = F21[p];
  e21[1] = dt * (s2 >= s1 ? 1.0 : -1.0);  // r[2,1] = dt * thesign(2,1)
  e22[0] = F22[p];
  e22[1] = 0.0;
}

__global__ void init_particles_kernel(const double* __restrict__ kL2, const double* __restrict__ n, double m,
                                      double dt, int V, double* __restrict__ F11, double* __restrict__ F21,
                                      double* __restrict__ F22) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= V) return;
  const double omega = sqrt(kL2[p] + m * m);
  const double np = n[p];
  F11[p] = (1.0 / omega) * (np + 0.5);
  F21[p] = (1.0 / omega) * (np + 0.5);
  F22[p] = (omega * (np + 0.5) * (dt * dt) + (1.0 / omega) * (np + 0.5));
}

// full deterministic window of free propagators (benchmark set-up);
// blockIdx.y = slot column c, threads over (site, slot row r >= c)
__global__ void fill_free_kernel(double* __restrict__ H, long NP, int V, int N, int tmax,
                                 const double* __restrict__ kL2, const double* __restrict__ n, double mass,
                                 double dt, int nb) {
  const long gid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int c = blockIdx.y;
  if (gid >= (long)nb * MB * N) return;
  const int r = (int)(gid % N);
  const int p = (int)(gid / N);
  if (r < c) return;
  const int mb = p / MB, lane = p % MB;
  double F = 0.0, rho = 0.0;
  if (p < V) {
    // times of the slots in the window [tmax-N+1, tmax]
    const int tmin = tmax - N + 1;
    const int smin = (tmin - 1) % N;
    const int th = tmin + (r - smin + N) % N;
    const int tl = tmin + (c - smin + N) % N;
    const double w = sqrt(kL2[p] + mass * mass);
    const double nn = n ? n[p] : 0.0;
    const double d = (double)(th - tl) * dt;
    F = (nn + 0.5) / w * cos(w * d);
    rho = sin(w * d) / w;  // rho(th, tl): the stored value for slots (r, c)
  }
  double* e = H + hoff(mb, pair_off(r, c, N), lane, NP);
  e[0] = F;
  e[1] = rho;
}

__global__ void finite_kernel(const double* __restrict__ H, size_t count, int* __restrict__ flag) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  int bad = 0;
  for (; i < count; i += stride) bad |= !isfinite(H[i]);
  if (bad) atomicOr(flag, 1);
}

}  // namespace qftkb
