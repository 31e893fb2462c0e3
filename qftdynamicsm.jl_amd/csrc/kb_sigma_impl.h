// kb_sigma_impl.h -- self-energy stage of the KB step by lattice transforms
// (TwoPIScalar_Evolution.jl:16-31).
//
// For every live t' the sunset needs Fx = real(rfft(F(t-1,t'))) and
// rx = real(rfft(rho(t-1,t'))), the pointwise products rx (Fx^2 - rx^2/12)
// and Fx (Fx^2 - 3/4 rx^2), and their inverse transforms.  real(rfft(X))
// only sees the inversion-even part X_e(p) = (X(p) + X(-p))/2, whose
// transform is real, so F_e + i rho_e is transformed as one complex lattice
// and both transforms come out as its real and imaginary parts.
//
// Modes.  SG_SUNSET, and SG_PLAIN on lattices of the caller.  SG_SUNSET_ADJ,
// the adjoint of the stage: the input is the adjoint self-energy pair
// (SigF_bar, Sigr_bar) per t', the pointwise step is the transpose of the
// sunset's Jacobian at the saved forward transforms (Fx, rx), and the output
// is added to the adjoint history row t-1.  The cosine transform C (real part
// of the DFT of an even lattice) is symmetric, so Sigma = pre C g(C F, C rho)
// has the adjoint
//   g_bar = pre C Sigma_bar,  F_bar += C (dg/dFx)^T g_bar,  rho_bar += C (dg/drx)^T g_bar.
// Two modes serve the 1/N expansion (NinverseNLO):
//   BUBBLE  gathers F(t-1,t'), rho(t-1,t') like the sunset, keeps (Fx, rx)
//           in X and transforms Fx^2 - rx^2/4 and Fx rx back: the bubbles
//           F2kr2 = ivol^2 C[Fx^2 - rx^2/4] and Fr = ivol^2 C[Fx rx] of the
//           pair (t-1, t') (calc_Fr_F2kr2!, SimDataStruct.jl:726-750), stored
//           as row t-1 of two slot triangles;
//   CHAIN   gathers the resummed kernels (IF, Ir)(t') in momentum space,
//           transforms them to Irx = ivol C Ir, IFx = ivol C IF and forms
//           Sigr = pre C[Fx Irx + rx IFx], SigF = pre C[Fx IFx - rx Irx / 4]
//           with the saved (Fx, rx) (calcSelfEnergyattp!, Evolution.jl:683-698).
//
// Passes.  A workgroup transforms the lines of a box in LDS.  With the sites
// (x, mid, outer) = (x, y, z) in 3D and (x, -, y) in 2D:
//   1D: one pass, KIND_ROW, a line per workgroup;
//   2D, Nx <= 64: one pass, KIND_ALL, a plane per workgroup;
//   3D, Nx <= 26: one pass, KIND_WHOLE, a whole row (its half space) per
//       workgroup; see SPREAD_MIN for 24^3 to 26^3 with few rows;
//   3D, Nx <= 64: KIND_FWD gathers plane z and its reflection -z and
//       transforms x and y; KIND_LAST transforms z, applies the pointwise
//       step and transforms back, on tiles of x; KIND_INV transforms y and x
//       back and writes the planes z and -z of the result;
//   larger lattices: the same with the x and y transforms in passes of their
//       own (KIND_MID; none in 2D), FWD and INV on batches of x rows.
// Every partial transform W of an even lattice is even under the point
// reflection of all indices, W(-x, -mid, -outer) = W(x, mid, outer), so
// between passes the workspace holds only outer in [0, n/2] of each row:
// KIND_LAST reads the other half of a line from the reflected one and writes
// both.
//
// Transforms.  n is cut into the fewest radices of 2 .. 11, 13, 17, 19 and 23 (two up to
// 100 or more; larger primes are a stage of their own), and one butterfly
// lives in one thread's registers.  Where a line is transformed forth and
// back, the last forward stage, the pointwise step and the first inverse stage
// (the same radix, so the same elements) run in registers: KIND_LAST crosses
// LDS twice.  All butterflies of a stage are held at once, so the stages work
// in place on one buffer, and a CU holds twice the workgroups it would with
// two.  Rows pass through LDS in memory order on their way in and out, planes
// and lines of W go straight between registers and memory.  The inverse
// transform is the forward one of swapped (re, im): values are swapped at the
// pointwise step and swapped back when written.
//
// Bound: latency (launch, LDS stages and barriers) up to some 20^3, then the
// gather of row t-1, the half-space round trip (L2 and the last-level cache
// hold most of it) and the result; past Nx = 64 the two passes more.
// Measured (stage of a step, N_mem rows less one; in brackets a Stockham
// form with radices up to 7 on two LDS buffers, three passes at every 3D size
// up to 64 and a line per workgroup past it): 8^3 N_mem 100 9.5 us (14.2),
// 16^3 202 18.2 (23.8), 24^3 150 35.5 (45.4), 26^3 100 50 (140), 32^3 400
// 161 (192), 42^3 96 127 (261), 48^3 100 154 (220), 66^3 16 131 (1178),
// 89^3 16 553 (9891), 112^3 16 453 (2435); 64^2 200 23 (29), 128^2 200 78
// (208), 251^2 60 374 (5717); 64^1 400 7.8 (8.1), 1024^1 200 12.3 (18.1).
#pragma once
#include <type_traits>

#include "kb_kernels.h"
#include "kb_twiddles.h"

namespace qftkb {

namespace {

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 swapped(double2 a) { return make_double2(a.y, a.x); }
__device__ __forceinline__ double2 mul_mi(double2 a) { return make_double2(a.y, -a.x); }  // -i a

// ---------------------------------------------------------------------------
// forward DFTs (exp(-2 pi i / R)) of R values in registers
// ---------------------------------------------------------------------------
// odd R: X_q, X_{R-q} = x_0 + sum_k (x_k + x_{R-k}) cos(2 pi q k / R) -+ i sum_k (x_k - x_{R-k}) sin(2 pi q k / R)
template <int R>
struct OddTable;
template <>
struct OddTable<3> {
  static constexpr double c[2] = {1.0, -0.5}, s[2] = {0.0, 0.86602540378443864676};
};
template <>
struct OddTable<5> {
  static constexpr double c[3] = {1.0, 0.30901699437494742410, -0.80901699437494742410};
  static constexpr double s[3] = {0.0, 0.95105651629515357212, 0.58778525229247312917};
};
template <>
struct OddTable<7> {
  static constexpr double c[4] = {1.0, 0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624};
  static constexpr double s[4] = {0.0, 0.78183148246802980871, 0.97492791218182360702, 0.43388373911755812048};
};
template <>
struct OddTable<11> {
  static constexpr double c[6] = {1.0, 0.84125353283118116886, 0.41541501300188642553, -0.14231483827328514044,
                                  -0.65486073394528506406, -0.95949297361449738989};
  static constexpr double s[6] = {0.0, 0.54064081745559758211, 0.90963199535451837141, 0.98982144188093273238,
                                  0.75574957435425828377, 0.28173255684142969771};
};
template <>
struct OddTable<13> {
  static constexpr double c[7] = {1.0, 0.8854560256532098959, 0.56806474673115580251, 0.12053668025532305335,
                                  -0.35460488704253562597, -0.74851074817110109863, -0.97094181742605202716};
  static constexpr double s[7] = {0.0, 0.46472317204376854566, 0.82298386589365639458, 0.9927088740980539928,
                                  0.93501624268541482344, 0.66312265824079520238, 0.23931566428755776715};
};
template <>
struct OddTable<17> {
  static constexpr double c[9] = {1.0, 0.93247222940435580457, 0.73900891722065911592, 0.4457383557765382674,
                                  0.09226835946330199524, -0.27366299007208286354, -0.60263463637925638918,
                                  -0.85021713572961415213, -0.98297309968390177828};
  static constexpr double s[9] = {0.0, 0.36124166618715294874, 0.67369564364655721171, 0.89516329135506232207,
                                  0.99573417629503452187, 0.96182564317281907041, 0.79801722728023950333,
                                  0.52643216287735580024, 0.18374951781657033157};
};
template <>
struct OddTable<19> {
  static constexpr double c[10] = {1.0, 0.94581724170063467902, 0.78914050939639359922, 0.54694815812242687471,
                                  0.24548548714079914892, -0.0825793454723323246, -0.40169542465296945752,
                                  -0.67728157162574107476, -0.87947375120648907139, -0.9863613034027223736};
  static constexpr double s[10] = {0.0, 0.32469946920468348741, 0.61421271268966781744, 0.83716647826252857481,
                                  0.96940026593933041674, 0.99658449300666984982, 0.91577332665505743992,
                                  0.73572391067313162477, 0.47594739303707354443, 0.16459459028073389414};
};
template <>
struct OddTable<23> {
  static constexpr double c[12] = {1.0, 0.96291728734779929502, 0.85441940454648855255, 0.68255314321865408287,
                                  0.46006503773115212604, 0.20345601305263378988, -0.068242413364670975921,
                                  -0.33487961217098615196, -0.57668032211486714125, -0.77571129070441980704,
                                  -0.91721130150545301784, -0.99068594603633075234};
  static constexpr double s[12] = {0.0, 0.26979677115702427125, 0.51958395003543357813, 0.73083596427812410165,
                                  0.88788521840237523498, 0.97908408768232287563, 0.99766876919053919845,
                                  0.94226092211882049562, 0.81696989301044201697, 0.63108794432605278937,
                                  0.398401089846241458, 0.13616664909624659076};
};

template <int R>
__device__ __forceinline__ void dft_odd(double2 (&v)[R]) {
  constexpr int H = (R - 1) / 2;
  double2 t[H + 1], d[H + 1];
#pragma unroll
  for (int k = 1; k <= H; ++k) {
    t[k] = cadd(v[k], v[R - k]);
    d[k] = csub(v[k], v[R - k]);
  }
  const double2 x0 = v[0];
#pragma unroll
  for (int q = 1; q <= H; ++q) {
    double2 a = x0, b = make_double2(0.0, 0.0);
#pragma unroll
    for (int k = 1; k <= H; ++k) {
      const int i = (q * k) % R;
      const double c = OddTable<R>::c[i <= H ? i : R - i];
      const double s = i <= H ? OddTable<R>::s[i <= H ? i : 0] : -OddTable<R>::s[i <= H ? 0 : R - i];
      a.x += c * t[k].x;
      a.y += c * t[k].y;
      b.x += s * d[k].y;
      b.y -= s * d[k].x;
    }
    v[q] = cadd(a, b);
    v[R - q] = csub(a, b);
  }
#pragma unroll
  for (int k = 1; k <= H; ++k) v[0] = cadd(v[0], t[k]);
}

template <int R>
__device__ __forceinline__ void dft(double2 (&v)[R]);

// A x B with coprime A, B: n = (B n1 + A n2) mod R, k = (k1 B B' + k2 A A') mod R
// (B B' = 1 mod A, A A' = 1 mod B); no twiddles
template <int A, int B>
__device__ __forceinline__ void dft_coprime(double2 (&v)[A * B]) {
  constexpr int R = A * B;
  constexpr auto inverse = [](int x, int m) {
    for (int i = 1; i < m; ++i)
      if (x * i % m == 1) return i;
    return 0;
  };
  constexpr int EB = B * inverse(B % A, A), EA = A * inverse(A % B, B);
  double2 w[R];
#pragma unroll
  for (int n2 = 0; n2 < B; ++n2) {
    double2 u[A];
#pragma unroll
    for (int n1 = 0; n1 < A; ++n1) u[n1] = v[(B * n1 + A * n2) % R];
    dft<A>(u);
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) w[k1 * B + n2] = u[k1];
  }
#pragma unroll
  for (int k1 = 0; k1 < A; ++k1) {
    double2 u[B];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) u[n2] = w[k1 * B + n2];
    dft<B>(u);
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) v[(k1 * EB + k2 * EA) % R] = u[k2];
  }
}

// exp(-2 pi i k / R) for the inner twiddles of R = 8, 9
template <int R>
__device__ __forceinline__ double2 inner_twiddle(int k) {
  if constexpr (R == 8) {
    constexpr double r = 0.70710678118654752440;
    constexpr double c[4] = {1.0, r, 0.0, -r}, s[4] = {0.0, r, 1.0, r};
    return make_double2(c[k], -s[k]);
  } else {
    static_assert(R == 9, "");
    constexpr double c[5] = {1.0, 0.76604444311897803520, 0.17364817766693034885, -0.5, -0.93969262078590838405};
    constexpr double s[5] = {0.0, 0.64278760968653932632, 0.98480775301220805937, 0.86602540378443864676,
                             0.34202014332566873304};
    return make_double2(c[k], -s[k]);
  }
}

// A x B with inner twiddles: n = B n1 + n2, k = k1 + A k2
template <int A, int B>
__device__ __forceinline__ void dft_twiddled(double2 (&v)[A * B]) {
  double2 w[A * B];
#pragma unroll
  for (int n2 = 0; n2 < B; ++n2) {
    double2 u[A];
#pragma unroll
    for (int n1 = 0; n1 < A; ++n1) u[n1] = v[B * n1 + n2];
    dft<A>(u);
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
      if (k1 * n2 == 0)
        w[k1 * B + n2] = u[k1];
      else if (A * B == 4 * k1 * n2)
        w[k1 * B + n2] = mul_mi(u[k1]);
      else
        w[k1 * B + n2] = cmul(u[k1], inner_twiddle<A * B>(k1 * n2));
    }
  }
#pragma unroll
  for (int k1 = 0; k1 < A; ++k1) {
    double2 u[B];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) u[n2] = w[k1 * B + n2];
    dft<B>(u);
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) v[k1 + A * k2] = u[k2];
  }
}

template <int R>
__device__ __forceinline__ void dft(double2 (&v)[R]) {
  if constexpr (R == 2) {
    const double2 a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
  } else if constexpr (R == 4) {
    const double2 a0 = cadd(v[0], v[2]), a1 = csub(v[0], v[2]);
    const double2 b0 = cadd(v[1], v[3]), b1 = mul_mi(csub(v[1], v[3]));
    v[0] = cadd(a0, b0);
    v[2] = csub(a0, b0);
    v[1] = cadd(a1, b1);
    v[3] = csub(a1, b1);
  } else if constexpr (R == 3 || R == 5 || R == 7 || R == 11 || R == 13 || R == 17 || R == 19 || R == 23) {
    dft_odd<R>(v);
  } else if constexpr (R == 6) {
    dft_coprime<2, 3>(v);
  } else if constexpr (R == 10) {
    dft_coprime<2, 5>(v);
  } else if constexpr (R == 8) {
    dft_twiddled<4, 2>(v);
  } else if constexpr (R == 9) {
    dft_twiddled<3, 3>(v);
  }  // R == 1: nothing
}

// ---------------------------------------------------------------------------
// pointwise steps and outputs of the modes
//
// The fused multiply-adds of the pointwise steps are written out, and their
// products are rounded: left to the compiler, they would be fused into the sums
// of the inverse butterfly where it follows in the same block of code (compiled
// lengths) and not elsewhere (run-time plans).  A row's values do not depend on
// the form that computes it: a row of kb_sunset has the bits of a step's.
// ---------------------------------------------------------------------------
// (Fx (Fx^2 - qF rx^2), rx (Fx^2 - qr rx^2)): qF = 3/4, qr = 1/12 for the
// quantum sunset (Evolution.jl:25-31), 0 for the classical one (:107-120)
__device__ __forceinline__ double2 sunset(double2 z, int classical) {
#pragma clang fp contract(off)
  const double qF = classical ? 0.0 : 0.75, qr = classical ? 0.0 : 1.0 / 12.0;
  const double Fx = z.x, rx = z.y;
  const double FF = Fx * Fx, rr = rx * rx;
  return make_double2(Fx * fma(-qF, rr, FF), rx * fma(-qr, rr, FF));
}

// transpose of the sunset's Jacobian at (Fx, rx) applied to
// (gF, gr) = (preF, preR) * (C SigF_bar, C Sigr_bar)
__device__ __forceinline__ double2 sunset_adj(double2 cs, double2 x, double preF, double preR, int classical) {
#pragma clang fp contract(off)
  const double a1 = classical ? 0.0 : 0.75, a2 = classical ? 0.0 : -1.5, a3 = classical ? 0.0 : 0.25;
  const double gF = preF * cs.x, gr = preR * cs.y;
  const double Fx = x.x, rx = x.y;
  const double FF = Fx * Fx, rr = rx * rx;
  return make_double2(fma(gF, fma(-a1, rr, 3.0 * FF), gr * (2.0 * rx * Fx)),
                      fma(gF, a2 * Fx * rx, gr * fma(-a3, rr, FF)));
}

// the pointwise step of each mode; the sunset and bubble save (Fx, rx) in X when it is set
template <int MODE>
__device__ __forceinline__ double2 pointwise(const SigmaArgs& a, double2 z, size_t xi) {
#pragma clang fp contract(off)
  if constexpr (MODE == SG_SUNSET_ADJ) {
    return sunset_adj(z, a.X[xi], a.preF, a.preR, a.classical);
  } else if constexpr (MODE == SG_BUBBLE) {
    if (a.X) a.X[xi] = z;
    return make_double2(fma(z.x, z.x, -0.25 * (z.y * z.y)), z.x * z.y);
  } else if constexpr (MODE == SG_CHAIN) {
    const double2 x = a.X[xi];  // (Fx, rx) of (t-1, t')
    const double IFx = a.ivol * z.x, Irx = a.ivol * z.y;
    return make_double2(fma(x.x, IFx, -0.25 * (x.y * Irx)), fma(x.x, Irx, x.y * IFx));
  } else {
    if (a.X) a.X[xi] = z;
    return sunset(z, a.classical);
  }
}

// one row of the stage: t' = tmin + q of the window, or lattice q of the caller
struct Row {
  size_t off;  // q V: site-indexed arrays
  int slot;
  double sg;   // sign of the stored rho(t-1, t')
  size_t pair, ppair;  // offsets of the slot pair (t-1, t') in a site block of the history, the bubble triangles
};

// offset in doubles of a site whose site block holds `pairs` slot pairs or
// slots of two values (pairs * 2 MB < 2^32: one 32 x 32 bit product)
__device__ __forceinline__ size_t block_off(int site, long pairs) {
  return (size_t)(unsigned)(site / MB) * (unsigned)(pairs * (2 * MB)) + (unsigned)(site % MB) * 2;
}

// offset in doubles of one-value slot pair (a, b) of a site block, lane 0
__device__ __forceinline__ size_t ppair_rel(int a, int b, int N) { return prel(ppair_off(a, b, N)); }

template <int MODE>
__device__ __forceinline__ int stage_rows(const SigmaArgs& a) {
  if constexpr (MODE == SG_PLAIN)
    return a.rows;
  else
    return a.st->L;
}

template <int MODE>
__device__ __forceinline__ Row row_of(const SigmaArgs& a, int q) {
  Row r{(size_t)q * a.V, 0, 1.0, 0, 0};
  if constexpr (MODE != SG_PLAIN) {
    const int s_tm1 = a.st->s_tm1;
    r.slot = a.st->s_min + q;
    if (r.slot >= a.N) r.slot -= a.N;
    r.sg = s_tm1 >= r.slot ? 1.0 : -1.0;
    if constexpr (MODE != SG_CHAIN) r.pair = (size_t)pair_off(s_tm1, r.slot, a.N) * (2 * MB);
    if constexpr (MODE == SG_BUBBLE) r.ppair = ppair_rel(s_tm1, r.slot, a.N);
  }
  return r;
}

// the input at sites s1 and s2 = -s1, symmetrised: physical F(t-1,t'),
// rho(t-1,t') from the history, a ring in self-energy layout -- (IF, Ir)(t')
// or (SigF_bar, Sigr_bar)(t') --, or the caller's lattices
template <int MODE>
__device__ __forceinline__ double2 gather(const SigmaArgs& a, const Row& r, int s1, int s2) {
  if constexpr (MODE == SG_PLAIN) {
    const double *F = a.Fin + r.off, *R = a.Rin + r.off;
    return make_double2(0.5 * (F[s1] + F[s2]), 0.5 * (R[s1] + R[s2]));
  } else {
    const int q1 = a.smap ? a.smap[s1] : s1, q2 = a.smap ? a.smap[s2] : s2;
    const double *h1, *h2;
    double sg = 1.0;
    if constexpr (MODE == SG_CHAIN || MODE == SG_SUNSET_ADJ) {
      const double* ring = MODE == SG_CHAIN ? a.Iring : a.Sbar;
      h1 = ring + block_off(q1, a.N) + r.slot * (2 * MB);
      h2 = ring + block_off(q2, a.N) + r.slot * (2 * MB);
    } else {
      h1 = a.H + block_off(q1, a.NP) + r.pair;
      h2 = a.H + block_off(q2, a.NP) + r.pair;
      sg = r.sg;
    }
    const double2 e1 = *reinterpret_cast<const double2*>(h1), e2 = *reinterpret_cast<const double2*>(h2);
    return make_double2(0.5 * (e1.x + e2.x), 0.5 * (e1.y + e2.y) * sg);
  }
}

// output of the stage at site s: Sigma into the ring, the adjoint added to
// (F_bar, rho_bar)(t-1, t'), or the bubbles of (t-1, t')
template <int MODE>
__device__ __forceinline__ void emit(const SigmaArgs& a, const Row& r, int s, double2 z) {
  if constexpr (MODE == SG_PLAIN) {
    a.SigFout[r.off + s] = a.preF * z.x;
    a.Sigrout[r.off + s] = a.preR * z.y;
  } else if constexpr (MODE == SG_SUNSET_ADJ) {
    double* o = a.Hbar + block_off(s, a.NP) + r.pair;
    o[0] += z.x;
    if (r.slot != a.st->s_tm1) o[1] += r.sg * z.y;  // rho(t-1,t-1) is not a variable
  } else {
    if (a.rmap) {
      s = a.rmap[s];  // orbit storage: the representative writes its orbit's value
      if (s < 0) return;
    }
    if constexpr (MODE == SG_BUBBLE) {
      const size_t o = poff(s / MB, 0, s % MB, a.PNP) + r.ppair;
      a.PF[o] = a.preF * z.x;
      a.PR[o] = r.sg * a.preR * z.y;  // sign-folded like rho
    } else {
      *reinterpret_cast<double2*>(a.S + block_off(s, a.N) + r.slot * (2 * MB)) = make_double2(a.preF * z.x, a.preR * z.y);
    }
  }
}

// ---------------------------------------------------------------------------
// a pass: the stages of its lines
// ---------------------------------------------------------------------------
enum PassKind { KIND_ROW, KIND_ALL, KIND_FWD, KIND_MID, KIND_LAST, KIND_INV, KIND_WHOLE };

enum StageFlags {
  ST_SRC = 1,     // inputs from W instead of LDS
  ST_SNK = 2,     // outputs to W
  ST_POINT = 4,   // last forward stage: pointwise step after it ...
  ST_TWICE = 8,   // ... and the first inverse stage, the same radix, at once
  ST_Y = 16,      // lines along the second index of the box (the line index is x)
  ST_Z = 32,      // KIND_WHOLE: lines along the third
  ST_ZIN = 64,    // their first stage, on the half space,
  ST_ZOUT = 128,  // and their last one, back to it
  ST_END = 256    // the last chunk of lines of its stage
};

struct Stage {
  short R, flags, ls, es;     // radix; line and element strides in LDS
  short Ns, m;                // span so far, n / R
  short first, lines, items;  // the chunk's lines, and its butterflies
  unsigned mg, mgNs;          // magic of `lines`, and of Ns
};

constexpr int MAX_STAGES = 48;
struct PassPlan {
  int n, nstages, threads;
  int lines;  // x rows, or x values, per workgroup
  int tiles;  // tiles of x (KIND_MID, KIND_LAST)
  int total;  // x rows of the half space (KIND_FWD, KIND_INV, KIND_WHOLE)
  int elements;  // complex values in LDS, after n twiddles
  int ls;        // LDS stride of an x row
  unsigned mgn;  // magic of n
  Stage st[MAX_STAGES];
};

constexpr int least(int a, int b) { return a < b ? a : b; }
constexpr int most(int a, int b) { return a > b ? a : b; }
// butterflies of radix R that a thread's registers hold
constexpr int held(int R) { return R == 1 ? 8 : most(1, 10 / R); }
// Prime stages: output pairs per item, and items per thread.  A line alone in
// its workgroup has an item for each pair: it has threads to spare, and a
// quarter of them each with four pairs take twice the time (a step's stage and
// the rest, N_mem = 8, us: 61^1 32 against 20, 251^1 80 against 37, 2039^1 501
// against 352; kb_sunset of 300 rows of 61^1 27 against 11).
constexpr int DIRECT_PAIRS = 4, DIRECT_HELD = 2;
constexpr int direct_pairs(int kind) { return kind == KIND_ROW ? 1 : DIRECT_PAIRS; }
constexpr int direct_groups(int kind, int R) { return ((R - 1) / 2 + direct_pairs(kind) - 1) / direct_pairs(kind); }

constexpr int RADICES[] = {23, 19, 17, 13, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2};
constexpr bool is_direct(int R) { return R > 23; }
constexpr size_t LDS_MAX = 160 * 1024;
constexpr int LDS_VALUES = (int)(LDS_MAX / sizeof(double2));

// x / d = umulhi(x, magic(d)) for x d < 2^32; 0 stands for d = 1
constexpr unsigned magic(int d) { return d > 1 ? (unsigned)(((unsigned long long)1 << 32) / d + 1) : 0u; }
__device__ __forceinline__ int div_magic(int x, unsigned mg) { return mg ? (int)__umulhi((unsigned)x, mg) : x; }
constexpr int odd(int n) { return n | 1; }  // LDS stride of a line: neighbouring lines on other banks

// How a pass knows its plan: a length NT > 0 is compiled in (whole rows up to
// 26^3, planes at multiples of 8 up to 64, lines at powers of two: with every
// index known a pass takes about two thirds of the time, 1024^1 N_mem = 200
// 12.3 against 18.1 us); PLAN_SMALL runs any plan of radices up to 8, PLAN_ANY
// any without 17, 19 and 23, PLAN_WIDE every plan.
enum { PLAN_SMALL = 0, PLAN_ANY = -1, PLAN_WIDE = -2 };
constexpr int SMALL_RADIX = 8, ANY_RADIX = 13;
// Waves per SIMD that the registers are cut for.  Six (80 registers) keep the
// memory busy where four (the passes' natural 100) leave it waiting: 48^3 x
// 100 rows 190 against 173 us; with the radices 9, 10 and the prime stages
// the code would spill (47^3 x 24: 160 -> 195 us), so those plans have four.
// A whole row has a CU to itself, or nearly, and 16 waves.
// The butterflies of 17, 19 and 23 need up to 230 registers: two waves, in
// workgroups of up to 512 (as prime stages, whose outputs are shared out in
// pairs, 17^3 N_mem = 100 took 55 us against 20, 34^3 N_mem = 60 over 200
// against 116; of 29 they would spill).
constexpr bool wide(const FFTPlan& pl) {
  for (int i = 0; i < pl.nf; ++i)
    if (pl.fac[i] > ANY_RADIX && !is_direct(pl.fac[i])) return true;
  return false;
}
constexpr bool plan_wide(int nt);
constexpr int plan_waves(int kind, int nt) {
  return plan_wide(nt) ? 2 : nt == PLAN_ANY || kind == KIND_WHOLE ? 4 : 6;
}
constexpr int plan_threads(bool wide) { return wide ? 512 : 1024; }

// the fewest radices with product m, descending; of those the smallest largest one
constexpr void best_radices(int m, int maxR, int depth, int* cur, int* best, int& nbest) {
  if (m == 1) {
    if (nbest < 0 || depth < nbest || (depth == nbest && cur[0] < best[0])) {
      nbest = depth;
      for (int i = 0; i < depth; ++i) best[i] = cur[i];
    }
    return;
  }
  if (depth == 8 || (nbest >= 0 && depth >= nbest)) return;
  for (int R : RADICES)
    if (R <= maxR && m % R == 0) {
      cur[depth] = R;
      best_radices(m / R, R, depth + 1, cur, best, nbest);
    }
}

constexpr FFTPlan make_plan(int n) {
  FFTPlan pl{};
  pl.n = n;
  int m = n, primes[FFT_MAXF] = {}, np = 0;
  for (int f : {2, 3, 5, 7, 11, 13, 17, 19, 23})
    while (m % f == 0) m /= f;
  const int smooth = n / m;
  for (int f = 29; m > 1; f += 2)
    while (m % f == 0) {
      primes[np++] = f;
      m /= f;
    }
  int cur[8] = {}, best[8] = {}, nbest = -1;
  if (smooth > 1) {
    best_radices(smooth, 23, 0, cur, best, nbest);
    for (int i = nbest - 1; i >= 0; --i) pl.fac[pl.nf++] = best[i];
  } else {
    pl.fac[pl.nf++] = 1;  // a prime stage does not read W
  }
  for (int i = 0; i < np; ++i) pl.fac[pl.nf++] = primes[i];
  return pl;
}

constexpr bool plan_wide(int nt) { return nt > 0 ? wide(make_plan(nt)) : nt == PLAN_WIDE; }

// The stages of one pass for workgroups of `threads`: a stage whose
// butterflies they do not hold at once runs in chunks of lines.
struct Builder {
  PassPlan pp{};
  FFTPlan pl{};
  int kind;

  constexpr Builder(int k, const FFTPlan& p, int lines, int elements, int threads) : pl(p), kind(k) {
    pp.n = p.n;
    pp.threads = threads;
    pp.lines = lines;
    pp.elements = elements;
    pp.ls = odd(p.n);
    pp.mgn = magic(p.n);
  }
  constexpr void add(int R, int Ns, int lines, int ls, int es, int flags) {
    if (R == 1 && !(flags & (ST_SRC | ST_SNK | ST_POINT))) return;  // (needed at W only)
    const int m = pp.n / R;
    const int per = m * (is_direct(R) ? direct_groups(kind, R) : 1);  // items of a line
    const int room = most(1, pp.threads * (is_direct(R) ? DIRECT_HELD : held(R)) / per);
    const int chunks = (lines + room - 1) / room, chunk = (lines + chunks - 1) / chunks;
    for (int first = 0; first < lines; first += chunk) {
      Stage& s = pp.st[pp.nstages++];
      s.R = (short)R;
      s.flags = (short)(flags | (first + chunk >= lines ? ST_END : 0));
      s.ls = (short)ls;
      s.es = (short)es;
      s.Ns = (short)Ns;
      s.m = (short)m;
      s.first = (short)first;
      s.lines = (short)least(chunk, lines - first);
      s.items = (short)(s.lines * per);
      s.mg = magic(s.lines);
      s.mgNs = magic(Ns);
    }
  }
  // one axis, or forth and back with the pointwise step between; src, snk:
  // what its first and last stage do besides
  constexpr void forward(int lines, int ls, int es, int flags, int src = 0, int snk = 0) {
    int Ns = 1;
    for (int i = 0; i < pl.nf; ++i) {
      add(pl.fac[i], Ns, lines, ls, es, flags | (i == 0 ? src : 0) | (i + 1 == pl.nf ? snk : 0));
      Ns *= pl.fac[i];
    }
  }
  constexpr void round_trip(int lines, int ls, int es, int flags, int src = 0, int snk = 0) {
    int Ns = 1;
    for (int i = 0; i + 1 < pl.nf; ++i) {
      add(pl.fac[i], Ns, lines, ls, es, flags | (i == 0 ? src : 0));
      Ns *= pl.fac[i];
    }
    // the last radix: forward, pointwise step, and (unless it is a prime
    // stage) its inverse at once
    int i = pl.nf - 1;
    const int R = pl.fac[i];
    const bool twice = !is_direct(R);
    add(R, Ns, lines, ls, es,
        flags | ST_POINT | (twice ? ST_TWICE : 0) | (i == 0 ? src : 0) | (twice && i == 0 ? snk : 0));
    Ns = 1;
    if (twice) {
      Ns = R;
      --i;
    }
    for (; i >= 0; --i) {
      add(pl.fac[i], Ns, lines, ls, es, flags | (i == 0 ? snk : 0));
      Ns *= pl.fac[i];
    }
  }
};

// workgroup size of a pass over `elements` values: what is asked for, but
// `fewest` (8) to sixteen values per thread, and never so few that a line
// would not be held.  Passes whose rows have a CU to themselves take 2 or 4
// (12^3 N_mem = 100 13.4 us with 2, 20 with 8; 16^3 N_mem = 202 18.3 with 4,
// 20.8 with 8, and 2 costs 16^3 N_mem = 600 45 against 37).
constexpr int pass_threads(int kind, const FFTPlan& pl, int elements, int want, int fewest = 8) {
  int per = 64;
  for (int i = 0; i < pl.nf; ++i) {
    const int R = pl.fac[i], m = pl.n / R;
    const int items = is_direct(R) ? m * direct_groups(kind, R) : m;
    const int h = is_direct(R) ? DIRECT_HELD : held(R);
    per = most(per, (items + h - 1) / h);
  }
  return (least(plan_threads(wide(pl)), most(per, least(most(want, elements / 16), elements / fewest))) + 63) / 64 * 64;
}

// lines per workgroup of a pass on batches: some 1536 values, and what LDS holds
constexpr int batch(int n, int limit) {
  const int lines = most(8, 1536 / n / 8 * 8);
  return most(1, least(least(limit, lines), (LDS_VALUES - n - (int)sizeof(PassPlan::st) / 16) / odd(n)));
}

// (LDS would hold planes up to 98 x 98, but one workgroup of them per CU is
// slower than batches: 96^3 N_mem = 16 313 against 293 us, 98^2 N_mem = 100 72
// against 47)
constexpr bool planes_fit(int n) { return n <= 64; }
// whole rows: the half space, and four lines that are their own reflection
constexpr int whole_values(int n) { return n * odd(n) * (n / 2 + 1) + 4 * n; }
constexpr bool whole_fits(int n) {
  return n >= 2 && whole_values(n) + n <= LDS_VALUES;  // n <= 26
}
constexpr int WHOLE_MAX = 26;
// From here on rows go by three passes, which fill the chip, while there are
// few of them: a whole row keeps one CU busy for 33 us at 24^3, three compiled
// passes take 14 us for 1 row, 18 for 24 and 31 for 96, as long as whole rows
// (at 16^3 the two take 16.5 us both for 8 rows, 17 and 19 for 64).  Lengths
// that have no compiled passes change over earlier: 25^3 22 against 29 us for 1
// row, 28 against 30 for 32, 32 against 31 for 48; 26^3 32 against 42, 38
// against 44, 42 against 45.  (Below 24 whole rows win there from the first
// row on: 22^3 28 against 32 us, 20^3 18 against 27.)  Beside other runs' stages,
// in an ensemble, these stay whole: the chip is filled and launches count (a step
// of six runs around 20^3, one of them 25^3, with N_mem = 9 104 against 111 us).
constexpr int ROW_MIN = 8, ROW_MAX = 1024;  // compiled lines: powers of two
constexpr int SPREAD_MIN = 24, SPREAD_ROWS = 96, SPREAD_PLAN_ROWS = 40;
// lines along z that stand for themselves and their reflection (-x, -y)
constexpr int whole_zlines(int n) { return (n % 2 ? 1 : 2) * (n / 2 + 1) + (n - 1) / 2 * n; }

// the plan of a pass; `three`: 3D (2D: the second index is the last one)
constexpr PassPlan pass_plan(const FFTPlan& pl, int kind, bool three, int want) {
  const int n = pl.n, ls = odd(n);
  const int nh = n / 2 + 1, xrows = three ? n * nh : nh;  // x rows of the half space
  if (kind == KIND_WHOLE) {
    const int ps = ls * n;
    Builder b(kind, pl, xrows, whole_values(n), pass_threads(kind, pl, n * n * nh, 1024, n < 16 ? 2 : 4));
    b.pp.total = xrows;
    b.forward(xrows, ls, 1, 0);
    b.forward(n * nh, 1, ls, ST_Y);
    b.round_trip(whole_zlines(n), 0, ps, ST_Z, ST_ZIN, ST_ZOUT);
    b.forward(n * nh, 1, ls, ST_Y);
    b.forward(xrows, ls, 1, 0);
    return b.pp;
  }
  if (kind == KIND_ROW) {  // a line: two values per thread
    Builder b(kind, pl, 1, ls, pass_threads(kind, pl, n, 1024, 2));
    b.pp.total = 1;
    b.round_trip(1, ls, 1, 0);
    return b.pp;
  }
  const bool planes = planes_fit(n);
  if (kind == KIND_LAST || kind == KIND_MID) {
    const int xt = batch(n, n);
    Builder b(kind, pl, xt, xt * ls, pass_threads(kind, pl, xt * n, want));
    b.pp.tiles = (n + xt - 1) / xt;
    if (kind == KIND_MID)
      b.forward(xt, ls, 1, 0, ST_SRC, ST_SNK);
    else
      b.round_trip(xt, ls, 1, 0, ST_SRC, ST_SNK);
    return b.pp;
  }
  const int xr = planes ? n : batch(n, xrows);
  Builder b(kind, pl, xr, xr * ls, pass_threads(kind, pl, xr * n, want, kind == KIND_ALL && n <= 32 ? 2 : 8));
  b.pp.total = kind == KIND_ALL ? n : xrows;
  if (kind == KIND_ALL) {
    b.forward(n, ls, 1, 0);
    b.round_trip(n, 1, ls, ST_Y);
    b.forward(n, ls, 1, 0);
  } else if (kind == KIND_FWD) {
    b.forward(xr, ls, 1, 0, 0, planes ? 0 : ST_SNK);
    if (planes) b.forward(n, 1, ls, ST_Y, 0, ST_SNK);
  } else {
    if (planes) b.forward(n, 1, ls, ST_Y, ST_SRC);
    b.forward(xr, ls, 1, 0, planes ? 0 : ST_SRC);
  }
  return b.pp;
}

// The lines of one workgroup: where the pass's inputs and outputs are.
template <int MODE, int KIND>
struct Box {
  const SigmaArgs& a;
  int n, nm, no, nh;  // sites along x, mid, outer; outer indices of the half space
  unsigned mgm;       // magic of nm
  Row row;
  size_t wrow;        // half-space workspace row
  int total;          // x rows of the whole pass
  int g0;             // FWD, INV: first x row
  int x0, mid, midn;  // LAST, MID: first x, the lines' mid index (MID: the outer one) and its reflection
  int xlim;           // lines x >= xlim take no part
  int ls;             // LDS stride of an x row

  __device__ __forceinline__ bool active(int line) const {
    if (KIND == KIND_LAST || KIND == KIND_MID) return x0 + line < xlim;
    if (KIND == KIND_ROW || KIND == KIND_ALL || KIND == KIND_WHOLE) return true;
    return g0 + line < total;
  }
  __device__ __forceinline__ int lines(int most) const { return min(most, total - g0); }
  __device__ __forceinline__ int mirror(int i, int len) const { return i ? len - i : 0; }

  // where element e of a line is in LDS (KIND_WHOLE: elements from `split` on
  // in the reflected line)
  struct Place {
    int b0, b1, es, split;
    __device__ __forceinline__ int operator()(int e) const {
      return KIND != KIND_WHOLE || e < split ? b0 + e * es : b1 - e * es;
    }
  };
  // KIND_WHOLE: line l along z stands for (x, y) and (-x, -y)
  __device__ __forceinline__ void zline(int l, int& x, int& y) const {
    const int half = n / 2 + 1, ns = n & 1 ? 1 : 2;
    if (l < ns * half) {  // rows y that are their own reflection
      y = l >= half ? n / 2 : 0;
      x = l >= half ? l - half : l;
    } else {
      const int t = l - ns * half, q = div_magic(t, mgm);
      y = 1 + q;
      x = t - q * n;
    }
  }
  __device__ __forceinline__ Place place(const Stage& s, int l, bool store) const {
    if constexpr (KIND == KIND_WHOLE) {
      if (s.flags & ST_Z) {
        int x, y;
        zline(l, x, y);
        const int xm = mirror(x, n), ym = mirror(y, n);
        if (xm == x && ym == y && (store || !(s.flags & ST_ZIN)))
          return Place{n + ls * n * nh + n * ((x ? 1 : 0) + (y ? 2 : 0)), 0, 1, n};  // a line of its own
        return Place{n + x + y * ls, n + xm + ym * ls + n * s.es, s.es, nh};
      }
      if (s.flags & ST_Y) {
        const int z = div_magic(l, mgm);
        return Place{n + (l - z * n) + z * ls * n, 0, s.es, n};
      }
    }
    return Place{n + l * s.ls, 0, s.es, n};
  }

  // the input of the x rows at position i of their memory order (line l,
  // element e), symmetrised
  __device__ __forceinline__ double2 input(int i, int l, int e) const {
    if (KIND == KIND_ROW) return gather<MODE>(a, row, e, mirror(e, n));
    const int g = g0 + l, o = div_magic(g, mgm), m = g - o * nm;
    return gather<MODE>(a, row, n * g0 + i, n * (mirror(m, nm) + nm * mirror(o, no)) + mirror(e, n));
  }
  // where a line starts in W, and its reflected one
  struct Line {
    size_t w1, w2;
  };
  __device__ __forceinline__ Line line(const Stage& s, int l) const {
    Line t{0, 0};
    if constexpr (KIND == KIND_LAST) {
      t.w1 = wrow + (x0 + l) + (size_t)n * mid;
      t.w2 = wrow + mirror(x0 + l, n) + (size_t)n * midn;
    } else if constexpr (KIND == KIND_MID) {
      t.w1 = wrow + (x0 + l) + (size_t)n * nm * mid;
    } else if constexpr (KIND == KIND_INV) {
      t.w1 = wrow + (s.flags & ST_Y ? (size_t)l + (size_t)n * g0 : (size_t)n * (g0 + l));
    }
    return t;
  }
  __device__ __forceinline__ double2 source(const Stage& s, const Line& t, int e) const {
    if constexpr (KIND == KIND_LAST) {
      return e < nh ? a.W[t.w1 + (size_t)n * nm * e] : a.W[t.w2 + (size_t)n * nm * (no - e)];
    } else if constexpr (KIND == KIND_MID) {
      return a.W[t.w1 + (size_t)n * e];
    } else if constexpr (KIND == KIND_INV) {
      return a.W[t.w1 + (s.flags & ST_Y ? (size_t)n * e : (size_t)e)];
    } else {
      return make_double2(0.0, 0.0);  // (their rows are staged in LDS)
    }
  }
  __device__ __forceinline__ void destination(int flags, int l, int e, double2 v) const {
    if constexpr (KIND == KIND_FWD) {
      a.W[wrow + (flags & ST_Y ? (size_t)l + (size_t)n * (g0 + e) : (size_t)e + (size_t)n * (g0 + l))] = v;
    } else if constexpr (KIND == KIND_MID) {
      a.W[wrow + (x0 + l) + (size_t)n * (e + nm * mid)] = v;
    } else if constexpr (KIND == KIND_LAST) {
      const int x = x0 + l, xn = mirror(x, n), en = mirror(e, no);
      if (e < nh) a.W[wrow + x + (size_t)n * (mid + nm * e)] = v;
      if (en < nh && (xn != x || midn != mid)) a.W[wrow + xn + (size_t)n * (midn + nm * en)] = v;
    } else {
      const double2 z = swapped(v);
      const int g = g0 + l;
      emit<MODE>(a, row, n * g + e, z);
      if constexpr (KIND == KIND_INV || KIND == KIND_WHOLE) {
        // the reflected row, if it lies outside the half space
        const int o = div_magic(g, mgm), m = g - o * nm, on = mirror(o, no);
        if (on != o) emit<MODE>(a, row, n * (mirror(m, nm) + nm * on) + mirror(e, n), z);
      }
    }
  }
  // the pointwise step at element e of a line; swapped for the way back
  __device__ __forceinline__ double2 point(int l, int e, double2 z) const {
    size_t xi;
    if (KIND == KIND_LAST) {
      xi = row.off + (x0 + l) + (size_t)n * (mid + nm * e);
    } else if (KIND == KIND_WHOLE) {
      int x, y;
      zline(l, x, y);
      xi = row.off + x + (size_t)n * (y + n * e);
    } else if (KIND == KIND_ROW) {
      xi = row.off + e;
    } else {
      xi = row.off + l + (size_t)n * e;
    }
    return swapped(pointwise<MODE>(a, z, xi));
  }
};

// n twiddles, then the lines.  Always indexed by name: through a pointer the
// accesses would be flat ones, whose waits also wait for global loads.
extern __shared__ double2 sigma_lds[];

// elements base + q stride of a line to where its stage leaves them
template <int R, int MODE, int KIND>
__device__ __forceinline__ void put_line(const Stage& s, const Box<MODE, KIND>& box, int line, int base, int stride,
                                         const double2 (&v)[R]) {
  if (s.flags & ST_SNK) {
#pragma unroll
    for (int q = 0; q < R; ++q) box.destination(s.flags, line, base + q * stride, v[q]);
    return;
  }
  if (KIND == KIND_WHOLE && (s.flags & ST_ZOUT)) {
    // the half z <= n/2 of this line and of its reflection
    const int n = box.n;
    int x, y;
    box.zline(line, x, y);
    const int xm = box.mirror(x, n), ym = box.mirror(y, n);
    const bool self = xm == x && ym == y;
    const int own = n + x + y * box.ls, refl = n + xm + ym * box.ls;
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int e = base + q * stride, en = box.mirror(e, n);
      if (e < box.nh) sigma_lds[own + e * s.es] = v[q];
      if (en < box.nh && !self) sigma_lds[refl + en * s.es] = v[q];
    }
    return;
  }
  const auto at = box.place(s, line, true);
#pragma unroll
  for (int q = 0; q < R; ++q) sigma_lds[at(base + q * stride)] = v[q];
}

template <int R, int MODE, int KIND>
__device__ __forceinline__ void run_stage(const Stage& s, const Box<MODE, KIND>& box) {
  constexpr int U = held(R);
  double2 v[U][R];
  const int T = blockDim.x;
  const int step = s.Ns > 1 ? s.m / s.Ns : 0;
  // neighbouring threads take the same butterfly of neighbouring lines
  auto split = [&](int u, int& line, int& j) {
    const int idx = (int)threadIdx.x + u * T;
    j = div_magic(idx, s.mg);
    line = s.first + idx - j * s.lines;
    return idx < s.items && box.active(line);
  };
#pragma unroll
  for (int u = 0; u < U; ++u) {
    int line, j;
    if (split(u, line, j)) {
      if (s.flags & ST_SRC) {
        const auto ln = box.line(s, line);
#pragma unroll
        for (int r = 0; r < R; ++r) v[u][r] = box.source(s, ln, j + r * s.m);
      } else {
        const auto at = box.place(s, line, false);
#pragma unroll
        for (int r = 0; r < R; ++r) v[u][r] = sigma_lds[at(j + r * s.m)];
      }
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    int line, j;
    if (split(u, line, j)) {
      if (step) {
        const int kk = (j - div_magic(j, s.mgNs) * s.Ns) * step;
#pragma unroll
        for (int r = 1; r < R; ++r) v[u][r] = cmul(v[u][r], sigma_lds[r * kk]);
      }
      dft<R>(v[u]);
      if (s.flags & ST_POINT) {
        // the last forward stage: element j + q m
#pragma unroll
        for (int q = 0; q < R; ++q) v[u][q] = box.point(line, j + q * s.m, v[u][q]);
        if (s.flags & ST_TWICE) dft<R>(v[u]);
      }
    }
  }
  if (!(s.flags & ST_SRC)) __syncthreads();  // in place: every input of these lines has been read
#pragma unroll
  for (int u = 0; u < U; ++u) {
    int line, j;
    if (split(u, line, j)) {
      // Stockham order; after ST_TWICE the inverse's first stage (span 1)
      int base = j * R, stride = 1;
      if (s.Ns > 1 && !(s.flags & ST_TWICE)) {
        const int jq = div_magic(j, s.mgNs);
        base = jq * s.Ns * R + (j - jq * s.Ns);
        stride = s.Ns;
      }
      put_line<R>(s, box, line, base, stride, v[u]);
    }
  }
  if ((s.flags & ST_END) && !(s.flags & ST_SNK)) __syncthreads();
}

// a prime radix above 23, from LDS: an item forms direct_pairs(KIND) output
// pairs q, R - q of one butterfly from the sums and differences of its inputs,
// X_q, X_{R-q} = A +- B (the odd DFT above with a table)
template <int MODE, int KIND>
__device__ __forceinline__ void run_direct(const Stage& s, const Box<MODE, KIND>& box) {
  constexpr int G = direct_pairs(KIND), U = DIRECT_HELD;
  const int R = s.R, H = (R - 1) / 2;
  const int T = blockDim.x;
  const int step = s.Ns > 1 ? s.m / s.Ns : 0;
  double2 A[U][G], B[U][G], dc[U];
  auto split = [&](int u, int& line, int& j, int& q0) {
    const int idx = (int)threadIdx.x + u * T;
    const int t = div_magic(idx, s.mg);  // lines fastest: a wave shares its butterfly
    line = s.first + idx - t * s.lines;
    const int g = t / s.m;
    j = t - g * s.m;
    q0 = 1 + g * G;
    return idx < s.items && box.active(line);
  };
#pragma unroll
  for (int u = 0; u < U; ++u) {
    int line, j, q0;
    if (split(u, line, j, q0)) {
      const auto at = box.place(s, line, false);
      const int kk = step ? (j - div_magic(j, s.mgNs) * s.Ns) * step : 0;
      const double2 x0 = sigma_lds[at(j)];
      dc[u] = x0;
      int iq[G];
#pragma unroll
      for (int g = 0; g < G; ++g) {
        A[u][g] = x0;
        B[u][g] = make_double2(0.0, 0.0);
        iq[g] = 0;
      }
      for (int r = 1; r <= H; ++r) {
        double2 a = sigma_lds[at(j + r * s.m)], b = sigma_lds[at(j + (R - r) * s.m)];
        if (step) {
          a = cmul(a, sigma_lds[r * kk]);
          b = cmul(b, sigma_lds[(R - r) * kk]);
        }
        const double2 t = cadd(a, b), d = csub(a, b);
        dc[u] = cadd(dc[u], t);
#pragma unroll
        for (int g = 0; g < G; ++g) {
          iq[g] += min(q0 + g, H);
          if (iq[g] >= R) iq[g] -= R;
          const double2 w = sigma_lds[iq[g] * s.m];  // (cos, -sin)(2 pi q r / R)
          A[u][g].x += w.x * t.x;
          A[u][g].y += w.x * t.y;
          B[u][g].x -= w.y * d.y;
          B[u][g].y += w.y * d.x;
        }
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < U; ++u) {
    int line, j, q0;
    if (split(u, line, j, q0)) {
      const int jq = s.Ns > 1 ? div_magic(j, s.mgNs) : j;
      const int base = jq * s.Ns * R + (j - jq * s.Ns);
      auto put = [&](int q, double2 v) {
        const int e = base + q * s.Ns;
        if (s.flags & ST_POINT) v = box.point(line, e, v);
        double2 one[1] = {v};
        put_line<1>(s, box, line, e, 0, one);
      };
      if (q0 == 1) put(0, dc[u]);
#pragma unroll
      for (int g = 0; g < G; ++g) {
        if (q0 + g <= H) {
          put(q0 + g, cadd(A[u][g], B[u][g]));
          put(R - q0 - g, csub(A[u][g], B[u][g]));
        }
      }
    }
  }
  if ((s.flags & ST_END) && !(s.flags & ST_SNK)) __syncthreads();
}

}  // namespace

namespace {

// one stage of a plan: run time, or (NT > 0) known when compiled
template <int CLASS, int MODE, int KIND>
__device__ __forceinline__ void any_stage(const Stage& s, const Box<MODE, KIND>& box) {
  switch (s.R) {
    case 1: run_stage<1>(s, box); break;
    case 2: run_stage<2>(s, box); break;
    case 3: run_stage<3>(s, box); break;
    case 4: run_stage<4>(s, box); break;
    case 5: run_stage<5>(s, box); break;
    case 6: run_stage<6>(s, box); break;
    case 7: run_stage<7>(s, box); break;
    case 8: run_stage<8>(s, box); break;
    default:
      if constexpr (CLASS == PLAN_WIDE) {
        if (s.R == 17)
          return run_stage<17>(s, box);
        else if (s.R == 19)
          return run_stage<19>(s, box);
        else if (s.R == 23)
          return run_stage<23>(s, box);
      }
      if constexpr (CLASS == PLAN_ANY || CLASS == PLAN_WIDE) {
        if (s.R == 9)
          run_stage<9>(s, box);
        else if (s.R == 10)
          run_stage<10>(s, box);
        else if (s.R == 11)
          run_stage<11>(s, box);
        else if (s.R == 13)
          run_stage<13>(s, box);
        else
          run_direct(s, box);
      }
  }
}

// threads of the passes on compiled lengths
constexpr int CT_WANT = 256;

template <int NT, int KIND>
struct CompiledPlan {
  static constexpr PassPlan pp = pass_plan(make_plan(NT), KIND, KIND != KIND_ROW && KIND != KIND_ALL, CT_WANT);
};

template <int NT, int I, int MODE, int KIND>
__device__ __forceinline__ void compiled_stages(const Box<MODE, KIND>& box) {
  if constexpr (I < CompiledPlan<NT, KIND>::pp.nstages) {
    constexpr Stage s = CompiledPlan<NT, KIND>::pp.st[I];
    if constexpr (is_direct(s.R))
      run_direct(s, box);
    else
      run_stage<s.R>(s, box);
    compiled_stages<NT, I + 1>(box);
  }
}

}  // namespace

// blockIdx.y: row q.  blockIdx.x: FWD and INV plane
// outer = x, or a batch of x rows; MID (tile of x, outer); LAST (tile of x, mid).
// NT: the length of a compiled plan, or the class of the one in `plan`.
struct NoPlan {};
constexpr int STAGE_WORDS = sizeof(Stage) / 4;
__shared__ int sigma_stages[MAX_STAGES * STAGE_WORDS];
__device__ __forceinline__ Stage stage_at(int i) {
  int w[STAGE_WORDS];
#pragma unroll
  for (int k = 0; k < STAGE_WORDS; ++k) w[k] = __builtin_amdgcn_readfirstlane(sigma_stages[i * STAGE_WORDS + k]);
  Stage s;
  __builtin_memcpy(&s, w, sizeof(s));
  return s;
}

template <int MODE, int KIND, int NT>
__global__ __launch_bounds__(plan_threads(plan_wide(NT))) __attribute__((amdgpu_waves_per_eu(plan_waves(KIND, NT)))) void sigma_pass(
    SigmaArgs a, std::conditional_t<(NT > 0), NoPlan, PassPlan> plan) {
  const PassPlan& pp = [&]() -> const PassPlan& {
    if constexpr (NT > 0)
      return CompiledPlan<NT, KIND>::pp;
    else
      return plan;
  }();
  const int n = pp.n;
  Box<MODE, KIND> box{a};
  box.n = n;
  box.nm = a.nz > 1 ? a.ny : 1;
  box.no = a.nz > 1 ? a.nz : a.ny;
  if constexpr (NT > 0) {
    box.nm = KIND == KIND_ROW || KIND == KIND_ALL ? 1 : n;
    box.no = KIND == KIND_ROW ? 1 : n;
  }
  box.nh = box.no / 2 + 1;
  box.mgm = (NT > 0 ? KIND != KIND_ROW && KIND != KIND_ALL : a.nz > 1) ? pp.mgn : 0u;
  box.ls = pp.ls;
  const int q = blockIdx.y;
  if (q >= stage_rows<MODE>(a)) return;
  box.row = row_of<MODE>(a, q);
  box.wrow = (size_t)q * n * box.nm * box.nh;
  box.g0 = KIND == KIND_FWD || KIND == KIND_INV ? blockIdx.x * pp.lines : 0;
  box.total = pp.total;
  if (KIND == KIND_LAST || KIND == KIND_MID) {
    box.mid = blockIdx.x / pp.tiles;
    box.x0 = (blockIdx.x - box.mid * pp.tiles) * pp.lines;
    box.midn = box.mid ? box.nm - box.mid : 0;
    // a mid index that is its own reflection pairs the lines x and -x of
    // its row: only x <= n/2 is taken
    box.xlim = KIND == KIND_LAST && box.midn == box.mid ? n / 2 + 1 : n;
    if (box.x0 >= box.xlim) return;
  }
  constexpr bool GATHER = KIND == KIND_ROW || KIND == KIND_FWD || KIND == KIND_ALL || KIND == KIND_WHOLE;
  // the stages, which would be read from the argument buffer one after another,
  // and the twiddles: on their way with the rows
  const int tid = threadIdx.x;
  const double2 tw0 = a.tw[min(tid, n - 1)];
  int stage0 = 0;
  if constexpr (NT <= 0) stage0 = reinterpret_cast<const int*>(plan.st)[min(tid, plan.nstages * STAGE_WORDS - 1)];
  if constexpr (GATHER) {
    // the x rows in memory order, four elements in flight per thread
    constexpr int U = 4;
    const int count = box.lines(pp.lines) * n;
    for (int i0 = threadIdx.x; i0 < count; i0 += U * blockDim.x) {
      double2 z[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = min(i0 + u * (int)blockDim.x, count - 1);
        const int l = div_magic(i, pp.mgn);
        z[u] = box.input(i, l, i - l * n);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = i0 + u * (int)blockDim.x;
        const int l = div_magic(i, pp.mgn);
        if (i < count) sigma_lds[n + l * pp.ls + (i - l * n)] = z[u];
      }
    }
  }
  if (tid < n) sigma_lds[tid] = tw0;
  for (int k = tid + blockDim.x; k < n; k += blockDim.x) sigma_lds[k] = a.tw[k];
  if constexpr (NT <= 0) {
    const int* from = reinterpret_cast<const int*>(plan.st);
    const int words = plan.nstages * STAGE_WORDS;
    if (tid < words) sigma_stages[tid] = stage0;
    for (int k = tid + blockDim.x; k < words; k += blockDim.x) sigma_stages[k] = from[k];
  }
  // (a first stage on W has no twiddles, and ends with a barrier unless it is
  // the only one)
  if constexpr (GATHER || NT <= 0) __syncthreads();
  if constexpr (NT > 0) {
    compiled_stages<NT, 0>(box);
  } else {
    for (int i = 0; i < pp.nstages; ++i) any_stage<NT>(stage_at(i), box);
  }
  if constexpr (KIND == KIND_ROW || KIND == KIND_INV || KIND == KIND_ALL || KIND == KIND_WHOLE) {
    // the x rows, in memory order
    const int count = box.lines(pp.lines) * n;
    for (int i = threadIdx.x; i < count; i += blockDim.x) {
      const int l = div_magic(i, pp.mgn), e = i - l * n;
      box.destination(0, l, e, sigma_lds[n + l * pp.ls + e]);
    }
  }
}

// ---------------------------------------------------------------------------
// host side: the launches of the stage
// ---------------------------------------------------------------------------
namespace {

template <int MODE, int KIND, int NT>
hipError_t launch_compiled(const SigmaArgs& a, dim3 grid, hipStream_t st) {
  constexpr PassPlan pp = CompiledPlan<NT, KIND>::pp;
  hipLaunchKernelGGL((sigma_pass<MODE, KIND, NT>), grid, dim3(pp.threads), sizeof(double2) * (pp.elements + pp.n), st, a,
                     NoPlan{});
  return hipGetLastError();
}

// the forms that the code of a mode comes in, each in an object file of its
// own: the compiled lengths, as lines and planes, whole rows or three passes, and
// the classes of run-time plans
constexpr int FORM_FLAT = 1, FORM_WHOLE = 2, FORM_PASSES = 3;

constexpr int plan_class(const FFTPlan& pl) {
  int top = 0;
  for (int i = 0; i < pl.nf; ++i) top = most(top, pl.fac[i]);
  return top <= SMALL_RADIX ? PLAN_SMALL : wide(pl) ? PLAN_WIDE : PLAN_ANY;
}
constexpr bool row_compiled(int n) { return n >= ROW_MIN && n <= ROW_MAX && (n & (n - 1)) == 0; }
constexpr bool by_whole_rows(int n, int rows, bool alone) {
  if (!whole_fits(n)) return false;
  return n < SPREAD_MIN || (n % 8 ? !alone || rows >= SPREAD_PLAN_ROWS : rows >= SPREAD_ROWS);
}
// the form of a stage over `rows` rows; alone: no other run's stages beside it
constexpr int stage_form(const FFTPlan& pl, int sdim, int rows, bool alone) {
  const int n = pl.n;
  if (sdim == 1 || n == 1) return row_compiled(n) ? FORM_FLAT : plan_class(pl);
  if (sdim == 3 && by_whole_rows(n, rows, alone)) return FORM_WHOLE;
  if (!planes_fit(n) || n % 8) return plan_class(pl);
  return sdim == 2 ? FORM_FLAT : FORM_PASSES;
}

template <int MODE, int KIND, int CLASS>
hipError_t launch_pass(const SigmaArgs& a, const PassPlan& pp, dim3 grid, hipStream_t st) {
  const size_t lds = sizeof(double2) * ((size_t)pp.elements + pp.n);
  if (lds + sizeof(pp.st) > LDS_MAX || pp.threads > plan_threads(CLASS == PLAN_WIDE) || pp.nstages > MAX_STAGES ||
      plan_class(a.plan) != CLASS)
    return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL((sigma_pass<MODE, KIND, CLASS>), grid, dim3(pp.threads), lds, st, a, pp);
  return hipGetLastError();
}

// the launch of the compiled length n in NT, NT + STEP (STEP = 0: 2 NT), ...
// LAST, if there is one
constexpr int next_length(int n, int step) { return step ? n + step : 2 * n; }
template <int MODE, int KIND, int NT, int LAST, int STEP>
hipError_t launch_length(const SigmaArgs& a, int n, dim3 grid, hipStream_t st) {
  constexpr int next = next_length(NT, STEP);
  if (n == NT) return launch_compiled<MODE, KIND, NT>(a, grid, st);
  if constexpr (next <= LAST)
    return launch_length<MODE, KIND, next, LAST, STEP>(a, n, grid, st);
  else
    return hipErrorInvalidConfiguration;
}

// the longest compiled line of a mode (SG_PLAIN has no lattice past TWIDDLE_MAX)
template <int MODE>
constexpr int row_last = MODE == SG_PLAIN ? TWIDDLE_MAX : ROW_MAX;

template <int MODE, int FORM>
hipError_t launch_compiled_stage(const SigmaArgs& a, int rows, hipStream_t st) {
  const int n = a.n;
  if constexpr (FORM == FORM_WHOLE) {
    return launch_length<MODE, KIND_WHOLE, 2, WHOLE_MAX, 1>(a, n, dim3(1, rows), st);
  } else if constexpr (FORM == FORM_FLAT) {
    if (a.ny == 1) return launch_length<MODE, KIND_ROW, ROW_MIN, row_last<MODE>, 0>(a, n, dim3(1, rows), st);
    return launch_length<MODE, KIND_ALL, 8, 64, 8>(a, n, dim3(1, rows), st);
  } else {
    const PassPlan last = pass_plan(a.plan, KIND_LAST, true, CT_WANT);
    const int nh = n / 2 + 1;
    const dim3 gx(nh, rows), gl(last.tiles * nh, rows);
    hipError_t e;
    if ((e = launch_length<MODE, KIND_FWD, SPREAD_MIN, 64, 8>(a, n, gx, st)) != hipSuccess) return e;
    if ((e = launch_length<MODE, KIND_LAST, SPREAD_MIN, 64, 8>(a, n, gl, st)) != hipSuccess) return e;
    return launch_length<MODE, KIND_INV, SPREAD_MIN, 64, 8>(a, n, gx, st);
  }
}

// want: threads per workgroup asked for
template <int MODE, int CLASS>
hipError_t launch_plan_stage(const SigmaArgs& a, int rows, int want, hipStream_t st) {
  const FFTPlan& pl = a.plan;
  const int n = a.n, nh = n / 2 + 1;
  if (a.ny == 1)
    return launch_pass<MODE, KIND_ROW, CLASS>(a, pass_plan(pl, KIND_ROW, false, want), dim3(1, rows), st);
  const bool three = a.nz > 1, planes = planes_fit(n);
  if (planes && !three)
    return launch_pass<MODE, KIND_ALL, CLASS>(a, pass_plan(pl, KIND_ALL, false, want), dim3(1, rows), st);
  const PassPlan fwd = pass_plan(pl, KIND_FWD, three, want), mid = pass_plan(pl, KIND_MID, three, want);
  const PassPlan last = pass_plan(pl, KIND_LAST, three, want), inv = pass_plan(pl, KIND_INV, three, want);
  const dim3 gx(planes ? nh : (fwd.total + fwd.lines - 1) / fwd.lines, rows), gm(mid.tiles * nh, rows),
      gl(last.tiles * (three ? nh : 1), rows);
  const bool between = three && !planes;
  auto middle = [&]() -> hipError_t {
    if constexpr (MODE == SG_PLAIN)
      return hipErrorInvalidConfiguration;  // (no lattice of that size)
    else
      return launch_pass<MODE, KIND_MID, CLASS>(a, mid, gm, st);
  };
  hipError_t e;
  if ((e = launch_pass<MODE, KIND_FWD, CLASS>(a, fwd, gx, st)) != hipSuccess) return e;
  if (between && (e = middle()) != hipSuccess) return e;
  if ((e = launch_pass<MODE, KIND_LAST, CLASS>(a, last, gl, st)) != hipSuccess) return e;
  if (between && (e = middle()) != hipSuccess) return e;
  return launch_pass<MODE, KIND_INV, CLASS>(a, inv, gx, st);
}

// the dynamic LDS that the larger passes need, per kernel
template <int MODE, int KIND, int NT>
hipError_t prepare_pass() {
  if constexpr (NT > 0) {
    constexpr PassPlan pp = CompiledPlan<NT, KIND>::pp;
    if (sizeof(double2) * (pp.elements + pp.n) <= 65536) return hipSuccess;
  }
  return hipFuncSetAttribute((const void*)sigma_pass<MODE, KIND, NT>, hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)(LDS_MAX - (NT > 0 ? 0 : sizeof(PassPlan::st))));
}
template <int MODE, int KIND, int NT, int LAST, int STEP>
hipError_t prepare_lengths() {
  const hipError_t e = prepare_pass<MODE, KIND, NT>();
  if constexpr (next_length(NT, STEP) <= LAST)
    return e == hipSuccess ? prepare_lengths<MODE, KIND, next_length(NT, STEP), LAST, STEP>() : e;
  else
    return e;
}
template <int MODE, int CLASS>
hipError_t prepare_plan_stage() {
  hipError_t e = prepare_pass<MODE, KIND_ROW, CLASS>();
  if (e == hipSuccess) e = prepare_pass<MODE, KIND_ALL, CLASS>();
  if (e == hipSuccess) e = prepare_pass<MODE, KIND_FWD, CLASS>();
  if constexpr (MODE != SG_PLAIN)
    if (e == hipSuccess) e = prepare_pass<MODE, KIND_MID, CLASS>();
  if (e == hipSuccess) e = prepare_pass<MODE, KIND_LAST, CLASS>();
  return e == hipSuccess ? prepare_pass<MODE, KIND_INV, CLASS>() : e;
}
template <int MODE, int FORM>
hipError_t prepare_compiled_stage() {
  if constexpr (FORM == FORM_WHOLE) {
    return prepare_lengths<MODE, KIND_WHOLE, 2, WHOLE_MAX, 1>();
  } else if constexpr (FORM == FORM_FLAT) {
    const hipError_t e = prepare_lengths<MODE, KIND_ROW, ROW_MIN, row_last<MODE>, 0>();
    return e == hipSuccess ? prepare_lengths<MODE, KIND_ALL, 8, 64, 8>() : e;
  } else {
    hipError_t e = prepare_lengths<MODE, KIND_FWD, SPREAD_MIN, 64, 8>();
    if (e == hipSuccess) e = prepare_lengths<MODE, KIND_LAST, SPREAD_MIN, 64, 8>();
    return e == hipSuccess ? prepare_lengths<MODE, KIND_INV, SPREAD_MIN, 64, 8>() : e;
  }
}

}  // namespace

// the stage of one mode in one form, and its preparation (kb_sigma_pass.hip)
template <int MODE, int FORM>
hipError_t sigma_form(const SigmaArgs& a, int rows, int want, hipStream_t st);
template <int MODE, int FORM>
hipError_t sigma_form_prepare();

}  // namespace qftkb
