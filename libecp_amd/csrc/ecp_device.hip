// HIP device layer of the ECP integral engine, written for gfx950 (MI355X).
//
// Pipeline of one job (all FP64; a main stream forks into worker streams
// and joins them, captured once into a HIP graph):
//   k_tables zero-fill of counters and flags; U_L(r_n) and r_n^k U_l(r_n) on
//            the 383-point small grid per (centre, channel, point chunk)
//            (evalECP / tabECP_FM06: ecp.c:41-60, type2.c:184-219); and
//            F_lambda(r_n) per (centre, shell) on its screened window
//            (calcF_FM06: type2.c:222-310)
//            and per-(centre, atom) angular tables (evalAngularIntegrals:
//            angular_integrals.c:104-142); the type-1 units
//   k_type1 / k_t1tail  type-1 radial integrals Q[l1][l2] per (triplet,
//            primitive pair) with the PS93 sequence (calcQ: type1.c:94-203):
//            lane-serial head, wave-cooperative tail for the open pairs,
//            which also redoes the failed ones with PSM92 on the FM06-mapped
//            large grid (type1.c:205-252)
//   k_type2 / k_type2_small  type-2 radial integrals T_l[l1][l2][l3] per
//            entry with PS93 (calcT_fast_FM06: type2.c:336-381)
//   k_fb2    PSM92 large-grid redo of failed type-2 entries (calcT_FM06:
//            type2.c:417-528)
//   k_asm1 / k_asm2  type-1 / type-2 blocks, binomial shift and norms
//            (calcChi: type1.c:211-302, calcGamma: type2.c:532-631,
//             calcPolynomials: util.c:246-334)
//
// The adaptive quadratures are evaluated lazily: one lane owns one integral
// (or one primitive pair's set of integrals) and visits the grid points in
// the integrator's own level order, replaying its recurrences and its
// convergence test after every level.  A lane stops at convergence, so only
// the points the reference's result depends on are evaluated; the reference
// tabulates every window point up front.  Summation order inside a level and
// the recurrences are those of gc_integrators.c:156-217 (PS93) and :38-86
// (PSM92).
//
// Large-grid fallback semantics: points past a screening break contribute
// zero (the reference reuses stale buffers there, type2.c:443-481).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <vector>

#include "../../include/libecp_ext.h"
#include "ecp_host.h"

#define ECP_CHECK(call)                                                            \
  do {                                                                             \
    hipError_t e_ = (call);                                                        \
    if (e_ != hipSuccess) {                                                        \
      snprintf(err, errlen, "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_), \
               __FILE__, __LINE__);                                                \
      return -1;                                                                   \
    }                                                                              \
  } while (0)

// Device scratch of the no-allocation entry point (ecp_dev_contract_noalloc):
// one array per GPU, held until the process ends.  Host code never uses the
// name `scratch` as an address: set-up looks up each device's copy with
// hipGetSymbolAddress, and every use goes through that pointer.
constexpr size_t kScratchBytes = (size_t)32 << 20;  // 32 MiB
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {

constexpr int kScratchDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kScratchDevices];

// An allocation; where memory has run out, once more after the idle contexts of
// the process cache have given theirs back.
template <typename Alloc>
hipError_t alloc_or_trim(Alloc alloc) {
  const hipError_t e = alloc();
  if (e != hipErrorOutOfMemory) return e;
  (void)hipGetLastError();
  libecp_cache_clear();
  return alloc();
}

// The scratch address on the current device, looked up once per device.
// 0, or -1 (message in err).
int scratch_setup(void **ptr, char *err, size_t errlen) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= kScratchDevices) {
    snprintf(err, errlen, "no-allocation scratch: no usable current device (%s)", hipGetErrorString(e));
    return -1;
  }
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      snprintf(err, errlen, "hipGetSymbolAddress(scratch) failed: %s", hipGetErrorString(e));
      return -1;
    }
    g_scratch_ptr[dev] = p;
  }
  *ptr = g_scratch_ptr[dev];
  return 0;
}

}  // namespace

namespace {

constexpr int SO = ECP_SMALL_ORDER;
constexpr int kMaxLMB = ECP_MAX_L - 1 + ECP_MAX_LBS;  // largest Bessel order of F / K_a / K_b

// A table that no kernel writes: its elements are read through the constant
// address space, so that a uniform index is a scalar load wherever it stands.
// Through a plain pointer the compiler falls back to vector loads behind
// every barrier and store, which wait in order with the data loads in
// flight.
template <typename V>
struct CPtr {
  const V *p;
  CPtr() = default;
  __host__ __device__ CPtr(const V *q) : p(q) {}
  __host__ __device__ operator const V *() const { return p; }
  template <typename I>
  __device__ __forceinline__ V operator[](I i) const {
    return at(p + i);
  }
  static __device__ __forceinline__ V at(const V *q) {
    if constexpr (sizeof(V) <= 8) {
      return *(const __attribute__((address_space(4))) V *)q;
    } else {
      static_assert(sizeof(V) % 4 == 0, "whole words");
      const __attribute__((address_space(4))) int *w = (const __attribute__((address_space(4))) int *)q;
      V out;
#pragma unroll
      for (size_t k = 0; k < sizeof(V) / 4; k++) {
        const int x = w[k];
        __builtin_memcpy((char *)&out + 4 * k, &x, 4);
      }
      return out;
    }
  }
};
// one element, or member, likewise
template <typename V>
__device__ __forceinline__ V cload(const V *q) {
  return CPtr<V>::at(q);
}

constexpr int kSphDim = 16;  // more than any l of the harmonics

// A point pair of the PS93 sequence, in visit order: its points, their
// weights, and the level it is the last pair of (0: none).  A level's last
// pair is its closest to the centre, so the level has a point in a window
// where this pair does.
struct Ps93Pair {
  double wl, wr;
  int li, ri, ends, pad;
};
constexpr int kPs93Pad = 16;  // copies of the last pair (ending nothing) past the end of the list

struct DevTables {
  CPtr<double> xs, ws, xl, wl;
  CPtr<int> p93l, p93r, p92l, p92r;
  CPtr<Ps93Pair> v93;
  CPtr<int> vis;  // a small-grid point's place in the PS93 visit order
  // harmonics: norms sqrt((l-m)!/(l+m)!) sqrt((2l+1)/(2 pi)) (m = 0: the
  // second factor) at [l * kSphDim + m], double factorials, 1 / n
  CPtr<double> snorm, dfac, inv;
  // position of the product of the monomials at positions r and q, of degree
  // up to the basis's each, at [r * prodN + q]
  CPtr<int> prod;
  int prodN;
  // the shift's terms (shift_table)
  const unsigned *shift;
  // T entries of a triplet (build_templates): packed (lambda1, lambda2, alpha + beta, l), channel after channel; those
  // of channel l < L at [toff(la, lb, l), toff(la, lb, l + 1)) (t2_off)
  CPtr<int> tmpl, toff;
  const double *bessel;
  const double *poly2sph;
  const double *omega;
  CPtr<int> ijk, ijkIndex;
  int ijkDim, tmDim, lorder;
  int omL, omLambda, omAlpha;
  double tol, lnAcc1, lnAcc2, accuracy;
  ecp_schedule s93, s92;
};

struct DevJob {
  CPtr<ecp_xyz> atoms;
  CPtr<int> atom_maxl;
  CPtr<ecp_shell> shells;
  CPtr<double> pa, pd;
  CPtr<ecp_centre> cent;
  CPtr<ecp_gauss> gauss;
  CPtr<ecp_window> win;
  CPtr<ecp_triplet> trip;
  int ntrip;
  double *UL, *Ut, *F, *ang;
  int FL, UK, angL, ang_lam, ang_c;
  int maxPairs;
  int deriv;  // derivative order: F slabs per run 0..deriv, angular tables to lmax + deriv
  CPtr<int> teoff;  // per triplet: its first T entry in the job's T arrays
  int US;            // U row stride: channels times powers
};

// ---------------------------------------------------------------------------
// numerical primitives

// The PS93 recurrences and test after level lv (gc_integrators.c:156-217);
// any: the level had a point in the window.  True when the integral has
// converged, to *res.  After level lv the rule has n = 3 2^(lv / 2) points in
// its estimate, and the levels take turns (j = 0 after odd ones): the
// divisions are by 9 2^h, three operations each (div_const's, with a
// reciprocal that is exact but for the factor 1 / 9).
__device__ __forceinline__ bool ps93_level(int lv, bool any, double tol, double I, double &p, double &q,
                                           double *res) {
  const int h = lv >> 1;
  const double b = (double)(9 << h), y = ldexp(1.0 / 9.0, -h);
  auto over = [&](double x) {
    const double d = x * y;
    return __builtin_fma(__builtin_fma(-b, d, x), y, d);
  };
  double err;
  if (lv & 1) {
    p += (I - q);
    err = over(16 * fabs(q - 3 * p / 2));
  } else {
    err = over(16 * fabs(I - 2 * q));
    q = I;
  }
  if (!(any && err < tol)) return false;
  *res = over(16 * q);
  return true;
}

// Radial powers other than 0, 1, 2 (rare in ECPs) through a call: inlined,
// pow's registers set the budget of the kernel around it (a type-1 fallback
// kernel of its own held 152 registers with it, 128 without)
__device__ __attribute__((noinline)) double ecp_pow_general(double r, double n) { return pow(r, n); }

__device__ __forceinline__ double ecp_pow(double r, double n) {
  // exact special cases of a correctly rounded pow
  if (n == 2.0) return r * r;
  if (n == 1.0) return r;
  if (n == 0.0) return 1.0;
  return ecp_pow_general(r, n);
}

// U_l(r): the channel's own Gaussians only (C.gl; the host orders a centre's
// Gaussians by channel), where a scan over all of them would read and test
// every one for each channel
__device__ __forceinline__ double eval_ecp(const DevJob &J, int centre, int l, double r) {
  double pot = 0.0;
  const double r2 = r * r;
  const ecp_centre *C = J.cent + centre;
  const ecp_gauss *g = J.gauss + cload(&C->g0);
  const int end = cload(&C->gl[l + 1]);
  for (int i = cload(&C->gl[l]); i < end; i++) {
    const ecp_gauss x = cload(g + i);
    pot += ecp_pow(r, x.n) * x.d * exp(-x.a * r2);
  }
  return pot;
}

// x / D, correctly rounded, in three operations: q = RN(x RN(1 / D)) is
// within one unit in the last place of the quotient, its remainder x - q D
// is exact in a fused multiply-add, and RN(q + r RN(1 / D)) is then the
// rounded quotient (Markstein, IBM J. Res. Dev. 34 (1990) 111).  The
// compiler's general FP64 division takes about a dozen instructions, one of
// them at a quarter of the rate.  Finite x away from the underflow range.
template <int D>
__device__ __forceinline__ double div_const(double x) {
  if constexpr ((D & (D - 1)) == 0) {
    return x * (1.0 / D);  // exact
  } else {
    constexpr double y = 1.0 / D;
    const double q = x * y;
    return __builtin_fma(__builtin_fma(-double(D), q, x), y, q);
  }
}

// K_0..K_LM at z (bessel.c:102-199): leading term below 1e-7, 5-term Taylor
// series about the nearest table abscissa below 16 (derivatives by the
// recurrence K_j' = j/(2j+1)(K_{j-1} - K_{j+1}) - K_j + K_{j+1}), asymptotic
// series above.
template <int LM, int L>
__device__ __forceinline__ void bessel_asymptotic(double (&A)[LM + 1], double (&K)[LM + 1]) {
  if constexpr (L <= LM) {
    double f = L * (L + 1);
#pragma unroll
    for (int i = 1; i < L; i++) {
      K[L] += f * A[i];
      f *= (L + i + 1) * (L - i);
    }
    A[L] = div_const<L>(-A[0] * A[L - 1]);
    K[L] += f * A[L];
    bessel_asymptotic<LM, L + 1>(A, K);
  }
}

template <int LM>
__device__ __forceinline__ void bessel_k(const double *__restrict__ tab, double z, double (&K)[LM + 1]) {
  if (z < 1.0E-7) {
    if (z <= 0) {
      K[0] = 1.0;
#pragma unroll
      for (int l = 1; l <= LM; l++) K[l] = 0.0;
    } else {
      K[0] = 1 - z;
#pragma unroll
      for (int l = 1; l <= LM; l++) K[l] = K[l - 1] * z / (2 * l + 1);
    }
  } else if (z < 16.0) {
    constexpr int ML = LM + 5;
    const int index = (int)floor(z * 100.0 + 0.5);
    const double dz = z - div_const<100>((double)index);
    const double *row = tab + (size_t)index * ECP_BESSEL_STRIDE;
    double d[ML + 2];
#pragma unroll
    for (int l = 0; l <= ML; l++) d[l] = row[l];
    d[ML + 1] = 0.0;
#pragma unroll
    for (int l = 0; l <= LM; l++) K[l] = d[l];
    // dz^i / i!, each factor divided in turn
    const double sc1 = dz, sc2 = div_const<2>(sc1 * dz), sc3 = div_const<3>(sc2 * dz), sc4 = div_const<4>(sc3 * dz),
                 sc5 = div_const<5>(sc4 * dz);
#pragma unroll
    for (int i = 1; i <= 5; i++) {
      const int top = ML - i;
      const double scale = i == 1 ? sc1 : i == 2 ? sc2 : i == 3 ? sc3 : i == 4 ? sc4 : sc5;
      double prev = d[0];
      d[0] = d[1] - d[0];
#pragma unroll
      for (int j = 1; j <= top; j++) {
        const double cur = d[j];
        double cj = double(j) / (2.0 * j + 1.0);
        d[j] = cj * (prev - d[j + 1]) - cur + d[j + 1];
        prev = cur;
      }
#pragma unroll
      for (int j = 0; j <= LM; j++) K[j] += scale * d[j];
    }
  } else {
    double A[LM + 1];
    A[0] = 0.5 / z;
#pragma unroll
    for (int l = 0; l <= LM; l++) K[l] = A[0];
    bessel_asymptotic<LM, 1>(A, K);
  }
}

// Column m >= 0 of the real spherical harmonics (entries (l, +-m), l =
// m..lmax) with the arithmetic of spherical_harmonics.c:15-114, a column per
// lane: associated Legendre recurrences without Condon-Shortley phase (s1^m
// by repeated multiplication, the diagonal, the first subdiagonal and the
// three-term recurrence in l), the normalisation sqrt((2l+1)/(2pi)
// (l-m)!/(l+m)!), 1/sqrt(2) for m = 0, and sin/cos(m phi) by the
// angle-addition recurrence from m = 1.
// x = cos(theta), sp = sin(phi), cp = cos(phi): the direction's trigonometric
// values, formed once per direction by the caller.  The norms come from a
// table and the divisions by l - m and sqrt(2) take three operations
// (div_const's): a square root and the divisions per entry were most of the
// type-1 assembly's instructions.
__device__ __forceinline__ void real_sph_column(const DevTables &T, int lmax, int m, double x, double phi, double sp,
                                                double cp, double *out) {
#define RSH(l, mm) ((l) * (l) + (l) + (mm))
  double sm = 0.0, cm = 1.0;
  for (int k = 1; k <= m; k++) {
    if (0.0 == phi) {
      sm = 0.0;
      cm = 1.0;
    } else if (k == 1) {
      sm = sp;
      cm = cp;
    } else {
      const double ns = sp * cm + cp * sm;
      cm = cp * cm - sp * sm;
      sm = ns;
    }
  }
  const bool pole = 1.0 == x || -1.0 == x;
  double p1 = 0.0, p2 = 0.0;  // P_(l-1)m, P_(l-2)m
  if (pole) {
    p1 = m == 0 ? 1.0 : 0.0;
  } else if (m == 0) {
    p1 = 1.0;
  } else {
    const double s1 = sqrt(1.0 - x * x);
    double sl = s1;
    for (int l = 2; l <= m; l++) sl = sl * s1;
    p1 = sl * T.dfac[2 * m - 1];
  }
  const double *__restrict__ nrm = T.snorm + m;
  const double rt2 = sqrt(2.0), irt2 = 1.0 / rt2;
  for (int l = m; l <= lmax; l++) {
    double P;
    if (l == m) {
      P = p1;
    } else {
      if (pole) {
        P = -1.0 == x ? -p1 : p1;
      } else if (l == m + 1) {
        P = x * (2 * m + 1) * p1;
      } else {
        const double a = x * (2 * l - 1) * p1 - (l + m - 1) * p2, b = l - m, y = T.inv[l - m];
        const double q = a * y;
        P = __builtin_fma(__builtin_fma(-b, q, a), y, q);
      }
      p2 = p1;
      p1 = P;
    }
    const double v = nrm[l * kSphDim] * P;
    if (m == 0) {
      const double q = v * irt2;
      out[RSH(l, 0)] = __builtin_fma(__builtin_fma(-rt2, q, v), irt2, q);
    } else {
      out[RSH(l, -m)] = v * sm;
      out[RSH(l, m)] = v * cm;
    }
  }
#undef RSH
}

// (r, theta, phi) of util.c:74-106
__device__ void sph_coords(double x, double y, double z, double &r, double &theta, double &phi) {
  const double acc = 1.0E-14;
  r = sqrt(x * x + y * y + z * z);
  theta = (r < acc) ? 0.0 : acos(z / r);
  if (fabs(x) < acc) {
    if (fabs(y) < acc) phi = 0.0;
    else if (y < 0.0) phi = 1.5 * M_PI;
    else phi = 0.5 * M_PI;
  } else {
    phi = (x > 0.0) ? atan(y / x) : atan(y / x) + M_PI;
  }
}

__device__ __forceinline__ double dist(const ecp_xyz &a, const ecp_xyz &b) {
  const double x = a.x - b.x, y = a.y - b.y, z = a.z - b.z;
  return sqrt(x * x + y * y + z * z);
}

// ---------------------------------------------------------------------------
// per-centre potential tables

// U tables of one (centre, row, chunk of 128 points): row C.L is the local
// channel U_L (type 1), rows l < L the semi-local channels times r^k,
// k < UK (type 2), zero past the channel's cut-off end[l].  The type-2 rows
// are Ut[vis(n)][l][k]: the type-2 small grid reads all of a point's values
// together, and the points in visit order, so that consecutive reads are
// consecutive in memory (three of four of its integrals read the first
// fifteen points only).
__device__ void utab_rows(const DevTables &T, const DevJob &J, int c, int row, int chunk) {
  const ecp_centre C = J.cent[c];
  if (row > C.L) return;
  const int n = chunk * 128 + (int)threadIdx.x;
  if (n >= SO) return;
  const double r = T.xs[n];
  if (row == C.L) {
    J.UL[C.UL_off + n] = eval_ecp(J, c, C.L, r);
    return;
  }
  const int l = row;
  double P = (n <= C.end[l]) ? eval_ecp(J, c, l, r) : 0.0;
  double *dst = J.Ut + C.Ut_off + (size_t)T.vis[n] * J.US + l * J.UK;
  dst[0] = P;
  for (int k = 1; k < J.UK; k++) {
    P = P * r;
    dst[k] = P;
  }
}

// F[centre][run][shell][vis(n)][lambda] (type2.c:263-303; points in visit
// order like the U rows), one block per non-skipped (centre, shell, run); the whole slab is written (zeros outside
// the window).
template <int LM>
__device__ void ftab_slab(const DevTables &T, const DevJob &J, const ecp_centre &C, int sl, int run,
                          const ecp_window &W) {
  const ecp_shell S = J.shells[C.shell0 + sl];
  const double dAC = dist(J.atoms[C.atom], J.atoms[S.atom]);
  double *slab = J.F + C.F_off + ((size_t)run * C.nsh + sl) * J.FL * SO;
  for (int n = threadIdx.x; n < SO; n += blockDim.x) {
    double acc[LM + 1];
#pragma unroll
    for (int i = 0; i <= LM; i++) acc[i] = 0.0;
    if (n >= W.start && n < W.end) {
      const double r = T.xs[n];
      for (int p = 0; p < S.K; p++) {
        const double zeta = J.pa[S.prim + p];
        double da = J.pd[S.prim + p];
        // derivatives: run n carries a^n (type2.c:286-289)
        for (int k = 0; k < run; k++) da *= zeta;
        double K[LM + 1];
        bessel_k<LM>(T.bessel, 2.0 * zeta * dAC * r, K);
        double e = dAC - r;
        e = exp(-zeta * e * e);
#pragma unroll
        for (int i = 0; i <= LM; i++) acc[i] += da * K[i] * e;
      }
    }
    double *row = slab + (size_t)T.vis[n] * J.FL;
#pragma unroll
    for (int i = 0; i <= LM; i++) row[i] = acc[i];
    for (int i = LM + 1; i < J.FL; i++) row[i] = 0.0;
  }
}

__device__ void ftab_item(const DevTables &T, const DevJob &J, int2 it) {
  const int sl = it.y >> 2, run = it.y & 3;  // (shell, run) packed
  const ecp_centre C = J.cent[it.x];
  const ecp_window W = J.win[C.win_off + sl];
  const int lm = C.L - 1 + J.shells[C.shell0 + sl].l + run;
  switch (lm) {
#define FT(k) \
  case k:     \
    ftab_slab<k>(T, J, C, sl, run, W); \
    break;
    FT(0) FT(1) FT(2) FT(3) FT(4) FT(5) FT(6) FT(7) FT(8) FT(9) FT(10) FT(11) FT(12)
#undef FT
    default:
      break;
  }
}

// per-(centre, atom) angular table ang[lambda][LM(l,m)][C(la,c)]
constexpr int kAngRsph = (ECP_MAX_L + ECP_MAX_LBS) * (ECP_MAX_L + ECP_MAX_LBS);

__device__ void ang_item(const DevTables &T, const DevJob &J, int2 it, double *rsph, double *s_dir, int part,
                         int nparts) {
  const ecp_centre C = J.cent[it.x];
  const int A = C.atom0 + it.y;
  const int lmax_a = J.atom_maxl[A] + J.deriv;
  const int lmax = C.L - 1 + lmax_a;
  if (threadIdx.x == 0) {
    const ecp_xyz a = J.atoms[A], c = J.atoms[C.atom];
    double r, th, ph;
    sph_coords(a.x - c.x, a.y - c.y, a.z - c.z, r, th, ph);
    s_dir[0] = cos(th);
    s_dir[1] = ph;
    s_dir[2] = sin(ph);
    s_dir[3] = cos(ph);
  }
  __syncthreads();
  // one column m of the harmonics per lane
  if ((int)threadIdx.x <= lmax)
    real_sph_column(T, lmax, threadIdx.x, s_dir[0], s_dir[1], s_dir[2], s_dir[3], rsph);
  __syncthreads();
  const int d1 = ECP_DIM_L(T.omLambda), d2 = ECP_DIM_C(T.omAlpha);
  const int nlm = C.L * C.L, nc = ECP_DIM_C(lmax_a);
  double *out = J.ang + C.ang_off + (size_t)it.y * J.ang_lam * J.angL * J.angL * J.ang_c;
  const int total = (lmax + 1) * nlm * nc;
  for (int idx = part * 128 + (int)threadIdx.x; idx < total; idx += 128 * nparts) {
    const int cc = idx % nc;
    const int lm = (idx / nc) % nlm;
    const int lambda = idx / (nc * nlm);
    double v = 0.0;
    for (int mu = 0; mu < 2 * lambda + 1; mu++)
      v += rsph[ECP_IDX_LM(lambda, mu)] * T.omega[((size_t)lm * d1 + ECP_IDX_LM(lambda, mu)) * d2 + cc];
    out[((size_t)lambda * J.angL * J.angL + lm) * J.ang_c + cc] = v;
  }
}

// ---------------------------------------------------------------------------
// type 1: PS93 over the window for all Q[l1][l2] of one primitive pair

__host__ __device__ constexpr int nq_of(int lab) {
  int n = 0;
  for (int l1 = 0; l1 <= lab; l1++) n += l1 / 2 + 1;
  return n;
}

struct T1Unit {
  int trip, pa, pb, qoff;
};

struct T1Geom {
  double za, zb, ca, cb, s, z, zd2, dAC, dBC;
  double P[3];
};

__device__ __forceinline__ void t1_geom(const DevJob &J, const ecp_triplet &tr, int pa, int pb, T1Geom &G) {
  const ecp_centre C = J.cent[tr.centre];
  const ecp_shell Sa = J.shells[tr.sa], Sb = J.shells[tr.sb];
  const ecp_xyz rc = J.atoms[C.atom], ra = J.atoms[Sa.atom], rb = J.atoms[Sb.atom];
  const double rAC[3] = {ra.x - rc.x, ra.y - rc.y, ra.z - rc.z};
  const double rBC[3] = {rb.x - rc.x, rb.y - rc.y, rb.z - rc.z};
  G.dAC = dist(rc, ra);
  G.dBC = dist(rc, rb);
  G.za = J.pa[Sa.prim + pa];
  G.ca = J.pd[Sa.prim + pa];
  G.zb = J.pa[Sb.prim + pb];
  G.cb = J.pd[Sb.prim + pb];
  // derivatives: coefficients times zeta^shift (type1.c:239-246)
  for (int k = 0; k < tr.powa; k++) G.ca *= G.za;
  for (int k = 0; k < tr.powb; k++) G.cb *= G.zb;
  for (int p = 0; p < 3; p++) G.P[p] = 2.0 * (G.za * rAC[p] + G.zb * rBC[p]);
  G.s = sqrt(G.P[0] * G.P[0] + G.P[1] * G.P[1] + G.P[2] * G.P[2]);
  G.zd2 = -G.za * G.dAC * G.dAC - G.zb * G.dBC * G.dBC;
  G.z = -G.za - G.zb;
}

// FM06 linear map of the large grid for zeta_p, P (gc_integrators.c:316-331)
struct Fm06 {
  double i1, i2;
};
__device__ __forceinline__ Fm06 fm06(double zeta_p, double P) {
  const double sigma = 1.0 / sqrt(zeta_p);
  const double t = P - 7.0 * sigma;
  const double rmin = (t > 0.0) ? t : 0.0;
  const double rmax = P + 9.0 * sigma;
  Fm06 m;
  m.i1 = 0.5 * (rmax - rmin);
  m.i2 = 0.5 * (rmax + rmin);
  return m;
}

// The exponents of the three points of PSM92 levels 0 and 1 are all below
// the numerical zero: every integral of the pair is then 0 at level 0 and
// converges with the result 0 at level 1 (0 <= 0 in its test).
template <typename Expo>
__device__ __forceinline__ bool psm92_dead(const DevTables &T, const Fm06 &M, double minExp, Expo expo) {
  if (T.s92.nlevels < 2) return false;
  const double e0 = expo(M.i1 * T.xl[T.s92.centre] + M.i2), e1 = expo(M.i1 * T.xl[T.p92l[0]] + M.i2),
               e2 = expo(M.i1 * T.xl[T.p92r[0]] + M.i2);
  return !(e0 >= minExp) && !(e1 >= minExp) && !(e2 >= minExp);
}

// psm92_dead of a type-1 unit (the large grid of fb1_body)
__device__ __forceinline__ bool t1_fb_dead(const DevTables &T, const T1Geom &G) {
  const double zeta_p = G.za + G.zb;
  const Fm06 M = fm06(zeta_p, (G.za * G.dAC + G.zb * G.dBC) / zeta_p);
  return psm92_dead(T, M, T.lnAcc1, [&](double r) { return (G.z * r + G.s) * r + G.zd2; });
}

// Beyond this exponent exp overflows (from 709.78 on), whatever its last
// bits: the point's integrand, exp(zd2) ... exp(expo) with exp(zd2) = 0 or
// not, is infinite or not a number, and so is every level sum that holds it.
constexpr double kOverflowExpo = 710.0;

// A level sum that is infinite or not a number stays so, and no later level
// passes the PS93 test: the entry has failed on the small grid.
__device__ __forceinline__ bool t1_lost(double I) { return !(fabs(I) < INFINITY); }

// A slot in a queue for every active lane: one atomic per wave
__device__ __forceinline__ int queue_slot(int *count) {
  const unsigned long long m = __ballot(true);
  const int lane = threadIdx.x & 63;
  int base = 0;
  if (lane == __ffsll((long long)m) - 1) base = atomicAdd(count, __popcll(m));
  return __builtin_amdgcn_readfirstlane(base) + __popcll(m & ((1ull << lane) - 1ull));
}

// Results of a finished primitive pair: converged entries, zeros for the
// others, which go to the large-grid fallback queue, unless the fallback
// would end with zeros at once (t1_fb_dead: nine tenths of the failed pairs,
// whose small-grid integrand overflows while the integral vanishes).
template <int NQ>
__device__ __forceinline__ void t1_finish(const DevTables &T, const T1Geom &G, int u, const T1Unit &U,
                                          const double (&p)[NQ], unsigned long long done, double *__restrict__ qout,
                                          unsigned long long *__restrict__ qfail, int *__restrict__ fbq,
                                          int *__restrict__ fbcount) {
  const unsigned long long all = (NQ >= 64) ? ~0ull : ((1ull << NQ) - 1ull);
  double *out = qout + U.qoff;
#pragma unroll
  for (int e = 0; e < NQ; e++) out[e] = (done & (1ull << e)) ? p[e] : 0.0;
  const unsigned long long failed = all & ~done;
  qfail[u] = failed;
  if (failed && !t1_fb_dead(T, G)) fbq[queue_slot(fbcount)] = u;
}

// Type-1 small grid, one lane per primitive pair: levels [0, head); a pair
// still open then saves its integrator state -- p per entry at its results'
// place, q and I in planes of `plane` doubles at state -- and its
// converged-entry mask and is queued
// for the tail (head >= the level count: the whole sequence, no tail).
// Within a level each point pair's sum T = (0 + f(left)) + f(right) is added
// to I in pair order, and the PS93 recurrences and test
// (gc_integrators.c:156-217) follow.  Four fifths of the integrals converge
// (nearly all to 0) by level 4, after 11 points, and hardly any at levels 5
// to 7: the head ends there.
template <int LAB>
__device__ __forceinline__ void type1_body(int bid, const DevTables &T, const DevJob &J,
                                           const T1Unit *__restrict__ units, int nunits, double *__restrict__ qout,
                                           unsigned long long *__restrict__ qfail, int *__restrict__ fbq,
                                           int *__restrict__ fbcount, int head, double *__restrict__ state,
                                           size_t plane, int *__restrict__ tq, int *__restrict__ tcount) {
  constexpr int NQ = nq_of(LAB);
  const int u = bid * 64 + (int)threadIdx.x;
  if (u < nunits) {
    const T1Unit U = units[u];
    const ecp_triplet tr = J.trip[U.trip];
    const ecp_centre Cn = J.cent[tr.centre];
    T1Geom G;
    t1_geom(J, tr, U.pa, U.pb, G);
    const double C0 = G.ca * G.cb * exp(G.zd2);
    const double *__restrict__ UL = J.UL + Cn.UL_off;
    const int gs = tr.gs, ge = tr.ge;
    const double minExp = T.lnAcc1;
    // a point's factors (type1.c:78-88 integrand, tabulated only on [gs, ge)
    // as type1.c:121-130): entry (l1, l2) is w ((C0 r^l1 U) K[l2]) g, all
    // zero where the point contributes nothing
    struct Point {
      double r, w, U, g, K[LAB + 1];
    };
    auto point = [&](int n, bool use) {
      Point Q;
      Q.r = Q.w = Q.U = Q.g = 0.0;
#pragma unroll
      for (int l = 0; l <= LAB; l++) Q.K[l] = 0.0;
      if (!use || n < gs || n >= ge) return Q;
      const double r = T.xs[n];
      const double expo = (G.z * r + G.s) * r;
      if (!(expo >= minExp)) return Q;
      Q.r = r;
      Q.g = exp(expo);
      bessel_k<LAB>(T.bessel, G.s * r, Q.K);
      Q.U = UL[n];
      Q.w = T.ws[n];
      return Q;
    };
    // each(e, (0 + f(left)) + f(right)) for every entry
    auto pair = [&](const Point &a, const Point &b, auto each) {
      double ra = 1.0, rb = 1.0;
      int e = 0;
#pragma unroll
      for (int l1 = 0; l1 <= LAB; l1++) {
        const double ca = (C0 * ra) * a.U, cb = (C0 * rb) * b.U;
#pragma unroll
        for (int l2 = l1; l2 >= 0; l2 -= 2, e++)
          each(e, (0.0 + a.w * ((ca * a.K[l2]) * a.g)) + b.w * ((cb * b.K[l2]) * b.g));
        ra *= a.r;
        rb *= b.r;
        // (many entries: no more of them in flight than registers hold)
        if constexpr (LAB > 8) __builtin_amdgcn_sched_barrier(0);
      }
    };
    double p[NQ], q[NQ], I[NQ];
    unsigned long long done = 0ull, lost = 0ull;
    const unsigned long long all = (NQ >= 64) ? ~0ull : ((1ull << NQ) - 1ull);
    const int lv1 = min(head, T.s93.nlevels);
    pair(point(T.s93.centre, true), point(0, false), [&](int e, double t) { p[e] = t; });
    pair(point(T.s93.first_l, true), point(T.s93.first_r, true), [&](int e, double t) {
      q[e] = t;
      I[e] = p[e] + t;
    });
    for (int lv = 2; lv < lv1; lv++) {
      int cnt = 0;
      for (int k = T.s93.lvl_begin[lv]; k < T.s93.lvl_begin[lv + 1]; k++) {
        const int li = T.p93l[k], ri = T.p93r[k];
        const bool useL = li >= gs, useR = ri <= ge;
        cnt += useL + useR;
        pair(point(li, useL), point(ri, useR), [&](int e, double t) { I[e] += t; });
      }
#pragma unroll
      for (int e = 0; e < NQ; e++) {
        if (done & (1ull << e)) continue;
        double res;
        if (ps93_level(lv, cnt > 0, T.tol, I[e], p[e], q[e], &res)) {
          done |= (1ull << e);
          p[e] = res;
        } else if (t1_lost(I[e])) {
          lost |= (1ull << e);
        }
      }
      if ((done | lost) == all) break;
    }
    if ((done | lost) != all && lv1 < T.s93.nlevels) {
      // an exponent that overflows in the tail's first level: nothing still
      // open can converge, so there is no tail to run
      for (int k = T.s93.lvl_begin[lv1]; k < T.s93.lvl_begin[lv1 + 1]; k++) {
        const int li = T.p93l[k], ri = T.p93r[k];
        const double rl = T.xs[li], rr = T.xs[ri];
        if ((li >= gs && li < ge && (G.z * rl + G.s) * rl > kOverflowExpo) ||
            (ri >= gs && ri < ge && (G.z * rr + G.s) * rr > kOverflowExpo))
          lost = all;
      }
    }
    if ((done | lost) != all && lv1 < T.s93.nlevels) {
#pragma unroll
      for (int e = 0; e < NQ; e++) {
        qout[U.qoff + e] = p[e];
        state[U.qoff + e] = q[e];
        state[plane + U.qoff + e] = I[e];
      }
      qfail[u] = done;
      tq[queue_slot(tcount)] = u;
      return;
    }
    t1_finish<NQ>(T, G, u, U, p, done, qout, qfail, fbq, fbcount);
  }
}

// two waves per SIMD up to class 6 (256 registers), one above
template <int LAB>
__global__ __launch_bounds__(64, LAB <= 6 ? 2 : 1) void k_type1(DevTables T, DevJob J,
                                                              const T1Unit *__restrict__ units, int nunits,
                                                              double *__restrict__ qout,
                                                              unsigned long long *__restrict__ qfail,
                                                              int *__restrict__ fbq, int *__restrict__ fbcount,
                                                              int head, double *__restrict__ state, size_t plane,
                                                              int *__restrict__ tq, int *__restrict__ tcount) {
  type1_body<LAB>(blockIdx.x, T, J, units, nunits, qout, qfail, fbq, fbcount, head, state, plane, tq, tcount);
}

// f + a[0] b[0] + a[sa] b[sb] + ... (n terms), accumulated in order; the
// reads of up to B terms are issued before their products are added
template <int B>
__device__ __forceinline__ double dot_in_order(double f, const double *a, int sa, const double *b, int sb, int n) {
  int m = 0;
  for (; m + B <= n; m += B) {
    double x[B], y[B];
#pragma unroll
    for (int i = 0; i < B; i++) {
      x[i] = a[(m + i) * sa];
      y[i] = b[(m + i) * sb];
    }
#pragma unroll
    for (int i = 0; i < B; i++) f += x[i] * y[i];
  }
  for (; m < n; m++) f += a[m * sa] * b[m * sb];
  return f;
}

// Wave-level helpers (blocks of exactly one 64-lane wave).
__device__ __forceinline__ bool wave_any(bool p) { return __ballot(p) != 0ull; }

// I + v[0] + v[1] + ... + v[n - 1], added left to right (the order of a
// lane-serial integrator); the reads (LDS or global) are issued eight
// (then four) at a time so that one wait covers several of them
__device__ __forceinline__ double sum_in_order(double I, const double *v, int n) {
  int k = 0;
  for (; k + 8 <= n; k += 8) {
    double x[8];
#pragma unroll
    for (int i = 0; i < 8; i++) x[i] = v[k + i];
#pragma unroll
    for (int i = 0; i < 8; i++) I += x[i];
  }
  if (k + 4 <= n) {
    double x[4];
#pragma unroll
    for (int i = 0; i < 4; i++) x[i] = v[k + i];
#pragma unroll
    for (int i = 0; i < 4; i++) I += x[i];
    k += 4;
  }
  for (; k < n; k++) I += v[k];
  return I;
}

// Point of slot `lane` in a round of PSM92 point pairs [c0, c1): pair c0 +
// lane / 2, left in even lanes, right in odd ones; in the first round (the
// pairs of levels 1 to 5, 31 of them) the centre is in lane 62.  -1: none.
__device__ __forceinline__ int psm92_point(const DevTables &T, int c0, int c1, int lane, bool first) {
  const int k = c0 + (lane >> 1);
  if (first && lane == 62) return T.s92.centre;
  if (k >= c1) return -1;
  return (lane & 1) ? T.p92r[k] : T.p92l[k];
}

// PSM92 levels [0, psm92_first) in the first round: centre and 31 pairs
__device__ __forceinline__ int psm92_first(const DevTables &T) { return min(6, T.s92.nlevels); }

// v(left) + v(right) of the wave's point pairs, in both lanes of each pair
__device__ __forceinline__ double pair_sum(double v) {
  // quad_perm [1, 0, 3, 2]: the neighbour's value
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0xB1, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0xB1, 0xF, 0xF, true);
  return v + __hiloint2double(hi, lo);
}

// An integral's PSM92 state (gc_integrators.c:38-86)
struct Psm92 {
  double I, p, q;
  __device__ __forceinline__ void step() {
    q = 2 * p;
    p = 2 * I;
  }
  // after a level: converged? (*res: the integral)
  __device__ __forceinline__ bool test(const DevTables &T, int l, double *res) const {
    const double N = T.s92.lvl_n[l];
    const double ee = I - p;
    if (!(16 * ee * ee <= 3 * N * fabs(I - q) * T.tol)) return false;
    *res = 16 * I / (3 * N);
    return true;
  }
  // the first round: pair sums v[0 .. 30] of levels 1 to 5, the centre v[31]
  __device__ __forceinline__ bool first_round(const DevTables &T, const double *v, double *res) {
    I = p = v[31];
    q = 0.0;
    const int l1 = psm92_first(T);
    for (int l = 1; l < l1; l++) {
      step();
      I = sum_in_order(I, v + T.s92.lvl_begin[l], T.s92.lvl_begin[l + 1] - T.s92.lvl_begin[l]);
      if (test(T, l, res)) return true;
    }
    return false;
  }
};

// type-1 fallback (type1.c:205-252) of one primitive pair with failed Q
// entries (mask), by one wave: results to out.  The wave's lanes evaluate the points of a round -- 31 point
// pairs and the centre (levels 0 to 5) together, then 32 pairs at a time --
// and form each open entry's pair sums (0 + f(left)) + f(right), a pair per
// two lanes, into LDS; lane e adds those of entry e in the integrator's
// order and applies the PSM92 test after each level.  (Pairs whose points
// of levels 0 and 1 are all numerically zero do not come here: t1_fb_dead.)
// The reference's screening break (type1.c:222-225: no points from the first
// one beyond both centres whose exponent is below the cut-off) needs no
// search: beyond both centres the exponent only decreases, so every point it
// drops is below the cut-off and contributes 0 here by its own test.
constexpr int kFbTS = 33;  // LDS stride of an entry's pair sums (at most 32 per round)

template <int LAB>
__device__ __forceinline__ void fb1_unit(const DevTables &T, const DevJob &J, const T1Unit &U, const ecp_triplet &tr,
                                         int L, const T1Geom &G, unsigned long long mask, double *__restrict__ out,
                                         unsigned char *__restrict__ status, double *s_t) {
  constexpr int NQ = nq_of(LAB);
  const int lane = threadIdx.x;
  const double Cc = G.ca * G.cb;
  const double zeta_p = G.za + G.zb;
  const Fm06 M = fm06(zeta_p, (G.za * G.dAC + G.zb * G.dBC) / zeta_p);
  const double minExp = T.lnAcc1;
  auto expo_of = [&](double r) { return (G.z * r + G.s) * r + G.zd2; };
  bool open = lane < NQ && ((mask >> lane) & 1ull);
  Psm92 S{0.0, 0.0, 0.0};
  double res = 0.0;
  // rounds of point pairs [c0, c1): levels 0 to 5 first, then 32 pairs of
  // level lv at a time
  int lv = psm92_first(T), c0 = 0, c1 = T.s92.lvl_begin[lv];
  for (;;) {
    const bool first = c0 == 0;
    const unsigned long long om = __ballot(open);
    const int n = psm92_point(T, c0, c1, lane, first);
    double w = 0.0, uu = 0.0, g = 0.0, r = 0.0;
    double K[LAB + 1];
#pragma unroll
    for (int l = 0; l <= LAB; l++) K[l] = 0.0;
    if (n >= 0) {
      r = M.i1 * T.xl[n] + M.i2;
      const double expo = expo_of(r);
      if (expo >= minExp) {
        g = exp(expo);
        bessel_k<LAB>(T.bessel, G.s * r, K);
        uu = eval_ecp(J, tr.centre, L, r);
        w = T.wl[n] * M.i1;
      }
    }
    // the open entries' pair sums
    double rn = 1.0;
    int e = 0;
#pragma unroll
    for (int l1 = 0; l1 <= LAB; l1++) {
      const double a = (Cc * rn) * uu;
#pragma unroll
      for (int l2 = l1; l2 >= 0; l2 -= 2, e++)
        if ((om >> e) & 1ull) {
          const double t = pair_sum(w * ((a * K[l2]) * g));
          if (!(lane & 1)) s_t[e * kFbTS + (lane >> 1)] = t;
        }
      rn = r * rn;
    }
    __syncthreads();
    const bool level_end = !first && c1 == T.s92.lvl_begin[lv + 1];
    if (open) {
      bool done;
      if (first) {
        done = S.first_round(T, s_t + lane * kFbTS, &res);
      } else {
        S.I = sum_in_order(S.I, s_t + lane * kFbTS, c1 - c0);
        done = level_end && S.test(T, lv, &res);
      }
      if (done) {
        out[lane] = res;
        open = false;
      }
    }
    __syncthreads();
    lv += level_end;
    if (lv >= T.s92.nlevels || !wave_any(open)) break;
    if (first || level_end) S.step();
    c0 = c1;
    c1 = min(c0 + 32, T.s92.lvl_begin[lv + 1]);
  }
  if (open) status[2 * U.trip] = 1;
}

// Tail: one wave per primitive pair left open by the head, levels [head,
// nlevels), in rounds of levels (at most 64 point pairs each; levels 5 to 11
// have 58, 12 and 13, and 14, 64).  Lane k looks at the k-th pair's two
// points; those inside the window whose exponent is above the cut-off -- a
// third of them, a contiguous range of r -- are dealt to the lanes densely,
// which evaluate them for every Q entry; the pair sums
// T_k = (0 + f(left)) + f(right) form in LDS, and lane e then adds each
// level's T_k to its entry's I in pair order and applies the PS93 test, so
// the arithmetic is that of the lane-serial integrator.  Where a point's
// exponent overflows, no entry can converge from its level on: nothing past
// it is evaluated.  The wave then runs the large-grid fallback of the
// entries that failed; the pairs that failed in the head (fbq) follow.
constexpr int kTS = 65;  // LDS stride of the per-entry pair sums (bank spread)

template <int LAB>
__device__ __forceinline__ void t1tail_body(int bid, int nb, const DevTables &T, const DevJob &J,
                                            const T1Unit *__restrict__ units, double *__restrict__ qout,
                                            unsigned long long *__restrict__ qfail, const int *__restrict__ fbq,
                                            const int *__restrict__ fbcount, int head,
                                            const double *__restrict__ state, size_t plane,
                                            const int *__restrict__ tq, const int *__restrict__ tcount,
                                            unsigned char *__restrict__ status, double *s_T, int *s_pt) {
  constexpr int NQ = nq_of(LAB);
  static_assert(NQ <= 64, "one lane per Q entry");
  const int ntail = cload(tcount), count = ntail + cload(fbcount);
  const int lane = threadIdx.x;
  for (int it = bid; it < count; it += nb) {
    const bool tail = it < ntail;
    const int u = cload(tail ? tq + it : fbq + (it - ntail));
    const T1Unit U = cload(units + u);
    const ecp_triplet tr = J.trip[U.trip];
    const ecp_centre Cn = J.cent[tr.centre];
    T1Geom G;
    t1_geom(J, tr, U.pa, U.pb, G);
    const double C0 = G.ca * G.cb * exp(G.zd2);
    const double *__restrict__ UL = J.UL + Cn.UL_off;
    const int gs = tr.gs, ge = tr.ge;
    const double minExp = T.lnAcc1;
    const unsigned long long done0 = qfail[u];
    double p = 0.0, q = 0.0, I = 0.0;
    bool mydone = true, lost = false;
    if (tail && lane < NQ) {
      p = qout[U.qoff + lane];
      q = state[U.qoff + lane];
      I = state[plane + U.qoff + lane];
      mydone = (done0 >> lane) & 1ull;
    }
    int lv = tail ? head : T.s93.nlevels;
    while (lv < T.s93.nlevels) {
      const int b0 = T.s93.lvl_begin[lv];
      int l1 = lv + 1;
      while (l1 < T.s93.nlevels && T.s93.lvl_begin[l1 + 1] - b0 <= 64) l1++;
      const int tot = T.s93.lvl_begin[l1] - b0;
      // the lane's pair: which of its points count, contribute, overflow
      bool in = false, liveL = false, liveR = false, over = false;
      if (lane < tot) {
        const int li = T.p93l[b0 + lane], ri = T.p93r[b0 + lane];
        const double rl = T.xs[li], rr = T.xs[ri];
        const double el = (G.z * rl + G.s) * rl, er = (G.z * rr + G.s) * rr;
        in = li >= gs || ri <= ge;
        liveL = li >= gs && li < ge && el >= minExp;
        liveR = ri >= gs && ri < ge && er >= minExp;
        over = (liveL && el > kOverflowExpo) || (liveR && er > kOverflowExpo);
      }
      // levels [lv, ls) are evaluated: those before the first overflow
      const unsigned long long ovm = __ballot(over);
      int ls = l1;
      if (ovm) {
        const int k = __ffsll((long long)ovm) - 1;
        ls = lv;
        while (T.s93.lvl_begin[ls + 1] - b0 <= k) ls++;
      }
      if (ls > lv) {
        const int ne = T.s93.lvl_begin[ls] - b0;
        const unsigned long long cmask = __ballot(in);
        const unsigned long long mL = __ballot(liveL && lane < ne), mR = __ballot(liveR && lane < ne);
        const int nL = __popcll(mL), n = nL + __popcll(mR);
        const unsigned long long below = (1ull << lane) - 1ull;
        if ((mL >> lane) & 1ull) s_pt[__popcll(mL & below)] = lane;
        if ((mR >> lane) & 1ull) s_pt[nL + __popcll(mR & below)] = lane | 64;
        if (lane < ne)
#pragma unroll
          for (int e = 0; e < NQ; e++) s_T[e * kTS + lane] = 0.0;
        __syncthreads();
        // live points, the left ones first (at most 64 of them)
        for (int b = 0; b < n; b += 64) {
          const int j = b + lane;
          int k = 0;
          double t[NQ];
          if (j < n) {
            k = s_pt[j] & 63;
            const int i = j < nL ? T.p93l[b0 + k] : T.p93r[b0 + k];
            const double r = T.xs[i];
            const double g = exp((G.z * r + G.s) * r);
            double K[LAB + 1];
            bessel_k<LAB>(T.bessel, G.s * r, K);
            const double Un = UL[i], wn = T.ws[i];
            double rn = 1.0;
            int e = 0;
#pragma unroll
            for (int a1 = 0; a1 <= LAB; a1++) {
              const double a = (C0 * rn) * Un;
#pragma unroll
              for (int a2 = a1; a2 >= 0; a2 -= 2, e++) t[e] = wn * ((a * K[a2]) * g);
              rn *= r;
            }
          }
          if (j < nL)
#pragma unroll
            for (int e = 0; e < NQ; e++) s_T[e * kTS + k] = 0.0 + t[e];
          __syncthreads();
          if (j >= nL && j < n)
#pragma unroll
            for (int e = 0; e < NQ; e++) s_T[e * kTS + k] += t[e];
          __syncthreads();
        }
        bool stop = false;
        for (int l = lv; l < ls; l++) {
          const int o = T.s93.lvl_begin[l] - b0, np = T.s93.lvl_begin[l + 1] - T.s93.lvl_begin[l];
          const unsigned long long lm = (np >= 64) ? ~0ull : (((1ull << np) - 1ull) << o);
          const bool any = (cmask & lm) != 0ull;
          // the level's sums from its first pair with a live point on (the
          // ones before it are 0)
          const unsigned long long lp = (mL | mR) & lm;
          if (lp && lane < NQ) {
            const int k = __ffsll((long long)lp) - 1;
            I = sum_in_order(I, s_T + lane * kTS + k, o + np - k);
          }
          if (!mydone) {
            double res;
            if (ps93_level(l, any, T.tol, I, p, q, &res)) {
              mydone = true;
              p = res;
            } else {
              lost = t1_lost(I);
            }
          }
          if (!wave_any(!mydone && !lost)) {
            stop = true;
            break;
          }
        }
        __syncthreads();
        if (stop) break;
      }
      if (ls < l1) break;
      lv = l1;
    }
    unsigned long long failed = done0;  // of a pair that failed in the head
    if (tail) {
      if (lane < NQ) qout[U.qoff + lane] = mydone ? p : 0.0;
      failed = __ballot(lane < NQ && !mydone);
      if (lane == 0) qfail[u] = failed;
      if (!failed || t1_fb_dead(T, G)) continue;
    }
    fb1_unit<LAB>(T, J, U, tr, Cn.L, G, failed, qout + U.qoff, status, s_T);
  }
}

template <int LAB>
__global__ __launch_bounds__(64) void k_t1tail(DevTables T, DevJob J, const T1Unit *__restrict__ units,
                                               double *__restrict__ qout, unsigned long long *__restrict__ qfail,
                                               const int *__restrict__ fbq, const int *__restrict__ fbcount, int head,
                                               const double *__restrict__ state, size_t plane,
                                               const int *__restrict__ tq, const int *__restrict__ tcount,
                                               unsigned char *__restrict__ status) {
  __shared__ double s_T[nq_of(LAB) * kTS];
  __shared__ int s_pt[128];
  t1tail_body<LAB>(blockIdx.x, gridDim.x, T, J, units, qout, qfail, fbq, fbcount, head, state, plane, tq, tcount,
                   status, s_T, s_pt);
}

// ---------------------------------------------------------------------------
// type 2: the small grid, a lane group per triplet; then the large grid

// first entry of channel l in the T entries of shells la, lb
__device__ __forceinline__ int t2_off(const DevTables &T, int la, int lb, int l) {
  return T.toff[(la * (ECP_MAX_LBS + 1) + lb) * (ECP_MAX_L + 1) + l];
}

struct T2Args {
  double *Tout;
  unsigned char *tfail;
  int *tnfail, *flist;  // per triplet: number of failed entries, listed at flist[teoff ...]
  int *fbq, *fbcount;   // per fallback class, the triplets with failed entries (qstride apart)
  int qstride;
  const unsigned char *tcls2;  // per triplet: its fallback class max(la, lb) + L - 1
};

// integrator state of a T entry
struct T2State {
  double p, q, I, res;
  bool done;
  __device__ __forceinline__ void level(const DevTables &T, int lv, bool any) {
    if (!done) done = ps93_level(lv, any, T.tol, I, p, q, &res);
  }
};

// Type-2 small grid: a lane group of 64 / G lanes per triplet, all channels.
// Every entry's integrand is a product of one value each of the triplet's
// rows at a point -- F_a (la + L of them), F_b, and r^k U_l (L (la + lb +
// 1)), 12 to 42 doubles up to f shells and projectors -- which the group reads
// once into LDS, one value per lane; the lanes then own the entries (R each
// per pass) and form the integrands from LDS.  Read per entry instead, the
// kernel was bound by the L1 cache's rate of accesses (1.9 G on 256 uneven
// molecules, 3.1 ms at one per clock and CU, of 3.3 ms).
// Levels 0 to 5, fifteen points read together, decide nearly all entries of
// most triplets; where entries stay open, the levels up to 14 follow in
// steps of NP = 4 point pairs (each ends its level or lies inside it; in
// steps of 8, the first takes levels 6 and 7, of 4 pairs each), the next
// step's values read ahead.  Point pairs
// are added in order, with the PS93 test at each level's end.  Points outside
// the pair's window need no test: F_a or F_b is 0 there; a step with all of
// its points outside is passed over.
constexpr int kT2Head = 6;      // levels of the first part
constexpr int kT2HeadPairs = 6; // their point pairs from level 2 on
constexpr int kT2HeadPts = 3 + 2 * kT2HeadPairs;
template <bool SMALL>
struct T2Shape {
  static constexpr int kStep = SMALL ? 8 : 4;  // point pairs of a later step
  static constexpr int kOwn = SMALL ? 1 : 2;   // entries a lane owns
};

// Workgroups go to the eight XCDs, each with its own L2, in turn: workgroup b
// of n takes the item that leaves runs of 64 consecutive items -- the
// triplets of one centre, which share its tables -- to one XCD.  (Items in
// turn, every XCD read every centre's F rows: 25 GB from HBM on 256 uneven
// molecules where the tables hold 1.8 GB, the type-2 small grid at 7.7 TB/s.)
__device__ __forceinline__ int xcd_item(int b, int n) {
  constexpr int S = 64, N = 8 * S;
  if (b >= n / N * N) return b;
  const int r = b % N;
  return b - r + (r % 8) * S + r / 8;
}

// doubles of LDS of a wave; CH: 16-byte chunks of a point's values
template <bool SMALL>
__host__ __device__ constexpr int t2_lds(int G, int CH) {
  constexpr int step = 2 * T2Shape<SMALL>::kStep;
  return G * 2 * CH * (step > kT2HeadPts ? step : kT2HeadPts);
}

typedef double dpair __attribute__((ext_vector_type(2)));

// LP: lanes that read a point together, two values (16 bytes) each; the F and
// U rows have even lengths, so that every chunk is aligned
template <int G, int CH, bool SMALL>
__device__ __forceinline__ void type2_body(int bid, const DevTables &T, const DevJob &J, const T2Args &A,
                                           const int *__restrict__ tlist, int ntl, int slice, int nslices,
                                           double *s_all) {
  constexpr int NP = T2Shape<SMALL>::kStep, R = T2Shape<SMALL>::kOwn;
  constexpr int W = 64 / G, LP = G == 1 ? 32 : 16, PT = W / LP, X = (CH + LP - 1) / LP, ROW = 2 * CH;
  const int grp = (int)threadIdx.x / W, lid = (int)threadIdx.x % W;
  const int pt = lid / LP, pl = lid % LP;  // point of a read, lane of the point
  double *s_v = s_all + grp * t2_lds<SMALL>(1, CH);
  const int ti = bid * G + grp;
  const bool active = ti < ntl;
  const int t = cload(tlist + (active ? ti : 0));
  const ecp_triplet tr = J.trip[t];
  const ecp_centre C = J.cent[tr.centre];
  const int L = C.L, la = tr.la, lb = tr.lb, na = la + L, nb = lb + L, nu = la + lb + 1;
  const int ca = (na + 1) >> 1, cb = (nb + 1) >> 1, cu = (nu + 1) >> 1;  // chunks of F_a, F_b, a channel's U
  const int nch = ca + cb + L * cu, gs = tr.gs, ge = tr.ge;
  const int t0 = t2_off(T, la, lb, 0), ne = active ? t2_off(T, la, lb, L) - t0 : 0, eoff = J.teoff[t];
  // this lane's chunks of a point: where they are, and their point stride
  const double *src[X];
  int st[X];
#pragma unroll
  for (int x = 0; x < X; x++) {
    const int v = pl + x * LP;
    if (v < ca + cb) {
      const bool b = v >= ca;
      const int run = b ? tr.powb : tr.powa, sh = (b ? tr.sb : tr.sa) - C.shell0;
      src[x] = J.F + C.F_off + ((size_t)run * C.nsh + sh) * J.FL * SO + 2 * (b ? v - ca : v);
      st[x] = J.FL;
    } else {
      const int y = v - ca - cb, l = (int)(((float)y + 0.5f) / (float)cu);
      src[x] = J.Ut + C.Ut_off + l * J.UK + 2 * (y - l * cu);
      st[x] = J.US;
    }
    if (v >= nch) {  // none: any readable place
      src[x] = J.Ut + C.Ut_off;
      st[x] = 0;
    }
  }
  for (int e0 = slice * W * R; __ballot(e0 < ne) != 0ull; e0 += nslices * W * R) {
    // LDS offsets of the entries' values, and their states
    int oa[R], ob[R], ou[R];
    T2State S[R];
#pragma unroll
    for (int i = 0; i < R; i++) {
      const int e = e0 + i * W + lid;
      S[i] = T2State{0.0, 0.0, 0.0, 0.0, e >= ne};
      const int code = e < ne ? T.tmpl[t0 + e] : 0;
      oa[i] = code & 0xff;
      ob[i] = 2 * ca + ((code >> 8) & 0xff);
      ou[i] = 2 * (ca + cb) + (code >> 24) * 2 * cu + ((code >> 16) & 0xff);
    }
    // value of point slot P of entry i, weighted
    auto f = [&](int i, int P, double w) {
      const double *v = s_v + P * ROW;
      return w * ((v[oa[i]] * v[ob[i]]) * v[ou[i]]);
    };
    Ps93Pair hp[kT2HeadPairs];
#pragma unroll
    for (int k = 0; k < kT2HeadPairs; k++) hp[k] = T.v93[k];
    {
      // rows in visit order: the centre, the first pair, the pairs hp
      constexpr int NI = (kT2HeadPts + PT - 1) / PT;
      dpair v[X][NI];
#pragma unroll
      for (int P = 0; P < NI; P++) {
        const int n = min(P * PT + pt, kT2HeadPts - 1);
#pragma unroll
        for (int x = 0; x < X; x++) v[x][P] = *(const dpair *)(src[x] + n * st[x]);
      }
#pragma unroll
      for (int P = 0; P < NI; P++)
#pragma unroll
        for (int x = 0; x < X; x++)
          if (pl + x * LP < CH && P * PT + pt < kT2HeadPts)
            *(dpair *)(s_v + (P * PT + pt) * ROW + 2 * (pl + x * LP)) = v[x][P];
    }
    __syncthreads();
    {
      const double w0 = T.ws[T.s93.centre], w1 = T.ws[T.s93.first_l], w2 = T.ws[T.s93.first_r];
#pragma unroll
      for (int i = 0; i < R; i++) {
        S[i].p = f(i, 0, w0);
        S[i].q = f(i, 1, w1) + f(i, 2, w2);
        S[i].I = S[i].p + S[i].q;
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < kT2HeadPairs; k++) {
        // (a few pairs' reads in flight at a time: registers)
        if (k & 1) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < R; i++) {
          S[i].I += (0.0 + f(i, 3 + 2 * k, hp[k].wl)) + f(i, 4 + 2 * k, hp[k].wr);
          if (hp[k].ends) S[i].level(T, hp[k].ends, hp[k].li >= gs || hp[k].ri <= ge);
        }
      }
    }
    __syncthreads();
    // the levels left, for the groups with an entry still open
    const int np = T.s93.npairs;
    int c0 = T.s93.lvl_begin[kT2Head];
    auto group_open = [&]() {
      bool o = false;
#pragma unroll
      for (int i = 0; i < R; i++) o = o || !S[i].done;
      const unsigned long long m = __ballot(o);
      return G == 1 ? m != 0ull : ((m >> (grp * W)) & ((1ull << (W & 63)) - 1ull)) != 0ull;
    };
    if (wave_any(group_open())) {
      // a step's pairs (read ahead with their values) and the values
      Ps93Pair pr[NP];
      constexpr int NI = 2 * NP / PT;
      dpair v[X][NI];
      auto read = [&](int b) {
#pragma unroll
        for (int j = 0; j < NP; j++) pr[j] = T.v93[b + j];
        // (opaque to the loop optimiser, which would keep an address per
        // read in registers, and spill)
        int n0 = 3 + 2 * b;
        asm volatile("" : "+s"(n0));
#pragma unroll
        for (int x = 0; x < X; x++) {
          const double *q = src[x] + (n0 + pt) * st[x];
          const int step = PT * st[x];
#pragma unroll
          for (int P = 0; P < NI; P++, q += step) v[x][P] = *(const dpair *)q;
        }
      };
      // the step from b on has a point in a group's window
      auto inside = [&](int b) {
        bool in = false;
#pragma unroll
        for (int j = 3; j < NP; j += 4) {
          const Ps93Pair z = T.v93[b + j];
          in = in || z.li >= gs || z.ri <= ge;
        }
        return wave_any(in);
      };
      bool on = inside(c0);
      if (on) read(c0);
      for (;;) {
        Ps93Pair cur[NP];
        const bool now = on;
        if (now) {
#pragma unroll
          for (int P = 0; P < NI; P++)
#pragma unroll
            for (int x = 0; x < X; x++)
              if (pl + x * LP < CH) *(dpair *)(s_v + (P * PT + pt) * ROW + 2 * (pl + x * LP)) = v[x][P];
#pragma unroll
          for (int j = 0; j < NP; j++) cur[j] = pr[j];
        }
        __syncthreads();
        const int b = c0;
        c0 += NP;
        const bool last = c0 >= np;
        on = !last && inside(c0);
        if (on) read(c0);
        if (now) {
#pragma unroll
          for (int i = 0; i < R; i++) {
            if (!wave_any(!S[i].done)) continue;
#pragma unroll
            for (int j0 = 0; j0 < NP; j0 += 4) {
              double t[4];
#pragma unroll
              for (int j = 0; j < 4; j++)
                t[j] = (0.0 + f(i, 2 * (j0 + j), cur[j0 + j].wl)) + f(i, 2 * (j0 + j) + 1, cur[j0 + j].wr);
#pragma unroll
              for (int j = 0; j < 4; j++) S[i].I += t[j];
              // level 6 ends with the first four pairs of its step
              const Ps93Pair &z = cur[j0 + 3];
              if (z.ends) S[i].level(T, z.ends, z.li >= gs || z.ri <= ge);
              __builtin_amdgcn_sched_barrier(0);
            }
          }
        } else {
#pragma unroll
          for (int j = 3; j < NP; j += 4) {
            const Ps93Pair z = T.v93[b + j];
            if (z.ends)
#pragma unroll
              for (int i = 0; i < R; i++) S[i].level(T, z.ends, false);
          }
        }
        __syncthreads();
        if (last || !wave_any(group_open())) break;
      }
    }
    // results; the pass's failed entries are listed together, and the first
    // to list any puts the triplet on its fallback queue
    bool fail[R];
    int below[R], nfail = 0;
#pragma unroll
    for (int i = 0; i < R; i++) {
      const int e = e0 + i * W + lid;
      fail[i] = e < ne && !S[i].done;
      if (e < ne) {
        A.Tout[eoff + e] = S[i].res;
        A.tfail[eoff + e] = fail[i];
      }
      unsigned long long m = __ballot(fail[i]);
      if (G > 1) m = (m >> (grp * W)) & ((1ull << (W & 63)) - 1ull);
      below[i] = nfail + __popcll(m & ((1ull << lid) - 1ull));
      nfail += __popcll(m);
    }
    if (wave_any(nfail != 0)) {
      int base = 0;
      if (lid == 0 && nfail) {
        base = atomicAdd(&A.tnfail[t], nfail);
        if (base == 0) {
          const int c = A.tcls2[t];
          A.fbq[(size_t)c * A.qstride + atomicAdd(&A.fbcount[c], 1)] = t;
        }
      }
      base = __shfl(base, grp * W);
#pragma unroll
      for (int i = 0; i < R; i++)
        if (fail[i]) A.flist[eoff + base + below[i]] = e0 + i * W + lid;
    }
  }
}

// The triplets of classes above kT2PackLab (tlist[m .. nt)), one per wave,
// then those up to it (tlist[0 .. m)), kT2Pack to a wave.  CH, CHP: 16-byte
// chunks of a point's values, of a triplet of either kind.
// A triplet of many entries takes one wave's passes in turn, kT2Pass entries
// each; jobs too small to fill the chip (kT2Fill waves, four times what it
// holds) split the passes over `nslices` waves per triplet.  A pass stages
// its points' rows in either case, so that the split adds no work: 17 atoms
// 231 -> 197 us an evaluation, 50 atoms 380 -> 342 us (at a quarter of
// kT2Fill: no gain on the latter), g shells shifted to h under L = 6 on
// three atoms 1331 -> 582 us (with the wide assembly below).
constexpr int kT2Pack = 2, kT2PackLab = 2, kT2Fill = 16384, kT2Pass = 128;

template <int CH, int CHP>
__global__ __launch_bounds__(64, CH <= 24 ? 4 : 3) void k_type2(DevTables T, DevJob J, T2Args A, const int *__restrict__ tlist,
                                                int m, int nslices) {
  __shared__ __align__(16) double s_v[t2_lds<false>(1, CH) > t2_lds<false>(kT2Pack, CHP) ? t2_lds<false>(1, CH)
                                                                                        : t2_lds<false>(kT2Pack, CHP)];
  const int n = J.ntrip - m, np = (m + kT2Pack - 1) / kT2Pack, b = blockIdx.x;
  if (b < n * nslices)
    type2_body<1, CH, false>(xcd_item(b % n, n), T, J, A, tlist + m, n, b / n, nslices, s_v);
  else
    type2_body<kT2Pack, CHP, false>(xcd_item(b - n * nslices, np), T, J, A, tlist, m, 0, 1, s_v);
}

// Jobs of up to kT2Small triplets, whose time is the chain of one wave's
// steps: an entry per lane, 64 a pass, every triplet in waves of its own, and
// steps of eight point pairs (half as many).  Alone, on a tiny molecule, 49 ->
// 29 us; replays of it 129 -> 109 us, 17 atoms (1167 triplets) 156 -> 144 us.
// From 50 atoms (8001 triplets) on the general shape is the better one, 306
// against 313 us, 24 674 triplets of a gradient 775 against 884 us.
constexpr int kT2Small = 4096;

template <int CH>
__global__ __launch_bounds__(64, 2) void k_type2_small(DevTables T, DevJob J, T2Args A, const int *__restrict__ tlist,
                                                       int nslices) {
  __shared__ __align__(16) double s_v[t2_lds<true>(1, CH)];
  const int n = J.ntrip;
  type2_body<1, CH, true>(blockIdx.x % n, T, J, A, tlist, n, blockIdx.x / n, nslices, s_v);
}

// type-2 fallback (calcT_FM06, type2.c:417-528): one wave per (triplet with
// failed T entries, slot).  The FM06-mapped points depend on the primitive
// pair only, so for each of its pairs the wave evaluates a round's points
// once (31 point pairs and the centre, levels 0 to 5, then 32 pairs at a
// time; a point per lane: exponential, weight and power of r in registers,
// K_a, K_b and U_l of the channels with failed entries in the lane's own LDS
// column) for all failed entries of all the triplet's channels.  The wave
// takes the entries one after another: every lane forms the entry's
// integrand at its point, two neighbouring lanes the pair sum, kFb2Chunk
// entries at a time into LDS; then each entry's owner lane adds its own in
// the integrator's order and tests after each level.
// The lanes own points, not entries, so a triplet with few failed entries
// keeps the wave as busy as one with many.  The primitive pairs whose points
// of levels 0 and 1 are all numerically zero (half of them) are found first,
// a pair per lane, and get their zeros without a wave's work; slot s of
// `nslot` takes every nslot-th of the others.
// Results per (entry, pair) go to fbT and are summed over pairs, in pair
// order, by the assembly.  No search for the screening break
// (type2.c:479-481), as in the type-1 fallback.
constexpr int kFb2Chunk = 16;  // entries whose pair sums are in LDS together
constexpr int kFb2Cnt = 52;  // fbc[kFb2Cnt + c]: triplets queued for the type-2 fallback, class c
constexpr int kFbcSlots = 80;  // queue counters per job
static_assert(ECP_MAX_LAB < 16 && kFb2Cnt + kMaxLMB < kFbcSlots, "queue counter slots");

// OWN: entries owned per lane and pass
template <int LMB, int OWN>
__device__ __forceinline__ void fb2_body(int bid, int nb, const DevTables &T, const DevJob &J,
                                         const int *__restrict__ fbq, const int *__restrict__ fbcount,
                                         double *__restrict__ fbT, unsigned char *__restrict__ status,
                                         const int *__restrict__ tnfail, const int *__restrict__ flist,
                                         int nslot, int nsplit, int share, double *s_cu,
                                         double *s_rn, double *s_ka, double *s_kb, double *s_t) {
  const int lane = threadIdx.x;
  const int count = cload(fbcount);
  // items (split, slot, triplet): split k takes the k-th share of the entries
  const long per_split = (long)count * nslot;
  const long total = per_split * nsplit;
  for (long it = bid; it < total; it += nb) {
    const int split = (int)(it / per_split);
    const int rest = (int)(it - split * per_split);
    const int slot = rest / count;
    const int t = cload(fbq + (rest - slot * count));
    const ecp_triplet tr = J.trip[t];
    const ecp_shell Sa = J.shells[tr.sa], Sb = J.shells[tr.sb];
    const int npairs = Sa.K * Sb.K;
    const ecp_centre Cn = J.cent[tr.centre];
    // the triplet's failed entries, and the channels they are of
    const int L = Cn.L, nfail = cload(tnfail + t), eoff = J.teoff[t], t0 = t2_off(T, tr.la, tr.lb, 0);
    unsigned int chan = 0;
    {
      unsigned int m = 0;
      for (int k = lane; k < nfail; k += 64) m |= 1u << (T.tmpl[t0 + flist[eoff + k]] >> 24);
      for (int l = 0; l < L; l++) chan |= wave_any((m >> l) & 1u) ? 1u << l : 0u;
    }
    const int lmax = 31 - __clz((int)chan);
    // shares of at least `share` entries, in whole chunks
    const int ns = max(1, min(nsplit, (nfail + share - 1) / share));
    const int per = ((nfail + ns - 1) / ns + kFb2Chunk - 1) / kFb2Chunk * kFb2Chunk;
    const int e0 = split * per, e1 = min(nfail, e0 + per);
    if (e0 >= e1) continue;
    const ecp_xyz rc = J.atoms[Cn.atom];
    const double dAC = dist(rc, J.atoms[Sa.atom]), dBC = dist(rc, J.atoms[Sb.atom]);
    const double minExp = T.lnAcc2;
    const int laC = tr.la + lmax, lbC = tr.lb + lmax, lab = tr.la + tr.lb;
    for (int w0 = e0; w0 < e1; w0 += 64 * OWN) {
      const int nhere = min(64 * OWN, e1 - w0);
      // this lane's entries: packed (lambda1, lambda2, lambda3, l) and index
      // in the job's T arrays
      int code[OWN], eo[OWN];
#pragma unroll
      for (int i = 0; i < OWN; i++) {
        code[i] = 0;
        eo[i] = -1;
        if (i * 64 + lane >= nhere) continue;
        const int e = flist[eoff + w0 + i * 64 + lane];
        code[i] = T.tmpl[t0 + e];
        eo[i] = eoff + e;
      }
      for (int pb0 = 0; pb0 < npairs; pb0 += 64) {
        bool mine_live = false;
        if (pb0 + lane < npairs) {
          const int pa = (pb0 + lane) / Sb.K, pb = (pb0 + lane) - pa * Sb.K;
          const double za = J.pa[Sa.prim + pa], zb = J.pa[Sb.prim + pb];
          const double zeta_p = za + zb;
          const Fm06 M = fm06(zeta_p, (za * dAC + zb * dBC) / zeta_p);
          mine_live = !psm92_dead(T, M, minExp, [&](double r) {
            const double d1 = dAC - r, d2 = dBC - r;
            return -za * d1 * d1 - zb * d2 * d2;
          });
        }
        const int nc64 = min(64, npairs - pb0);
        unsigned long long live = __ballot(mine_live);
        unsigned long long dead = ~live & (nc64 == 64 ? ~0ull : (1ull << nc64) - 1ull);
        // the zeros of the dead pairs: shared among the slots
        for (int k = 0; dead; dead &= dead - 1ull, k++) {
          if (k % nslot != slot) continue;
          const int pair = pb0 + __ffsll((long long)dead) - 1;
#pragma unroll
          for (int i = 0; i < OWN; i++)
            if (eo[i] >= 0) fbT[(size_t)eo[i] * J.maxPairs + pair] = 0.0;
        }
        for (int k = 0; live; live &= live - 1ull, k++) {
          if (k % nslot != slot) continue;
          const int pair = pb0 + __ffsll((long long)live) - 1;
          const int pa = pair / Sb.K, pb = pair - pa * Sb.K;
          const double za = J.pa[Sa.prim + pa], zb = J.pa[Sb.prim + pb];
          const double s1 = 2.0 * za * dAC, s2 = 2.0 * zb * dBC;
          double Cc = J.pd[Sa.prim + pa] * J.pd[Sb.prim + pb];
          // derivatives: times zeta^shift (type2.c:457-462)
          for (int x = 0; x < tr.powa; x++) Cc *= za;
          for (int x = 0; x < tr.powb; x++) Cc *= zb;
          const double zeta_p = za + zb;
          const Fm06 M = fm06(zeta_p, (za * dAC + zb * dBC) / zeta_p);
          Psm92 S[OWN];
          bool open[OWN];
#pragma unroll
          for (int i = 0; i < OWN; i++) {
            S[i] = Psm92{0.0, 0.0, 0.0};
            open[i] = eo[i] >= 0;
          }
          // rounds of point pairs [c0, c1): levels 0 to 5 first, then 32
          // pairs of level lv at a time
          int lv = psm92_first(T), c0 = 0, c1 = T.s92.lvl_begin[lv];
          for (;;) {
            const bool first = c0 == 0;
            const int n = psm92_point(T, c0, c1, lane, first);
            double r = 0.0, w = 0.0, ex = 0.0;
            bool on = false;
            if (n >= 0) {
              r = M.i1 * T.xl[n] + M.i2;
              const double d1 = dAC - r, d2 = dBC - r;
              const double expo = -za * d1 * d1 - zb * d2 * d2;
              if (expo >= minExp) {
                on = true;
                ex = exp(expo);
                w = T.wl[n] * M.i1;
              }
            }
            for (int l = 0; l < L; l++)
              if ((chan >> l) & 1u) s_cu[l * 64 + lane] = on ? Cc * eval_ecp(J, tr.centre, l, r) : 0.0;
            {
              double rn = 1.0;
              for (int x = 0; x <= lab; x++) {
                s_rn[x * 64 + lane] = rn;
                rn = r * rn;
              }
            }
            // one Bessel vector live at a time (register pressure)
            {
              double K[LMB + 1];
#pragma unroll
              for (int l = 0; l <= LMB; l++) K[l] = 0.0;
              if (on) bessel_k<LMB>(T.bessel, s1 * r, K);
#pragma unroll
              for (int l = 0; l <= LMB; l++)
                if (l <= laC) s_ka[l * 64 + lane] = K[l];
            }
            {
              double K[LMB + 1];
#pragma unroll
              for (int l = 0; l <= LMB; l++) K[l] = 0.0;
              if (on) bessel_k<LMB>(T.bessel, s2 * r, K);
#pragma unroll
              for (int l = 0; l <= LMB; l++)
                if (l <= lbC) s_kb[l * 64 + lane] = K[l];
            }
            const bool level_end = !first && c1 == T.s92.lvl_begin[lv + 1];
            bool any = false;
#pragma unroll
            for (int i = 0; i < OWN; i++) {
              const unsigned long long om = __ballot(open[i]);
              for (int o = 0; o < 64; o += kFb2Chunk) {
                unsigned int m = (unsigned int)(om >> o) & ((1u << kFb2Chunk) - 1u);
                if (!m) continue;
                // four entries at a time, so that their LDS reads overlap
                // (fewer left: the last one again)
                while (m) {
                  int j[4];
                  double cu[4], ka[4], kb[4], rn[4];
#pragma unroll
                  for (int x = 0; x < 4; x++) {
                    j[x] = __ffs((int)m) - 1;
                    if (m & (m - 1u)) m &= m - 1u;
                    else if (x == 3) m = 0;
                    const int cd = __builtin_amdgcn_readlane(code[i], o + j[x]);
                    cu[x] = s_cu[(cd >> 24) * 64 + lane];
                    rn[x] = s_rn[((cd >> 16) & 0xff) * 64 + lane];
                    ka[x] = s_ka[(cd & 0xff) * 64 + lane];
                    kb[x] = s_kb[((cd >> 8) & 0xff) * 64 + lane];
                  }
#pragma unroll
                  for (int x = 0; x < 4; x++) {
                    const double v = pair_sum(w * ((((cu[x] * rn[x]) * ka[x]) * kb[x]) * ex));
                    if (!(lane & 1)) s_t[j[x] * kFbTS + (lane >> 1)] = v;
                  }
                }
                __syncthreads();
                if (open[i] && (unsigned)(lane - o) < (unsigned)kFb2Chunk) {
                  const double *row = s_t + (lane - o) * kFbTS;
                  double res = 0.0;
                  bool done;
                  if (first) {
                    done = S[i].first_round(T, row, &res);
                  } else {
                    S[i].I = sum_in_order(S[i].I, row, c1 - c0);
                    done = level_end && S[i].test(T, lv, &res);
                  }
                  if (done) {
                    open[i] = false;
                    fbT[(size_t)eo[i] * J.maxPairs + pair] = res;
                  }
                }
                __syncthreads();
              }
              any = any || open[i];
            }
            lv += level_end;
            if (lv >= T.s92.nlevels || !wave_any(any)) break;
            if (first || level_end)
#pragma unroll
              for (int i = 0; i < OWN; i++) S[i].step();
            c0 = c1;
            c1 = min(c0 + 32, T.s92.lvl_begin[lv + 1]);
          }
#pragma unroll
          for (int i = 0; i < OWN; i++) {
            if (open[i]) status[2 * t + 1] = 1;
          }
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Fused launches: one grid covers every class (lambda = la + lb for type 1,
// lambda_max = max(la, lb) + l for the type-2 fallback), each class owning a
// contiguous range of workgroups; the class bodies are those of the
// per-class kernels.  For small jobs, where each per-class launch holds only
// a few waves, this turns ~40 dependent launches into a handful.

struct ClassMap {
  int n;                     // classes with work
  int cls[16];               // class id of entry i
  int bbeg[17];              // workgroup range of entry i: [bbeg[i], bbeg[i+1])
};

__device__ __forceinline__ int class_entry(const ClassMap &cm, int b) {
  int i = 0;
  while (i + 1 < cm.n && b >= cm.bbeg[i + 1]) i++;
  return i;
}

// per-class views of the type-1 work arrays
struct T1Set {
  const T1Unit *units;
  double *q;
  unsigned long long *qf;
  int *fbq, *fbc, *tq;
  double *st;
  size_t plane;
  unsigned char *stat;
  int ubeg[ECP_MAX_LAB + 1], ucnt[ECP_MAX_LAB + 1];
  int head;  // PS93 levels of the head (>= the level count: no tail)
};

#define ECP_CASES_LAB(X) X(0) X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12)
#define ECP_CASES_LMB(X) X(0) X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12)

template <int MAXLAB>
__global__ __launch_bounds__(64, MAXLAB <= 6 ? 2 : 1) void k_type1_fused(DevTables T, DevJob J, T1Set S, ClassMap cm) {
  const int i = class_entry(cm, blockIdx.x);
  const int c = cm.cls[i], bid = blockIdx.x - cm.bbeg[i];
  const int ub = S.ubeg[c];
  switch (c) {
#define X(L)                                                                                                     \
  case L:                                                                                                        \
    if constexpr (L <= MAXLAB)                                                                                   \
      type1_body<L>(bid, T, J, S.units + ub, S.ucnt[c], S.q, S.qf + ub, S.fbq + ub, S.fbc + c, S.head, S.st,     \
                    S.plane, S.tq + ub, S.fbc + 32 + c);                                                         \
    break;
    ECP_CASES_LAB(X)
#undef X
  }
}

template <int MAXLAB>
__global__ __launch_bounds__(64) void k_t1tail_fused(DevTables T, DevJob J, T1Set S, ClassMap cm) {
  __shared__ double s_T[nq_of(MAXLAB) * kTS];
  __shared__ int s_pt[128];
  const int i = class_entry(cm, blockIdx.x);
  const int c = cm.cls[i], bid = blockIdx.x - cm.bbeg[i], nb = cm.bbeg[i + 1] - cm.bbeg[i];
  const int ub = S.ubeg[c];
  switch (c) {
#define X(L)                                                                                                     \
  case L:                                                                                                        \
    if constexpr (L <= MAXLAB)                                                                                   \
      t1tail_body<L>(bid, nb, T, J, S.units + ub, S.q, S.qf + ub, S.fbq + ub, S.fbc + c, S.head, S.st, S.plane,  \
                     S.tq + ub, S.fbc + 32 + c, S.stat, s_T, s_pt);                                              \
    break;
    ECP_CASES_LAB(X)
#undef X
  }
}

struct T2Set {
  const int *fbq2;  // per class, the triplets with failed entries (nt apart)
  const int *fbc;
  double *fbT;
  unsigned char *stat;
  int nt;
  const int *tnfail, *flist;
  int nslot, nsplit, share;
  int cu_rows, rn_rows, k_rows;  // LDS rows: U_l of the job's channels, powers of r, K of its largest class
};

// two entries per lane where registers set the waves per SIMD (three), four
// in the larger classes, where the LDS rows do (two)
template <int MAXLMB, int OWN = MAXLMB <= 7 ? 2 : 4>
__global__ __launch_bounds__(64, MAXLMB <= 7 ? 3 : 2) void k_fb2_fused(DevTables T, DevJob J, T2Set S, ClassMap cm) {
  // pair sums, then the points' columns: U rows for the job's channels, K
  // rows for its largest class (fb2_lds)
  extern __shared__ double lds[];
  double *s_t = lds, *s_cu = lds + kFb2Chunk * kFbTS, *s_rn = s_cu + S.cu_rows * 64, *s_ka = s_rn + S.rn_rows * 64,
         *s_kb = s_ka + S.k_rows * 64;
  const int i = class_entry(cm, blockIdx.x);
  const int c = cm.cls[i], bid = blockIdx.x - cm.bbeg[i], nb = cm.bbeg[i + 1] - cm.bbeg[i];
  switch (c) {
#define X(L)                                                                                                     \
  case L:                                                                                                        \
    if constexpr (L <= MAXLMB)                                                                                   \
      fb2_body<L, OWN>(bid, nb, T, J, S.fbq2 + (size_t)L * S.nt, S.fbc + kFb2Cnt + L, S.fbT, S.stat, S.tnfail,   \
                       S.flist, S.nslot, S.nsplit, S.share, s_cu, s_rn, s_ka, s_kb, s_t);                       \
    break;
    ECP_CASES_LMB(X)
#undef X
  }
}

// ---------------------------------------------------------------------------
// assembly: type-1 block (calcChi), type-2 block (calcGamma), binomial shift
// (calcPolynomials) and norms (libecp.c:234-235)

constexpr int kAsmThreads = 64;
constexpr int kAsmPack = 4, kAsmPackLab = 2;  // packed type-1 assembly: triplets per wave, largest la + lb

struct AsmArgs {
  const T1Unit *units1;
  const int *t1first;        // per triplet: first type-1 unit
  const double *qout;
  const double *Tout;
  const unsigned char *tfail;
  const double *fbT;
  double *blocks;
  // dynamic LDS layout (doubles): J is shared; the type-1 region (rsph, H)
  // and the type-2 region (blk, T) overlap
  int lds_blk, lds_H, lds_J, lds_rsph, lds_T, lds_rs_stride, pair_chunk, lds_Q;
  int lds_S1, lds_S2, shift_lm;  // shift factor tables (aliasing rsph/Q resp. T) for shells up to shift_lm
  const double *udir;             // type 1: per unit, cos theta, phi, sin phi, cos phi of its pair direction
  int lds_group;                  // packed type-1 assembly: LDS doubles per triplet
};

// binomial shift of a block over C-centred monomials to the IJK(la) x IJK(lb)
// output (util.c:246-334).  The block is read through get(r, q): row r is an
// ordering position of degree <= la, column q a position of degree <= lb.
struct V3 {
  double x, y, z;
};

// Nonzero binomial factors of the shift (util.c:246-334), listed once per
// triplet: for component c of shell l (ordering position), the factors
// C(a,alpha) (C-A)^(a-alpha) over alpha in the loop order of util.c:277-320,
// each formed exactly as the per-element loops would (powers by repeated
// multiplication, binomials left to right, factors |f| <= accuracy dropped,
// the norm applied to the B side), with the position of alpha.
__host__ __device__ constexpr int shift_mt(int l) {
  int best = 1;
  for (int ax = 0; ax <= l; ax++)
    for (int ay = 0; ax + ay <= l; ay++) {
      const int v = (ax + 1) * (ay + 1) * (l - ax - ay + 1);
      best = v > best ? v : best;
    }
  return best;
}

// doubles of LDS for the factor tables of both sides for shells up to LM
__host__ __device__ constexpr int shift_tab_doubles(int LM) {
  const int n = ECP_DIM_IJK(LM) * shift_mt(LM);
  return 2 * (n + (n + 1) / 2 + (ECP_DIM_IJK(LM) + 1) / 2);
}

struct ShiftTab {
  double *f;
  int *r, *n;
  int mt;
};

__device__ __forceinline__ ShiftTab shift_tab_at(double *base, int LM, int side) {
  const int n = ECP_DIM_IJK(LM) * shift_mt(LM);
  double *b = base + side * (n + (n + 1) / 2 + (ECP_DIM_IJK(LM) + 1) / 2);
  ShiftTab S;
  S.f = b;
  S.r = (int *)(b + n);
  S.n = (int *)(b + n + (n + 1) / 2);
  S.mt = shift_mt(LM);
  return S;
}

// (component, alpha) terms of a shell l, and of the shells before it
__host__ __device__ constexpr int shift_terms(int l) {
  return (l + 1) * (l + 2) * (l + 3) * (l + 4) * (l + 5) / 120;
}
__host__ __device__ constexpr int shift_terms_before(int l) {
  return l * (l + 1) * (l + 2) * (l + 3) * (l + 4) * (l + 5) / 720;
}

// One side's factors, a term per lane of the W (8 to 64) lanes lid of a
// group, from the term table (shift_table); the terms kept move up inside
// their component.  (A component per lane took its up to 27 terms one after
// another, each behind two table reads.  The assembly of 256 molecules,
// alone: type 1 1978 + 461 -> 1276 + 338 us, type 2 2857 + 682 -> 2177 + 476;
// waits were 0.6 of its wave cycles.)
__device__ __forceinline__ void shift_factors(const DevTables &T, int l, const V3 v, bool with_norm, double norm,
                                              ShiftTab S, int lid, int W) {
  const int n = shift_terms(l);
  const unsigned *tab = T.shift + shift_terms_before(l);
  const double tol = T.accuracy;
  const int base = (int)(threadIdx.x & 63) & ~(W - 1);
  const unsigned long long group = W == 64 ? ~0ull : (1ull << W) - 1ull;
  unsigned long long prev = 0;
  for (int e0 = 0; e0 < n; e0 += W) {
    const bool in = e0 + lid < n;
    const unsigned z = tab[min(e0 + lid, n - 1)];
    const int c = z & 31, r = (z >> 14) & 127, dist = (z >> 26) & 31;
    double px = 1.0, py = 1.0, pz = 1.0;
    for (int i = (z >> 5) & 7; i > 0; i--) px = -px * v.x;
    for (int i = (z >> 8) & 7; i > 0; i--) py = -py * v.y;
    for (int i = (z >> 11) & 7; i > 0; i--) pz = -pz * v.z;
    const double factor = (double)((z >> 21) & 31) * ((px * py) * pz);
    const bool keep = in && !(fabs(factor) <= tol);
    const unsigned long long m = (__ballot(keep) >> base) & group;
    // kept terms of the component before this one; its first term may have
    // been in the previous round
    const int first = lid - dist;
    int pos = __popcll(m & ((1ull << lid) - 1ull) & (~0ull << max(first, 0)));
    if (first < 0) pos += __popcll(prev >> (W + first));
    if (keep) {
      S.f[c * S.mt + pos] = with_norm ? factor * norm : factor;
      S.r[c * S.mt + pos] = r;
    }
    if (in && z >> 31) S.n[c] = pos + keep;
    prev = m;
  }
}

// sum of f[t] get(r[t]) over t < n, in order; the reads of up to four terms
// are issued together
template <typename Get>
__device__ __forceinline__ double shift_sum(const double *f, const int *r, int n, Get get) {
  double acc = 0.0;
  int t = 0;
  for (; t + 4 <= n; t += 4) {
    double x[4], y[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      x[i] = f[t + i];
      y[i] = get(r[t + i]);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) acc += x[i] * y[i];
  }
  for (; t < n; t++) acc += f[t] * get(r[t]);
  return acc;
}

// binomial shift of a block over C-centred monomials to the IJK(la) x IJK(lb)
// output (util.c:246-334).  The block is read through get(r, q): row r is an
// ordering position of degree <= la, column q a position of degree <= lb.
// tab: LDS for the factor tables (shift_tab_doubles(LM) doubles, LM >= la,
// lb), free to overwrite; Jbuf: LDS for the half-shifted block.  The lanes
// lid = 0 .. nlanes - 1 of the workgroup do the work; every lane of the
// workgroup calls it (it synchronises the workgroup), those of an inactive
// lane group with active = false.
template <typename Get>
__device__ void shift_block(const DevTables &T, Get get, int la, int lb, const V3 rA, const V3 rB, double norm,
                            double *Jbuf, double *tab, int LM, double *out, int lid = -1, int nlanes = 0,
                            bool active = true) {
  if (lid < 0) {
    lid = threadIdx.x;
    nlanes = blockDim.x;
  }
  const int ncb = ECP_DIM_C(lb), nia = active ? ECP_DIM_IJK(la) : 0, nib = ECP_DIM_IJK(lb);
  const ShiftTab SA = shift_tab_at(tab, LM, 0), SB = shift_tab_at(tab, LM, 1);
  __syncthreads();
  if (active) {
    // the sides beside each other where the lanes suffice
    const int W = min(nlanes, 64), h = W / 2;
    if (nlanes > 64) {
      if (lid < 64) shift_factors(T, la, rA, false, 1.0, SA, lid, 64);
      else if (lid < 128) shift_factors(T, lb, rB, true, norm, SB, lid - 64, 64);
    } else if (max(shift_terms(la), shift_terms(lb)) <= h) {
      const bool b = lid >= h;
      shift_factors(T, b ? lb : la, b ? rB : rA, b, norm, b ? SB : SA, lid & (h - 1), h);
    } else {
      shift_factors(T, la, rA, false, 1.0, SA, lid, W);
      shift_factors(T, lb, rB, true, norm, SB, lid, W);
    }
  }
  __syncthreads();
  for (int idx = lid; idx < nia * ncb; idx += nlanes) {
    const int c1 = idx / ncb, q = idx % ncb;
    const double *f = SA.f + c1 * SA.mt;
    const int *r = SA.r + c1 * SA.mt;
    const int n = SA.n[c1];
    Jbuf[idx] = shift_sum(f, r, n, [&](int x) { return get(x, q); });
  }
  __syncthreads();
  for (int idx = lid; idx < nia * nib; idx += nlanes) {
    const int c1 = idx / nib, c2 = idx % nib;
    const double *f = SB.f + c2 * SB.mt;
    const int *r = SB.r + c2 * SB.mt;
    const int n = SB.n[c2];
    out[idx] = shift_sum(f, r, n, [&](int x) { return Jbuf[c1 * ncb + x]; });
  }
  __syncthreads();
}

// One C-centred monomial's sum over the chunk's pairs: acc, then per pair the
// blocks l = deg, deg - 2, .. of its poly2sph row times the pair's harmonics,
// each times its Q value, in that order.  The lanes of a wave hold monomials
// of every degree up to lab <= MAXD: block b is l = 2 b for even degrees and
// l = 2 b - 1 for odd ones, so that all degrees go through one pass of at most
// (MAXD + 1)(MAXD + 2) / 2 terms, the last two of a block for even degrees
// only.  (A pass per degree, with its lanes alone, kept 0.20 of the lanes
// busy: 84 terms a pair for class 6 instead of 28; 256 molecules 2111 ->
// 1978 us.)  Terms a lane does not have are computed and not taken.
template <int MAXD>
__device__ __forceinline__ double asm1_monomial(double acc, int deg, int lab, const double *__restrict__ pm,
                                                const double *rsph, int rs_stride, const double *Qs, int nql,
                                                int nc) {
  constexpr int NB = (MAXD + 1) / 2 + 1, NT = 4 * (NB - 1) + 1;
  const int odd = deg & 1;
  double pmv[NB][NT];
  int off[NB];  // the block's first harmonic
  bool on[NB];
#pragma unroll
  for (int b = 0; b < NB; b++) {
    const int l = 2 * b - odd;
    on[b] = l >= 0 && l <= deg;
    off[b] = on[b] ? l * l : 0;
    if (2 * b - 1 <= lab)
#pragma unroll
      for (int m = 0; m < 4 * b + 1; m++)
        if (2 * b <= MAXD || m < 4 * b - 1) pmv[b][m] = pm[off[b] + (on[b] ? min(m, 2 * l) : 0)];
  }
  for (int k = 0; k < nc; k++) {
    const double *rs = rsph + k * rs_stride;
    const double *Q = Qs + k * nql;
#pragma unroll
    for (int b = NB - 1; b >= 0; b--) {
      if (2 * b - 1 > lab) continue;
      const double q = Q[on[b] ? (deg - 2 * b + odd) >> 1 : 0];
      double f = 0.0;
#pragma unroll
      for (int m = 0; m < 4 * b + 1; m++) {
        if (2 * b > MAXD && m >= 4 * b - 1) continue;
        const double x = f + rs[off[b] + m] * pmv[b][m];
        f = m < 4 * b - 1 || !odd ? x : f;
      }
      const double a = acc + f * q;
      acc = on[b] ? a : acc;
    }
  }
  return acc;
}

// The block of a triplet whose integration failed: zeros, whatever an earlier
// job left in the memory (a contraction sums every block and reports the
// failure beside its result).
__device__ __forceinline__ void zero_block(const DevJob &J, int t, double *blk, int lid, int nlanes) {
  const ecp_triplet &tr = J.trip[t];
  const int n = ECP_DIM_IJK(tr.oa) * ECP_DIM_IJK(tr.ob);
  for (int i = lid; i < n; i += nlanes) blk[i] = 0.0;
}

// Type-1 block of one triplet per wave (the triplets tlist[0 .. ntl), in
// class order lambda = la + lb).  chi[i][j] depends on (i, j) only
// through the monomial p = i + j, so H[p] = sum_pairs sum_l F_pair[p][l]
// Q[deg p][l] with F_pair[p][l] = sum_m S_lm(k^_pair) poly2sph[p][lm] is
// formed once per monomial (same terms, same order as type1.c:266-295 per
// element), then shifted to the output block (util.c:246-334).
// G > 1 (classes la + lb <= 2, where a triplet has at most 10 monomials):
// G triplets per wave, kAsmThreads / G lanes and an LDS slice of
// A.lds_group doubles each; the wave's lane groups run the same phases and
// synchronise together, an inactive group with empty loops.
// MAXD: the largest monomial degree whose poly2sph row goes to registers
// (the triplets' la + lb when a launch covers one class); higher degrees
// take the general loop.  Registers, without spills: 64 (rows up to degree
// 3 in registers) to 98 (degree 6), 92 for the packed variant; the pair
// directions come from the tables kernel, so no trigonometric code sits
// here.
template <int G = 1, int MAXD = 6>
__global__ __launch_bounds__(kAsmThreads, 3) void k_asm1(DevTables T, DevJob J, AsmArgs A,
                                                      const unsigned char *__restrict__ status,
                                                      const int *__restrict__ tlist, int ntl) {
  extern __shared__ double lds_all[];
  constexpr int W = kAsmThreads / G;
  const int grp = G == 1 ? 0 : (int)threadIdx.x / W;
  const int lid = G == 1 ? (int)threadIdx.x : (int)threadIdx.x % W;
  double *lds = lds_all + (size_t)grp * A.lds_group;
  double *H = lds + A.lds_H;
  double *Jbuf = lds + A.lds_J;
  double *rsph = lds + A.lds_rsph;
  double *Qs = lds + A.lds_Q;
  int t;
  bool active = true;
  if constexpr (G == 1) {
    t = tlist[blockIdx.x];
    if (status[2 * t]) {
      zero_block(J, t, A.blocks + J.trip[t].blk1, lid, W);
      return;
    }
  } else {
    const int ti = blockIdx.x * G + grp;
    active = ti < ntl;
    t = active ? tlist[ti] : tlist[0];
    if (active && status[2 * t]) {
      zero_block(J, t, A.blocks + J.trip[t].blk1, lid, W);
      active = false;
    }
    if (!wave_any(active)) return;
  }
  const ecp_triplet tr = J.trip[t];
  const ecp_centre Cn = J.cent[tr.centre];
  const ecp_shell Sa = J.shells[tr.sa], Sb = J.shells[tr.sb];
  const int la = tr.la, lb = tr.lb, lab = la + lb;  // shifted for derivatives
  const ecp_xyz rc = J.atoms[Cn.atom], ra = J.atoms[Sa.atom], rb = J.atoms[Sb.atom];
  const V3 vA{ra.x - rc.x, ra.y - rc.y, ra.z - rc.z}, vB{rb.x - rc.x, rb.y - rc.y, rb.z - rc.z};
  const int tmd = ECP_DIM_L(T.tmDim);

  const int np = active ? ECP_DIM_C(lab) : 0;
  const int nql = nq_of(lab);
  const int npairs = active ? Sa.K * Sb.K : 0;
  int npmax = npairs;
  if (G > 1)
    for (int o = 32; o > 0; o >>= 1) npmax = max(npmax, __shfl_xor(npmax, o, 64));
  const int u0 = A.t1first[t];
  int qstart = 0;
  for (int idx = lid; idx < np; idx += W) H[idx] = 0.0;
  for (int c0 = 0; c0 < npmax; c0 += A.pair_chunk) {
    const int nc = G == 1 ? min(A.pair_chunk, npairs - c0) : max(0, min(A.pair_chunk, npairs - c0));
    // the harmonics of the chunk's pair directions (formed by the tables
    // kernel), one (pair, m) column per lane; the pairs' Q values staged
    // alongside
    for (int it = lid; it < nc * (lab + 1); it += W) {
      const int k = it / (lab + 1), m = it - k * (lab + 1);
      const double *d = A.udir + 4 * (size_t)(u0 + c0 + k);
      real_sph_column(T, lab, m, d[0], d[1], d[2], d[3], rsph + k * A.lds_rs_stride);
    }
    for (int it = lid; it < nc * nql; it += W) {
      const int k = it / nql, e = it - k * nql;
      Qs[k * nql + e] = A.qout[A.units1[u0 + c0 + k].qoff + e];
    }
    __syncthreads();
    for (int p = lid; p < np; p += W) {
      const int *e = T.ijk + 3 * p;
      const int deg = e[0] + e[1] + e[2];
      qstart = 0;
      for (int l1 = 0; l1 < deg; l1++) qstart += l1 / 2 + 1;
      const double *pm = T.poly2sph + (size_t)p * tmd;
      double acc = H[p];
      if (deg <= MAXD) {
        acc = asm1_monomial<MAXD>(acc, deg, lab, pm, rsph, A.lds_rs_stride, Qs + qstart, nql, nc);
        H[p] = acc;
        continue;
      }
      for (int k = 0; k < nc; k++) {
        const double *rs = rsph + k * A.lds_rs_stride;
        const double *Q = Qs + k * nql + qstart;
        for (int l = deg; l >= 0; l -= 2) {
          double f = 0.0;
          f = dot_in_order<2>(f, rs + ECP_IDX_LM(l, 0), 1, pm + ECP_IDX_LM(l, 0), 1, 2 * l + 1);
          acc += f * Q[(deg - l) / 2];
        }
      }
      H[p] = acc;
    }
    __syncthreads();
  }
  const double norm1 = 4.0 * M_PI;
  auto get1 = [&](int r, int q) { return H[T.prod[r * T.prodN + q]]; };
  if constexpr (G == 1)
    shift_block(T, get1, tr.oa, tr.ob, vA, vB, norm1, Jbuf, lds + A.lds_S1, A.shift_lm, A.blocks + tr.blk1);
  else
    shift_block(T, get1, tr.oa, tr.ob, vA, vB, norm1, Jbuf, lds + A.lds_S1, A.shift_lm, A.blocks + tr.blk1, lid, W,
                active);
}

// degree of the C-centred monomial at ordering position p (l <= 6)
__device__ __forceinline__ int deg_of(int p) {
  return (p >= 1) + (p >= 4) + (p >= 10) + (p >= 20) + (p >= 35) + (p >= 56);
}

// T values of a triplet in LDS, every channel: entry (l, lambda1, lambda2,
// k = alpha + beta).  lambda1 + alpha, lambda2 + beta and l have the same
// parity, so k and lambda1 + lambda2 do too, and half of the k suffice.
__device__ __forceinline__ int t2_slot(int la, int lb, int l, int l1, int l2, int k) {
  const int a = la + 1, b = lb + 1, d3 = (la + lb + 2) >> 1;
  // the channels before l: sum of (a + i)(b + i), i < l
  const int before = l * a * b + (a + b) * (l * (l - 1) >> 1) + (l - 1) * l * (2 * l - 1) / 6;
  return (before + l1 * (b + l) + l2) * d3 + (k >> 1);
}
__host__ __device__ constexpr int t2_slots(int la, int lb, int L) {
  int n = 0;
  for (int l = 0; l < L; l++) n += (la + l + 1) * (lb + l + 1);
  return n * ((la + lb + 2) / 2);
}

// One channel's part of element (pp, qq) of a type-2 block (type2.c:583-623):
// the sum over lambda1 and lambda2 of (sum_m A[lambda1][m][pp]
// B[lambda2][m][qq]) T[lambda1][lambda2].  The channel is a template
// argument, so that its 2 l + 1 factors and its at most (NB - 1 + l) / 2 + 1
// values of lambda2 are the only ones in the code: with both padded to the
// largest channel's, the kernel's time was that of instructions for absent
// values.
// NB > 0 (basis l < NB): the angular factors of atom B for every lambda2 in
// registers, those of atom A for the next lambda1 read ahead; NB = 0: both
// read for each pair.
template <int NB, int L>
__device__ __forceinline__ double asm2_channel(const double *__restrict__ pA, const double *__restrict__ pB,
                                               int ang_c, int lam_stride, const double *Tl, int la, int lb, int alpha,
                                               int beta) {
  constexpr int NM = 2 * L + 1;
  constexpr int NBL = NB == 0 ? 1 : (NB - 1 + L) / 2 + 1 < NB ? (NB - 1 + L) / 2 + 1 : NB;
  const int ll1 = max((alpha + L) & 1, L - alpha), ll2 = max((beta + L) & 1, L - beta);
  const int ds = (la + lb + 2) >> 1, d2 = (lb + L + 1) * ds;
  const double *Te = Tl + t2_slot(la, lb, L, ll1, ll2, alpha + beta);
  pA += L * L * ang_c + ll1 * lam_stride;
  pB += L * L * ang_c + ll2 * lam_stride;
  const int n1 = (la + L - ll1) >> 1, n2 = (lb + L - ll2) >> 1;  // values of lambda1, lambda2, less one
  double tmp = 0.0;
  if constexpr (NB > 0) {
    double Bv[NBL][NM], Av[NM];
#pragma unroll
    for (int m = 0; m < NM; m++) Av[m] = pA[m * ang_c];
#pragma unroll
    for (int i = 0; i < NBL; i++) {
      const double *pb = pB + 2 * min(i, n2) * lam_stride;
#pragma unroll
      for (int m = 0; m < NM; m++) Bv[i][m] = pb[m * ang_c];
    }
    for (int i1 = 0; i1 <= n1; i1++, Te += 2 * d2) {
      double An[NM];
      pA += i1 < n1 ? 2 * lam_stride : 0;
#pragma unroll
      for (int m = 0; m < NM; m++) An[m] = pA[m * ang_c];
#pragma unroll
      for (int i = 0; i < NBL; i++)
        if (i <= n2) {
          double factor = 0.0;
#pragma unroll
          for (int m = 0; m < NM; m++) factor += Av[m] * Bv[i][m];
          tmp += factor * Te[2 * i * ds];
        }
#pragma unroll
      for (int m = 0; m < NM; m++) Av[m] = An[m];
    }
  } else {
    for (int i1 = 0; i1 <= n1; i1++, pA += 2 * lam_stride, Te += 2 * d2)
      for (int i = 0; i <= n2; i++) {
        const double *pb = pB + 2 * i * lam_stride;
        double x[NM], y[NM];
#pragma unroll
        for (int m = 0; m < NM; m++) {
          x[m] = pA[m * ang_c];
          y[m] = pb[m * ang_c];
        }
        double factor = 0.0;
#pragma unroll
        for (int m = 0; m < NM; m++) factor += x[m] * y[m];
        tmp += factor * Te[2 * i * ds];
      }
  }
  return tmp;
}

// Type-2 blocks, a lane group of 64 / G lanes and an LDS slice per triplet
// (tlist[0 .. ntl); G = kAsmPack: classes la + lb <= kAsmPackLab, at most 9
// elements): the T values of every channel (small-grid results, or the sum
// of the per-pair fallback results) are read together and placed in LDS, the
// lanes form the elements, contracting them with the angular tables of both
// atoms (type2.c:583-623), and the block is shifted (util.c:246-334).
// NB: as in asm2_channel; channels l < MAXL.
template <int G, int NB, int MAXL, int NT = kAsmThreads>
__global__ __launch_bounds__(NT) void k_asm2(DevTables T, DevJob J, AsmArgs A,
                                                      const unsigned char *__restrict__ status,
                                                      const int *__restrict__ tlist, int ntl) {
  extern __shared__ double lds_all[];
  constexpr int W = NT / G;
  const int grp = G == 1 ? 0 : (int)threadIdx.x / W, lid = (int)threadIdx.x % W;
  double *lds = lds_all + (G == 1 ? 0 : (size_t)grp * A.lds_group);
  double *blk = lds + A.lds_blk, *Jbuf = lds + A.lds_J, *Tl = lds + A.lds_T;
  const int ti = xcd_item(blockIdx.x, gridDim.x) * G + grp;
  bool active = ti < ntl;
  const int t = cload(tlist + (active ? ti : 0));
  if (active && status[2 * t + 1]) {
    zero_block(J, t, A.blocks + J.trip[t].blk2, lid, W);
    active = false;
  }
  if (!wave_any(active)) return;
  const ecp_triplet tr = J.trip[t];
  const ecp_centre Cn = J.cent[tr.centre];
  const ecp_shell Sa = J.shells[tr.sa], Sb = J.shells[tr.sb];
  const int la = tr.la, lb = tr.lb;  // shifted for derivatives
  const int nca = ECP_DIM_C(la), ncb = ECP_DIM_C(lb);
  const ecp_xyz rc = J.atoms[Cn.atom], ra = J.atoms[Sa.atom], rb = J.atoms[Sb.atom];
  const V3 vA{ra.x - rc.x, ra.y - rc.y, ra.z - rc.z}, vB{rb.x - rc.x, rb.y - rc.y, rb.z - rc.z};
  const int t0 = t2_off(T, la, lb, 0), eoff = J.teoff[t];
  const int ne = active ? t2_off(T, la, lb, Cn.L) - t0 : 0, npairs = Sa.K * Sb.K;
  const int nslots = active ? t2_slots(la, lb, Cn.L) : 0;
  for (int i = lid; i < nslots; i += W) Tl[i] = 0.0;
  __syncthreads();
  for (int e0 = lid; e0 < ne; e0 += 4 * W) {
    double v[4];
    int code[4];
    unsigned char f[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int e = min(e0 + i * W, ne - 1);
      v[i] = A.Tout[eoff + e];
      f[i] = A.tfail[eoff + e];
      code[i] = T.tmpl[t0 + e];
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int e = e0 + i * W;
      if (e >= ne) break;
      if (f[i]) v[i] = sum_in_order(0.0, A.fbT + (size_t)(eoff + e) * J.maxPairs, npairs);
      Tl[t2_slot(la, lb, code[i] >> 24, code[i] & 0xff, (code[i] >> 8) & 0xff, (code[i] >> 16) & 0xff)] = v[i];
    }
  }
  __syncthreads();
  const int lam_stride = J.angL * J.angL * J.ang_c;
  const double *angA = J.ang + Cn.ang_off + (size_t)(Sa.atom - Cn.atom0) * J.ang_lam * lam_stride;
  const double *angB = J.ang + Cn.ang_off + (size_t)(Sb.atom - Cn.atom0) * J.ang_lam * lam_stride;
  const float inv_ncb = 1.0f / ncb;
  for (int idx = active ? lid : nca * ncb; idx < nca * ncb; idx += W) {
    const int pp = (int)(((float)idx + 0.5f) * inv_ncb), qq = idx - pp * ncb;
    const int alpha = deg_of(pp), beta = deg_of(qq);
    double v = 0.0;
#define CH(x)                                                                                          \
  if constexpr (x < MAXL)                                                                              \
    if (x < Cn.L) v += asm2_channel<NB, x>(angA + pp, angB + qq, J.ang_c, lam_stride, Tl, la, lb, alpha, beta);
    CH(0) CH(1) CH(2) CH(3) CH(4) CH(5) CH(6)
#undef CH
    blk[idx] = v;
  }
  __syncthreads();
  const double norm2 = (4.0 * M_PI) * (4.0 * M_PI);
  auto get2 = [&](int r, int q) { return blk[r * ncb + q]; };
  shift_block(T, get2, tr.oa, tr.ob, vA, vB, norm2, Jbuf, lds + A.lds_S2, A.shift_lm, A.blocks + tr.blk2, lid, W,
              active);
}

// ---------------------------------------------------------------------------
// host-side orchestration

template <typename T>
struct DBuf {
  T *p = nullptr;
  size_t n = 0;
};

size_t align_up(size_t x) { return (x + 255) & ~(size_t)255; }

// The per-job tables in one launch of 128-thread blocks: the zero-fill of
// per-run counters and flags (a kernel, so that the sequence can be captured
// in a HIP graph without memset nodes), the U tables per (centre, row, point
// chunk), the F slabs per (centre, shell, run), the pair directions of
// the type-1 units and the angular tables per (centre, atom).  They are independent of each other; every consumer is
// a later launch.
struct TabArgs {
  unsigned int *zero_base;
  size_t zero_words;
  int nzb, nub, nfit, rows;  // rows: U-table rows per centre (largest L + 1)
  const int2 *fit;
  // the type-1 units (class after class, in triplet order) and their pair
  // directions, one (triplet, pair) item per lane
  T1Unit *units;
  double *udir;
  const int *t1first;
  int cls_begin[ECP_MAX_LAB + 1];
  size_t cls_qbase[ECP_MAX_LAB + 1];
  const int2 *ait;           // (centre, atom) pairs of the angular tables, aparts workgroups each
  int nait, aparts;
};

// The pair direction k = 2 (za rAC + zb rBC) of a type-1 unit (type1.c:
// 211-302 via util.c:74-106), stored as cos theta, phi, sin phi, cos phi,
// the values spherical_harmonics.c:15-114 forms from it.  Formed with the
// tables, so that the type-1 assembly carries no trigonometric code (with
// it, it held 168 registers and spilled; 111 when it was taken out).
__device__ void unit_dir(const DevJob &J, const T1Unit &U, double *out) {
  const ecp_triplet tr = J.trip[U.trip];
  const ecp_centre Cn = J.cent[tr.centre];
  const ecp_shell Sa = J.shells[tr.sa], Sb = J.shells[tr.sb];
  const ecp_xyz rc = J.atoms[Cn.atom], ra = J.atoms[Sa.atom], rb = J.atoms[Sb.atom];
  const double za = J.pa[Sa.prim + U.pa], zb = J.pa[Sb.prim + U.pb];
  double r, th, ph;
  sph_coords(2.0 * (za * (ra.x - rc.x) + zb * (rb.x - rc.x)), 2.0 * (za * (ra.y - rc.y) + zb * (rb.y - rc.y)),
             2.0 * (za * (ra.z - rc.z) + zb * (rb.z - rc.z)), r, th, ph);
  out[0] = cos(th);
  out[1] = ph;
  out[2] = sin(ph);
  out[3] = cos(ph);
}

constexpr int kUtabChunks = (SO + 127) / 128;

__global__ __launch_bounds__(128, 4) void k_tables(DevTables T, DevJob J, TabArgs A) {
  __shared__ double rsph[kAngRsph], s_dir[4];
  int b = blockIdx.x;
  // the longest items first
  if (b < A.nait * A.aparts) {
    ang_item(T, J, A.ait[b / A.aparts], rsph, s_dir, b % A.aparts, A.aparts);
    return;
  }
  b -= A.nait * A.aparts;
  if (b < A.nzb) {
    for (size_t i = (size_t)b * 128 + threadIdx.x; i < A.zero_words; i += (size_t)A.nzb * 128) A.zero_base[i] = 0u;
    return;
  }
  b -= A.nzb;
  if (b < A.nub) {
    const int per_c = A.rows * kUtabChunks;
    const int c = b / per_c, rem = b - c * per_c;
    utab_rows(T, J, c, rem / kUtabChunks, rem % kUtabChunks);
    return;
  }
  b -= A.nub;
  if (b < A.nfit) {
    ftab_item(T, J, A.fit[b]);
    return;
  }
  b -= A.nfit;
  const size_t item = (size_t)b * 128 + threadIdx.x;
  const int t = (int)(item / J.maxPairs), k = (int)(item - (size_t)t * J.maxPairs);
  if (t >= J.ntrip) return;
  const ecp_triplet tr = J.trip[t];
  const int Kb = J.shells[tr.sb].K;
  if (k >= J.shells[tr.sa].K * Kb) return;
  const int c = tr.la + tr.lb, u = A.t1first[t] + k;
  // entries of a class: sum of l / 2 + 1 over l <= c
  const int nq = (c + 2) * (c + 2) / 4;
  const T1Unit U{t, k / Kb, k % Kb, (int)(A.cls_qbase[c] + (size_t)(u - A.cls_begin[c]) * nq)};
  A.units[u] = U;
  unit_dir(J, U, A.udir + 4 * (size_t)u);
}

// byte offsets of a job's arrays inside its device block: inputs (uploaded)
// first, then device-only buffers
struct JobLayout {
  size_t i_atoms = 0, i_amaxl = 0, i_sh = 0, i_pa = 0, i_pd = 0, i_cent = 0, i_gauss = 0, i_win = 0, i_trip = 0,
         i_t1f = 0, i_teoff = 0, i_fit = 0, i_ait = 0, i_tcls = 0, i_tcls2 = 0,
         in_bytes = 0;
  size_t d_zero = 0, d_fbc = 0, d_stat = 0, d_zero_end = 0, d_UL = 0, d_Ut = 0, d_F = 0, d_ang = 0,
         d_q = 0, d_t1s = 0, d_tq1 = 0, d_qf = 0, d_u1 = 0, d_udir = 0, d_fbq1 = 0, d_T = 0, d_tf = 0, d_flist = 0, d_tnf = 0, d_fbq2 = 0, d_fbT = 0, d_blk = 0, total = 0;
  int FL = 0, UK = 0, US = 0, angL = 0, ang_lam = 0, ang_c = 0, deriv = 0;
};

struct Prepared {
  int nt = 0;
  int ncent = 0;
  int nfit = 0, nait = 0;
  int cls_begin[ECP_MAX_LAB + 2] = {0};
  int cls_count[ECP_MAX_LAB + 1] = {0};
  int ntot2 = 0, maxPairs = 0;
  size_t nblk = 0;
  // device pointers
  DevJob J{};
  T1Unit *u1 = nullptr;
  size_t cls_qbase[ECP_MAX_LAB + 2] = {0};  // first Q value of each class
  double *q = nullptr;
  size_t nq = 0;
  double *t1s = nullptr;  // type-1 head -> tail state: q, I planes of nq doubles (p in q)
  int *tq1 = nullptr;     // type-1 tail queues (per class, indexed like the units)
  unsigned long long *qf = nullptr;
  double *udir = nullptr;  // per type-1 unit: its pair direction (4 values)
  int *fbq1 = nullptr, *fbc = nullptr;
  unsigned char *stat = nullptr;
  int max_lab = 0;
  int tcount2[kMaxLMB + 1] = {0};  // triplets per type-2 fallback class
  int max_cls2 = 0;
  int max_ent2 = 0;  // T entries of a triplet, at most
  const unsigned char *tcls2 = nullptr;
  int max_lbs = 0, max_L = 0;  // largest basis l and ECP local label of the job
  double *Tout = nullptr;
  unsigned char *tf = nullptr;
  int *tnfail = nullptr, *fbq2 = nullptr;
  int *flist = nullptr;  // per triplet: its failed T entries (tnfail[t] of them) at teoff[t]
  double *fbT = nullptr;
  const int2 *fit = nullptr, *ait = nullptr;
  AsmArgs aa{};
  AsmArgs aa4{};  // packed type-1 assembly of classes la + lb <= kAsmPackLab
  unsigned int *zero_base = nullptr;
  size_t zero_words = 0;
  double *blk = nullptr;
  size_t asm1_lds = 0, asm2_lds = 0, asm1_lds4 = 0, asm2_lds4 = 0;
  AsmArgs aa2p{};  // packed type-2 assembly of classes la + lb <= kAsmPackLab
  int tcls_begin[ECP_MAX_LAB + 2] = {0};  // triplets of each class lambda = la + lb in tcls
  const int *tcls = nullptr;
  // algorithmic FLOPs per evaluation (the per-unit models of the reference's
  // eager algorithm): type-1 radial work per class, type-2 radial work
  double flops_t1[ECP_MAX_LAB + 1] = {0};
};

}  // namespace

constexpr int kWorkers = 3;
constexpr int kSpanGraphs = 8;  // graph copies with their own quadrature event pair

constexpr ecp_tuning kTuningDefaults{5, 8, 100000, 8192, 2, 1, 15, 2048, 0, 1, 0};

struct ecp_dev {
  hipStream_t stream = nullptr;
  hipStream_t workers[kWorkers] = {};
  hipEvent_t fork = nullptr, join[kWorkers] = {};
  // the type-1 small-grid quadrature (head and tail launches), recorded on
  // its stream: event pair k belongs to captured graph k (replays cycle over
  // the graphs, so the last kSpanGraphs replays can be read); the eager
  // evaluation uses pair 0
  hipEvent_t span[kSpanGraphs][2] = {};
  int span_k = 0;
  bool span_valid = false;
  bool capturing = false;  // enqueue runs under stream capture
  hipError_t seq_err = hipSuccess;  // first error of the sequence being enqueued (seq)
  bool last_eager = false;  // the last execute ran no replay
  long long replays = 0;    // replays since the graphs were captured
  int last_replays = 0;     // replays of the last execute
  DevTables T{};
  void *static_mem = nullptr;
  char *arena = nullptr;
  size_t arena_cap = 0;
  char *pin_in = nullptr;
  size_t pin_in_cap = 0;
  char *pin_out = nullptr;
  size_t pin_out_cap = 0;
  int lds_max = 64 * 1024;  // LDS per workgroup of the device (160 KiB on gfx950)
  hipEvent_t ev[8] = {};
  float last_ms[8] = {};
  int nev = 0;
  std::vector<int> tmpl, toff;
  Prepared P;
  JobLayout L;
  ecp_tuning tune = kTuningDefaults;
  bool planned = false, prepared = false, eager_done = false;
  bool uploading = false;  // a copy from pin_in may be in flight on stream
  hipGraph_t graph[kSpanGraphs] = {};
  hipGraphExec_t gexec[kSpanGraphs] = {};
  int ngraph = 0;
  // per-launch profiling (eager runs only)
  bool profiling = false;
  std::vector<hipEvent_t> pev;
  std::vector<int> pfam;
  int npev = 0;
  // density contraction: index tables, densities, partial sums, results
  char *con_mem = nullptr;
  size_t con_cap = 0;
  hipEvent_t con_ev[2] = {};
  std::vector<char> con_idx;  // index tables last uploaded to con_mem at con_idx_at
  size_t con_idx_at = 0;
  double *fbf = nullptr;      // the profile's fallback FLOP sums
  void *scratch = nullptr;    // this device's no-allocation scratch (scratch_setup)
};

namespace {
// kernel families reported by the profiler
enum { FAM_TABLES = 0, FAM_TYPE1, FAM_TYPE2, FAM_FB1, FAM_FB2, FAM_ASM, FAM_T1TAIL, FAM_N };
const char *kFamName[FAM_N] = {"tables", "type1", "type2", "fallback1", "fallback2", "assemble", "type1_tail"};

// keeps the first error of the calls of a kernel sequence (run_sequence)
void seq(ecp_dev *d, hipError_t e) {
  if (d->seq_err == hipSuccess) d->seq_err = e;
}

// records an event pair around one launch on stream s when profiling
struct Span {
  ecp_dev *d;
  hipStream_t s;
  int i;
  Span(ecp_dev *d_, hipStream_t s_, int fam) : d(d_), s(s_), i(-1) {
    if (!d->profiling) return;
    if ((size_t)(2 * d->npev + 2) > d->pev.size()) {
      hipEvent_t a = nullptr, b = nullptr;
      seq(d, hipEventCreate(&a));
      seq(d, hipEventCreate(&b));
      d->pev.push_back(a);
      d->pev.push_back(b);
      d->pfam.push_back(fam);
    }
    i = d->npev++;
    d->pfam[i] = fam;
    seq(d, hipEventRecord(d->pev[2 * i], s));
  }
  ~Span() {
    if (i >= 0) seq(d, hipEventRecord(d->pev[2 * i + 1], s));
  }
};
}  // namespace

namespace {

int toff_key(int la, int lb, int l) { return (la * (ECP_MAX_LBS + 1) + lb) * (ECP_MAX_L + 1) + l; }

// T_l entries (lambda1, lambda2, alpha+beta) with a possibly non-zero angular
// factor: lambda1 from max((alpha+l) mod 2, l-alpha) to l+alpha in steps of 2
// (the lower limit of type2.c:590-592; the angular table vanishes above
// l+alpha, angular_integrals.c:77), likewise lambda2 with beta.
void build_templates(ecp_dev *d) {
  d->tmpl.clear();
  d->toff.clear();
  for (int la = 0; la <= ECP_MAX_LBS; la++)
    for (int lb = 0; lb <= ECP_MAX_LBS; lb++) {
      for (int l = 0; l < ECP_MAX_L; l++) {
        d->toff.push_back((int)d->tmpl.size());
        const int d1 = la + l + 1, d2 = lb + l + 1, d3 = la + lb + 1;
        std::vector<char> used((size_t)d1 * d2 * d3, 0);
        for (int alpha = 0; alpha <= la; alpha++)
          for (int beta = 0; beta <= lb; beta++)
            for (int l1 = std::max((alpha + l) % 2, l - alpha); l1 <= l + alpha; l1 += 2)
              for (int l2 = std::max((beta + l) % 2, l - beta); l2 <= l + beta; l2 += 2)
                used[((size_t)l1 * d2 + l2) * d3 + alpha + beta] = 1;
        for (int l1 = 0; l1 < d1; l1++)
          for (int l2 = 0; l2 < d2; l2++)
            for (int l3 = 0; l3 < d3; l3++)
              if (used[((size_t)l1 * d2 + l2) * d3 + l3]) d->tmpl.push_back(l1 | (l2 << 8) | (l3 << 16) | (l << 24));
      }
      d->toff.push_back((int)d->tmpl.size());
    }
}

void reset_graph(ecp_dev *d) {
  for (int k = 0; k < d->ngraph; k++) {
    if (d->gexec[k]) (void)hipGraphExecDestroy(d->gexec[k]);
    if (d->graph[k]) (void)hipGraphDestroy(d->graph[k]);
    d->gexec[k] = nullptr;
    d->graph[k] = nullptr;
  }
  d->ngraph = 0;
  d->replays = 0;
}

}  // namespace

// The terms of the shift of shells l = 0 .. 6, component after component,
// alpha in the loop order of util.c:277-320, a word each: component (5 bits),
// a - alpha (3 bits an axis), position of alpha (7), product of the binomials
// C(a, alpha) (5: at most 20), distance from the component's first term (5)
// and whether it is the component's last.
static std::vector<unsigned> shift_table(const ecp_static *st) {
  std::vector<unsigned> tab;
  double f[8] = {1.0};
  for (int i = 1; i < 8; i++) f[i] = f[i - 1] * i;
  auto binom = [&](int n, int k) { return (unsigned)(f[n] / (f[n - k] * f[k])); };
  for (int l = 0; l <= 6 && l < st->ijkDim; l++)
    for (int c = 0; c < ECP_DIM_IJK(l); c++) {
      const int *e = st->ijk + 3 * ECP_IDX_C(l, c);
      unsigned d = 0;
      for (int x = 0; x <= e[0]; x++)
        for (int y = 0; y <= e[1]; y++)
          for (int z = 0; z <= e[2]; z++, d++) {
            const unsigned r = (unsigned)st->ijkIndex[(x * st->ijkDim + y) * st->ijkDim + z];
            const unsigned b = binom(e[0], x) * binom(e[1], y) * binom(e[2], z);
            const bool last = x == e[0] && y == e[1] && z == e[2];
            tab.push_back((unsigned)c | (unsigned)(e[0] - x) << 5 | (unsigned)(e[1] - y) << 8 |
                          (unsigned)(e[2] - z) << 11 | r << 14 | b << 21 | d << 26 | (unsigned)last << 31);
          }
    }
  return tab;
}

extern "C" ecp_dev *ecp_dev_create(const ecp_static *st, char *err, size_t errlen) {
  ecp_dev *d = new ecp_dev();
  auto fail = [&](const char *what, hipError_t e) {
    snprintf(err, errlen, "%s: %s", what, hipGetErrorString(e));
    ecp_dev_destroy(d);
    return (ecp_dev *)nullptr;
  };
  hipError_t e;
  int ndev = 0;
  if ((e = hipGetDeviceCount(&ndev)) != hipSuccess || ndev == 0) {
    snprintf(err, errlen, "no HIP device available (%s)", hipGetErrorString(e));
    delete d;
    return nullptr;
  }
  {
    int dev = 0, v = 0;
    if ((e = hipGetDevice(&dev)) != hipSuccess) return fail("hipGetDevice", e);
    if ((e = hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev)) != hipSuccess)
      return fail("hipDeviceGetAttribute", e);
    d->lds_max = v;
  }
  if ((e = hipStreamCreateWithFlags(&d->stream, hipStreamNonBlocking)) != hipSuccess) return fail("hipStreamCreate", e);
  for (int i = 0; i < kWorkers; i++) {
    if ((e = hipStreamCreateWithFlags(&d->workers[i], hipStreamNonBlocking)) != hipSuccess)
      return fail("hipStreamCreate", e);
    if ((e = hipEventCreateWithFlags(&d->join[i], hipEventDisableTiming)) != hipSuccess)
      return fail("hipEventCreate", e);
  }
  if ((e = hipEventCreateWithFlags(&d->fork, hipEventDisableTiming)) != hipSuccess) return fail("hipEventCreate", e);
  for (int k = 0; k < kSpanGraphs; k++)
    for (int i = 0; i < 2; i++)
      if ((e = hipEventCreate(&d->span[k][i])) != hipSuccess) return fail("hipEventCreate", e);
  for (int i = 0; i < 8; i++)
    if ((e = hipEventCreate(&d->ev[i])) != hipSuccess) return fail("hipEventCreate", e);
  for (int i = 0; i < 2; i++)
    if ((e = hipEventCreate(&d->con_ev[i])) != hipSuccess) return fail("hipEventCreate", e);
  if (scratch_setup(&d->scratch, err, errlen)) {
    ecp_dev_destroy(d);
    return nullptr;
  }
  build_templates(d);
  const int so = ECP_SMALL_ORDER, lo = st->lorder;
  const size_t nbess = (size_t)(ECP_BESSEL_N + 1) * ECP_BESSEL_STRIDE;
  const size_t npoly = (size_t)ECP_DIM_C(st->tmDim) * ECP_DIM_L(st->tmDim);
  const size_t nom = (size_t)ECP_DIM_L(st->omL) * ECP_DIM_L(st->omLambda) * ECP_DIM_C(st->omAlpha);
  const size_t nijk = 3 * (size_t)ECP_DIM_C(st->ijkDim - 1);
  const size_t nidx = (size_t)st->ijkDim * st->ijkDim * st->ijkDim;
  const size_t nfac = 2 * (size_t)st->tmDim + 6;
  size_t off = 0;
  auto take = [&](size_t bytes) {
    size_t o = off;
    off += align_up(bytes);
    return o;
  };
  const size_t o_xs = take(so * 8), o_ws = take(so * 8), o_xl = take(lo * 8), o_wl = take(lo * 8);
  const size_t o_p93l = take(so * 4), o_p93r = take(so * 4), o_p92l = take(lo * 4), o_p92r = take(lo * 4);
  const size_t o_vis = take(so * 4), o_v93 = take((st->s93.npairs + kPs93Pad) * sizeof(Ps93Pair));
  const size_t o_bess = take(nbess * 8), o_poly = take(npoly * 8), o_om = take(nom * 8);
  const size_t o_ijk = take(nijk * 4), o_idx = take(nidx * 4);
  const size_t o_snorm = take(kSphDim * kSphDim * 8), o_dfac = take(nfac * 8), o_inv = take(kSphDim * 8);
  const std::vector<unsigned> shift = shift_table(st);
  const size_t o_shift = take(shift.size() * 4 + 4);
  const int prodN = ECP_DIM_C(st->omAlpha);
  const size_t o_prod = take((size_t)prodN * prodN * 4);
  const size_t o_tmpl = take(d->tmpl.size() * 4 + 4), o_toff = take(d->toff.size() * 4);
  std::vector<char> h(off, 0);
  auto put = [&](size_t o, const void *src, size_t bytes) { memcpy(h.data() + o, src, bytes); };
  put(o_xs, st->xs, so * 8);
  put(o_ws, st->ws, so * 8);
  put(o_xl, st->xl, lo * 8);
  put(o_wl, st->wl, lo * 8);
  put(o_p93l, st->p93l, so * 4);
  put(o_p93r, st->p93r, so * 4);
  put(o_p92l, st->p92l, lo * 4);
  put(o_p92r, st->p92r, lo * 4);
  {
    std::vector<Ps93Pair> v(st->s93.npairs + kPs93Pad);
    for (int k = 0; k < (int)v.size(); k++) {
      const int i = std::min(k, st->s93.npairs - 1), li = st->p93l[i], ri = st->p93r[i];
      v[k] = Ps93Pair{st->ws[li], st->ws[ri], li, ri, 0, 0};
    }
    for (int lv = 2; lv < st->s93.nlevels; lv++) {
      v[st->s93.lvl_begin[lv + 1] - 1].ends = lv;
      // what ps93_level relies on
      if (3 * st->s93.lvl_n[lv] != 9 << (lv >> 1) || st->s93.lvl_j[lv] != 1 - (lv & 1)) {
        snprintf(err, errlen, "unexpected PS93 schedule");
        ecp_dev_destroy(d);
        return nullptr;
      }
    }
    put(o_v93, v.data(), v.size() * sizeof(Ps93Pair));
    std::vector<int> vis(so, -1);
    vis[st->s93.centre] = 0;
    vis[st->s93.first_l] = 1;
    vis[st->s93.first_r] = 2;
    for (int k = 0; k < st->s93.npairs; k++) {
      vis[st->p93l[k]] = 3 + 2 * k;
      vis[st->p93r[k]] = 4 + 2 * k;
    }
    put(o_vis, vis.data(), so * 4);
  }
  put(o_bess, st->bessel, nbess * 8);
  put(o_poly, st->poly2sph, npoly * 8);
  put(o_om, st->omega, nom * 8);
  put(o_ijk, st->ijk, nijk * 4);
  put(o_idx, st->ijkIndex, nidx * 4);
  {
    std::vector<double> nrm(kSphDim * kSphDim, 0.0), inv(kSphDim, 0.0);
    for (int l = 0; l < kSphDim; l++) {
      const double norm0 = sqrt((2.0 * l + 1.0) / (2.0 * M_PI));
      for (int m = 0; m <= l && l + m < (int)nfac; m++)
        nrm[l * kSphDim + m] = m == 0 ? norm0 : sqrt(st->fac[l - m] / st->fac[l + m]) * norm0;
      if (l > 0) inv[l] = 1.0 / l;
    }
    put(o_snorm, nrm.data(), nrm.size() * 8);
    put(o_inv, inv.data(), inv.size() * 8);
    std::vector<int> prod((size_t)prodN * prodN);
    for (int r = 0; r < prodN; r++)
      for (int q = 0; q < prodN; q++) {
        const int *a = st->ijk + 3 * r, *c = st->ijk + 3 * q, D = st->ijkDim;
        prod[(size_t)r * prodN + q] = st->ijkIndex[((a[0] + c[0]) * D + a[1] + c[1]) * D + a[2] + c[2]];
      }
    put(o_prod, prod.data(), prod.size() * 4);
    put(o_shift, shift.data(), shift.size() * 4);
  }
  put(o_dfac, st->dfac, nfac * 8);
  put(o_tmpl, d->tmpl.data(), d->tmpl.size() * 4);
  put(o_toff, d->toff.data(), d->toff.size() * 4);
  if ((e = alloc_or_trim([&] { return hipMalloc(&d->static_mem, off); })) != hipSuccess)
    return fail("hipMalloc(static tables)", e);
  if ((e = hipMemcpy(d->static_mem, h.data(), off, hipMemcpyHostToDevice)) != hipSuccess)
    return fail("hipMemcpy(static tables)", e);
  char *b = (char *)d->static_mem;
  DevTables &T = d->T;
  T.xs = (const double *)(b + o_xs);
  T.ws = (const double *)(b + o_ws);
  T.xl = (const double *)(b + o_xl);
  T.wl = (const double *)(b + o_wl);
  T.p93l = (const int *)(b + o_p93l);
  T.p93r = (const int *)(b + o_p93r);
  T.p92l = (const int *)(b + o_p92l);
  T.p92r = (const int *)(b + o_p92r);
  T.v93 = (const Ps93Pair *)(b + o_v93);
  T.vis = (const int *)(b + o_vis);
  T.bessel = (const double *)(b + o_bess);
  T.poly2sph = (const double *)(b + o_poly);
  T.omega = (const double *)(b + o_om);
  T.ijk = (const int *)(b + o_ijk);
  T.ijkIndex = (const int *)(b + o_idx);
  T.snorm = (const double *)(b + o_snorm);
  T.dfac = (const double *)(b + o_dfac);
  T.inv = (const double *)(b + o_inv);
  T.prod = (const int *)(b + o_prod);
  T.prodN = prodN;
  T.shift = (const unsigned *)(b + o_shift);
  T.tmpl = (const int *)(b + o_tmpl);
  T.toff = (const int *)(b + o_toff);
  T.ijkDim = st->ijkDim;
  T.tmDim = st->tmDim;
  T.lorder = st->lorder;
  T.omL = st->omL;
  T.omLambda = st->omLambda;
  T.omAlpha = st->omAlpha;
  T.tol = st->tolerance;
  T.lnAcc1 = st->lnAcc1;
  T.lnAcc2 = st->lnAcc2;
  T.accuracy = st->accuracy;
  T.s93 = st->s93;
  T.s92 = st->s92;
  return d;
}

extern "C" void ecp_dev_destroy(ecp_dev *d) {
  if (!d) return;
  if (d->stream) (void)hipStreamSynchronize(d->stream);
  reset_graph(d);
  if (d->static_mem) (void)hipFree(d->static_mem);
  if (d->arena) (void)hipFree(d->arena);
  if (d->pin_in) (void)hipHostFree(d->pin_in);
  if (d->pin_out) (void)hipHostFree(d->pin_out);
  if (d->fbf) (void)hipFree(d->fbf);
  for (int i = 0; i < 8; i++)
    if (d->ev[i]) (void)hipEventDestroy(d->ev[i]);
  for (int i = 0; i < kWorkers; i++) {
    if (d->workers[i]) (void)hipStreamSynchronize(d->workers[i]);
    if (d->workers[i]) (void)hipStreamDestroy(d->workers[i]);
    if (d->join[i]) (void)hipEventDestroy(d->join[i]);
  }
  if (d->fork) (void)hipEventDestroy(d->fork);
  for (int k = 0; k < kSpanGraphs; k++)
    for (int i = 0; i < 2; i++)
      if (d->span[k][i]) (void)hipEventDestroy(d->span[k][i]);
  for (auto e : d->pev) (void)hipEventDestroy(e);
  if (d->con_mem) (void)hipFree(d->con_mem);
  for (int i = 0; i < 2; i++)
    if (d->con_ev[i]) (void)hipEventDestroy(d->con_ev[i]);
  if (d->stream) (void)hipStreamDestroy(d->stream);
  delete d;
}

extern "C" int ecp_dev_last_timing(ecp_dev *d, double *ms, int n) {
  int k = std::min(n, d->nev);
  for (int i = 0; i < k; i++) ms[i] = d->last_ms[i];
  return k;
}

namespace {

// chunks of a point's values in the type-2 small grid: basis l <= 3 with
// projectors l <= 3 (24; packed triplets 14), basis l <= 4 with projectors
// l <= 4 (35; 17), and the largest (63; 23)
void launch_type2(ecp_dev *d, hipStream_t s) {
  const Prepared &P = d->P;
  if (P.ntot2 <= 0) return;
  T2Args A{P.Tout, P.tf, P.tnfail, P.flist, P.fbq2, P.fbc + kFb2Cnt, P.nt, P.tcls2};
  Span sp(d, s, FAM_TYPE2);
  if (P.nt <= kT2Small && P.max_lbs <= 4 && P.max_L <= 5) {
    const int ns = std::max(1, std::min((P.max_ent2 + 63) / 64, kT2Fill / P.nt));
    if (P.max_lbs <= 3 && P.max_L <= 4) k_type2_small<24><<<P.nt * ns, 64, 0, s>>>(d->T, P.J, A, P.tcls, ns);
    else k_type2_small<35><<<P.nt * ns, 64, 0, s>>>(d->T, P.J, A, P.tcls, ns);
    return;
  }
  const int m = P.tcls_begin[kT2PackLab + 1];
  const int n = P.nt - m, npass = (P.max_ent2 + kT2Pass - 1) / kT2Pass;
  const int ns = std::max(1, std::min(npass, kT2Fill / std::max(n, 1)));
  const int grid = n * ns + (m + kT2Pack - 1) / kT2Pack;
  if (P.max_lbs <= 3 && P.max_L <= 4) k_type2<24, 14><<<grid, 64, 0, s>>>(d->T, P.J, A, P.tcls, m, ns);
  else if (P.max_lbs <= 4 && P.max_L <= 5) k_type2<35, 17><<<grid, 64, 0, s>>>(d->T, P.J, A, P.tcls, m, ns);
  else k_type2<63, 23><<<grid, 64, 0, s>>>(d->T, P.J, A, P.tcls, m, ns);
}

// Jobs of up to this many type-2 blocks (of classes above kAsmPackLab) give
// each 256 threads: 17 atoms 197 -> 180 us an evaluation; 50 atoms (1000 to
// 4000 such blocks) lose, 379 -> 398 us, and 256 molecules are unchanged to
// 19 % slower.
constexpr int kAsm2Wide = 1024;

// type-2 assembly: the register-cached variant fits basis l <= 3 with
// projectors l <= 3, or basis l <= 4 with projectors l <= 4; larger jobs (and
// asm2_cache 0) read the tables directly.  The triplets of classes la + lb
// <= kAsmPackLab (the first of the class-ordered list) go kAsmPack to a
// wave, the others one per workgroup: a wave where the job fills the chip,
// 256 threads where it does not and for the largest classes, whose LDS lets
// few workgroups share a CU (i shells, L = 7: 5477 -> 2092 us with the split
// small grid).
void launch_asm2(ecp_dev *d, hipStream_t s) {
  const Prepared &P = d->P;
  Span sp(d, s, FAM_ASM);
  const bool cache = d->tune.asm2_cache != 0;
  const int m = P.tcls_begin[kAsmPackLab + 1], n = P.nt - m;
  auto go = [&](auto kernel, int g, size_t lds, const AsmArgs &aa, const int *tl, int ntl, int nt = kAsmThreads) {
    if (g > 0) kernel<<<g, nt, lds, s>>>(d->T, P.J, aa, P.stat, tl, ntl);
  };
  const int *tl = P.tcls + m;
  const bool wide = n <= kAsm2Wide;
  if (cache && P.max_lbs <= 3 && P.max_L <= 4 && wide) go(k_asm2<1, 4, 4, 256>, n, P.asm2_lds, P.aa, tl, n, 256);
  else if (cache && P.max_lbs <= 4 && P.max_L <= 5 && wide)
    go(k_asm2<1, 5, 5, 256>, n, P.asm2_lds, P.aa, tl, n, 256);
  else if (cache && P.max_lbs <= 3 && P.max_L <= 4) go(k_asm2<1, 4, 4>, n, P.asm2_lds, P.aa, tl, n);
  else if (cache && P.max_lbs <= 4 && P.max_L <= 5) go(k_asm2<1, 5, 5>, n, P.asm2_lds, P.aa, tl, n);
  else go(k_asm2<1, 0, 7, 256>, n, P.asm2_lds, P.aa, tl, n, 256);
  const int gp = (m + kAsmPack - 1) / kAsmPack;
  if (P.max_L <= 4) go(k_asm2<kAsmPack, kAsmPackLab + 1, 4>, gp, P.asm2_lds4, P.aa2p, P.tcls, m);
  else if (P.max_L == 5) go(k_asm2<kAsmPack, kAsmPackLab + 1, 5>, gp, P.asm2_lds4, P.aa2p, P.tcls, m);
  else go(k_asm2<kAsmPack, 0, 7>, gp, P.asm2_lds4, P.aa2p, P.tcls, m);
}

// type-1 assembly of the triplets tcls[b .. e) (class-ordered), one per
// wave, those of classes la + lb <= kAsmPackLab kAsmPack to a wave
// cls >= 0: every triplet of the range is of class la + lb = cls (per-class
// launches), which bounds the monomial degrees the kernel holds in registers
void launch_asm1(ecp_dev *d, hipStream_t s, int b, int e, int cls = -1) {
  const Prepared &P = d->P;
  Span sp(d, s, FAM_ASM);
  const int m = std::min(std::max(b, P.tcls_begin[kAsmPackLab + 1]), e);
  if (m > b)
    k_asm1<kAsmPack, kAsmPackLab><<<(m - b + kAsmPack - 1) / kAsmPack, kAsmThreads, P.asm1_lds4, s>>>(
        d->T, P.J, P.aa4, P.stat, P.tcls + b, m - b);
  if (e <= m) return;
  const dim3 g(e - m);
  switch (cls) {
#define ASM1(D)                                                                              \
  case D:                                                                                  \
    k_asm1<1, D><<<g, kAsmThreads, P.asm1_lds, s>>>(d->T, P.J, P.aa, P.stat, P.tcls + m, e - m); \
    break;
    ASM1(3) ASM1(4) ASM1(5)
#undef ASM1
    default:
      // classes above 5 and mixed-class launches: rows up to degree 6 in
      // registers (the uneven batch's class-6 chain 0.7 ms slower with
      // degree 6 in the general loop)
      k_asm1<1, 6><<<g, kAsmThreads, P.asm1_lds, s>>>(d->T, P.J, P.aa, P.stat, P.tcls + m, e - m);
  }
}

T1Set t1_set(const ecp_dev *d) {
  const Prepared &P = d->P;
  T1Set S{};
  S.units = P.u1;
  S.q = P.q;
  S.qf = P.qf;
  S.fbq = P.fbq1;
  S.fbc = P.fbc;
  S.tq = P.tq1;
  S.st = P.t1s;
  S.plane = P.nq;
  S.stat = P.stat;
  for (int c = 0; c <= ECP_MAX_LAB; c++) {
    S.ubeg[c] = P.cls_begin[c];
    S.ucnt[c] = P.cls_count[c];
  }
  // the head always takes levels 0 and 1, so the tail starts at 2 or later
  S.head = std::max(2, d->tune.t1_head_coop);
  return S;
}

// Type-1 quadrature of one class: the head, then the tail and the large-grid
// fallbacks in one persistent launch
template <int LAB>
void launch_type1(ecp_dev *d, hipStream_t s, const T1Set &S) {
  const int n = S.ucnt[LAB], ub = S.ubeg[LAB];
  if (n <= 0) return;
  {
    Span sp(d, s, FAM_TYPE1);
    k_type1<LAB><<<(n + 63) / 64, 64, 0, s>>>(d->T, d->P.J, S.units + ub, n, S.q, S.qf + ub, S.fbq + ub, S.fbc + LAB,
                                              S.head, S.st, S.plane, S.tq + ub, S.fbc + 32 + LAB);
  }
  Span sp(d, s, FAM_T1TAIL);
  k_t1tail<LAB><<<std::min(n, d->tune.t1_tail_grid), 64, 0, s>>>(d->T, d->P.J, S.units + ub, S.q, S.qf + ub,
                                                                 S.fbq + ub, S.fbc + LAB, S.head, S.st, S.plane,
                                                                 S.tq + ub, S.fbc + 32 + LAB, S.stat);
}

// workgroup ranges of the classes with work; blocks(c) = workgroups of class c
template <typename F>
ClassMap class_map(int ncls, const int *count, F blocks) {
  ClassMap cm{};
  int b = 0;
  for (int c = 0; c < ncls; c++) {
    if (count[c] <= 0) continue;
    const int nb = blocks(c);
    if (nb <= 0) continue;
    cm.cls[cm.n] = c;
    cm.bbeg[cm.n] = b;
    b += nb;
    cm.n++;
  }
  cm.bbeg[cm.n] = b;
  return cm;
}

// the type-2 fallback classes of cm in one grid; like the type-1 kernels,
// four tiers bound the Bessel orders the grid holds: up to 7, 8, 11 and 12
void launch_fb2_fused(ecp_dev *d, hipStream_t s, const T2Set &S2, const ClassMap &cm) {
  const Prepared &P = d->P;
  const int nb = cm.bbeg[cm.n];
  // 13.1 KB for projectors up to f and class 6: twelve waves per CU, what
  // the registers (148) allow
  const size_t lds = sizeof(double) * (kFb2Chunk * kFbTS + (S2.cu_rows + S2.rn_rows + 2 * S2.k_rows) * 64);
  if (P.max_cls2 > 11) k_fb2_fused<12><<<nb, 64, lds, s>>>(d->T, P.J, S2, cm);
  // (class 8, g shells under L = 5, without class 11's scratch: 20 atoms
  // 4450 -> 3864 us an evaluation)
  else if (P.max_cls2 > 8) k_fb2_fused<11><<<nb, 64, lds, s>>>(d->T, P.J, S2, cm);
  else if (P.max_cls2 > 7) k_fb2_fused<8><<<nb, 64, lds, s>>>(d->T, P.J, S2, cm);
  else k_fb2_fused<7><<<nb, 64, lds, s>>>(d->T, P.J, S2, cm);
}

// Waves per triplet of the type-2 fallback (nslot: its primitive pairs are
// dealt to them) and the entries per wave (share), by the job's (triplet,
// pair) items.  Many short waves where the fallback's latency counts, few
// long ones where the wave's set-up (triplet, shells, entry list: a chain of
// dependent reads) and the points evaluated once per share are what the chip
// spends its time on.  Fallback alone, one wave per pair / three / one per
// triplet at the shares given: the 50-atom cluster (72 k items) 120 / 150 /
// 432 us, its gradient (222 k) 260 / 319 / 576, 20 atoms with g shells
// (445 k) 1910 / 1557 / 2176, 256 uneven molecules (6.2 M) 5916 / 4208 /
// 3917.  fb2_split > 0 sets the number of shares instead.
void fb2_slots(const ecp_dev *d, T2Set &S) {
  const int maxPairs = d->P.maxPairs;
  long items = 0;
  for (int c = 0; c <= kMaxLMB; c++) items += (long)d->P.tcount2[c] * maxPairs;
  S.nslot = items <= 300000 ? maxPairs : items <= 2000000 ? std::min(maxPairs, 3) : 1;
  S.share = items <= 100000 ? 64 : items <= 300000 || d->P.max_cls2 <= 7 ? 128 : 256;
  const int v = d->tune.fb2_split;
  S.nsplit = v > 0 ? std::min(v, 8) : (d->P.max_ent2 + S.share - 1) / S.share;
  S.cu_rows = d->P.max_L;
  S.rn_rows = d->P.max_lab + 1;
  S.k_rows = d->P.max_cls2 + 1;
}

ClassMap fb2_classes(const ecp_dev *d, const T2Set &S) {
  return class_map(kMaxLMB + 1, d->P.tcount2, [&](int c) {
    return (int)std::min<long>((long)d->P.tcount2[c] * S.nslot * S.nsplit, 8192);
  });
}

void enqueue_fused(ecp_dev *d, hipStream_t s, hipEvent_t *evs);

// parts of the tables launch: what type 1 needs (with the zero-fill), and
// the rest, which only type 2 reads
constexpr int kTabFront = 1, kTabBack = 2;

void launch_tables(ecp_dev *d, hipStream_t s, int parts) {
  const Prepared &P = d->P;
  TabArgs A{};
  A.zero_base = P.zero_base;
  A.zero_words = P.zero_words;
  A.nzb = (int)std::max<size_t>(1, std::min<size_t>((P.zero_words + 127) / 128, 2048));
  A.rows = P.max_L + 1;
  A.nub = P.ncent * A.rows * kUtabChunks;
  A.nfit = P.nfit;
  A.fit = P.fit;
  A.units = P.u1;
  A.udir = P.udir;
  A.t1first = P.aa.t1first;
  for (int c = 0; c <= ECP_MAX_LAB; c++) {
    A.cls_begin[c] = P.cls_begin[c];
    A.cls_qbase[c] = P.cls_qbase[c];
  }
  A.ait = P.ait;
  A.nait = P.nait;
  // few pairs: several workgroups each (20 atoms with g shells, 160 pairs:
  // the launch 116 us at one, 4556 workgroups in all)
  A.aparts = P.nait < 1024 ? 4 : 1;
  int units = (int)(((size_t)P.nt * P.maxPairs + 127) / 128);
  if (!(parts & kTabFront)) A.nzb = A.nub = units = 0;
  if (!(parts & kTabBack)) A.nait = A.nfit = 0;
  const int grid = A.nait * A.aparts + A.nzb + A.nub + A.nfit + units;
  if (grid == 0) return;
  Span sp(d, s, FAM_TABLES);
  k_tables<<<grid, 128, 0, s>>>(d->T, P.J, A);
}

// fuse = 2 (automatic), by the job's type-1 primitive pairs.  Up to
// kFuseAutoSmall fused launches: per-class ones hold few waves each.  Up to
// kFuseAutoLarge per class, each class with its own registers.  Above, fused
// again where the largest class is 6: every stage fills the chip by itself.
// Replays, us, fused / per class: 8001 pairs 135 / 214, 119 934 348 / 361,
// 149 436 443 / 433, 196 659 567 / 556, 290 133 687 / 662, 328 707 865 / 888,
// 548 541 1146 / 1244, 852 570 1834 / 2003; classes up to 8: 459 360 4823 /
// 4571, 880 656 7228 / 7503.  So the lower edge is at the crossing; the upper
// one is above it, and the class limit holds back jobs of classes up to 8.
constexpr int kFuseAutoSmall = 150000, kFuseAutoLarge = 800000;

bool fuse_auto(int units, int max_lab) {
  return units <= kFuseAutoSmall || (units > kFuseAutoLarge && max_lab <= 6);
}

// The tables, and the fork of the first nw workers, which take the type-1
// work, off the main stream.  Captured small jobs split the launch, so that
// the type-1 chain does not wait for the tables of type 2: replays of a tiny
// molecule 146 -> 137 us, 17 atoms 174 -> 165 us, 50 atoms 330 -> 314 us.
// Eager, the second launch costs what it gains (tiny molecule 234 -> 242 us a
// call), and large jobs gain nothing (50-atom gradient 784 -> 799 us, 20
// atoms with g shells 3509 -> 3523 us, 256 molecules 12458 -> 12392 us).
void fork_tables(ecp_dev *d, hipStream_t s, int nw, hipEvent_t *evs) {
  const bool split = d->capturing && d->P.cls_begin[ECP_MAX_LAB + 1] <= kFuseAutoSmall;
  launch_tables(d, s, split ? kTabFront : kTabFront | kTabBack);
  seq(d, hipEventRecord(d->fork, s));
  for (int i = 0; i < nw; i++) seq(d, hipStreamWaitEvent(d->workers[i], d->fork, 0));
  if (split) launch_tables(d, s, kTabBack);
  if (evs) seq(d, hipEventRecord(evs[1], s));
}

// one type-1 class of the per-class sequence: quadrature, assembly
template <int c>
void enqueue_t1_class_t(ecp_dev *d, hipStream_t ws) {
  const Prepared &P = d->P;
  launch_type1<c>(d, ws, t1_set(d));
  if (P.tcls_begin[c + 1] > P.tcls_begin[c]) launch_asm1(d, ws, P.tcls_begin[c], P.tcls_begin[c + 1], c);
}

void enqueue_t1_class(ecp_dev *d, hipStream_t ws, int c) {
  switch (c) {
#define T1(c) \
  case c:     \
    enqueue_t1_class_t<c>(d, ws); \
    break;
    T1(0) T1(1) T1(2) T1(3) T1(4) T1(5) T1(6) T1(7) T1(8) T1(9) T1(10) T1(11) T1(12)
#undef T1
  }
}

// The kernel sequence of one evaluation, on resident inputs: fused launches
// (enqueue_fused), or tables on the main stream, then there the type-2 chain
// and beside it, on the workers, the type-1 classes, each as head -> tail and
// large-grid fallback -> assembly.  With evs, stage boundaries are recorded on
// the main stream: start, tables done, end, end (assembly overlaps the
// quadratures).
void enqueue(ecp_dev *d, hipStream_t s, hipEvent_t *evs) {
  const int units = d->P.cls_begin[ECP_MAX_LAB + 1];
  const bool fused = d->tune.fuse == 1 || (d->tune.fuse == 2 && fuse_auto(units, d->P.max_lab));
  if (fused) {
    enqueue_fused(d, s, evs);
    return;
  }
  const Prepared &P = d->P;
  const DevTables &T = d->T;
  const DevJob &J = P.J;
  hipStream_t *w = d->workers;
  d->span_valid = false;  // type-1 classes run on several streams
  if (evs) seq(d, hipEventRecord(evs[0], s));
  fork_tables(d, s, kWorkers, evs);
  // the type-2 chain (small grid, fallbacks, assembly) on the main stream,
  // beside it the type-1 classes on three workers: one stream per hardware
  // queue the device gives a process
  const int nw1 = kWorkers;
  if (P.ntot2 > 0) {
    launch_type2(d, s);
    // every fallback class in one persistent grid: the classes' items run
    // side by side instead of one class after another on this stream
    T2Set S2{P.fbq2, P.fbc, P.fbT, P.stat, P.nt, P.tnfail, P.flist, 1, 1, 1, 0, 0, 0};
    fb2_slots(d, S2);
    const ClassMap cm2 = fb2_classes(d, S2);
    if (cm2.n > 0) {
      Span sp(d, s, FAM_FB2);
      launch_fb2_fused(d, s, S2, cm2);
    }
    launch_asm2(d, s);
  }
  // type-1 classes, each followed by its assembly, on one of the
  // workers: the costliest class first, each on the worker with the
  // least work so far (the cost of a class: its algorithmic small-grid
  // FLOPs), so that no large class starts last and runs alone at the end
  int order[ECP_MAX_LAB + 1], nord = 0;
  for (int c = 0; c <= ECP_MAX_LAB; c++)
    if (P.cls_count[c] > 0) order[nord++] = c;
  std::stable_sort(order, order + nord, [&](int a, int b) { return P.flops_t1[a] > P.flops_t1[b]; });
  double load[kWorkers] = {};
  for (int i = 0; i < nord; i++) {
    int k = 0;
    for (int j = 1; j < nw1; j++)
      if (load[j] < load[k]) k = j;
    load[k] += P.flops_t1[order[i]];
    enqueue_t1_class(d, w[k], order[i]);
  }
  for (int i = 0; i < kWorkers; i++) {
    seq(d, hipEventRecord(d->join[i], w[i]));
    seq(d, hipStreamWaitEvent(s, d->join[i], 0));
  }
  if (evs) {
    seq(d, hipEventRecord(evs[2], s));
    seq(d, hipEventRecord(evs[3], s));
  }
}

// Event i of the quadrature's pair, on stream s.  Under capture an event
// record node of the graph, so that replays record it too: added to the graph
// itself, since hipEventRecordWithFlags with hipEventRecordExternal is refused
// by HIP 7.0 runtimes (one may be in the process before this library).
hipError_t record_span(ecp_dev *d, hipStream_t s, int i) {
  hipEvent_t ev = d->span[d->span_k][i];
  if (!d->capturing) return hipEventRecord(ev, s);
  hipStreamCaptureStatus st;
  hipGraph_t g = nullptr;
  const hipGraphNode_t *dep = nullptr;
  size_t ndep = 0;
  hipError_t e = hipStreamGetCaptureInfo_v2(s, &st, nullptr, &g, &dep, &ndep);
  if (e != hipSuccess) return e;
  if (st != hipStreamCaptureStatusActive) return hipErrorStreamCaptureInvalidated;
  hipGraphNode_t node;
  e = hipGraphAddEventRecordNode(&node, g, dep, ndep, ev);
  return e != hipSuccess ? e : hipStreamUpdateCaptureDependencies(s, &node, 1, hipStreamSetCaptureDependencies);
}

// The fused sequence: tables on the main stream, then the two chains side by
// side, each stage one launch over every class.  Type 1: head, then tail and
// large-grid fallbacks, then assembly.  Type 2: small grid, fallbacks,
// assembly.  evs: stage boundaries as in enqueue.
void enqueue_fused(ecp_dev *d, hipStream_t s, hipEvent_t *evs) {
  const Prepared &P = d->P;
  const DevTables &T = d->T;
  const DevJob &J = P.J;
  hipStream_t w = d->workers[0];
  d->span_valid = false;
  if (evs) seq(d, hipEventRecord(evs[0], s));
  fork_tables(d, s, 1, evs);
  // ---- type 1 ----
  const T1Set S = t1_set(d);
  // the fused kernels hold the registers of their largest class: four
  // instantiations, classes up to 6, 8, 10 and 12 (8 without spills; with
  // class 10's registers for a class-8 job the evaluation took 2 % longer)
  auto launch = [&](auto f6, auto f8, auto f10, auto f12, const ClassMap &cm) {
    auto f = P.max_lab <= 6 ? f6 : P.max_lab <= 8 ? f8 : P.max_lab <= 10 ? f10 : f12;
    f<<<cm.bbeg[cm.n], 64, 0, w>>>(T, J, S, cm);
  };
  const ClassMap cmh = class_map(ECP_MAX_LAB + 1, P.cls_count, [&](int c) { return (P.cls_count[c] + 63) / 64; });
  if (cmh.n > 0) {
    seq(d, record_span(d, w, 0));
    {
      Span sp(d, w, FAM_TYPE1);
      launch(k_type1_fused<6>, k_type1_fused<8>, k_type1_fused<10>, k_type1_fused<12>, cmh);
    }
    {
      const ClassMap cmt = class_map(ECP_MAX_LAB + 1, P.cls_count,
                                     [&](int c) { return std::min(P.cls_count[c], d->tune.t1_tail_grid); });
      Span sp(d, w, FAM_T1TAIL);
      launch(k_t1tail_fused<6>, k_t1tail_fused<8>, k_t1tail_fused<10>, k_t1tail_fused<12>, cmt);
    }
    seq(d, record_span(d, w, 1));
    d->span_valid = true;
    launch_asm1(d, w, 0, P.nt);
  }
  // ---- type 2 ----
  if (P.ntot2 > 0) {
    launch_type2(d, s);
    T2Set S2{P.fbq2, P.fbc, P.fbT, P.stat, P.nt, P.tnfail, P.flist, 1, 1, 1, 0, 0, 0};
    fb2_slots(d, S2);
    const ClassMap cm2 = fb2_classes(d, S2);
    if (cm2.n > 0) {
      Span sp(d, s, FAM_FB2);
      launch_fb2_fused(d, s, S2, cm2);
    }
    launch_asm2(d, s);
  }
  seq(d, hipEventRecord(d->join[0], w));
  seq(d, hipStreamWaitEvent(s, d->join[0], 0));
  if (evs) {
    seq(d, hipEventRecord(evs[2], s));
    seq(d, hipEventRecord(evs[3], s));
  }
}

// enqueue, with every call's and launch's error looked at: under capture a
// launch that failed would be missing from every replay.  0, or -1 (message
// in err) with nothing of the sequence left running.
int run_sequence(ecp_dev *d, hipStream_t s, hipEvent_t *evs, char *err, size_t errlen) {
  // a stale error of an earlier, unrelated call must not be taken for one of
  // this sequence's
  (void)hipGetLastError();
  d->seq_err = hipSuccess;
  enqueue(d, s, evs);
  seq(d, hipGetLastError());
  if (d->seq_err == hipSuccess) return 0;
  snprintf(err, errlen, "kernel sequence failed: %s", hipGetErrorString(d->seq_err));
  if (!d->capturing) (void)ecp_dev_sync(d);
  return -1;
}

}  // namespace

// Host half of preparing a job: class grouping of the type-1 units, type-2
// entry groups, table work items, the algorithmic FLOP model, and the byte
// layout of the job's device block; the inputs are staged in pinned host
// memory.  *bytes = size of the device block the job needs.
extern "C" int ecp_dev_plan(ecp_dev *d, const ecp_job *job, size_t *bytes, char *err, size_t errlen) {
  Prepared &P = d->P;
  JobLayout &Ly = d->L;
  d->prepared = false;
  d->planned = false;
  d->eager_done = false;
  reset_graph(d);
  if (d->uploading) {
    ECP_CHECK(hipStreamSynchronize(d->stream));
    d->uploading = false;
  }
  P = Prepared();
  Ly = JobLayout();
  const int nt = job->ntrip;
  P.nt = nt;
  P.ncent = job->ncent;
  P.nblk = job->nblk;
  if (bytes) *bytes = 0;
  if (nt == 0) {
    d->planned = true;
    return 0;
  }
  // type-1 units are grouped by class lab, inside a class in triplet order;
  // the tables launch writes them
  for (int t = 0; t < nt; t++) {
    const ecp_triplet &tr = job->trip[t];
    const int c = tr.la + tr.lb, KK = job->shells[tr.sa].K * job->shells[tr.sb].K;
    P.cls_count[c] += KK;
    P.tcls_begin[c + 1]++;
    // per primitive pair: G (31 lambda + 74 + 4 n_Q) + 150 n_Q
    P.flops_t1[c] += KK * ((tr.ge - tr.gs) * (31.0 * c + 74 + 4.0 * nq_of(c)) + 150.0 * nq_of(c));
  }
  for (int c = 0; c <= ECP_MAX_LAB; c++) {
    P.cls_begin[c + 1] = P.cls_begin[c] + P.cls_count[c];
    P.cls_qbase[c + 1] = P.cls_qbase[c] + (size_t)P.cls_count[c] * nq_of(c);
    P.tcls_begin[c + 1] += P.tcls_begin[c];
    if (P.cls_count[c]) P.max_lab = c;
  }
  const size_t nunits = P.cls_begin[ECP_MAX_LAB + 1], nq = P.cls_qbase[ECP_MAX_LAB + 1];
  for (int c = 0; c < job->ncent; c++) {
    const ecp_centre &C = job->cent[c];
    for (int s = 0; s < C.nsh; s++) P.nfit += !job->win[C.win_off + s].skip;
    P.nait += C.nat;
  }
  P.nfit *= job->deriv + 1;
  P.maxPairs = job->maxK * job->maxK;
  // layout: inputs (copied), then device-only buffers; the per-run zeroed
  // counters and flags are contiguous
  size_t in_off = 0;
  auto in_take = [&](size_t b) {
    size_t o = in_off;
    in_off += align_up(b);
    return o;
  };
  Ly.i_atoms = in_take(sizeof(ecp_xyz) * job->nat);
  Ly.i_amaxl = in_take(4 * (size_t)job->nat);
  Ly.i_sh = in_take(sizeof(ecp_shell) * job->nsh);
  Ly.i_pa = in_take(8 * (size_t)job->nprim);
  Ly.i_pd = in_take(8 * (size_t)job->nprim);
  Ly.i_cent = in_take(sizeof(ecp_centre) * job->ncent);
  Ly.i_gauss = in_take(sizeof(ecp_gauss) * job->ngauss);
  Ly.i_win = in_take(sizeof(ecp_window) * job->nwin);
  Ly.i_trip = in_take(sizeof(ecp_triplet) * nt);
  Ly.i_t1f = in_take(4 * (size_t)nt);
  Ly.i_teoff = in_take(4 * (size_t)nt);
  Ly.i_tcls2 = in_take((size_t)nt);
  Ly.i_fit = in_take(sizeof(int2) * P.nfit);
  Ly.i_ait = in_take(sizeof(int2) * P.nait);
  Ly.i_tcls = in_take(4 * (size_t)nt);
  Ly.in_bytes = in_off;
  if (Ly.in_bytes > d->pin_in_cap) {
    if (d->pin_in) ECP_CHECK(hipHostFree(d->pin_in));
    d->pin_in = nullptr;
    d->pin_in_cap = 0;
    ECP_CHECK(alloc_or_trim([&] { return hipHostMalloc(&d->pin_in, Ly.in_bytes + Ly.in_bytes / 4); }));
    d->pin_in_cap = Ly.in_bytes + Ly.in_bytes / 4;
  }
  // the inputs, straight into the staging memory
  char *H = d->pin_in;
  auto cp = [&](size_t o, const void *src, size_t b) {
    if (b) memcpy(H + o, src, b);
  };
  cp(Ly.i_atoms, job->atoms, sizeof(ecp_xyz) * job->nat);
  cp(Ly.i_amaxl, job->atom_maxl, 4 * (size_t)job->nat);
  cp(Ly.i_sh, job->shells, sizeof(ecp_shell) * job->nsh);
  cp(Ly.i_pa, job->pa, 8 * (size_t)job->nprim);
  cp(Ly.i_pd, job->pd, 8 * (size_t)job->nprim);
  cp(Ly.i_cent, job->cent, sizeof(ecp_centre) * job->ncent);
  cp(Ly.i_gauss, job->gauss, sizeof(ecp_gauss) * job->ngauss);
  cp(Ly.i_win, job->win, sizeof(ecp_window) * job->nwin);
  cp(Ly.i_trip, job->trip, sizeof(ecp_triplet) * nt);
  int ntot2 = 0;
  {
    int *t1first = (int *)(H + Ly.i_t1f), *teoff = (int *)(H + Ly.i_teoff), *tcls = (int *)(H + Ly.i_tcls);
    unsigned char *tcls2 = (unsigned char *)(H + Ly.i_tcls2);
    int ufill[ECP_MAX_LAB + 1], tfill[ECP_MAX_LAB + 1];
    for (int c = 0; c <= ECP_MAX_LAB; c++) {
      ufill[c] = P.cls_begin[c];
      tfill[c] = P.tcls_begin[c];
    }
    for (int t = 0; t < nt; t++) {
      const ecp_triplet &tr = job->trip[t];
      const int la = tr.la, lb = tr.lb, c = la + lb, L = job->cent[tr.centre].L;
      t1first[t] = ufill[c];
      ufill[c] += job->shells[tr.sa].K * job->shells[tr.sb].K;
      tcls[tfill[c]++] = t;
      const int c2 = std::max(la, lb) + L - 1;
      tcls2[t] = (unsigned char)c2;
      P.tcount2[c2]++;
      P.max_cls2 = std::max(P.max_cls2, c2);
      const int ne = d->toff[toff_key(la, lb, L)] - d->toff[toff_key(la, lb, 0)];
      teoff[t] = ntot2;
      ntot2 += ne;
      P.max_ent2 = std::max(P.max_ent2, ne);
    }
    int2 *fit = (int2 *)(H + Ly.i_fit), *ait = (int2 *)(H + Ly.i_ait);
    for (int c = 0; c < job->ncent; c++) {
      const ecp_centre &C = job->cent[c];
      for (int run = 0; run <= job->deriv; run++)
        for (int s = 0; s < C.nsh; s++)
          if (!job->win[C.win_off + s].skip) *fit++ = make_int2(c, s * 4 + run);
      for (int a = 0; a < C.nat; a++) *ait++ = make_int2(c, a);
    }
  }
  P.ntot2 = ntot2;
  size_t dv_off = align_up(Ly.in_bytes);
  auto dv_take = [&](size_t b) {
    size_t o = dv_off;
    dv_off += align_up(b);
    return o;
  };
  Ly.d_zero = dv_off;
  Ly.d_fbc = dv_take(4 * kFbcSlots);
  Ly.d_stat = dv_take(2 * (size_t)nt);
  Ly.d_tnf = dv_take(4 * (size_t)nt);
  Ly.d_zero_end = dv_off;
  Ly.d_UL = dv_take(8 * job->nUL);
  Ly.d_Ut = dv_take(8 * job->nUt);
  Ly.d_F = dv_take(8 * job->nF);
  Ly.d_ang = dv_take(8 * job->nang);
  Ly.d_q = dv_take(8 * nq);
  P.nq = nq;
  Ly.d_qf = dv_take(8 * nunits);
  Ly.d_u1 = dv_take(sizeof(T1Unit) * nunits);
  Ly.d_fbq1 = dv_take(4 * nunits);
  Ly.d_T = dv_take(8 * (size_t)ntot2);
  Ly.d_tf = dv_take((size_t)ntot2);
  Ly.d_flist = dv_take(4 * (size_t)ntot2);
  Ly.d_fbq2 = dv_take(4 * (size_t)(kMaxLMB + 1) * nt);
  Ly.d_fbT = dv_take(8 * (size_t)ntot2 * P.maxPairs);
  Ly.d_blk = dv_take(8 * job->nblk);
  Ly.d_t1s = dv_take(2 * 8 * nq);
  Ly.d_tq1 = dv_take(4 * nunits);
  Ly.d_udir = dv_take(32 * nunits);
  Ly.total = dv_off;
  Ly.FL = job->FL;
  Ly.UK = job->UK;
  Ly.US = job->maxL * job->UK;
  Ly.angL = job->angL;
  Ly.ang_lam = job->ang_lam;
  Ly.ang_c = job->ang_c;
  Ly.deriv = job->deriv;
  {
    int LM = 0, LC = 1;
    for (int i = 0; i < job->nsh; i++) LM = std::max(LM, job->shells[i].l + job->deriv);
    for (int c = 0; c < job->ncent; c++) LC = std::max(LC, job->cent[c].L);
    P.max_lbs = LM;
    P.max_L = LC;
    AsmArgs &aa = P.aa;
    aa.pair_chunk = std::min((LM <= 4) ? 16 : 8, std::max(1, P.maxPairs));
    aa.lds_rs_stride = (2 * LM + 1) * (2 * LM + 1);
    int o = 0;
    aa.shift_lm = LM;
    const int ns = shift_tab_doubles(LM);
    aa.lds_J = o; o += ECP_DIM_IJK(LM) * ECP_DIM_C(LM);
    const int base = o;
    // type 1: H stays for the shift; the shift tables reuse rsph and Q
    aa.lds_H = o; o += ECP_DIM_C(2 * LM);
    aa.lds_S1 = o;
    aa.lds_rsph = o; o += aa.pair_chunk * aa.lds_rs_stride;
    aa.lds_Q = o; o += aa.pair_chunk * nq_of(2 * LM);
    const int end1 = std::max(o, aa.lds_S1 + ns);
    // type 2: blk stays for the shift; the shift tables reuse T
    o = base;
    aa.lds_blk = o; o += ECP_DIM_C(LM) * ECP_DIM_C(LM);
    aa.lds_S2 = o;
    aa.lds_T = o; o += t2_slots(LM, LM, LC);
    const int end2 = std::max(o, aa.lds_S2 + ns);
    P.asm1_lds = (size_t)end1 * sizeof(double);
    // packed type 1 (la + lb <= kAsmPackLab): one slice of LDS per triplet
    {
      AsmArgs &a4 = P.aa4;
      const int LS = std::min(LM, kAsmPackLab), LQ = std::min(2 * LM, kAsmPackLab);
      a4.pair_chunk = aa.pair_chunk;
      a4.lds_rs_stride = (LQ + 1) * (LQ + 1);
      a4.shift_lm = LS;
      int o4 = 0;
      a4.lds_J = o4; o4 += ECP_DIM_IJK(LS) * ECP_DIM_C(LS);
      a4.lds_H = o4; o4 += ECP_DIM_C(LQ);
      a4.lds_S1 = o4;
      a4.lds_rsph = o4; o4 += a4.pair_chunk * a4.lds_rs_stride;
      a4.lds_Q = o4; o4 += a4.pair_chunk * nq_of(LQ);
      a4.lds_group = std::max(o4, a4.lds_S1 + shift_tab_doubles(LS));
      P.asm1_lds4 = (size_t)kAsmPack * a4.lds_group * sizeof(double);
    }
    // packed type 2 likewise: blk stays for the shift, whose tables reuse T
    {
      AsmArgs &a2 = P.aa2p;
      const int LS = std::min(LM, kAsmPackLab);
      a2.shift_lm = LS;
      int o2 = 0;
      a2.lds_J = o2; o2 += ECP_DIM_IJK(LS) * ECP_DIM_C(LS);
      a2.lds_blk = o2; o2 += ECP_DIM_C(LS) * ECP_DIM_C(LS);
      a2.lds_S2 = o2;
      a2.lds_T = o2;
      int ts = 0;
      for (int x = 0; x <= LS; x++)
        for (int y = 0; y <= LS; y++)
          if (x + y <= kAsmPackLab) ts = std::max(ts, t2_slots(x, y, LC));
      o2 += ts;
      a2.lds_group = std::max(o2, a2.lds_S2 + shift_tab_doubles(LS));
      P.asm2_lds4 = (size_t)kAsmPack * a2.lds_group * sizeof(double);
    }
    P.asm2_lds = (size_t)end2 * sizeof(double);
    if (std::max(P.asm1_lds, P.asm2_lds) > (size_t)d->lds_max) {
      snprintf(err, errlen, "assembly needs %zu bytes of LDS, the device has %d per workgroup",
               std::max(P.asm1_lds, P.asm2_lds), d->lds_max);
      return -1;
    }
  }
  const size_t out_bytes = 8 * job->nblk + 2 * (size_t)nt;
  if (out_bytes > d->pin_out_cap) {
    if (d->pin_out) ECP_CHECK(hipHostFree(d->pin_out));
    d->pin_out = nullptr;
    d->pin_out_cap = 0;
    ECP_CHECK(alloc_or_trim([&] { return hipHostMalloc(&d->pin_out, out_bytes + out_bytes / 4); }));
    d->pin_out_cap = out_bytes + out_bytes / 4;
  }
  if (bytes) *bytes = Ly.total;
  d->planned = true;
  return 0;
}

// Device half: places the planned job at `mem` (capacity cap; NULL = the
// context's own grow-only arena) and queues the upload of the staged inputs;
// nothing waits for it here.
extern "C" int ecp_dev_bind(ecp_dev *d, void *mem, size_t cap, char *err, size_t errlen) {
  if (!d->planned) {
    snprintf(err, errlen, "ecp_dev_bind before ecp_dev_plan");
    return -1;
  }
  Prepared &P = d->P;
  const JobLayout &Ly = d->L;
  d->prepared = false;
  d->eager_done = false;
  reset_graph(d);
  if (P.nt == 0) {
    d->prepared = true;
    return 0;
  }
  char *A = (char *)mem;
  if (!A) {
    if (Ly.total > d->arena_cap) {
      if (d->arena) ECP_CHECK(hipFree(d->arena));
      d->arena = nullptr;
      d->arena_cap = 0;
      const size_t c2 = Ly.total + Ly.total / 4;
      ECP_CHECK(alloc_or_trim([&] { return hipMalloc(&d->arena, c2); }));
      d->arena_cap = c2;
    }
    A = d->arena;
  } else if (Ly.total > cap) {
    snprintf(err, errlen, "job needs %zu bytes of device memory, %zu given", Ly.total, cap);
    return -1;
  }
  // the evaluation follows on the same stream; the staging memory is not
  // written again before ecp_dev_plan has waited for the copy
  ECP_CHECK(hipMemcpyAsync(A, d->pin_in, Ly.in_bytes, hipMemcpyHostToDevice, d->stream));
  d->uploading = true;
  DevJob &J = P.J;
  J.atoms = (const ecp_xyz *)(A + Ly.i_atoms);
  J.atom_maxl = (const int *)(A + Ly.i_amaxl);
  J.shells = (const ecp_shell *)(A + Ly.i_sh);
  J.pa = (const double *)(A + Ly.i_pa);
  J.pd = (const double *)(A + Ly.i_pd);
  J.cent = (const ecp_centre *)(A + Ly.i_cent);
  J.gauss = (const ecp_gauss *)(A + Ly.i_gauss);
  J.win = (const ecp_window *)(A + Ly.i_win);
  J.trip = (const ecp_triplet *)(A + Ly.i_trip);
  J.ntrip = P.nt;
  J.UL = (double *)(A + Ly.d_UL);
  J.Ut = (double *)(A + Ly.d_Ut);
  J.F = (double *)(A + Ly.d_F);
  J.ang = (double *)(A + Ly.d_ang);
  J.FL = Ly.FL;
  J.UK = Ly.UK;
  J.angL = Ly.angL;
  J.ang_lam = Ly.ang_lam;
  J.ang_c = Ly.ang_c;
  J.deriv = Ly.deriv;
  J.maxPairs = P.maxPairs;
  J.teoff = (const int *)(A + Ly.i_teoff);
  J.US = Ly.US;
  P.u1 = (T1Unit *)(A + Ly.d_u1);
  P.q = (double *)(A + Ly.d_q);
  P.t1s = (double *)(A + Ly.d_t1s);
  P.tq1 = (int *)(A + Ly.d_tq1);
  P.qf = (unsigned long long *)(A + Ly.d_qf);
  P.udir = (double *)(A + Ly.d_udir);
  P.fbq1 = (int *)(A + Ly.d_fbq1);
  P.fbc = (int *)(A + Ly.d_fbc);  // [0..12] type-1 fallback queues, [32..44] type-1 tails,
                                  // [kFb2Cnt + 0..12] type-2 fallback queues
  P.stat = (unsigned char *)(A + Ly.d_stat);
  P.Tout = (double *)(A + Ly.d_T);
  P.tf = (unsigned char *)(A + Ly.d_tf);
  P.tnfail = (int *)(A + Ly.d_tnf);
  P.flist = (int *)(A + Ly.d_flist);
  P.fbq2 = (int *)(A + Ly.d_fbq2);
  P.tcls2 = (const unsigned char *)(A + Ly.i_tcls2);
  P.fbT = (double *)(A + Ly.d_fbT);
  P.fit = (const int2 *)(A + Ly.i_fit);
  P.ait = (const int2 *)(A + Ly.i_ait);
  P.tcls = (const int *)(A + Ly.i_tcls);
  P.blk = (double *)(A + Ly.d_blk);
  P.zero_base = (unsigned int *)(A + Ly.d_zero);
  P.zero_words = (Ly.d_zero_end - Ly.d_zero) / 4;
  for (AsmArgs *x : {&P.aa, &P.aa4, &P.aa2p}) {
    AsmArgs &aa = *x;
    aa.units1 = P.u1;
    aa.udir = P.udir;
    aa.t1first = (const int *)(A + Ly.i_t1f);
    aa.qout = P.q;
    aa.Tout = P.Tout;
    aa.tfail = P.tf;
    aa.fbT = P.fbT;
    aa.blocks = P.blk;
  }
  d->prepared = true;
  return 0;
}

extern "C" int ecp_dev_prepare(ecp_dev *d, const ecp_job *job, char *err, size_t errlen) {
  if (ecp_dev_plan(d, job, nullptr, err, errlen)) return -1;
  return ecp_dev_bind(d, nullptr, 0, err, errlen);
}

// Runs the prepared evaluation `repeats` times and waits.  The first
// evaluation of a job runs eagerly and records the stage timings; when more
// evaluations follow (in this call or a later one) the kernel sequence is
// captured once into a HIP graph and replayed.
extern "C" int ecp_dev_execute(ecp_dev *d, int repeats, double *ms_total, char *err, size_t errlen) {
  if (!d->prepared) {
    snprintf(err, errlen, "ecp_dev_execute before ecp_dev_prepare");
    return -1;
  }
  d->nev = 0;
  if (ms_total) *ms_total = 0.0;
  if (d->P.nt == 0 || repeats <= 0) return 0;
  hipStream_t s = d->stream;
  int remaining = repeats;
  double total = 0.0;
  d->last_eager = false;
  if (!d->eager_done) {
    d->span_k = 0;
    d->last_eager = true;
    if (run_sequence(d, s, d->ev, err, errlen)) return -1;
    ECP_CHECK(hipStreamSynchronize(s));
    for (int i = 1; i < 4; i++) {
      float ms = 0.f;
      (void)hipEventElapsedTime(&ms, d->ev[i - 1], d->ev[i]);
      d->last_ms[i - 1] = ms;
    }
    d->nev = 3;
    total = d->last_ms[0] + d->last_ms[1] + d->last_ms[2];
    d->eager_done = true;
    remaining--;
  }
  if (remaining > 0 && d->ngraph == 0) {
    // fused launches: kSpanGraphs copies, each recording its own quadrature
    // event pair; per-class launches: one graph
    for (int k = 0; k < kSpanGraphs; k++) {
      d->span_k = k;
      // a first host-side record, so that the pair reads as recorded before
      // the graph's event nodes overwrite it
      ECP_CHECK(hipEventRecord(d->span[k][0], s));
      ECP_CHECK(hipEventRecord(d->span[k][1], s));
      ECP_CHECK(hipStreamSynchronize(s));
      ECP_CHECK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
      d->capturing = true;
      const int rc = run_sequence(d, s, nullptr, err, errlen);
      d->capturing = false;
      hipError_t ec = hipStreamEndCapture(s, &d->graph[k]);
      if (!rc && ec == hipSuccess) ec = hipGraphInstantiate(&d->gexec[k], d->graph[k], nullptr, nullptr, 0);
      if (rc || ec != hipSuccess) {
        // copy k does not exist (an invalidated capture gives no graph)
        (void)hipGetLastError();
        if (d->graph[k]) (void)hipGraphDestroy(d->graph[k]);
        d->graph[k] = nullptr;
        d->gexec[k] = nullptr;
        if (!rc) snprintf(err, errlen, "capturing the kernel sequence failed: %s", hipGetErrorString(ec));
        return -1;
      }
      d->ngraph = k + 1;
      if (!d->span_valid) break;
    }
    d->span_k = 0;
    d->replays = 0;
  }
  if (remaining > 0) {
    d->last_eager = false;
    d->last_replays = remaining;
    ECP_CHECK(hipEventRecord(d->ev[5], s));
    for (int r = 0; r < remaining; r++) {
      ECP_CHECK(hipGraphLaunch(d->gexec[d->replays % d->ngraph], s));
      d->replays++;
    }
    ECP_CHECK(hipEventRecord(d->ev[6], s));
    ECP_CHECK(hipStreamSynchronize(s));
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, d->ev[5], d->ev[6]);
    total = ms / remaining;
    d->last_ms[3] = (float)total;
    d->nev = 4;
  }
  if (ms_total) *ms_total = total;
  return 0;
}

namespace {
// Algorithmic FLOPs of the large-grid fallbacks of the last evaluation
// (ecp_fb1_flops per failed primitive pair, ecp_fb2_flops per primitive pair of
// a (triplet, channel) with failed entries): every term is an integer below
// 2^53, so the atomic sum is exact in any order.
__global__ __launch_bounds__(256) void k_fb_flops(DevJob J, const T1Unit *__restrict__ units,
                                                  const unsigned long long *__restrict__ qf, int nunits,
                                                  DevTables T, const int *__restrict__ tnfail,
                                                  const int *__restrict__ flist, int N, double *out) {
  double s1 = 0.0, s2 = 0.0;
  const int stride = gridDim.x * blockDim.x;
  for (int u = blockIdx.x * blockDim.x + threadIdx.x; u < nunits; u += stride) {
    const int f = __popcll(qf[u]);
    if (!f) continue;
    const ecp_triplet tr = J.trip[units[u].trip];
    s1 += ecp_fb1_flops(tr.la + tr.lb, f, N);
  }
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < J.ntrip; t += stride) {
    const int nf = tnfail[t];
    if (!nf) continue;
    const ecp_triplet tr = J.trip[t];
    const ecp_centre *C = J.cent + tr.centre;
    const int KK = J.shells[tr.sa].K * J.shells[tr.sb].K, t0 = t2_off(T, tr.la, tr.lb, 0);
    // one term per channel with failed entries: counted first, since the
    // waves that share a triplet's passes list their entries in any order
    int f[ECP_MAX_L] = {0};
    for (int k = 0; k < nf; k++) {
      const int l = T.tmpl[t0 + flist[J.teoff[t] + k]] >> 24;
#pragma unroll
      for (int i = 0; i < ECP_MAX_L; i++) f[i] += l == i;
    }
#pragma unroll
    for (int l = 0; l < ECP_MAX_L; l++)
      if (f[l]) s2 += KK * ecp_fb2_flops(tr.la, tr.lb, l, C->gl[l + 1] - C->gl[l], f[l], N);
  }
  if (s1 != 0.0) atomicAdd(&out[0], s1);
  if (s2 != 0.0) atomicAdd(&out[1], s2);
}

}  // namespace

// One eager evaluation with an event pair around every kernel launch on its
// own stream; per family: launches, summed duration (ms), algorithmic FLOPs.
// The type-1 large grid runs in the tail's launches: its FLOPs are under
// FAM_FB1, its time is in FAM_T1TAIL's.
extern "C" int ecp_dev_profile(ecp_dev *d, const ecp_job *job, int *launches, double *ms, double *flops, char *err,
                               size_t errlen) {
  if (!d->prepared) {
    snprintf(err, errlen, "ecp_dev_profile before ecp_dev_prepare");
    return -1;
  }
  for (int f = 0; f < FAM_N; f++) {
    launches[f] = 0;
    ms[f] = 0.0;
    flops[f] = 0.0;
  }
  if (d->P.nt == 0) return FAM_N;
  d->profiling = true;
  d->npev = 0;
  d->span_k = 0;
  d->last_eager = true;
  const int rc = run_sequence(d, d->stream, nullptr, err, errlen);
  d->profiling = false;
  if (rc) return -1;
  ECP_CHECK(hipStreamSynchronize(d->stream));
  for (int i = 0; i < d->npev; i++) {
    float t = 0.f;
    (void)hipEventElapsedTime(&t, d->pev[2 * i], d->pev[2 * i + 1]);
    launches[d->pfam[i]]++;
    ms[d->pfam[i]] += t;
  }
  // algorithmic FLOPs per family: the model's terms known before the
  // evaluation, and the fallbacks from this evaluation's failed integrals
  const Prepared &P = d->P;
  double model[ECP_FL_N];
  ecp_model_flops(job, model);
  flops[FAM_TABLES] = model[ECP_FL_FTAB];
  flops[FAM_TYPE1] = model[ECP_FL_T1];
  flops[FAM_TYPE2] = model[ECP_FL_T2];
  flops[FAM_ASM] = model[ECP_FL_ASM1] + model[ECP_FL_ASM2] + model[ECP_FL_SHIFT];
  if (!d->fbf) ECP_CHECK(hipMalloc(&d->fbf, 2 * sizeof(double)));
  ECP_CHECK(hipMemsetAsync(d->fbf, 0, 2 * sizeof(double), d->stream));
  const int nunits = P.cls_begin[ECP_MAX_LAB + 1];
  const int nb = std::max(1, std::min(1024, (std::max(nunits, P.nt) + 255) / 256));
  k_fb_flops<<<nb, 256, 0, d->stream>>>(P.J, P.u1, P.qf, nunits, d->T, P.tnfail, P.flist, d->T.lorder, d->fbf);
  ECP_CHECK(hipGetLastError());
  double fb[2] = {0.0, 0.0};
  ECP_CHECK(hipMemcpyAsync(fb, d->fbf, sizeof(fb), hipMemcpyDeviceToHost, d->stream));
  ECP_CHECK(hipStreamSynchronize(d->stream));
  flops[FAM_FB1] = fb[0];
  flops[FAM_FB2] = fb[1];
  return FAM_N;
}

extern "C" const char *ecp_dev_family_name(int f) { return (f >= 0 && f < FAM_N) ? kFamName[f] : ""; }

extern "C" int ecp_dev_fetch(ecp_dev *d, double **blocks, unsigned char **status, char *err, size_t errlen) {
  const Prepared &P = d->P;
  *blocks = nullptr;
  *status = nullptr;
  if (P.nt == 0) return 0;
  ECP_CHECK(hipMemcpyAsync(d->pin_out, P.blk, 8 * P.nblk, hipMemcpyDeviceToHost, d->stream));
  ECP_CHECK(hipMemcpyAsync(d->pin_out + 8 * P.nblk, P.stat, 2 * (size_t)P.nt, hipMemcpyDeviceToHost, d->stream));
  ECP_CHECK(hipStreamSynchronize(d->stream));
  *blocks = (double *)d->pin_out;
  *status = (unsigned char *)(d->pin_out + 8 * P.nblk);
  return 0;
}

// Zeros for a job's results, which a context of an earlier job holds other
// values in (a fetch or contraction before the first evaluation reads them).
extern "C" int ecp_dev_clear(ecp_dev *d, char *err, size_t errlen) {
  const Prepared &P = d->P;
  if (P.nt == 0) return 0;
  ECP_CHECK(hipMemsetAsync(P.blk, 0, 8 * P.nblk, d->stream));
  ECP_CHECK(hipMemsetAsync(P.stat, 0, 2 * (size_t)P.nt, d->stream));
  return 0;
}

// bytes of device and pinned memory a context holds for jobs
extern "C" size_t ecp_dev_held(const ecp_dev *d) {
  return d->arena_cap + d->con_cap + d->pin_in_cap + d->pin_out_cap;
}

// ---------------------------------------------------------------------------
// Density contraction of the evaluated blocks on the device, the consumer
// that getIntegrals.c:15-18 anticipates (a density P and a gradient in
// place of the AO matrix): no blocks leave the device.
//   n = 0: E_m = sum_{mu nu} P_{mu nu} V_{mu nu}; a block of shells a != b
//          stands for itself and its transpose (weight 2), a diagonal shell
//          block (a = b) for itself (weight 1).
//   n = 1: dE_m/dR_{X,d}.  A primitive's derivative is
//          d/dA_d g(a) = 2 zeta g(a + 1_d) - a_d g(a - 1_d) (libecp.c:242-245),
//          whose zeta factor the (+1) blocks already carry; the potential's
//          own derivative follows from translational invariance,
//          d/dC = -(d/dA + d/dB), so each block's contribution s goes to the
//          atom of its shifted shell with +s and to the ECP centre with -s.
//          Blocks the screening skips (A = B = C; the side on the centre,
//          libecp.c:305-306,326-330) would cancel in that sum.
// Partial sums per triplet are reduced by a fixed butterfly, and the
// per-molecule / per-atom sums run over triplets in a fixed order, so
// results do not depend on scheduling.

namespace {
struct ConArgs {
  const ecp_triplet *trip;
  const ecp_shell *shells;
  const ecp_centre *cent;
  const double *blocks;
  const unsigned char *stat;
  const int *aoff;        // AO offset of each global shell within its molecule
  const double *P;        // densities, packed by molecule
  const long long *poff;  // [nmol] offset of each molecule's density
  const int *prow;        // [nmol] its row stride
  const int *tmb;         // [nmol + 1] triplet range of each molecule
  const int *umol;        // [nunits] molecule of each output unit
  const int *uatom;       // [nunits] global atom of each output unit (n = 1)
  const int *uout;        // [nunits] output offset of each unit
  double *part;           // [ntrip * nd] weighted partial sums
  double *out;
  int *codes;             // [nmol] first failed integration: 0, 1 or 2
  int ntrip, nd, nunits, nmol;
};

__device__ __forceinline__ double wave_sum_fixed(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

__global__ __launch_bounds__(64) void k_con_part(DevTables T, ConArgs A) {
  const int lane = threadIdx.x;
  const int D = T.ijkDim;
  for (int t = blockIdx.x; t < A.ntrip; t += gridDim.x) {
    const ecp_triplet tr = A.trip[t];
    const ecp_shell Sa = A.shells[tr.sa], Sb = A.shells[tr.sb];
    const double *__restrict__ Pm = A.P + A.poff[Sa.mol];
    const int R = A.prow[Sa.mol];
    const int a0 = A.aoff[tr.sa], b0 = A.aoff[tr.sb];
    const int la = Sa.l, lb = Sb.l, nb = ECP_DIM_IJK(lb), nab = ECP_DIM_IJK(la) * nb;
    const int no = ECP_DIM_IJK(tr.ob);
    const double *__restrict__ b1 = A.blocks + tr.blk1;
    const double *__restrict__ b2 = A.blocks + tr.blk2;
    const bool bra = tr.shifta != 0;
    const int sh = bra ? tr.shifta : tr.shiftb, ls = bra ? la : lb;
    double acc[3] = {0.0, 0.0, 0.0};
    for (int e = lane; e < nab; e += 64) {
      const int i = e / nb, j = e - i * nb;
      const double p = Pm[(size_t)(a0 + i) * R + b0 + j];
      if (A.nd == 1) {
        acc[0] += p * (b1[i * no + j] + b2[i * no + j]);
        continue;
      }
      const int *ex = T.ijk + 3 * ECP_IDX_C(ls, bra ? i : j);
#pragma unroll
      for (int dd = 0; dd < 3; dd++) {
        int x[3] = {ex[0], ex[1], ex[2]};
        double coef;
        if (sh > 0) {
          coef = 2.0;
          x[dd] += 1;
        } else {
          if (x[dd] == 0) continue;
          coef = -(double)x[dd];
          x[dd] -= 1;
        }
        const int c = T.ijkIndex[(x[0] * D + x[1]) * D + x[2]] - ECP_IDX_C(ls + sh, 0);
        const int o = bra ? c * no + j : i * no + c;
        acc[dd] += coef * (p * (b1[o] + b2[o]));
      }
    }
    const double w = (tr.sa == tr.sb) ? 1.0 : 2.0;
    for (int k = 0; k < A.nd; k++) {
      const double v = wave_sum_fixed(acc[k]);
      if (lane == 0) A.part[(size_t)t * A.nd + k] = w * v;
    }
  }
}

constexpr int kConThreads = 256;

__global__ __launch_bounds__(kConThreads) void k_con_reduce(ConArgs A) {
  __shared__ double red[3][kConThreads];
  __shared__ int fmin[kConThreads];
  const int u = blockIdx.x, tid = threadIdx.x;
  const int m = A.umol[u], g = A.uatom[u];
  const int t0 = A.tmb[m], t1 = A.tmb[m + 1];
  double s[3] = {0.0, 0.0, 0.0};
  int first = INT_MAX;
  for (int t = t0 + tid; t < t1; t += kConThreads) {
    if (A.stat[2 * t]) first = min(first, 2 * t);
    else if (A.stat[2 * t + 1]) first = min(first, 2 * t + 1);
    if (A.nd == 1) {
      s[0] += A.part[t];
      continue;
    }
    const ecp_triplet tr = A.trip[t];
    const int X = A.shells[tr.shifta != 0 ? tr.sa : tr.sb].atom, C = A.cent[tr.centre].atom;
    const double *v = A.part + (size_t)t * 3;
    if (X == g)
      for (int k = 0; k < 3; k++) s[k] += v[k];
    if (C == g)
      for (int k = 0; k < 3; k++) s[k] -= v[k];
  }
  for (int k = 0; k < 3; k++) red[k][tid] = s[k];
  fmin[tid] = first;
  __syncthreads();
  for (int w = kConThreads / 2; w > 0; w >>= 1) {
    if (tid < w) {
      for (int k = 0; k < 3; k++) red[k][tid] += red[k][tid + w];
      fmin[tid] = min(fmin[tid], fmin[tid + w]);
    }
    __syncthreads();
  }
  if (tid < A.nd) A.out[A.uout[u] + tid] = red[tid][0];
  // one unit per molecule reports its first failure (callback order)
  if (tid == 0 && (u == 0 || A.umol[u - 1] != m))
    A.codes[m] = fmin[0] == INT_MAX ? 0 : 1 + (fmin[0] & 1);
}
}  // namespace

namespace {

// Index tables of a contraction (device layout, one block of `bytes`): the
// density offsets and row strides per molecule, the AO offset of every
// shell, the triplet range of every molecule, and the output units (one
// per molecule for the energy, one per atom for the gradient: molecule,
// global atom, output offset).  img == nullptr: sizes only.
struct ConImage {
  size_t poff = 0, aoff = 0, prow = 0, tmb = 0, umol = 0, uatom = 0, uout = 0, bytes = 0;
  int nunits = 0;
  size_t nout = 0;
};

ConImage con_image(const ecp_job *job, const long long *poff, const int *prow, char *img) {
  ConImage c;
  const int nmol = job->nmol, nd = job->deriv == 0 ? 1 : 3;
  c.nunits = nd == 1 ? nmol : job->mol_atom0[nmol];
  c.nout = (size_t)c.nunits * nd;
  size_t q = 0;
  auto take = [&](size_t bytes) {
    const size_t o = q;
    q += (bytes + 7) & ~(size_t)7;
    return o;
  };
  c.poff = take(8 * (size_t)nmol);
  c.aoff = take(4 * ((size_t)job->nsh + 1));
  c.prow = take(4 * (size_t)nmol);
  c.tmb = take(4 * ((size_t)nmol + 1));
  c.umol = take(4 * (size_t)c.nunits);
  c.uatom = take(4 * (size_t)c.nunits);
  c.uout = take(4 * (size_t)c.nunits);
  c.bytes = q;
  if (!img) return c;
  memcpy(img + c.poff, poff, 8 * (size_t)nmol);
  ecp_job_ao_offsets(job, (int *)(img + c.aoff));
  memcpy(img + c.prow, prow, 4 * (size_t)nmol);
  memcpy(img + c.tmb, job->trip_mol_begin, 4 * ((size_t)nmol + 1));
  int *um = (int *)(img + c.umol), *ua = (int *)(img + c.uatom), *uo = (int *)(img + c.uout);
  int u = 0;
  for (int m = 0; m < nmol; m++) {
    if (nd == 1) {
      um[u] = m;
      ua[u] = -1;
      uo[u] = u;
      u++;
      continue;
    }
    for (int g = job->mol_atom0[m]; g < job->mol_atom0[m + 1]; g++, u++) {
      um[u] = m;
      ua[u] = g;
      uo[u] = 3 * u;
    }
  }
  return c;
}

// Launches the contraction over a prepared image at base + o_idx, partial
// sums at part, codes at codes_dev; P and out are device pointers.
int con_launch(ecp_dev *d, const ecp_job *job, const ConImage &c, char *idx, const double *P, double *part,
               double *out, int *codes_dev, char *err, size_t errlen) {
  const Prepared &Pp = d->P;
  ConArgs A{};
  A.trip = Pp.J.trip;
  A.shells = Pp.J.shells;
  A.cent = Pp.J.cent;
  A.blocks = Pp.blk;
  A.stat = Pp.stat;
  A.aoff = (const int *)(idx + c.aoff);
  A.P = P;
  A.poff = (const long long *)(idx + c.poff);
  A.prow = (const int *)(idx + c.prow);
  A.tmb = (const int *)(idx + c.tmb);
  A.umol = (const int *)(idx + c.umol);
  A.uatom = (const int *)(idx + c.uatom);
  A.uout = (const int *)(idx + c.uout);
  A.part = part;
  A.out = out;
  A.codes = codes_dev;
  A.ntrip = Pp.nt;
  A.nd = job->deriv == 0 ? 1 : 3;
  A.nunits = c.nunits;
  A.nmol = job->nmol;
  // a stale error of an earlier, unrelated call must not be taken for one of
  // these launches
  (void)hipGetLastError();
  ECP_CHECK(hipEventRecord(d->con_ev[0], d->stream));
  if (Pp.nt > 0) {
    k_con_part<<<std::min(Pp.nt, 65536), 64, 0, d->stream>>>(d->T, A);
    ECP_CHECK(hipGetLastError());
  }
  if (c.nunits > 0) {
    k_con_reduce<<<c.nunits, kConThreads, 0, d->stream>>>(A);
    ECP_CHECK(hipGetLastError());
  }
  ECP_CHECK(hipEventRecord(d->con_ev[1], d->stream));
  return 0;
}

}  // namespace

extern "C" int ecp_dev_contract(ecp_dev *d, const ecp_job *job, const double *P, size_t nP, int P_on_device,
                                const long long *poff, const int *prow, double *out, int out_on_device,
                                int *codes, double *ms, char *err, size_t errlen) {
  const Prepared &Pp = d->P;
  if (!d->prepared) {
    snprintf(err, errlen, "no evaluated job to contract");
    return -1;
  }
  if (job->deriv > 1) {
    snprintf(err, errlen, "density contraction supports derivative orders 0 and 1");
    return -1;
  }
  const int nmol = job->nmol, nd = job->deriv == 0 ? 1 : 3;
  const ConImage ci = con_image(job, poff, prow, nullptr);
  std::vector<char> h(ci.bytes);
  con_image(job, poff, prow, h.data());
  // device layout
  auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
  size_t o = 0;
  const size_t o_part = o; o += al(8 * (size_t)std::max(1, Pp.nt) * nd);
  const size_t o_out = o; o += al(8 * std::max<size_t>(1, ci.nout));
  const size_t o_codes = o; o += al(4 * (size_t)nmol);
  const size_t o_idx = o; o += al(ci.bytes);
  const size_t o_P = o; o += P_on_device ? 0 : al(8 * nP);
  if (o > d->con_cap) {
    if (d->con_mem) ECP_CHECK(hipFree(d->con_mem));
    d->con_mem = nullptr;
    d->con_cap = 0;
    ECP_CHECK(alloc_or_trim([&] { return hipMalloc(&d->con_mem, o); }));
    d->con_cap = o;
    d->con_idx.clear();
  }
  char *b = d->con_mem;
  // the index tables change with the job or the density layout only
  if (d->con_idx_at != o_idx || d->con_idx != h) {
    ECP_CHECK(hipMemcpyAsync(b + o_idx, h.data(), h.size(), hipMemcpyHostToDevice, d->stream));
    ECP_CHECK(hipStreamSynchronize(d->stream));
    d->con_idx = h;
    d->con_idx_at = o_idx;
  }
  if (!P_on_device && nP) ECP_CHECK(hipMemcpyAsync(b + o_P, P, 8 * nP, hipMemcpyHostToDevice, d->stream));
  double *outp = out_on_device ? out : (double *)(b + o_out);
  if (con_launch(d, job, ci, b + o_idx, P_on_device ? P : (const double *)(b + o_P), (double *)(b + o_part), outp,
                 (int *)(b + o_codes), err, errlen))
    return -1;
  if (!out_on_device && ci.nout)
    ECP_CHECK(hipMemcpyAsync(out, b + o_out, 8 * ci.nout, hipMemcpyDeviceToHost, d->stream));
  ECP_CHECK(hipMemcpyAsync(codes, b + o_codes, 4 * (size_t)nmol, hipMemcpyDeviceToHost, d->stream));
  ECP_CHECK(hipStreamSynchronize(d->stream));
  if (ms) {
    float f = 0.f;
    ECP_CHECK(hipEventElapsedTime(&f, d->con_ev[0], d->con_ev[1]));
    *ms = f;
  }
  return 0;
}

extern "C" size_t ecp_dev_contract_image(const ecp_job *job, const long long *poff, const int *prow, char *img,
                                         size_t cap) {
  const ConImage c = con_image(job, poff, prow, nullptr);
  if (img && cap >= c.bytes) con_image(job, poff, prow, img);
  return c.bytes;
}

extern "C" int ecp_dev_contract_noalloc(ecp_dev *d, const ecp_job *job, const char *img, size_t img_bytes,
                                        const double *P, double *out, int *codes, double *ms, char *err,
                                        size_t errlen) {
  const Prepared &Pp = d->P;
  if (!d->prepared) {
    snprintf(err, errlen, "no evaluated job to contract");
    return -1;
  }
  if (job->deriv > 1) {
    snprintf(err, errlen, "density contraction supports derivative orders 0 and 1");
    return -1;
  }
  if (!d->scratch) {
    snprintf(err, errlen, "the no-allocation scratch of this device is not set up");
    return -1;
  }
  const int nmol = job->nmol, nd = job->deriv == 0 ? 1 : 3;
  // the image's sizes, from the same layout function that wrote it (no
  // allocation: sizes only)
  const ConImage ci = con_image(job, nullptr, nullptr, nullptr);
  if (ci.bytes != img_bytes) {
    snprintf(err, errlen, "contraction index image of %zu bytes does not match the job (%zu)", img_bytes, ci.bytes);
    return -1;
  }
  // scratch layout: partial sums, codes, index tables
  auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
  size_t o = 0;
  const size_t o_part = o; o += al(8 * (size_t)std::max(1, Pp.nt) * nd);
  const size_t o_codes = o; o += al(4 * (size_t)nmol);
  const size_t o_idx = o; o += al(ci.bytes);
  if (o > kScratchBytes) {
    snprintf(err, errlen,
             "the contraction needs %zu bytes of scratch (%d triplets, %d molecules); the no-allocation "
             "entry point holds %zu",
             o, Pp.nt, nmol, kScratchBytes);
    return -1;
  }
  char *b = (char *)d->scratch;
  // nothing in the scratch has to start at zero: the kernels write every
  // partial sum, output and code they read
  ECP_CHECK(hipMemcpyAsync(b + o_idx, img, ci.bytes, hipMemcpyHostToDevice, d->stream));
  if (con_launch(d, job, ci, b + o_idx, P, (double *)(b + o_part), out, (int *)(b + o_codes), err, errlen))
    return -1;
  if (codes) ECP_CHECK(hipMemcpyAsync(codes, b + o_codes, 4 * (size_t)nmol, hipMemcpyDeviceToHost, d->stream));
  ECP_CHECK(hipStreamSynchronize(d->stream));
  if (ms) {
    float f = 0.f;
    ECP_CHECK(hipEventElapsedTime(&f, d->con_ev[0], d->con_ev[1]));
    *ms = f;
  }
  return 0;
}

extern "C" int ecp_dev_span_ms(ecp_dev *d, double *ms, int *samples, char *err, size_t errlen) {
  if (!d->prepared || !d->span_valid || (!d->last_eager && d->replays == 0)) {
    snprintf(err, errlen, "no single-stream type-1 quadrature span in the last evaluation");
    return -1;
  }
  // the eager evaluation, or the last replays (one per graph copy)
  const int n = d->last_eager ? 1 : std::min(d->ngraph, d->last_replays);
  double sum = 0.0;
  for (int i = 0; i < n; i++) {
    const int k = d->last_eager ? 0 : (int)((d->replays - 1 - i) % d->ngraph);
    float f = 0.f;
    ECP_CHECK(hipEventElapsedTime(&f, d->span[k][0], d->span[k][1]));
    sum += f;
  }
  *ms = sum / n;
  if (samples) *samples = n;
  return 0;
}

extern "C" int ecp_dev_mem_alloc(void **p, size_t bytes, char *err, size_t errlen) {
  *p = nullptr;
  ECP_CHECK(alloc_or_trim([&] { return hipMalloc(p, bytes); }));
  return 0;
}

extern "C" void ecp_dev_mem_free(void *p) {
  if (p) (void)hipFree(p);
}

extern "C" int ecp_dev_sync(ecp_dev *d) {
  int rc = 0;
  if (d->stream && hipStreamSynchronize(d->stream) != hipSuccess) rc = -1;
  for (int k = 0; k < kWorkers; k++)
    if (d->workers[k] && hipStreamSynchronize(d->workers[k]) != hipSuccess) rc = -1;
  return rc;
}

extern "C" int ecp_dev_current(void) {
  int dv = 0;
  return hipGetDevice(&dv) == hipSuccess ? dv : -1;
}

extern "C" int ecp_dev_use(int device) { return hipSetDevice(device) == hipSuccess ? 0 : -1; }

extern "C" void ecp_dev_renew(ecp_dev *d) {
  ecp_dev_set_tuning(d, &kTuningDefaults);
  d->planned = d->prepared = false;
  d->nev = 0;
  d->span_valid = false;
  d->last_eager = false;
  d->last_replays = 0;
  d->P = Prepared();
  d->L = JobLayout();
}

extern "C" void ecp_dev_get_tuning(const ecp_dev *d, ecp_tuning *t) { *t = d->tune; }

extern "C" void ecp_dev_set_tuning(ecp_dev *d, ecp_tuning const *t) {
  d->tune = *t;
  d->tune.t1_tail_grid = std::max(1, d->tune.t1_tail_grid);
  reset_graph(d);
  d->eager_done = false;
}
