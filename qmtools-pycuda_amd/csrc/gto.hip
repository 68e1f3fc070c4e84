// Analytic potential of the GTO density plus nuclei (FP64).
//
// Reference kernel_hartree.cu:288-869 evaluates, per grid node C and per
// basis-function pair (p >= q), hand-derived closed forms of
//   int phi_p(r) phi_q(r) / |r - C| d^3r
// for each (La, Lb) class up to D-D.  Here the same integrals come from
// McMurchie-Davidson Hermite expansions (Helgaker, Jorgensen, Olsen,
// "Molecular Electronic-Structure Theory", sec. 9.5, 9.9):
//
//   phi_a phi_b = sum_tuv E^ab_t E^ab_u E^ab_v Lambda_tuv(p, P),
//   int Lambda_tuv / r_C = (2 pi / p) R_tuv(p, P - C).
//
// The density-matrix contraction is done once per molecule on the host: every
// primitive pair becomes a Hermite charge distribution (p, P, D_tuv) with
//   D_tuv = -f (2 pi/p) K c_a c_b sum_{ma,mb} P_(a ma),(b mb) sum_cart E_t E_u E_v
// (f = 2 for distinct shells), so that V_el(C) = sum_dist sum_tuv D_tuv R_tuv.  Shells of one nucleus and L
// with the same exponents (a general contraction) share their primitive pairs: their D_tuv are added
// before anything is evaluated, and on one nucleus the pairs (i, j) and (j, i) are one distribution too.
// cc-pVDZ: 196 instead of 484 pairs for two carbon atoms.
// The device kernel then only evaluates Boys functions and R_tuv per point.
// This has no singularity at T = 0 (the reference's closed forms divide by
// powers of T = gamma |PC|^2 and lose precision there).
//
// Boys function F_n(T): for T < 40, Taylor expansion (8 terms) around the
// nearest point of a 0.1-spaced table of F_L+k / k! (one table per L, so that a term is one multiply-add) and
// e^-T (computed on the host from the all-positive series e^-T sum (2T)^k / ((2n+1)...(2n+2k+1))), then
// downward recursion F_{n-1} = (2T F_n + e^-T)/(2n-1); for T >= 40,
// F_0 = sqrt(pi/T)/2 and upward recursion (e^-40 is below FP64 resolution of F).
#include <algorithm>
#include <atomic>
#include <cmath>
#include <system_error>
#include <thread>
#include <vector>

#include "qm_internal.h"

namespace {

constexpr int kLmax = 4;                 // La + Lb <= 4
constexpr int kNTUV = 35;                // (t,u,v) with t+u+v <= 4
constexpr int kTaylor = 8;               // terms F_L+k / k! of a table row, then e^-T
constexpr int kBoysN = kTaylor + 1;
constexpr int kBoysPts = 401;            // T = 0, 0.1, ..., 40
constexpr double kBoysStep = 0.1;
constexpr double kBoysTmax = 40.0;
constexpr double kGtoScreen = 1e-17;      // largest dropped contribution of one distribution (hartree)

__host__ __device__ constexpr int ntuv(int L) { return (L + 1) * (L + 2) * (L + 3) / 6; }
__host__ __device__ constexpr int tuv_index(int t, int u, int v) {
  return (t + u + v) * (t + u + v + 1) * (t + u + v + 2) / 6 + (u + v) * (u + v + 1) / 2 + v;
}

// A distribution of L = La + Lb in the table: p, Px, Py, Pz, then D_tuv for t + u + v <= L (tuv_index order).
__host__ __device__ constexpr int dist_doubles(int L) { return 4 + ntuv(L); }

// ------------------------------------------------------------------ device
// 1 / (2n - 1) for the recursion and 1 / k! for e^d: multiplications by rounded reciprocals instead of FP64
// divisions (each a ~10-instruction sequence)
__device__ constexpr double kInvInt[8] = {0.0, 1.0, 1.0 / 2, 1.0 / 3, 1.0 / 4, 1.0 / 5, 1.0 / 6, 1.0 / 7};
__device__ constexpr double kInvFact[10] = {1.0, 1.0, 1.0 / 2, 1.0 / 6, 1.0 / 24, 1.0 / 120, 1.0 / 720, 1.0 / 5040,
                                            1.0 / 40320, 1.0 / 362880};

template <int L>
__device__ __forceinline__ void boys(double T, const double* __restrict__ tab, double* F) {
  if (T < kBoysTmax) {
    const int i = (int)(T * (1.0 / kBoysStep) + 0.5);
    const double d = i * kBoysStep - T;       // T = Ti - d, |d| <= 0.05
    const double* row = tab + i * kBoysN;
    // F_L(T) = sum_k F_{L+k}(Ti) d^k / k!
    double f = row[kTaylor - 1];
#pragma unroll
    for (int k = kTaylor - 2; k >= 0; --k) f = fma(f, d, row[k]);
    F[L] = f;
    // e^-T = e^-Ti e^d: the table's last column holds e^-Ti, e^d is its Taylor series to d^9
    // (remainder below 3e-20)
    double ed = kInvFact[9];
#pragma unroll
    for (int k = 8; k >= 0; --k) ed = fma(ed, d, kInvFact[k]);
    const double ex = row[kTaylor] * ed;
#pragma unroll
    for (int n = L; n >= 1; --n) F[n - 1] = (2.0 * T * F[n] + ex) * kInvInt[2 * n - 1];
  } else {
    // F_0 = sqrt(pi / T) / 2 from one reciprocal square root (no FP64 division or sqrt), 1/T = r^2
    const double r = rsqrt(T);
    const double inv = r * r;
    F[0] = 0.88622692545275801365 * r;   // sqrt(pi) / 2
#pragma unroll
    for (int n = 1; n <= L; ++n) F[n] = F[n - 1] * ((double)(2 * n - 1) * 0.5 * inv);
  }
}

// The table is constant during a launch and its address wave uniform: read through scalar loads.
typedef const double __attribute__((address_space(4))) TableDouble;

// sum_tuv D_tuv R^0_tuv for t+u+v <= L, R from the Hermite recursion (Helgaker eq. 9.9.18-20)
template <int L>
__device__ __forceinline__ double hermite_contract(double X, double Y, double Z, const double* rn,
                                                   TableDouble* D) {
  constexpr int N = ntuv(L);
  double cur[N], nxt[N];
  cur[0] = rn[L];
#pragma unroll
  for (int n = L - 1; n >= 0; --n) {
    const int dmax = L - n;
    nxt[0] = rn[n];
#pragma unroll
    for (int d = 1; d <= L; ++d) {
      if (d > dmax) break;
#pragma unroll
      for (int t = d; t >= 0; --t) {
#pragma unroll
        for (int u = d - t; u >= 0; --u) {
          const int v = d - t - u;
          double val;
          if (t > 0) {
            val = X * cur[tuv_index(t - 1, u, v)];
            if (t > 1) val += (double)(t - 1) * cur[tuv_index(t - 2, u, v)];
          } else if (u > 0) {
            val = Y * cur[tuv_index(t, u - 1, v)];
            if (u > 1) val += (double)(u - 1) * cur[tuv_index(t, u - 2, v)];
          } else {
            val = Z * cur[tuv_index(t, u, v - 1)];
            if (v > 1) val += (double)(v - 1) * cur[tuv_index(t, u, v - 2)];
          }
          nxt[tuv_index(t, u, v)] = val;
        }
      }
    }
#pragma unroll
    for (int q = 0; q < N; ++q) cur[q] = nxt[q];
  }
  double acc = 0.0;
#pragma unroll
  for (int q = 0; q < N; ++q) acc += D[q] * cur[q];
  return acc;
}

template <int L>
__device__ __forceinline__ double dist_sum(const double* __restrict__ ds, int lo, int hi, double cx, double cy,
                                           double cz, const double* __restrict__ tab) {
  double acc = 0.0;
  for (int d = lo; d < hi; ++d) {
    TableDouble* h = (TableDouble*)(uintptr_t)(ds + (int64_t)d * dist_doubles(L));
    const double p = h[0];
    const double X = h[1] - cx, Y = h[2] - cy, Z = h[3] - cz;
    const double T = p * (X * X + Y * Y + Z * Z);
    double F[L + 1];
    boys<L>(T, tab, F);
    double rn[L + 1];
    double m = 1.0;
#pragma unroll
    for (int n = 0; n <= L; ++n) {
      rn[n] = m * F[n];
      m *= -2.0 * p;
    }
    acc += hermite_contract<L>(X, Y, Z, rn, h + 4);
  }
  return acc;
}

struct DistLists {
  const double* d[kLmax + 1];
  int n[kLmax + 1];
  int cost;                 // of all lists (dist_cost)
};

// cost of a distribution, about proportional to its FP64 operations
__host__ __device__ constexpr int dist_cost(int L) { return L == 0 ? 5 : L == 1 ? 6 : L == 2 ? 8 : L == 3 ? 12 : 20; }

// Point of thread t of workgroup b: a list or a grid's nodes in order, or (blocks) a grid in blocks of 8^3 per workgroup
// and 4^3 per wave, so that the points of a wave mostly take the same branch of the Boys function.  idx < 0: none.
__device__ __forceinline__ int64_t gto_point(const double* __restrict__ pts, const GeomView& g, int64_t npts, int64_t b,
                                             int t, int blocks, double& cx, double& cy, double& cz) {
  if (!blocks) {
    const int64_t idx = b * 512 + t, u = idx < npts ? idx : npts - 1;
    if (!pts) {
      cx = g.ox + (double)(u % g.nx) * g.h;
      cy = g.oy + (double)((u / g.nx) % g.ny) * g.h;
      cz = g.oz + (double)(u / ((int64_t)g.nx * g.ny)) * g.h;
      return idx < npts ? idx : -1;
    }
    cx = pts[3 * u];
    cy = pts[3 * u + 1];
    cz = pts[3 * u + 2];
    return idx < npts ? idx : -1;
  }
  const int nbx = (g.nx + 7) / 8, nby = (g.ny + 7) / 8;
  const int64_t q = b / nbx;
  const int i = (int)(b - q * nbx) * 8 + (t & 3) + 4 * ((t >> 6) & 1);
  const int j = (int)(q % nby) * 8 + ((t >> 2) & 3) + 4 * ((t >> 7) & 1);
  const int k = (int)(q / nby) * 8 + ((t >> 4) & 3) + 4 * (t >> 8);
  const int ic = min(i, g.nx - 1), jc = min(j, g.ny - 1), kc = min(k, g.nz - 1);
  cx = g.ox + ic * g.h;
  cy = g.oy + jc * g.h;
  cz = g.oz + kc * g.h;
  return i < g.nx && j < g.ny && k < g.nz ? i + (int64_t)g.nx * (j + (int64_t)g.ny * k) : -1;
}

// partial[chunk][pt] = sum over this chunk's slice of every L list
// 512 threads share one 29 KB LDS copy of the table of one L at a time.  FP64 VALU bound.  60 atoms, 10^4
// points: 3.1 -> 1.7 ms with shared primitive pairs and one multiply-add per Taylor term; 16 atoms,
// 48 x 40 x 56 nodes: 2.9 -> 1.3 ms, with the nodes taken in 4^3 blocks.
constexpr int kGtoThreads = 512;
// SHARES: a chunk takes an equal share of lists.cost, else a slice of every list (as a branch in one kernel this cost the
// long chunks 1 %)
template <bool SHARES>
__global__ __launch_bounds__(kGtoThreads) void k_gto(DistLists lists, const double* __restrict__ boys_tab,
                                                     const double* __restrict__ pts, GeomView g, int64_t npts,
                                                     int blocks, int nchunk, double* __restrict__ partial) {
  __shared__ double tab[kBoysPts * kBoysN];
  const int chunk = blockIdx.y;
  double cx, cy, cz;
  const int64_t idx = gto_point(pts, g, npts, blockIdx.x, threadIdx.x, blocks, cx, cy, cz);
  double acc = 0.0;
  int c0 = (int)((int64_t)lists.cost * chunk / nchunk), c1 = (int)((int64_t)lists.cost * (chunk + 1) / nchunk);
#define QM_GTO_L(LL)                                                                                                 \
  {                                                                                                                  \
    const int n = lists.n[LL];                                                                                       \
    const int per = (n + nchunk - 1) / nchunk;                                                                       \
    int lo = min(n, chunk * per), hi = min(n, lo + per);                                                             \
    if (SHARES) {                                                                                                    \
      lo = min(n, max(0, (c0 + dist_cost(LL) - 1) / dist_cost(LL)));                                                 \
      hi = min(n, max(0, (c1 + dist_cost(LL) - 1) / dist_cost(LL)));                                                 \
      c0 -= n * dist_cost(LL);                                                                                       \
      c1 -= n * dist_cost(LL);                                                                                       \
    }                                                                                                                \
    if (hi > lo) { /* the same for the whole workgroup */                                                            \
      __syncthreads();                                                                                               \
      for (int i = threadIdx.x; i < kBoysPts * kBoysN; i += kGtoThreads) tab[i] = boys_tab[LL * kBoysPts * kBoysN + i]; \
      __syncthreads();                                                                                               \
      acc += dist_sum<LL>(lists.d[LL], lo, hi, cx, cy, cz, tab);                                                     \
    }                                                                                                                \
  }
  QM_GTO_L(0)
  QM_GTO_L(1)
  QM_GTO_L(2)
  QM_GTO_L(3)
  QM_GTO_L(4)
#undef QM_GTO_L
  if (idx >= 0) partial[(int64_t)chunk * npts + idx] = acc;
}

// out[t] = sum_chunks partial + sum_A Z_A / |C - R_A| (|C - R_A| > 1e-8, kernel_hartree.cu:851-865)
template <typename TO>
__global__ void k_gto_finish(const double* __restrict__ partial, int nchunk, const double4* __restrict__ atoms,
                             int natoms, const double* __restrict__ pts, GeomView g, int64_t npts,
                             TO* __restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= npts) return;
  double cx, cy, cz;
  if (pts) {
    cx = pts[3 * t];
    cy = pts[3 * t + 1];
    cz = pts[3 * t + 2];
  } else {
    const int64_t i = t % g.nx, j = (t / g.nx) % g.ny, k = t / ((int64_t)g.nx * g.ny);
    cx = g.ox + i * g.h;
    cy = g.oy + j * g.h;
    cz = g.oz + k * g.h;
  }
  double v = 0.0;
  for (int c = 0; c < nchunk; ++c) v += partial[(int64_t)c * npts + t];
  for (int a = 0; a < natoms; ++a) {
    const double4 A = atoms[a];
    const double dx = cx - A.x, dy = cy - A.y, dz = cz - A.z;
    const double r = sqrt(dx * dx + dy * dy + dz * dz);
    if (r > 1e-8) v += A.w / r;
  }
  out[t] = (TO)v;
}

// ------------------------------------------------------------------ host: tables
std::vector<double> make_boys_table() {
  constexpr int nf = kLmax + kTaylor;   // F_0 .. F_11
  std::vector<double> tab((size_t)(kLmax + 1) * kBoysPts * kBoysN);
  for (int i = 0; i < kBoysPts; ++i) {
    const double T = i * kBoysStep;
    long double F[nf];
    const long double e = std::exp(-(long double)T);
    for (int n = 0; n < nf; ++n) {
      // e^-T sum_k (2T)^k / ((2n+1)(2n+3)...(2n+2k+1)): positive terms, no cancellation
      long double term = 1.0L / (2 * n + 1), s = term;
      for (int k = 1; k < 2000; ++k) {
        term *= 2.0L * T / (2 * n + 2 * k + 1);
        s += term;
        if (term < s * 1e-21L) break;
      }
      F[n] = e * s;
    }
    for (int L = 0; L <= kLmax; ++L) {
      double* row = &tab[((size_t)L * kBoysPts + i) * kBoysN];
      long double fact = 1.0L;
      for (int k = 0; k < kTaylor; ++k) {
        row[k] = (double)(F[L + k] / fact);
        fact *= k + 1;
      }
      row[kTaylor] = (double)e;
    }
  }
  return tab;
}

// Cartesian expansion of the reference's solid harmonics (kernel_density.cu:14-31), m order (0,+1,-1,+2,-2)
struct CartTerm {
  double c;
  int e[3];
};
constexpr double C00 = 0.28209479177387814, C1 = 0.4886025119029199, C2A = 1.0925484305920792,
                 C20 = 0.31539156525252005, C22 = 0.5462742152960396;

std::vector<CartTerm> cart_terms(int L, int mi) {
  if (L == 0) return {{C00, {0, 0, 0}}};
  if (L == 1) {
    if (mi == 0) return {{C1, {0, 0, 1}}};
    if (mi == 1) return {{C1, {1, 0, 0}}};
    return {{C1, {0, 1, 0}}};
  }
  switch (mi) {
    case 0: return {{2 * C20, {0, 0, 2}}, {-C20, {2, 0, 0}}, {-C20, {0, 2, 0}}};
    case 1: return {{C2A, {1, 0, 1}}};
    case 2: return {{C2A, {0, 1, 1}}};
    case 3: return {{C22, {2, 0, 0}}, {-C22, {0, 2, 0}}};
    default: return {{C2A, {1, 1, 0}}};
  }
}

// E[i][j][t] for one axis, i,j <= 2, t <= 4 (Helgaker eq. 9.5.6-9.5.7), without K
void hermite_E(double a, double b, double XAB, double E[3][3][6]) {
  const double p = a + b;
  const double XPA = -b / p * XAB, XPB = a / p * XAB, i2p = 0.5 / p;
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j)
      for (int t = 0; t < 6; ++t) E[i][j][t] = 0.0;
  E[0][0][0] = 1.0;
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j) {
      if (i == 0 && j == 0) continue;
      for (int t = 0; t <= i + j; ++t) {
        double v;
        if (i > 0) {
          v = XPA * E[i - 1][j][t] + (t + 1) * E[i - 1][j][t + 1];
          if (t > 0) v += i2p * E[i - 1][j][t - 1];
        } else {
          v = XPB * E[i][j - 1][t] + (t + 1) * E[i][j - 1][t + 1];
          if (t > 0) v += i2p * E[i][j - 1][t - 1];
        }
        E[i][j][t] = v;
      }
    }
}

// f(i) for every i in [0, n), taken in increasing i by up to 16 host threads (the calling thread
// included; with fewer threads available it takes what the others leave)
template <typename F>
void host_parallel(int n, F&& f) {
  std::atomic<int> next{0};
  auto runner = [&]() {
    for (int i = next.fetch_add(1); i < n; i = next.fetch_add(1)) f(i);
  };
  const int nthr = std::max(1, std::min(16, (int)std::thread::hardware_concurrency()));
  std::vector<std::thread> pool;
  try {
    for (int t = 1; t < nthr && t < n; ++t) pool.emplace_back(runner);
  } catch (const std::system_error&) {
  }
  runner();
  for (auto& t : pool) t.join();
}

struct GtoCache {
  double* dev = nullptr;
  size_t off[kLmax + 1] = {0, 0, 0, 0, 0};   // first double of each L's distributions
  int n[kLmax + 1] = {0, 0, 0, 0, 0};
  double* boys = nullptr;
};

// Shells of one nucleus and L with the same exponents, evaluated as one: their primitive pairs coincide.
struct ShellSet {
  int atom, L, nprim, poff;
  std::vector<int> shells;
};

int build_distributions(qm_ctx* ctx, qm_mol* mol, hipStream_t s, GtoCache& c) {
  const int nbf = mol->nbf;
  // Cartesian term lists per (L, m index)
  std::vector<CartTerm> terms[3][5];
  for (int L = 0; L <= 2; ++L)
    for (int mi = 0; mi < 2 * L + 1; ++mi) terms[L][mi] = cart_terms(L, mi);
  std::vector<ShellSet> sets;
  {
    std::vector<std::vector<int>> of_atom(mol->natoms);   // sets of each nucleus
    for (int k = 0; k < mol->nshell; ++k) {
      const DevShell& sh = mol->h_shells[k];
      int found = -1;
      for (int i : of_atom[sh.atom]) {
        bool same = sets[i].L == sh.L && sets[i].nprim == sh.nprim;
        for (int q = 0; same && q < sh.nprim; ++q)
          same = mol->h_alpha[sets[i].poff + q] == mol->h_alpha[sh.poff + q];
        if (same) found = i;
      }
      if (found < 0) {
        of_atom[sh.atom].push_back((int)sets.size());
        sets.push_back({sh.atom, sh.L, sh.nprim, sh.poff, {k}});
      } else {
        sets[found].shells.push_back(k);
      }
    }
  }
  const int nset = (int)sets.size();
  // distributions of set A with the sets B <= A, per L, in the order (B, primitive of A, primitive of B);
  // the table is the concatenation over A in increasing order, the same whether the sets are built by one
  // thread or several
  struct SetOut {
    std::vector<double> l[kLmax + 1];
  };
  std::vector<SetOut> per(nset);
  auto build_set = [&](int sa) {
    const ShellSet& A = sets[sa];
    const double* RA = &mol->xyz[3 * A.atom];
    // Cartesian pair (exponents ea, eb) with its weight sum_{ma,mb} P_ab fa fb for every pair of shells of the sets
    struct CW {
      int ea[3], eb[3];
      std::vector<double> w;   // [shell of A][shell of B]
    };
    for (int sb = 0; sb <= sa; ++sb) {
      const ShellSet& B = sets[sb];
      const double* RB = &mol->xyz[3 * B.atom];
      const size_t na = A.shells.size(), nb = B.shells.size();
      std::vector<CW> cw;
      double wmax = 0.0;
      for (size_t ka = 0; ka < na; ++ka)
        for (size_t kb = 0; kb < nb; ++kb) {
          const DevShell &SA = mol->h_shells[A.shells[ka]], &SB = mol->h_shells[B.shells[kb]];
          for (int ma = 0; ma < 2 * A.L + 1; ++ma)
            for (int mb = 0; mb < 2 * B.L + 1; ++mb) {
              const double P = mol->h_P[(size_t)(SA.bf + ma) * nbf + (SB.bf + mb)];
              if (P == 0.0) continue;
              for (const CartTerm& ta : terms[A.L][ma])
                for (const CartTerm& tb : terms[B.L][mb]) {
                  CW* x = nullptr;
                  for (CW& y : cw)
                    if (y.ea[0] == ta.e[0] && y.ea[1] == ta.e[1] && y.ea[2] == ta.e[2] && y.eb[0] == tb.e[0] &&
                        y.eb[1] == tb.e[1] && y.eb[2] == tb.e[2])
                      x = &y;
                  if (!x) {
                    cw.push_back({{ta.e[0], ta.e[1], ta.e[2]}, {tb.e[0], tb.e[1], tb.e[2]},
                                  std::vector<double>(na * nb, 0.0)});
                    x = &cw.back();
                  }
                  x->w[ka * nb + kb] += P * ta.c * tb.c;
                }
            }
        }
      for (const CW& x : cw)
        for (double w : x.w) wmax = std::max(wmax, std::fabs(w));
      if (cw.empty() || wmax == 0.0) continue;
      const int L = A.L + B.L;
      const double AB[3] = {RA[0] - RB[0], RA[1] - RB[1], RA[2] - RB[2]};
      const double AB2 = AB[0] * AB[0] + AB[1] * AB[1] + AB[2] * AB[2];
      double D[kNTUV];
      // adds the pair (ia, ib) to D; false if it contributes nothing (exp underflow or zero coefficients)
      auto add_pair = [&](int ia, int ib, double f) -> bool {
        const double a = mol->h_alpha[A.poff + ia], b = mol->h_alpha[B.poff + ib], p = a + b;
        const double pref = -f * 2.0 * M_PI / p * std::exp(-a * b / p * AB2);
        bool any = false;
        double E[3][3][3][6];
        for (const CW& x : cw) {
          double w = 0.0;
          for (size_t ka = 0; ka < na; ++ka)
            for (size_t kb = 0; kb < nb; ++kb)
              w += mol->h_coeff[mol->h_shells[A.shells[ka]].poff + ia] * mol->h_coeff[mol->h_shells[B.shells[kb]].poff + ib] *
                   x.w[ka * nb + kb];
          w *= pref;
          if (w == 0.0) continue;
          if (!any)
            for (int d = 0; d < 3; ++d) hermite_E(a, b, AB[d], E[d]);
          any = true;
          for (int t = 0; t <= x.ea[0] + x.eb[0]; ++t) {
            const double et = E[0][x.ea[0]][x.eb[0]][t];
            if (et == 0.0) continue;
            for (int u = 0; u <= x.ea[1] + x.eb[1]; ++u) {
              const double eu = E[1][x.ea[1]][x.eb[1]][u];
              if (eu == 0.0) continue;
              for (int v = 0; v <= x.ea[2] + x.eb[2]; ++v)
                D[tuv_index(t, u, v)] += w * et * eu * E[2][x.ea[2]][x.eb[2]][v];
            }
          }
        }
        return any;
      };
      for (int ia = 0; ia < A.nprim; ++ia) {
        // one set with itself: (ia, ib) and (ib, ia) have the same centre and exponent
        for (int ib = 0; ib < (sa == sb ? ia + 1 : B.nprim); ++ib) {
          std::fill(D, D + kNTUV, 0.0);
          bool any = add_pair(ia, ib, sa == sb ? 1.0 : 2.0);
          if (sa == sb && ia != ib) any = add_pair(ib, ia, 1.0) || any;
          if (!any) continue;
          const double a = mol->h_alpha[A.poff + ia], b = mol->h_alpha[B.poff + ib], p = a + b;
          // Screening: |sum_tuv D_tuv R_tuv(C)| <= sum_tuv |D_tuv| (2p)^{n/2} 2^n n! for every point C
          // (n = t+u+v; Hermite-function bound on the derivatives of F_0), so a distribution whose
          // bound is below kGtoScreen changes no potential by more than that.
          double bound = 0.0, g = 1.0;
          for (int n = 0, k = 0; n <= L; ++n) {
            for (; k < ntuv(n); ++k) bound += std::fabs(D[k]) * g;
            g *= std::sqrt(2.0 * p) * 2.0 * (n + 1);
          }
          if (bound < kGtoScreen) continue;
          std::vector<double>& out = per[sa].l[L];
          const double head[4] = {p, (a * RA[0] + b * RB[0]) / p, (a * RA[1] + b * RB[1]) / p, (a * RA[2] + b * RB[2]) / p};
          out.insert(out.end(), head, head + 4);
          out.insert(out.end(), D, D + ntuv(L));
        }
      }
    }
  };
  // sets taken largest first (set A pairs with A + 1 sets)
  host_parallel(nset, [&](int k) { build_set(nset - 1 - k); });
  // table offsets: L-major, sets in increasing order within each L
  std::vector<size_t> at((size_t)(kLmax + 1) * nset);
  size_t tot = 0;
  for (int L = 0; L <= kLmax; ++L) {
    c.off[L] = tot;
    for (int sa = 0; sa < nset; ++sa) {
      at[(size_t)L * nset + sa] = tot;
      tot += per[sa].l[L].size();
    }
    c.n[L] = (int)((tot - c.off[L]) / dist_doubles(L));
  }
  // stream-ordered: kernels queued earlier on s still read the previous table
  if (c.dev) {
    QM_CHECK_HIP(ctx, hipFreeAsync(c.dev, s));
    c.dev = nullptr;
  }
  if (tot) {
    // the context's pinned staging buffer (the last upload from it finished: synchronised below)
    const size_t bytes = sizeof(double) * tot;
    if (bytes > ctx->gto_staged_bytes) {
      if (ctx->gto_staged) QM_CHECK_HIP(ctx, hipHostFree(ctx->gto_staged));
      ctx->gto_staged = nullptr;
      ctx->gto_staged_bytes = 0;
      QM_CHECK_HIP(ctx, hipHostMalloc(&ctx->gto_staged, bytes, hipHostMallocDefault));
      ctx->gto_staged_bytes = bytes;
    }
    double* staged = (double*)ctx->gto_staged;
    // the sets' lists go to their places in the staging buffer
    host_parallel(nset, [&](int sa) {
      for (int L = 0; L <= kLmax; ++L)
        if (!per[sa].l[L].empty())
          std::copy(per[sa].l[L].begin(), per[sa].l[L].end(), staged + at[(size_t)L * nset + sa]);
    });
    QM_CHECK_HIP(ctx, hipMallocAsync((void**)&c.dev, bytes, s));
    QM_CHECK_HIP(ctx, hipMemcpyAsync(c.dev, staged, bytes, hipMemcpyHostToDevice, s));
    QM_CHECK_HIP(ctx, hipStreamSynchronize(s));   // the staging buffer is rewritten by the next build
  }
  mol->n_gto_builds++;
  if (!c.boys) {
    const std::vector<double> tab = make_boys_table();
    QM_CHECK_HIP(ctx, hipMalloc(&c.boys, sizeof(double) * tab.size()));
    QM_CHECK_HIP(ctx, hipMemcpy(c.boys, tab.data(), sizeof(double) * tab.size(), hipMemcpyHostToDevice));
  }
  return QM_OK;
}

int get_cache(qm_ctx* ctx, qm_mol* mol, hipStream_t s, GtoCache** out) {
  if (!mol->gto) mol->gto = new GtoCache();
  GtoCache* c = (GtoCache*)mol->gto;
  if (mol->gto_dirty) {
    int rc = build_distributions(ctx, mol, s, *c);
    if (rc) return rc;
    mol->gto_dirty = false;
  }
  *out = c;
  return QM_OK;
}

template <typename TO>
int gto_eval(qm_ctx* ctx, qm_mol* mol, hipStream_t s, const double* pts, const GeomView& gv, int64_t npts,
             TO* out) {
  GtoCache* c = nullptr;
  int rc = get_cache(ctx, mol, s, &c);
  if (rc) return rc;
  DistLists dl;
  int total = 0;
  for (int L = 0; L <= kLmax; ++L) {
    dl.d[L] = c->dev ? c->dev + c->off[L] : nullptr;
    dl.n[L] = c->n[L];
    total += c->n[L];
  }
  // Nodes in blocks cost 4 to 7 % less than in order (16 atoms, 48 x 40 x 56: 1302 and 1359 us; 64^3: 3089 and 3320), so
  // they are taken so only where the blocks' padding is less than that: 33^3 (1.76 times the nodes) 759 and 473 us,
  // 256 x 256 x 1 (8 times) 6040 and 810, a line of 20000 (62 times) 14670 and 276.
  const int64_t linear = (npts + kGtoThreads - 1) / kGtoThreads;
  const int64_t blocked = pts ? 0 : (int64_t)((gv.nx + 7) / 8) * ((gv.ny + 7) / 8) * ((gv.nz + 7) / 8);
  const bool blocks = !pts && 20 * blocked <= 21 * linear;
  const int64_t pblocks = blocks ? blocked : linear;
  // Enough workgroups for 256 CUs: the distributions are split over chunks when points are few, at least 64 of them to a
  // chunk, or 32 of up to 2048 (the last kernel adds the chunks up one after the other).  Short chunks take a share of the
  // total cost, so that they run one or two of the lists, since each refills the table in LDS; long ones a slice of every
  // list.  2, 5, 9, 12 atoms (185, 1148, 3292, 5347 distributions), 700 points, us: slices of 64 36, 40, 53, 62; shares
  // of 64 34, 33, 46, 56; of 32 20, 28, 49, 66.
  const int few = total / (total <= 2048 ? 32 : 64);
  const int64_t fill = std::min<int64_t>(256, 2048 / std::max<int64_t>(pblocks, 1));
  const int nchunk = (int)std::max<int64_t>(1, std::min<int64_t>(fill, few));
  const bool shares = total < 256 * nchunk;
  dl.cost = 0;
  for (int L = 0; shares && L <= kLmax; ++L) dl.cost += dl.n[L] * dist_cost(L);
  double* partial = nullptr;
  if ((rc = qm_ws(ctx, s, WS_GTO, sizeof(double) * (size_t)nchunk * npts, (void**)&partial))) return rc;
  QM_REQUIRE(ctx, pblocks <= 0x7fffffff, QM_ELIMIT, "gto: too many points");
  {
    ProfScope ps(ctx, s, QM_K_GTO);
    hipLaunchKernelGGL(shares ? k_gto<true> : k_gto<false>, dim3((unsigned)pblocks, nchunk), dim3(kGtoThreads), 0, s, dl,
                       (const double*)c->boys, pts, gv, npts, blocks ? 1 : 0, nchunk, partial);
  }
  QM_CHECK_LAUNCH(ctx);
  hipLaunchKernelGGL(k_gto_finish<TO>, dim3((unsigned)((npts + 255) / 256)), dim3(256), 0, s,
                     (const double*)partial, nchunk, (const double4*)mol->atoms, mol->natoms, pts, gv, npts, out);
  QM_CHECK_LAUNCH(ctx);
  return QM_OK;
}

}  // namespace

void qm_gto_cache_free(void* p) {
  GtoCache* c = (GtoCache*)p;
  if (!c) return;
  if (c->dev) {
    (void)hipFreeAsync(c->dev, nullptr);
    (void)hipStreamSynchronize(nullptr);
  }
  if (c->boys) (void)hipFree(c->boys);
  delete c;
}

extern "C" {

int qm_hartree_gto_points(qm_ctx* ctx, qm_mol* mol, void* stream, const double* pts, int64_t npts, double* out) {
  int rc = qm_enter(ctx);
  if (rc) return rc;
  QM_REQUIRE(ctx, mol && pts && out, QM_EINVAL, "gto: null argument");
  QM_REQUIRE(ctx, mol->has_dm, QM_EINVAL, "gto: molecule has no density matrix");
  QM_REQUIRE(ctx, npts > 0, QM_EINVAL, "gto: no points");
  GeomView gv{};
  return gto_eval<double>(ctx, mol, (hipStream_t)stream, pts, gv, npts, out);
}

int qm_hartree_gto_grid(qm_ctx* ctx, qm_mol* mol, void* stream, const qm_geom* g, int dtype, void* out) {
  int rc = qm_enter(ctx);
  if (rc) return rc;
  if ((rc = qm_check_geom(ctx, g))) return rc;
  QM_REQUIRE(ctx, mol && out, QM_EINVAL, "gto: null argument");
  QM_REQUIRE(ctx, mol->has_dm, QM_EINVAL, "gto: molecule has no density matrix");
  const GeomView gv = geom_view(g);
  if (dtype == QM_F64) return gto_eval<double>(ctx, mol, (hipStream_t)stream, nullptr, gv, npoints(g), (double*)out);
  if (dtype == QM_F32) return gto_eval<float>(ctx, mol, (hipStream_t)stream, nullptr, gv, npoints(g), (float*)out);
  return qm_fail(ctx, QM_EINVAL, "gto: bad dtype");
}

}  // extern "C"
