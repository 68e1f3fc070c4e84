// Sine transforms (DST-I) of the interior of a grid, as FP64 matrix products.
//
// Both relaxations of the library are linear and act on the interior points only, with the outer layer
// held: the Jacobi sweep (reference kernel_hartree.cu:85-171) and the diffusion V_ne sweep (kernel_vne.cu:13-128).
// Their neighbour sums are diagonal in the products of sin(pi k n / (m + 1)) along each axis (m interior
// points), so a given number of sweeps has a closed form: with increments d_j = A^j d_0 the field after n
// sweeps is V_0 + sum_{j<n} d_j, a multiplication by (1 - a^n) / (1 - a) between two transforms, a being the
// eigenvalue of the sweep.  A fixed sweep count is then 6 one-axis transforms whatever the count, and the
// change of the n-th sweep (the convergence test) is 3 transforms of a^(n-1) times the stored spectrum.
//
// One axis is a product with the symmetric m x m matrix S_kn = sqrt(2 / (m + 1)) sin(pi k n / (m + 1)), which
// is its own inverse.  Its rows are even or odd under n -> m + 1 - n in turn, so the product is two of half the
// size: the rows of odd k take the sums u_j = x_j + x_m+1-j, those of even k the differences, m flops per point.
// An FFT would take about 2.5 log2 m per real point, but this runs on the FP64 matrix cores for any m (an FFT of
// the odd extension has length 2 (m + 1) = 510 for 256 points, with factors 17 and 51), and one pass reads and
// writes each value once like an FFT pass: 256^3, 6 transforms: 25 GFLOP, 1.6 GB.
//
// Kernel: a workgroup of 8 waves owns 16 LT lines and keeps their sums and differences in LDS ([line tile][j]
// [16 lines]: an MFMA operand row is 128 contiguous bytes, and 4 consecutive rows cover all 64 banks; the lines of
// row j are permuted by j mod 16, so that 16 values of one line spread over the banks too, as lines along x are
// loaded and stored); waves 0-3 own the rows of odd k, waves 4-7 those of even k, and read S from L2 (64 points:
// 16 KB, 254: 258 KB) straight into operands.  Lines are read whole before anything is stored, so a pass works
// in place.  254^3, with all of S and rows shared out among 8 waves -> these: x from the residual 242 -> 188 us, y 192 ->
// 128, z forward, factor and back 448 -> 314, x added to V 228 -> 160 (262 MB a pass: 53 us of copying; the products
// 58 us at the rate of a large one); load, product and store of a workgroup follow each other, two share a CU.
#include <algorithm>
#include <cmath>

#include <type_traits>

#include "qm_sine.h"

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 512;
constexpr int kMaxM = 1024;       // interior points per axis (131 KB of LDS)
// Residuals from here on, and those that are not finite, are left to the sweeps.  A transform grows values by at most
// m sqrt(2 / (m + 1)) < 46 an axis and the factor is below 1 / (1 - a) < 2.2e5, so six transforms stay below 2.1e15
// times the residual, 2.1e305; sweeps reach the end of the range only where the field itself does.
constexpr double kMaxResidual = 1e290;

enum Load { LOAD_PLAIN, LOAD_RESIDUAL, LOAD_SCALED };
enum Store { STORE_PLAIN, STORE_ADD, STORE_SUM, STORE_SUMV };

struct Args {
  SinePlan p;
  const double* in;
  double* out;              // STORE_ADD: the field that receives the sum; STORE_SUMV: the field
  const double* rho;        // LOAD_RESIDUAL: in is V, the result is one Jacobi sweep minus V
  double hinv;
  SineFactor f;
  double* part;             // STORE_SUM: sum |x|, STORE_SUMV: sum |out + x|, one per workgroup
  const double* gate;       // STORE_ADD: nothing is added if sine_undecided(*gate, tol, delta)
  double tol, delta;
};

// q = 1 - a and c = 1 + a of the sweep's eigenvalue a at mode (kx, ky, kz) (0-based), from sin^2 of the half
// angles, without cancellation where they are small: a = (cos x + cos y + cos z) / 3 (Jacobi), or one minus the
// row sum's distance from 1 and the weights times 1 - cos, 1 - cos cos', 1 - cos cos' cos'' (V_ne, where c stays near 2).
// Returns a^n (SINE_POWER) or (1 - a^n) / (1 - a) (SINE_SUM).
__device__ __forceinline__ double factor(const SinePlan& p, const SineFactor& f, int kx, int ky, int kz) {
  double q, c;
  const double sx = p.s2[0][kx], sy = p.s2[1][ky], sz = p.s2[2][kz];   // sin^2(theta / 2)
  if (f.sweep == SINE_JACOBI) {
    q = (sx + sy + sz) * (2.0 / 3.0);
    c = (p.s2[0][p.m[0] - 1 - kx] + p.s2[1][p.m[1] - 1 - ky] + p.s2[2][p.m[2] - 1 - kz]) * (2.0 / 3.0);
  } else {
    const double yz = 2.0 * (sy + sz - 2.0 * sy * sz);   // 1 - cos y cos z
    q = f.w0 + f.w1 * (2.0 * (sx + sy + sz)) + f.w2 * (2.0 * (sx + sy - 2.0 * sx * sy) + 2.0 * (sx + sz - 2.0 * sx * sz) + yz) +
        f.w3 * (2.0 * sx + (1.0 - 2.0 * sx) * yz);
    c = 2.0 - q;
  }
  // log |a| from the smaller of 1 - a and 1 + a (with a near 0 both may round to just above 1)
  const bool pos = q < 1.0;
  const double la = log1p(-fmin(pos ? q : c, 1.0));
  if (f.kind == SINE_POWER) {
    const double v = exp(f.n * la);
    return !pos && f.odd ? -v : v;
  }
  if (fabs(q) < 1e-290) return f.n;
  if (pos) return -expm1(f.n * la) / q;
  const double v = exp(f.n * la);
  return (1.0 - (f.odd ? -v : v)) / q;
}

template <int LT, int RT, int AX, int LOAD, bool MID, int STORE>
__global__ __launch_bounds__(kThreads) void k_sine(Args a) {
  constexpr int HP = 64 * RT;         // rows 0 ..: sums, rows HP ..: differences
  __shared__ __align__(16) double x[LT][2 * HP][16];
  __shared__ int64_t base[16 * LT];   // first interior point of each line
  __shared__ int2 mode[16 * LT];      // its indices along the two other axes
  const SinePlan& p = a.p;
  // left to qm_sine_sweeps_if or to the caller
  if (STORE == STORE_ADD && (*p.flag || (a.gate && sine_undecided(*a.gate, a.tol, a.delta)))) return;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int li = lane & 15, lk = lane >> 4;
  const int m = p.m[AX], ld = p.ld[AX];
  const int half = (m + 1) / 2;       // sums; m / 2 differences
  const int m0 = AX == 0 ? p.m[1] : p.m[0];   // fast one of the other axes
  const int m1 = AX == 2 ? p.m[1] : p.m[2];
  const int64_t nx = p.nx, nxy = (int64_t)p.nx * p.ny;
  const int64_t stride = AX == 0 ? 1 : AX == 1 ? nx : nxy;
  const int64_t nl = (int64_t)m0 * m1, l0 = (int64_t)blockIdx.x * (16 * LT);
  if (t < 16 * LT) {
    const int64_t l = min(l0 + t, nl - 1);
    const int u = (int)(l % m0), w = (int)(l / m0);
    base[t] = AX == 0 ? 1 + nx * (1 + u) + nxy * (1 + w)
                      : AX == 1 ? (1 + u) + nx + nxy * (1 + w) : (1 + u) + nx * (1 + w) + nxy;
    mode[t] = make_int2(u, w);
  }
  __syncthreads();
  auto at = [&](int line, int row) __attribute__((always_inline)) -> double& {
    return x[line >> 4][row][(line ^ row) & 15];
  };
  // mode (kx, ky, kz) of element n of line t
  auto fac = [&](int line, int n) __attribute__((always_inline)) -> double {
    const int2 u = mode[line];
    return AX == 0 ? factor(p, a.f, n, u.x, u.y) : AX == 1 ? factor(p, a.f, u.x, n, u.y) : factor(p, a.f, u.x, u.y, n);
  };
  bool bad = false;
  auto load = [&](int line, int n) __attribute__((always_inline)) -> double {
    const int64_t idx = base[line] + n * stride;
    if (LOAD == LOAD_RESIDUAL) {
      const double* __restrict__ V = a.in;
      double s = V[idx - 1] + V[idx + 1];
      s += V[idx + nx];
      s += V[idx - nx];
      s += V[idx + nxy];
      s += V[idx - nxy];
      const double v = fma(-a.rho[idx], a.hinv, s) * (1.0 / 6.0) - V[idx];
      bad = bad || !(fabs(v) < kMaxResidual);
      return v;
    }
    const double v = a.in[idx];
    if (LOAD != LOAD_SCALED) return v;
    {
#pragma clang fp contract(off)   // the product is rounded before the sums, as where it is kept in between (MID)
      const double scaled = v * fac(line, n);
      return scaled;
    }
  };
  // element e of the workgroup's count * 16 LT: lines along x: 16 threads per 128 bytes of a line; else
  // consecutive threads take neighbouring lines
  auto split = [&](int e, int& line, int& n) __attribute__((always_inline)) {
    line = AX == 0 ? (e >> 4) % (16 * LT) : e % (16 * LT);
    n = AX == 0 ? (e & 15) + 16 * ((e >> 4) / (16 * LT)) : e / (16 * LT);
  };
  const int rows = (half + 15) / 16 * 16;
  for (int e = t; e < rows * 16 * LT; e += kThreads) {
    int line, j;
    split(e, line, j);
    double u = 0.0, v = 0.0;
    if (j < half) {
      u = load(line, j);
      const int n = m - 1 - j;
      if (n != j) {
        const double w = load(line, n);
        v = u - w;
        u += w;
      }
    }
    at(line, j) = u;
    at(line, HP + j) = v;
  }
  if (LOAD == LOAD_RESIDUAL && bad) atomicOr(p.flag, 1);
  __syncthreads();

  const int odd = wave >> 2, w4 = wave & 3;   // odd: differences, rows k = 2 r + 1 (0-based)
  const int kk = odd ? m / 2 : half;
  const double* __restrict__ S = odd ? p.So[AX] : p.S[AX];
  d4 acc[RT][LT];
  auto product = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int l = 0; l < LT; ++l) acc[r][l] = d4{0, 0, 0, 0};
    const double* __restrict__ Sw = S + (int64_t)lk * ld + 16 * w4 + li;
    const int lx = li ^ lk;
    auto run = [&](auto nrc) __attribute__((always_inline)) {
      constexpr int NR = decltype(nrc)::value;
#pragma unroll 4
      for (int n0 = 0; n0 < kk; n0 += 4) {   // rows beyond the half of S and of x are zero
        double b[LT], s[NR > 0 ? NR : 1];
#pragma unroll
        for (int r = 0; r < NR; ++r) s[r] = Sw[(int64_t)n0 * ld + 64 * r];
#pragma unroll
        for (int l = 0; l < LT; ++l) b[l] = x[l][HP * odd + n0 + lk][lx ^ (n0 & 12)];
#pragma unroll
        for (int r = 0; r < NR; ++r)
#pragma unroll
          for (int l = 0; l < LT; ++l) acc[r][l] = __builtin_amdgcn_mfma_f64_16x16x4f64(s[r], b[l], acc[r][l], 0, 0, 0);
      }
    };
    // row tiles of this wave: w4 + 4 r < (kk + 15) / 16 (uniform)
    const int nr = max(0, ((kk + 15) / 16 - w4 + 3) / 4);
    if (nr == RT) run(std::integral_constant<int, RT>());
    else if (RT > 1 && nr == RT - 1) run(std::integral_constant<int, RT - 1>());
    else if (RT > 2 && nr == RT - 2) run(std::integral_constant<int, (RT > 2 ? RT - 2 : 0)>());
    else if (RT > 3 && nr == RT - 3) run(std::integral_constant<int, (RT > 3 ? RT - 3 : 0)>());
    else if (RT > 4 && nr == RT - 4) run(std::integral_constant<int, (RT > 4 ? RT - 4 : 0)>());
  };
  // element of acc[r][l][q]: line 16 l + li, n = 2 (16 (w4 + 4 r) + 4 q + lk) + odd
  auto each = [&](auto&& f) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int l = 0; l < LT; ++l)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int n = 2 * (16 * (w4 + 4 * r) + 4 * q + lk) + odd;
          if (n < m) f(16 * l + li, n, acc[r][l][q]);
        }
  };
  product();
  if (MID) {
    // scaled values at the rows of their sums and differences, then folded in place
    __syncthreads();
    each([&](int line, int n, double v) { at(line, n < half ? n : HP + m - 1 - n) = v * fac(line, n); });
    __syncthreads();
    for (int e = t; e < half * 16 * LT; e += kThreads) {
      const int line = e % (16 * LT), j = e / (16 * LT);
      double u = at(line, j), v = 0.0;
      if (m - 1 - j != j) {
        const double w = at(line, HP + j);
        v = u - w;
        u += w;
      }
      at(line, j) = u;
      at(line, HP + j) = v;
    }
    __syncthreads();
    product();
  }
  double sum = 0.0;
  auto store = [&](int line, int n, double v) __attribute__((always_inline)) {
    if (l0 + line >= nl) return;
    const int64_t idx = base[line] + n * stride;
    if (STORE == STORE_PLAIN) a.out[idx] = v;
    else if (STORE == STORE_ADD) a.out[idx] += v;
    else if (STORE == STORE_SUM) sum += fabs(v);
    else sum += fabs(a.out[idx] + v);
  };
  if (AX == 0 && STORE != STORE_SUM) {
    // along x a wave's values are every other point: through LDS, so that whole cache lines are stored
    __syncthreads();
    each([&](int line, int n, double v) { at(line, n) = v; });
    __syncthreads();
    for (int e = t; e < (m + 15) / 16 * 16 * 16 * LT; e += kThreads) {
      int line, n;
      split(e, line, n);
      if (n < m) store(line, n, at(line, n));
    }
  } else {
    each(store);
  }
  if (STORE == STORE_SUM || STORE == STORE_SUMV) {
    __shared__ double red[8];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_down(sum, off, 64);
    if (lane == 0) red[wave] = sum;
    __syncthreads();
    if (t == 0) {
      double s = 0.0;
      for (int w = 0; w < 8; ++w) s += red[w];
      a.part[blockIdx.x] = s;
    }
  }
}

// The halves of S (row j: input, column r: output 2 r or 2 r + 1, 0-based) with zero columns up to ld and zero rows
// up to a multiple of 4, and sin^2(pi k / (2 (m + 1)))
__global__ __launch_bounds__(256) void k_sine_tables(SinePlan p) {
  const int ax = blockIdx.y, m = p.m[ax], ld = p.ld[ax];
  const int half = (m + 1) / 2, rows = (half + 3) / 4 * 4;
  double* __restrict__ s2 = const_cast<double*>(p.s2[ax]);
  if (ax == 0 && blockIdx.x == 0 && threadIdx.x == 0) {
    *p.flag = 0;
    p.ctl[0] = p.ctl[1] = p.ctl[2] = 0;
  }
  const double scale = sqrt(2.0 / (m + 1));
  for (int i = blockIdx.x * 256 + threadIdx.x; i < 2 * rows * ld; i += gridDim.x * 256) {
    const int odd = i >= rows * ld, q = i - odd * rows * ld;
    const int j = q / ld, r = q - j * ld, k = 2 * r + odd;
    const int64_t a = (int64_t)(j + 1) * (k + 1) % (2 * (m + 1));
    const bool in = k < m && j < (odd ? m / 2 : half);
    const_cast<double*>(odd ? p.So[ax] : p.S[ax])[q] = in ? scale * sinpi((double)a / (m + 1)) : 0.0;
  }
  for (int i = blockIdx.x * 256 + threadIdx.x; i < m; i += gridDim.x * 256) {
    const double h = sinpi((double)(i + 1) / (2 * (m + 1)));
    s2[i] = h * h;
  }
}

// The sweeps of a relaxation whose residual is left to them, in one launch behind the closed form, so that the host
// need not wait for the flag: without it the workgroups return at once (3 us; a wait for the flag held the caller
// for all earlier work of the stream).  A sweep is followed by a barrier of the workgroups that take part.  These are
// the ones that run when the first of them closes the count; a workgroup that starts later returns, so a barrier only
// waits for workgroups that are running and every wait ends, whatever else the GPU runs.  The arithmetic of a
// point is that of the sweep kernels.
constexpr unsigned long long kClosed = 1ull << 32;
__global__ __launch_bounds__(kThreads) void k_sweeps_if(const int* flag, unsigned long long* ctl, const double* rho,
                                                        double* v, double* tmp, int nx, int ny, int nz, double hinv,
                                                        int64_t sweeps) {
  if (*flag == 0) return;
  __shared__ unsigned long long in;   // this workgroup's number and, once closed, the count
  if (threadIdx.x == 0) {
    unsigned long long at = __hip_atomic_fetch_add(&ctl[0], 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (at == 0) {   // the first one gives the others some time
      for (int i = 0; i < 4096; ++i) {
        if (__hip_atomic_load(&ctl[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x) break;
        __builtin_amdgcn_s_sleep(8);
      }
      const unsigned long long n = __hip_atomic_fetch_or(&ctl[0], kClosed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      // the count at closing, for the others (ctl[0] may grow by late ones)
      __hip_atomic_store(&ctl[2], n, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    }
    in = at;
  }
  __syncthreads();
  const unsigned long long me = in;
  if (me & kClosed) return;   // late
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long n;
    while ((n = __hip_atomic_load(&ctl[2], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT)) == 0) __builtin_amdgcn_s_sleep(8);
    in = n;
  }
  __syncthreads();
  const int64_t count = (int64_t)in;
  const int64_t sz = (int64_t)nx * ny, n = sz * nz;
  const int64_t lo = n * (int64_t)me / count, hi = n * ((int64_t)me + 1) / count;
  unsigned long long target = 0;
  auto barrier = [&]() {
    target += count;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");   // every wave's own stores, before thread 0 arrives
    __syncthreads();
    if (threadIdx.x == 0) {
      __hip_atomic_fetch_add(&ctl[1], 1ull, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
      while (__hip_atomic_load(&ctl[1], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT) < target) __builtin_amdgcn_s_sleep(1);
    }
    __syncthreads();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  };
  double *src = v, *dst = tmp;
  for (int64_t q = 0; q < sweeps; ++q) {
    for (int64_t e = lo + threadIdx.x; e < hi; e += kThreads) {
      const int i = (int)(e % nx), j = (int)(e / nx % ny), k = (int)(e / sz);
      double r = src[e];
      if (i > 0 && i < nx - 1 && j > 0 && j < ny - 1 && k > 0 && k < nz - 1) {
        double s = src[e - 1] + src[e + 1];
        s += src[e + nx];
        s += src[e - nx];
        s += src[e + sz];
        s += src[e - sz];
        r = fma(-rho[e], hinv, s) * (1.0 / 6.0);
      }
      dst[e] = r;
    }
    barrier();
    double* t = src;
    src = dst;
    dst = t;
  }
  if (src != v)
    for (int64_t e = lo + threadIdx.x; e < hi; e += kThreads) v[e] = src[e];
}

template <int LT, int RT, int AX, int LOAD, bool MID, int STORE>
void launch(hipStream_t s, const Args& a) {
  const int64_t nl = (int64_t)(AX == 0 ? a.p.m[1] : a.p.m[0]) * (AX == 2 ? a.p.m[1] : a.p.m[2]);
  hipLaunchKernelGGL((k_sine<LT, RT, AX, LOAD, MID, STORE>), dim3((unsigned)((nl + 16 * LT - 1) / (16 * LT))),
                     dim3(kThreads), 0, s, a);
}

// 32 lines per workgroup (33 or 66 KB of LDS, two workgroups per CU) up to 256 points, 16 beyond
template <int AX, int LOAD, bool MID, int STORE>
int pass(qm_ctx* ctx, hipStream_t s, const Args& a) {
  const int m = a.p.m[AX];
  if (m <= 128) launch<2, 1, AX, LOAD, MID, STORE>(s, a);
  else if (m <= 256) launch<2, 2, AX, LOAD, MID, STORE>(s, a);
  else if (m <= 512) launch<1, 4, AX, LOAD, MID, STORE>(s, a);
  else launch<1, 8, AX, LOAD, MID, STORE>(s, a);
  QM_CHECK_LAUNCH(ctx);
  return QM_OK;
}

Args plain_args(const SinePlan& p, const double* in, double* out) {
  Args a{};
  a.p = p;
  a.in = in;
  a.out = out;
  return a;
}

}  // namespace

int qm_sine_first_below(int64_t n, double dn, double tol, const std::function<int(int64_t, double*)>& delta_at,
                        int64_t* at, double* delta) {
  int64_t lo = 0, hi = n;   // delta(lo) > tol >= delta(hi); 0 stands for "no check yet"
  double dlo = 0.0, dhi = dn;
  for (int step = 0; hi - lo > 1; ++step) {
    int64_t c = lo + (hi - lo) / 2;
    if (lo > 0 && step % 3 != 2 && dhi > 0.0 && tol > 0.0) {
      // where the line through (lo, log dlo) and (hi, log dhi) meets log tol
      const double f = (std::log(dlo) - std::log(tol)) / (std::log(dlo) - std::log(dhi));
      c = lo + (int64_t)std::llround(f * (double)(hi - lo));
      c = std::max(lo + 1, std::min(hi - 1, c));
    }
    double d = 0.0;
    const int rc = delta_at(c, &d);
    if (rc) return rc;
    if (d <= tol) {
      hi = c;
      dhi = d;
    } else {
      lo = c;
      dlo = d;
    }
  }
  *at = hi;
  *delta = dhi;
  return QM_OK;
}

int SineUse::begin() {
  // orders streams of this device only: without fences to the host and other devices 200 sweeps of 64^3 take 51.5
  // instead of 57 us
  if (!ctx->sine_done)
    QM_CHECK_HIP(ctx, hipEventCreateWithFlags(&ctx->sine_done, hipEventDisableTiming | hipEventDisableSystemFence));
  if (ctx->sine_pending) QM_CHECK_HIP(ctx, hipStreamWaitEvent(s, ctx->sine_done, 0));
  held = true;
  return QM_OK;
}

bool qm_sine_fits(const qm_geom* g) {
  const int n[3] = {g->nx, g->ny, g->nz};
  for (int d = 0; d < 3; ++d)
    if (n[d] < 3 || n[d] - 2 > kMaxM) return false;
  return true;
}

int qm_sine_plan(qm_ctx* ctx, hipStream_t s, const qm_geom* g, SinePlan* p) {
  const int n[3] = {g->nx, g->ny, g->nz};
  p->nx = g->nx;
  p->ny = g->ny;
  size_t doubles = 0, off[3], table[3], most = 0;
  for (int d = 0; d < 3; ++d) {
    p->m[d] = n[d] - 2;
    const int half = (p->m[d] + 1) / 2;
    p->ld[d] = (half + 15) / 16 * 16;
    table[d] = (size_t)((half + 3) / 4 * 4) * p->ld[d];
    off[d] = doubles;
    most = std::max(most, 2 * table[d]);
    doubles += 2 * table[d] + p->m[d];
  }
  // partial sums of an x pass, their reduction's, its result, then the flag
  const size_t nparts = ((size_t)p->m[1] * p->m[2] + 15) / 16;
  double* w = nullptr;
  int rc = qm_ws(ctx, s, WS_SINE, sizeof(double) * (doubles + nparts + kRedMaxBlocks + 8), (void**)&w);
  if (rc) return rc;
  for (int d = 0; d < 3; ++d) {
    p->S[d] = w + off[d];
    p->So[d] = p->S[d] + table[d];
    p->s2[d] = p->So[d] + table[d];
  }
  p->part = w + doubles;
  p->red = p->part + nparts;
  p->sum = p->red + kRedMaxBlocks;
  p->flag = (int*)(p->sum + 1);
  p->ctl = (unsigned long long*)(p->sum + 2);
  hipLaunchKernelGGL(k_sine_tables, dim3((unsigned)std::min<size_t>(512, (most + 255) / 256), 3), dim3(256), 0, s, *p);
  QM_CHECK_LAUNCH(ctx);
  return QM_OK;
}

int qm_sine_residual_xy(qm_ctx* ctx, hipStream_t s, const SinePlan& p, const double* rho, const double* v, double h,
                        double* out) {
  Args a = plain_args(p, v, out);
  a.rho = rho;
  a.hinv = 1.0 / h;
  int rc = pass<0, LOAD_RESIDUAL, false, STORE_PLAIN>(ctx, s, a);
  if (rc) return rc;
  return pass<1, LOAD_PLAIN, false, STORE_PLAIN>(ctx, s, plain_args(p, out, out));
}

int qm_sine_x(qm_ctx* ctx, hipStream_t s, const SinePlan& p, double* a) {
  return pass<0, LOAD_PLAIN, false, STORE_PLAIN>(ctx, s, plain_args(p, a, a));
}

int qm_sine_xy(qm_ctx* ctx, hipStream_t s, const SinePlan& p, double* a) {
  int rc = qm_sine_x(ctx, s, p, a);
  if (rc) return rc;
  return pass<1, LOAD_PLAIN, false, STORE_PLAIN>(ctx, s, plain_args(p, a, a));
}

int qm_sine_z(qm_ctx* ctx, hipStream_t s, const SinePlan& p, double* a) {
  return pass<2, LOAD_PLAIN, false, STORE_PLAIN>(ctx, s, plain_args(p, a, a));
}

int qm_sine_z_scale_zy(qm_ctx* ctx, hipStream_t s, const SinePlan& p, const SineFactor& f, double* a) {
  Args r = plain_args(p, a, a);
  r.f = f;
  int rc = pass<2, LOAD_PLAIN, true, STORE_PLAIN>(ctx, s, r);
  if (rc) return rc;
  return pass<1, LOAD_PLAIN, false, STORE_PLAIN>(ctx, s, plain_args(p, a, a));
}

int qm_sine_scale_zy(qm_ctx* ctx, hipStream_t s, const SinePlan& p, const SineFactor& f, const double* spectrum,
                     double* out) {
  Args r = plain_args(p, spectrum, out);
  r.f = f;
  int rc = pass<2, LOAD_SCALED, false, STORE_PLAIN>(ctx, s, r);
  if (rc) return rc;
  return pass<1, LOAD_PLAIN, false, STORE_PLAIN>(ctx, s, plain_args(p, out, out));
}

int qm_sine_x_add(qm_ctx* ctx, hipStream_t s, const SinePlan& p, const double* a, double* v) {
  return pass<0, LOAD_PLAIN, false, STORE_ADD>(ctx, s, plain_args(p, a, v));
}

int qm_sine_x_add_decided(qm_ctx* ctx, hipStream_t s, const SinePlan& p, const double* a, double* v, double tol,
                          double delta) {
  Args r = plain_args(p, a, v);
  r.gate = p.sum;
  r.tol = tol;
  r.delta = delta;
  return pass<0, LOAD_PLAIN, false, STORE_ADD>(ctx, s, r);
}

int qm_sine_sweeps_if(qm_ctx* ctx, hipStream_t s, const SinePlan& p, const qm_geom* g, const double* rho, double* v,
                      double* tmp, int64_t sweeps) {
  hipLaunchKernelGGL(k_sweeps_if, dim3((unsigned)ctx->ncu), dim3(kThreads), 0, s, (const int*)p.flag, p.ctl, rho, v, tmp,
                     g->nx, g->ny, g->nz, 1.0 / g->step, sweeps);
  QM_CHECK_LAUNCH(ctx);
  return QM_OK;
}

int qm_sine_x_sum(qm_ctx* ctx, hipStream_t s, const SinePlan& p, const double* a, const double* v) {
  Args r = plain_args(p, a, const_cast<double*>(v));
  r.part = p.part;
  int rc = v ? pass<0, LOAD_PLAIN, false, STORE_SUMV>(ctx, s, r) : pass<0, LOAD_PLAIN, false, STORE_SUM>(ctx, s, r);
  if (rc) return rc;
  const int64_t nl = (int64_t)p.m[1] * p.m[2], lines = p.m[0] <= 256 ? 32 : 16;
  return qm_reduce_part_dev(ctx, s, QM_RED_SUM, QM_F64, p.part, nullptr, (nl + lines - 1) / lines, p.red, p.sum);
}

int qm_sine_sum(qm_ctx* ctx, hipStream_t s, const SinePlan& p, double* host_sum) {
  QM_CHECK_HIP(ctx, hipMemcpyAsync(ctx->host_scalars + 2, p.sum, sizeof(double), hipMemcpyDeviceToHost, s));
  QM_CHECK_HIP(ctx, hipStreamSynchronize(s));
  *host_sum = ctx->host_scalars[2];
  return QM_OK;
}
