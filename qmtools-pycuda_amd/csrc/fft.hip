// FFT Poisson solve of the total charge: hand-written mixed-radix Stockham FFT.
//
// Reference kernel_fft.cu:23-106 + cuFFT (qmtools.py:2578-2639):
//   rhs = -( -Q/h^3 + sum_A Z_A (2 pi s^2)^-3/2 exp(-r^2/2s^2) [r^2 <= (cutoff s)^2] ) / eps0
//   (Angstrom / volt units; voxel centres (i+1/2) h + origin; nuclei at coords * 0.529177211;
//   Q read x-fastest, rhs written C order [i][j][k])
//   periodic:  V^ = rhs^ * (-1/(4 pi^2 |k|^2)), V^(0) = 0, k in cycles/Angstrom
//   free space (no reference counterpart): V = rhs (*) G on the 2x zero-padded grid,
//     G(d) = -h^3/(4 pi |d|), G(0) = -h^3 C0/(4 pi h), C0 = 2 (3 asinh(1/sqrt2) - pi/4)
//     (the average of 1/|u| over the voxel), G^ cached per geometry.
//
// The charge is real, so its transform is Hermitian and half of it is kept: complex work buffer
// [n0][m1][hs] in C order, the k <= m2 / 2 of axis 2 (hs: that count rounded up to 128 bytes, so the
// groups of adjacent lines of the other two axes start on cache lines).  One kernel per pass:
//   z    two real lines packed as one complex line, separated by symmetry on the way out
//   y    complex lines of i < n0, k <= m2 / 2
//   x    forward, factor in k space, inverse, on the lines held on chip
//   y    inverse, keeping j < n1
//   z    the two half lines of a pair joined as one complex line, its real and imaginary parts stored
//        as the two lines of the potential
// Zero padding is never stored or cleared: positions beyond the grid are read as zero and only
// positions that are read later are written.
//
// A workgroup takes B lines.  The first stage of a transform reads its inputs from memory straight
// into registers and the last stage writes its outputs from registers (both touch positions i + j n / R
// for one i, adjacent lanes adjacent addresses), so only the exchanges between stages go through LDS;
// in the x pass the last forward and first inverse stage have the same radix and so the same points,
// and the product with the factor happens in registers between the two.  Twiddles
// exp(-2 pi i m/n) come from a per-length table in LDS.
#include <algorithm>
#include <cmath>
#include <map>
#include <tuple>
#include <vector>

#include "qm_internal.h"

namespace {

constexpr double kRBohr = 0.529177211;       // kernel_fft.cu:15
constexpr double kEps0 = 0.0055263494;       // kernel_fft.cu:16, e/(V Angstrom)
constexpr double kAng2Bor = 1.8897259886;
constexpr int kThreads = 256;
constexpr int kFftThreads = 512;   // threads of an axis-pass workgroup
// points per workgroup (B lines of n): 8 per thread for complex128, 16 for complex64, so that a
// workgroup's LDS is about the same and a strided axis reads 128 contiguous bytes (B adjacent lines)
// (power-of-two lengths only: the mixed-radix kernel's register staging would spill)
template <typename R, bool POW2>
struct FftPts {
  static constexpr int kMax = sizeof(R) == 4 && POW2 ? 8192 : 4096;
};
constexpr int kMaxStages = 12;   // 4096 = 2^12

template <typename R>
struct Cx {
  R x, y;
};

template <typename R>
__device__ __forceinline__ Cx<R> cmul(Cx<R> a, Cx<R> b) {
  return Cx<R>{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}

// a times the table value b = exp(-i t) (DIR -1, forward) or its conjugate (DIR 1, inverse)
template <int DIR, typename R>
__device__ __forceinline__ Cx<R> twiddle(Cx<R> a, Cx<R> b) {
  return cmul(a, Cx<R>{b.x, DIR < 0 ? b.y : -b.y});
}

// LDS index skew: one empty slot after every 32 complex values, so that the strided accesses of the
// stages (stride RR in the first stage's writes) and of the twiddle table spread over the banks, and an
// odd number of slots per line, so that adjacent lines at one position do too.  FP64, 240 x 256 x 200
// in free space, whole solve: 1011 us; lines 2 (4, 8) slots past a multiple of 16: 1032 (1097, 1337);
// a slot after every 8 (16) values: 1143 (1025), none: 1056.  Complex64 differs by less than 1 %.
__host__ __device__ __forceinline__ int sk(int i) { return i + (i >> 5); }
__host__ __device__ __forceinline__ int line_slots(int n) { return (n + (n >> 5) + 15) / 16 * 16 + 1; }
__host__ __device__ __forceinline__ int table_slots(int n) { return n + (n >> 5) + 1; }

// Division by a run-time divisor 1 <= d < 2^16 of dividends x < 2^16: q = umulhi(x, ceil(2^32 / d))
// is exact (the product overshoots x / d by less than x / 2^32 < 2^-16 <= 1 / d, which cannot reach
// the next integer since frac(x / d) <= 1 - 1 / d); d = 1 is stored as 0.  The mixed-radix passes
// divide every element and butterfly index by the length, the lines per workgroup, the butterfly
// count and the span; these take one multiply instead of a division sequence.
struct FastDiv {
  uint32_t mul;
  __host__ static FastDiv of(int d) {
    FastDiv f;
    f.mul = d <= 1 ? 0u : (uint32_t)((((uint64_t)1 << 32) + (uint64_t)d - 1) / (uint64_t)d);
    return f;
  }
};
__device__ __forceinline__ int fdiv(int x, FastDiv f) { return f.mul ? (int)__umulhi((uint32_t)x, f.mul) : x; }

struct AxisPlan {
  int n;              // transform length
  int nstage;
  int radix[kMaxStages];
  int span[kMaxStages];
  FastDiv ndiv;                 // by n
  FastDiv mdiv[kMaxStages];     // by n / radix (butterflies per line)
  FastDiv pdiv[kMaxStages];     // by the span
};

// What one axis pass does with its lines.  TURN_*: forward, k-space factor, inverse (axis 0).
enum Kind { FORWARD, INVERSE, TURN_FREE, TURN_PERIODIC, FROM_REAL, TO_REAL };
// How: power-of-two lengths; other lengths of radices <= 10; any length (two LDS planes).
enum Path { POW2, RADIX, GENERIC };

struct AxisLines {
  int64_t stride;     // distance between consecutive elements of a line
  int nl0, nl1;       // lines: l0 in [0, nl0), l1 in [0, nl1); real passes: l1 counts pairs of lines
  int64_t s0, s1;     // line base = l0 * s0 + l1 * s1
  int B;              // lines per workgroup (consecutive l1)
  FastDiv bdiv;       // by B
  FastDiv hdiv;       // by n / 2 + 1
  int nin;            // positions >= nin of a line are zero on input (not loaded)
  int nout;           // positions >= nout are not needed after the pass (not stored)
  int nr1, nr2;       // real passes: lines per l0 and points per line of the real array
};

// Transform of the free-space Green's function for one padded shape, computed at unit grid step:
// the transform is real and even in every axis, so one octant is kept, o1 = m1 / 2 + 1 and
// o2 = m2 / 2 + 1 wide; the value at grid step h is g[min(i, m0 - i)][min(j, m1 - j)][min(k, m2 - k)]
// times scale = h^2 (Angstrom), since g(d) = 1 / |d| scales as 1 / h and the voxel volume as h^3.
// TURN_PERIODIC reads the shape, the grid step and the normalisation of the inverse transform.
template <typename R>
struct FactorView {
  const R* g;
  int m0, m1, m2;
  int o1, o2;
  R scale;
  double step, norm;
};

// R-point DFT of x with W = exp(i DIR 2 pi / R), DIR = -1 (forward) or 1.  The odd radices pair x_q with
// x_R-q: real parts of W^k multiply the sums, imaginary parts the differences (radix 5: 16 multiplications
// and no table read, against 16 complex products with table values for the plain sum).  Radices 6 and 10 are radix 3 and 5 of the sums and differences of opposite points, in the
// prime-factor order, which needs no inner twiddles.
template <typename R, int RR, int DIR>
__device__ __forceinline__ void dft(Cx<R>* x) {
  constexpr R dir = (R)DIR;
  if (RR == 2) {
    const Cx<R> a = x[0], b = x[1];
    x[0] = Cx<R>{a.x + b.x, a.y + b.y};
    x[1] = Cx<R>{a.x - b.x, a.y - b.y};
  } else if (RR == 4 || RR == 8) {
    // out_r = sum_m c_m W4^(m r), W4 = i dir
    auto dft4 = [&](const Cx<R>& c0, const Cx<R>& c1, const Cx<R>& c2, const Cx<R>& c3, Cx<R>& o0, Cx<R>& o1, Cx<R>& o2,
                    Cx<R>& o3) __attribute__((always_inline)) {
      const Cx<R> d0{c0.x + c2.x, c0.y + c2.y}, d1{c0.x - c2.x, c0.y - c2.y};
      const Cx<R> d2{c1.x + c3.x, c1.y + c3.y};
      const Cx<R> d3{-dir * (c1.y - c3.y), dir * (c1.x - c3.x)};
      o0 = Cx<R>{d0.x + d2.x, d0.y + d2.y};
      o1 = Cx<R>{d1.x + d3.x, d1.y + d3.y};
      o2 = Cx<R>{d0.x - d2.x, d0.y - d2.y};
      o3 = Cx<R>{d1.x - d3.x, d1.y - d3.y};
    };
    if (RR == 4) {
      const Cx<R> c0 = x[0], c1 = x[1], c2 = x[2], c3 = x[3];
      dft4(c0, c1, c2, c3, x[0], x[1], x[2], x[3]);
    } else {
      // X_2r = DFT4(x_m + x_m+4)_r, X_2r+1 = DFT4((x_m - x_m+4) W8^m)_r, W8 = (1 + i dir) / sqrt 2
      Cx<R> a[4], b[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        a[q] = Cx<R>{x[q].x + x[q + 4].x, x[q].y + x[q + 4].y};
        b[q] = Cx<R>{x[q].x - x[q + 4].x, x[q].y - x[q + 4].y};
      }
      const R h = (R)0.70710678118654752440, hd = h * dir;
      b[1] = Cx<R>{h * b[1].x - hd * b[1].y, h * b[1].y + hd * b[1].x};
      b[2] = Cx<R>{-dir * b[2].y, dir * b[2].x};
      b[3] = Cx<R>{-h * b[3].x - hd * b[3].y, -h * b[3].y + hd * b[3].x};
      dft4(a[0], a[1], a[2], a[3], x[0], x[2], x[4], x[6]);
      dft4(b[0], b[1], b[2], b[3], x[1], x[3], x[5], x[7]);
    }
  } else if (RR == 6 || RR == 10) {
    // m = H a + 2 b, r = H c + (H + 1) d (mod 2H, H odd): W_2H^(m r) = (-1)^(a c) W_H^(b d)
    constexpr int H = RR / 2;
    Cx<R> u[H], v[H];
#pragma unroll
    for (int b = 0; b < H; ++b) {
      const Cx<R> p = x[2 * b], q = x[(2 * b + H) % RR];
      u[b] = Cx<R>{p.x + q.x, p.y + q.y};
      v[b] = Cx<R>{p.x - q.x, p.y - q.y};
    }
    dft<R, RR == 6 ? 3 : 5, DIR>(u);
    dft<R, RR == 6 ? 3 : 5, DIR>(v);
#pragma unroll
    for (int d = 0; d < H; ++d) {
      x[(H + 1) * d % RR] = u[d];
      x[(H + (H + 1) * d) % RR] = v[d];
    }
  } else {
    constexpr int H = RR / 2;
    // cos and sin of 2 pi k / RR, k = 0 .. H
    constexpr double C3[2] = {1.0, -0.5}, S3[2] = {0.0, 0.86602540378443864676};
    constexpr double C5[3] = {1.0, 0.30901699437494742410, -0.80901699437494742410};
    constexpr double S5[3] = {0.0, 0.95105651629515357212, 0.58778525229247312917};
    constexpr double C7[4] = {1.0, 0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624};
    constexpr double S7[4] = {0.0, 0.78183148246802980871, 0.97492791218182360702, 0.43388373911755812048};
    Cx<R> sum[H + 1], dif[H + 1];
    Cx<R> y0 = x[0];
#pragma unroll
    for (int q = 1; q <= H; ++q) {
      sum[q] = Cx<R>{x[q].x + x[RR - q].x, x[q].y + x[RR - q].y};
      dif[q] = Cx<R>{x[q].x - x[RR - q].x, x[q].y - x[RR - q].y};
      y0.x += sum[q].x;
      y0.y += sum[q].y;
    }
    Cx<R> lo[H + 1], hi[H + 1];
#pragma unroll
    for (int j = 1; j <= H; ++j) {
      Cx<R> a = x[0], b{0, 0};
#pragma unroll
      for (int q = 1; q <= H; ++q) {
        const int k = j * q % RR, kk = k <= H ? k : RR - k;
        const double cd = RR == 3 ? C3[kk] : RR == 5 ? C5[kk] : C7[kk];
        const double sd = RR == 3 ? S3[kk] : RR == 5 ? S5[kk] : S7[kk];
        const R c = (R)cd, sn = (R)(k <= H ? sd : -sd);
        a.x += c * sum[q].x;
        a.y += c * sum[q].y;
        b.x += sn * dif[q].x;
        b.y += sn * dif[q].y;
      }
      // a + i dir b and its mirror
      lo[j] = Cx<R>{a.x - dir * b.y, a.y + dir * b.x};
      hi[j] = Cx<R>{a.x + dir * b.y, a.y - dir * b.x};
    }
    x[0] = y0;
#pragma unroll
    for (int j = 1; j <= H; ++j) {
      x[j] = lo[j];
      x[RR - j] = hi[j];
    }
  }
}

// One radix-RR Stockham stage on a workgroup's B lines.  EDGE 0: LDS to LDS in place (all inputs of the
// thread's butterflies are read into registers, then, after a barrier, the outputs are written).
// EDGE 1: the first stage, inputs through io.load, no twiddles.  EDGE 2: the last stage, outputs through
// io.store.  EDGE 3: the last forward stage, io.factor and the first inverse stage (span 1) in one.
// Butterflies of the first and last stage follow the order of the lines in memory (ROWS: line-major,
// else line-minor).  P2: n, p, B and RR are powers of two, so the line / butterfly / twiddle indices
// come from shifts and masks instead of divisions by run-time values.
template <typename R, int RR, int DIR, int EDGE, bool P2, typename IO>
__device__ __forceinline__ void stage(const IO& io, Cx<R>* buf, const Cx<R>* __restrict__ tw, int n, int B, int LS,
                                      int p, FastDiv mdiv, FastDiv pdiv) {
  constexpr int MAXB = (FftPts<R, P2>::kMax / kFftThreads + RR - 1) / RR;   // butterflies per thread (B n <= kMax)
  const int m = n / RR;
  const int tstep = n / (p * RR);
  const int total = B * m;
  const int lm = P2 ? __builtin_ctz(m) : 0, lb = P2 ? __builtin_ctz(B) : 0;
  const bool rows = EDGE == 0 || io.rows();
  auto split = [&](int bf, int& l, int& i) __attribute__((always_inline)) {   // bf < B n <= kMax
    if (rows) {
      l = P2 ? bf >> lm : fdiv(bf, mdiv);
      i = P2 ? bf & (m - 1) : bf - l * m;
    } else {
      i = P2 ? bf >> lb : fdiv(bf, io.bdiv());
      l = P2 ? bf & (B - 1) : bf - i * B;
    }
  };
  // the span of the last stage is m, of the first stage 1
  auto rem = [&](int i) __attribute__((always_inline)) {
    return EDGE == 1 ? 0 : EDGE >= 2 ? i : P2 ? i & (p - 1) : i - fdiv(i, pdiv) * p;
  };
  Cx<R> x[MAXB][RR];
#pragma unroll
  for (int b = 0; b < MAXB; ++b) {
    const int bf = threadIdx.x + b * kFftThreads;
    if (bf < total) {
      int l, i;
      split(bf, l, i);
      if (EDGE == 1) {
        io.template load<RR>(l, i, m, x[b]);
      } else {
        const int k = rem(i);
        const Cx<R>* src = buf + l * LS;
#pragma unroll
        for (int j = 0; j < RR; ++j) {
          const Cx<R> v = src[sk(i + j * m)];
          // j k tstep <= (RR - 1)(p - 1) n / (p RR) < n: the twiddle index needs no reduction
          x[b][j] = j ? twiddle<DIR>(v, tw[sk(j * k * tstep)]) : v;
        }
      }
    }
  }
#pragma unroll
  for (int b = 0; b < MAXB; ++b) {
    const int bf = threadIdx.x + b * kFftThreads;
    if (bf < total) {
      dft<R, RR, DIR>(x[b]);
      if (EDGE >= 2) {
        int l, i;
        split(bf, l, i);
        if (EDGE == 2) {
          io.template store<RR>(l, i, m, x[b]);
        } else {
          io.template factor<RR>(l, i, m, x[b]);
          dft<R, RR, -DIR>(x[b]);
        }
      }
    }
  }
  if (EDGE == 2) return;
  if (EDGE != 1) __syncthreads();
#pragma unroll
  for (int b = 0; b < MAXB; ++b) {
    const int bf = threadIdx.x + b * kFftThreads;
    if (bf < total) {
      int l, i;
      split(bf, l, i);
      const int k = EDGE == 3 ? 0 : rem(i), q = EDGE == 3 ? 1 : p;
      Cx<R>* dst = buf + l * LS;
      const int o = (i - k) * RR + k;
#pragma unroll
      for (int j = 0; j < RR; ++j) dst[sk(o + j * q)] = x[b][j];
    }
  }
  __syncthreads();
}

// Any radix, out of place between two LDS planes (used when a length has a prime factor > 7).
// Indices as in stage (quotients by multiply-high, twiddle index below n); the DFT table
// index (j q mod RR) m is carried from one q to the next.
template <typename R, int DIR>
__device__ __forceinline__ void stage_generic(const Cx<R>* in, Cx<R>* out, const Cx<R>* __restrict__ tw, int n,
                                              int B, int LS, int RR, int p, FastDiv mdiv, FastDiv pdiv) {
  const int m = n / RR;
  const int tstep = n / (p * RR);
  for (int bf = threadIdx.x; bf < B * m; bf += kFftThreads) {
    const int l = fdiv(bf, mdiv), i = bf - l * m, k = i - fdiv(i, pdiv) * p;
    const Cx<R>* src = in + l * LS;
    Cx<R>* dst = out + l * LS;
    const int o = (i - k) * RR + k;
    for (int j = 0; j < RR; ++j) {
      Cx<R> acc{0, 0};
      int jq = 0;   // j q mod RR
      for (int q = 0; q < RR; ++q) {
        Cx<R> v = src[sk(i + q * m)];
        if (k) v = twiddle<DIR>(v, tw[sk(q * k * tstep)]);
        const Cx<R> t = twiddle<DIR>(v, tw[sk(jq * m)]);
        acc.x += t.x;
        acc.y += t.y;
        jq += j;
        if (jq >= RR) jq -= RR;
      }
      dst[sk(o + j * p)] = acc;
    }
  }
  __syncthreads();
}

template <typename R, int DIR, int EDGE, bool P2, typename IO>
__device__ __forceinline__ void run_stage(const IO& io, const AxisPlan& plan, int s, Cx<R>* buf, const Cx<R>* tw,
                                          int B, int LS) {
  const int n = plan.n, p = plan.span[s];
  const FastDiv md = plan.mdiv[s], pd = plan.pdiv[s];
  if (P2) {
    switch (plan.radix[s]) {
      case 2: stage<R, 2, DIR, EDGE, P2>(io, buf, tw, n, B, LS, p, md, pd); break;
      case 4: stage<R, 4, DIR, EDGE, P2>(io, buf, tw, n, B, LS, p, md, pd); break;
      default: stage<R, 8, DIR, EDGE, P2>(io, buf, tw, n, B, LS, p, md, pd); break;
    }
  } else {
    switch (plan.radix[s]) {
      case 2: stage<R, 2, DIR, EDGE, P2>(io, buf, tw, n, B, LS, p, md, pd); break;
      case 3: stage<R, 3, DIR, EDGE, P2>(io, buf, tw, n, B, LS, p, md, pd); break;
      case 4: stage<R, 4, DIR, EDGE, P2>(io, buf, tw, n, B, LS, p, md, pd); break;
      case 5: stage<R, 5, DIR, EDGE, P2>(io, buf, tw, n, B, LS, p, md, pd); break;
      case 6: stage<R, 6, DIR, EDGE, P2>(io, buf, tw, n, B, LS, p, md, pd); break;
      case 7: stage<R, 7, DIR, EDGE, P2>(io, buf, tw, n, B, LS, p, md, pd); break;
      case 8: stage<R, 8, DIR, EDGE, P2>(io, buf, tw, n, B, LS, p, md, pd); break;
      default: stage<R, 10, DIR, EDGE, P2>(io, buf, tw, n, B, LS, p, md, pd); break;
    }
  }
}

template <typename R, int DIR>
__device__ __forceinline__ Cx<R>* run_generic(const AxisPlan& plan, Cx<R>* in, Cx<R>* out, const Cx<R>* tw, int B,
                                              int LS) {
  for (int s = 0; s < plan.nstage; ++s) {
    stage_generic<R, DIR>(in, out, tw, plan.n, B, LS, plan.radix[s], plan.span[s], plan.mdiv[s], plan.pdiv[s]);
    Cx<R>* t = in;
    in = out;
    out = t;
  }
  return in;
}

__device__ __forceinline__ double periodic_freq(int i, int n, double step) {
  return (i > n / 2 - 1 ? (double)(i - n) : (double)i) / (n * step);
}

// Memory side of a pass: element j of butterfly i of workgroup line l is position i + j m.
template <typename R, typename TO, int KIND>
struct LineIO {
  Cx<R>* data;          // the workgroup's first line (complex side)
  const R* rin;         // FROM_REAL: the workgroup's first pair
  TO* rout;             // TO_REAL
  const AxisLines& ln;
  const FactorView<R>& fv;
  int n, l0, l1b, nb;

  __device__ __forceinline__ bool rows() const {
    return KIND == FROM_REAL || KIND == TO_REAL || ln.stride == 1;
  }
  __device__ __forceinline__ FastDiv bdiv() const { return ln.bdiv; }
  // the second line of the last pair may not exist
  __device__ __forceinline__ bool second(int l) const { return 2 * (l1b + l) + 1 < ln.nr1; }

  template <int RR>
  __device__ __forceinline__ void load(int l, int i, int m, Cx<R>* x) const {
    if (KIND == FROM_REAL) {
      const R* a = rin + (int64_t)(2 * l) * ln.nr2;
      const bool two = second(l);
#pragma unroll
      for (int j = 0; j < RR; ++j) {
        const int e = i + j * m;
        x[j] = Cx<R>{0, 0};
        if (l < nb && e < ln.nin) {
          x[j].x = a[e];
          if (two) x[j].y = a[e + ln.nr2];
        }
      }
    } else if (KIND == TO_REAL) {
      // X = A + i B of the Hermitian halves A and B; their first and middle values are real
      const Cx<R>* a = data + (int64_t)(2 * l) * ln.s1;
      const bool two = second(l);
#pragma unroll
      for (int j = 0; j < RR; ++j) {
        const int e = i + j * m, k = min(e, n - e);
        x[j] = Cx<R>{0, 0};
        if (l < nb) {
          Cx<R> u = a[k], v{0, 0};
          if (two) v = a[k + ln.s1];
          const R sg = 2 * k == n || k == 0 ? (R)0 : e == k ? (R)1 : (R)-1;
          x[j] = Cx<R>{u.x - sg * v.y, sg * u.y + v.x};
        }
      }
    } else {
      const Cx<R>* a = data + (int64_t)l * ln.s1 + (int64_t)i * ln.stride;
#pragma unroll
      for (int j = 0; j < RR; ++j) {
        x[j] = Cx<R>{0, 0};
        if (l < nb && i + j * m < ln.nin) x[j] = a[(int64_t)(j * m) * ln.stride];
      }
    }
  }

  template <int RR>
  __device__ __forceinline__ void store(int l, int i, int m, const Cx<R>* x) const {
    if (l >= nb) return;
    if (KIND == TO_REAL) {
      TO* a = rout + (int64_t)(2 * l) * ln.nr2;
      const bool two = second(l);
#pragma unroll
      for (int j = 0; j < RR; ++j) {
        const int e = i + j * m;
        if (e < ln.nout) {
          a[e] = (TO)x[j].x;
          if (two) a[e + ln.nr2] = (TO)x[j].y;
        }
      }
    } else {
      Cx<R>* a = data + (int64_t)l * ln.s1 + (int64_t)i * ln.stride;
#pragma unroll
      for (int j = 0; j < RR; ++j)
        if (i + j * m < ln.nout) a[(int64_t)(j * m) * ln.stride] = x[j];
    }
  }

  // TURN_*: line (j, k) = (l0, l1b + l) with k <= m2 / 2, position along axis 0
  template <int RR>
  __device__ __forceinline__ void factor(int l, int i, int m, Cx<R>* x) const {
    if (l >= nb) return;
    const int k = l1b + l;
    if (KIND == TURN_FREE) {
      const R* g = fv.g + (int64_t)min(l0, fv.m1 - l0) * fv.o2 + k;
      const int64_t gs = (int64_t)fv.o1 * fv.o2;
#pragma unroll
      for (int j = 0; j < RR; ++j) {
        const int e = i + j * m;
        const R f = g[min(e, n - e) * gs] * fv.scale;
        x[j].x *= f;
        x[j].y *= f;
      }
    } else {
      // -1 / (4 pi^2 |k|^2), 0 at k = 0 (kernel_fft.cu:82-106).  The frequency of an odd axis is not
      // antisymmetric there (index n / 2 counts as -(n + 1) / 2); the real part of the full inverse
      // transform, which is the result, has the mean of the factors at k and -k.
      const double ky = periodic_freq(l0, fv.m1, fv.step), kz = periodic_freq(k, fv.m2, fv.step);
      const double kyz = ky * ky, kz2 = kz * kz;
      const bool odd = (fv.m0 | fv.m1 | fv.m2) & 1;
      double my = ky, mz = kz;
      if (odd) {
        my = periodic_freq(l0 ? fv.m1 - l0 : 0, fv.m1, fv.step);
        mz = periodic_freq(k ? fv.m2 - k : 0, fv.m2, fv.step);
      }
#pragma unroll
      for (int j = 0; j < RR; ++j) {
        const int e = i + j * m;
        if ((e | l0 | k) == 0) {
          x[j] = Cx<R>{0, 0};
          continue;
        }
        const double kx = periodic_freq(e, n, fv.step);
        double f = -1.0 / (4.0 * M_PI * M_PI * (kx * kx + kyz + kz2)) * fv.norm;
        if (odd) {
          const double mx = periodic_freq(e ? n - e : 0, n, fv.step);
          f = 0.5 * (f + -1.0 / (4.0 * M_PI * M_PI * (mx * mx + my * my + mz * mz)) * fv.norm);
        }
        x[j].x = (R)(x[j].x * f);
        x[j].y = (R)(x[j].y * f);
      }
    }
  }
};

// One pass along one axis (unnormalised transforms).  PATH GENERIC (a prime factor above 7, or a
// single stage): the lines are loaded into LDS, the stages run between two planes and the result
// is stored from there.  FP64, 240 x 256 x 200 in free space (480 x 512 x 400), complex passes on all of
// the padded axis 2 with an LDS exchange at both ends -> these: x 1840 -> 590 us (0.8 GB moved), y 300 -> 125 and
// 121, z 260 -> 106 and 100.  What is left in x: LDS busy for 55 % of the time, arithmetic for 39 %.
template <typename R, typename TO, int KIND, int PATH>
__global__ __launch_bounds__(kFftThreads) void k_fft_axis(Cx<R>* __restrict__ data, const R* __restrict__ rin,
                                                       TO* __restrict__ rout, const Cx<R>* __restrict__ twg,
                                                       AxisPlan plan, AxisPlan back, AxisLines ln,
                                                       FactorView<R> fv) {
  extern __shared__ unsigned char smem[];
  constexpr bool TURN = KIND == TURN_FREE || KIND == TURN_PERIODIC;
  constexpr int DIR = KIND == INVERSE || KIND == TO_REAL ? 1 : -1;
  constexpr bool P2 = PATH == POW2;
  const int n = plan.n;
  const int B = ln.B;
  const int LS = line_slots(n);
  Cx<R>* tw = (Cx<R>*)smem;
  Cx<R>* buf0 = tw + table_slots(n);
  Cx<R>* buf1 = buf0 + (int64_t)B * LS;
  const int lines_per_row = (ln.nl1 + B - 1) / B;
  const int l0 = blockIdx.x / lines_per_row;
  const int l1b = (blockIdx.x % lines_per_row) * B;
  constexpr bool REAL = KIND == FROM_REAL || KIND == TO_REAL;
  const int64_t first = (int64_t)l0 * ln.s0 + (int64_t)(REAL ? 2 * l1b : l1b) * ln.s1;
  const int64_t rfirst = REAL ? ((int64_t)l0 * ln.nr1 + 2 * l1b) * ln.nr2 : 0;
  const LineIO<R, TO, KIND> io{data + first, rin + rfirst, rout + rfirst, ln, fv, n, l0, l1b,
                               min(B, ln.nl1 - l1b)};
  for (int q = threadIdx.x; q < n; q += kFftThreads) tw[sk(q)] = twg[q];
  Cx<R>* res = buf0;
  if (PATH == GENERIC) {
    const bool rows = io.rows();
    auto split = [&](int e) __attribute__((always_inline)) {   // (line, position)
      if (rows) {
        const int l = fdiv(e, plan.ndiv);
        return make_int2(l, e - l * n);
      }
      const int a = fdiv(e, ln.bdiv);
      return make_int2(e - a * B, a);
    };
    for (int e = threadIdx.x; e < B * n; e += kFftThreads) {
      const int2 la = split(e);
      io.template load<1>(la.x, la.y, 0, buf0 + la.x * LS + sk(la.y));
    }
    __syncthreads();
    res = run_generic<R, DIR>(plan, buf0, buf1, tw, B, LS);
    if (TURN) {
      for (int e = threadIdx.x; e < B * n; e += kFftThreads) {
        const int2 la = split(e);
        io.template factor<1>(la.x, la.y, 0, res + la.x * LS + sk(la.y));
      }
      __syncthreads();
      res = run_generic<R, 1>(plan, res, res == buf0 ? buf1 : buf0, tw, B, LS);
    }
    if (KIND != FROM_REAL) {
      for (int e = threadIdx.x; e < B * n; e += kFftThreads) {
        const int2 la = split(e);
        io.template store<1>(la.x, la.y, 0, res + la.x * LS + sk(la.y));
      }
    }
  } else {
    const int last = plan.nstage - 1;   // >= 1
    run_stage<R, DIR, 1, P2>(io, plan, 0, buf0, tw, B, LS);
    for (int s = 1; s < last; ++s) run_stage<R, DIR, 0, P2>(io, plan, s, buf0, tw, B, LS);
    if (TURN) {
      run_stage<R, DIR, 3, P2>(io, plan, last, buf0, tw, B, LS);
      for (int s = 1; s < last; ++s) run_stage<R, 1, 0, P2>(io, back, s, buf0, tw, B, LS);
      run_stage<R, 1, 2, P2>(io, back, last, buf0, tw, B, LS);
    } else if (KIND == FROM_REAL) {
      run_stage<R, DIR, 0, P2>(io, plan, last, buf0, tw, B, LS);
    } else {
      run_stage<R, DIR, 2, P2>(io, plan, last, buf0, tw, B, LS);
    }
  }
  if (KIND == FROM_REAL) {
    // Z = A + i B: A_k = (Z_k + conj Z_-k) / 2, B_k = (Z_k - conj Z_-k) / 2i
    const int h = n / 2 + 1;
    for (int e = threadIdx.x; e < B * h; e += kFftThreads) {
      const int l = fdiv(e, ln.hdiv), k = e - l * h;
      if (l < io.nb) {
        const Cx<R>* z = res + l * LS;
        const Cx<R> u = z[sk(k)], v = z[sk(k ? n - k : 0)];
        Cx<R>* a = io.data + (int64_t)(2 * l) * ln.s1 + k;
        a[0] = Cx<R>{(R)0.5 * (u.x + v.x), (R)0.5 * (u.y - v.y)};
        if (io.second(l)) a[ln.s1] = Cx<R>{(R)0.5 * (u.y + v.y), (R)0.5 * (v.x - u.x)};
      }
    }
  }
}

// rhs, C order [n0][n1][n2].  Tile: 32 i x 32 k at fixed j; Q is read along i (x-fastest) and written
// along k.  The nuclei whose cutoff sphere reaches the tile's box are listed first (in order, 256 at a
// time): 50 atoms at 240 x 256 x 200, 253 us testing every atom at every voxel, 79 us so.
template <typename R, typename TI>
__global__ __launch_bounds__(kThreads) void k_rhs(const TI* __restrict__ q, const double4* __restrict__ atoms,
                                                  int natoms, GeomView g, double sigma, double cut2,
                                                  R* __restrict__ out) {
  __shared__ double tile[32][33];
  __shared__ double4 near[kThreads];
  __shared__ int cnt[kThreads / 64];
  const int i0 = blockIdx.x * 32, k0 = blockIdx.z * 32, j = blockIdx.y;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;   // 32 x 8
  const double step = g.h / kAng2Bor;
  const double norm = 1.0 / (sigma * sigma * sigma * 2.0 * M_PI * sqrt(2.0 * M_PI));
  const double inv2s2 = 1.0 / (2.0 * sigma * sigma);
#pragma unroll
  for (int r = ty; r < 32; r += 8) {
    const int i = i0 + tx, k = k0 + r;
    double v = 0.0;
    if (i < g.nx && k < g.nz) v = (double)q[i + (int64_t)g.nx * (j + (int64_t)g.ny * k)];
    tile[r][tx] = v;
  }
  __syncthreads();
  const double y = g.oy / kAng2Bor + (j + 0.5) * step;
  const double z = g.oz / kAng2Bor + (k0 + tx + 0.5) * step;
  double rho[4], x[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int r = ty + 8 * c;
    rho[c] = tile[tx][r] / (-(step * step * step));
    x[c] = g.ox / kAng2Bor + (i0 + r + 0.5) * step;
  }
  const double xm = g.ox / kAng2Bor + (i0 + 16) * step, zm = g.oz / kAng2Bor + (k0 + 16) * step, hw = 16.0 * step;
  for (int a0 = 0; a0 < natoms; a0 += kThreads) {
    // the box around the voxel centres, half a step wider: rounding cannot lose an atom
    double4 A{0, 0, 0, 0};
    bool in = false;
    if (a0 + (int)threadIdx.x < natoms) {
      A = atoms[a0 + threadIdx.x];
      A.x *= kRBohr;
      A.y *= kRBohr;
      A.z *= kRBohr;
      const double bx = fmax(fabs(A.x - xm) - hw, 0.0), by = fmax(fabs(A.y - y) - 0.5 * step, 0.0),
                   bz = fmax(fabs(A.z - zm) - hw, 0.0);
      in = bx * bx + by * by + bz * bz <= cut2;
    }
    const uint64_t ball = __ballot(in);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) cnt[wave] = __popcll(ball);
    __syncthreads();
    int at = __popcll(ball & (((uint64_t)1 << lane) - 1)), n = 0;
#pragma unroll
    for (int w = 0; w < kThreads / 64; ++w) {
      at += w < wave ? cnt[w] : 0;
      n += cnt[w];
    }
    if (in) near[at] = A;
    __syncthreads();
    for (int t = 0; t < n; ++t) {
      const double4 C = near[t];
      const double dy = y - C.y, dz = z - C.z;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const double dx = x[c] - C.x;
        const double r2 = dx * dx + dy * dy + dz * dz;
        if (r2 <= cut2) rho[c] += C.w * norm * exp(-r2 * inv2s2);
      }
    }
    __syncthreads();
  }
  const int k = k0 + tx;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int i = i0 + ty + 8 * c;
    if (i < g.nx && k < g.nz) out[((int64_t)i * g.ny + j) * g.nz + k] = (R)(-rho[c] / kEps0);
  }
}

// g(d) at unit grid step on the m0 x m1 x m2 cyclic grid (m >= 2n), C order: |d_i| = min(i, m - i),
// g(0) = C0.  Distances between two voxels of the grid are below n, so only |d| < n is ever used.
template <typename R>
__global__ void k_green(Cx<R>* __restrict__ a, int m0, int m1, int m2) {
  const int64_t N = (int64_t)m0 * m1 * m2;
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= N) return;
  const int k = (int)(idx % m2), j = (int)((idx / m2) % m1), i = (int)(idx / ((int64_t)m1 * m2));
  const double x = min(i, m0 - i);
  const double y = min(j, m1 - j);
  const double z = min(k, m2 - k);
  const double r = sqrt(x * x + y * y + z * z);
  const double c0 = 2.0 * (3.0 * asinh(1.0 / sqrt(2.0)) - M_PI / 4.0);
  const double g = (idx == 0) ? c0 : 1.0 / r;
  a[idx] = Cx<R>{(R)g, (R)0};
}

// the octant i <= m0 / 2, j <= m1 / 2, k <= m2 / 2 of the transform's real part, times scale
template <typename R>
__global__ void k_green_store(const Cx<R>* __restrict__ a, R* __restrict__ gh, int m1, int m2, int o0, int o1,
                              int o2, double scale) {
  const int64_t N = (int64_t)o0 * o1 * o2;
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= N) return;
  const int k = (int)(idx % o2), j = (int)((idx / o2) % o1), i = (int)(idx / ((int64_t)o1 * o2));
  gh[idx] = (R)((double)a[((int64_t)i * m1 + j) * m2 + k].x * scale);
}

// ------------------------------------------------------------------ host: plans
// Stage radices of a length, largest first.  Powers of two and lengths without a prime factor above 7:
// as few stages as radices up to 8 (10) allow, of those the smallest sum (480 = 10 8 6, 400 = 10 8 5,
// 1024 = 8 8 4 4); otherwise 8, 4, 2, 3, 5, 7 and the larger primes.
void best_radices(int n, bool pow2, std::vector<int>& cur, std::vector<int>& best) {
  if (n == 1) {
    auto sum = [](const std::vector<int>& v) {
      int t = 0;
      for (int r : v) t += r;
      return t;
    };
    if (best.empty() || cur.size() < best.size() || (cur.size() == best.size() && sum(cur) < sum(best))) best = cur;
    return;
  }
  if (!best.empty() && cur.size() + 1 > best.size()) return;
  for (int r : {10, 8, 7, 6, 5, 4, 3, 2}) {
    if (n % r || (!cur.empty() && r > cur.back()) || (pow2 && (r & (r - 1)))) continue;
    cur.push_back(r);
    best_radices(n / r, pow2, cur, best);
    cur.pop_back();
  }
}

std::vector<int> factorize(int n) {
  std::vector<int> f, cur;
  best_radices(n, (n & (n - 1)) == 0, cur, f);
  // the first and the last stage hold the two ends of a pass, so 4, 6, 8 and 10 take two stages as well instead of the
  // generic path (8^3, periodic, FP64: 61 -> 27 us)
  if (f.size() == 1 && f[0] % 2 == 0 && f[0] > 2) f = {f[0] / 2, 2};
  if (!f.empty()) return f;
  for (int r : {8, 4, 2, 3, 5, 7}) {
    while (n % r == 0) {
      f.push_back(r);
      n /= r;
    }
  }
  for (int p = 11; n > 1; p += 2)
    while (n % p == 0) {
      f.push_back(p);
      n /= p;
    }
  return f;
}

}  // namespace

// Transforms of the free-space Green's function at unit step, one octant per (padded shape,
// precision), are kept up to kGreenCacheBytes per context; beyond that the least recently used
// are released (stream-ordered, from the stream-ordered allocator).
constexpr size_t kGreenCacheBytes = (size_t)4 << 30;

struct FftPlanCache {
  std::map<std::pair<int, int>, void*> twiddles;            // (n, bytes per real) -> device table
  size_t twiddle_bytes = 0;
  struct Green {
    int m0, m1, m2;   // padded shape
    int rbytes;
    void* gh;
    size_t bytes;
    uint64_t used;   // last use (cache clock)
  };
  std::vector<Green> greens;
  size_t green_bytes = 0;
  uint64_t clock = 0;
};

size_t qm_fft_cache_bytes(const FftPlanCache* c) { return c ? c->twiddle_bytes + c->green_bytes : 0; }

void qm_fft_cache_free(FftPlanCache* c) {
  if (!c) return;
  for (auto& kv : c->twiddles) (void)hipFree(kv.second);
  for (auto& g : c->greens) (void)hipFreeAsync(g.gh, nullptr);
  (void)hipStreamSynchronize(nullptr);
  delete c;
}

namespace {

template <typename R>
int twiddle_table(qm_ctx* ctx, int n, const Cx<R>** out) {
  if (!ctx->fft) ctx->fft = new FftPlanCache();
  auto key = std::make_pair(n, (int)sizeof(R));
  auto it = ctx->fft->twiddles.find(key);
  if (it != ctx->fft->twiddles.end()) {
    *out = (const Cx<R>*)it->second;
    return QM_OK;
  }
  std::vector<Cx<R>> h(n);
  for (int m = 0; m < n; ++m) {
    // exp(-2 pi i m / n) with the angle reduced exactly in integers
    const long double ang = -2.0L * 3.141592653589793238462643383279502884L * (long double)m / (long double)n;
    h[m] = Cx<R>{(R)std::cos(ang), (R)std::sin(ang)};
  }
  void* d = nullptr;
  QM_CHECK_HIP(ctx, hipMalloc(&d, sizeof(Cx<R>) * n));
  QM_CHECK_HIP(ctx, hipMemcpy(d, h.data(), sizeof(Cx<R>) * n, hipMemcpyHostToDevice));
  ctx->fft->twiddles[key] = d;
  ctx->fft->twiddle_bytes += sizeof(Cx<R>) * n;
  *out = (const Cx<R>*)d;
  return QM_OK;
}

// Free-space padding: the smallest length >= 2n with no prime factor above 7.  A cyclic length of
// at least 2n - 1 holds the linear convolution of two n-point signals exactly, and such a length
// keeps every pass on the in-place radices (2n = 304 = 16 x 19 would take the generic stage; 315 = 3^2 5 7).
int freespace_len(int n) {
  for (int v = 2 * n;; ++v) {
    int x = v;
    for (int r : {2, 3, 5, 7})
      while (x % r == 0) x /= r;
    if (x == 1) return v;
  }
}

AxisPlan make_plan(int n, const std::vector<int>& f) {
  AxisPlan plan{};
  plan.n = n;
  plan.nstage = (int)f.size();
  plan.ndiv = FastDiv::of(n);
  int span = 1;
  for (size_t q = 0; q < f.size(); ++q) {
    plan.radix[q] = f[q];
    plan.span[q] = span;
    plan.mdiv[q] = FastDiv::of(n / f[q]);
    plan.pdiv[q] = FastDiv::of(span);
    span *= f[q];
  }
  return plan;
}

// One pass along `axis` (length n) of a C-order [..][m1][row] complex buffer, on the lines whose other
// two indices are below (lim_a, lim_b) (in increasing axis order); positions >= nin are read as zero and
// positions >= nout are not written.  FROM_REAL / TO_REAL (axis 2): rin / rout is a real
// [lim_a][lim_b][nin / nout] array, the complex lines hold n / 2 + 1 values.
template <typename R, typename TO, int KIND>
int fft_pass(qm_ctx* ctx, hipStream_t s, Cx<R>* data, const R* rin, TO* rout, int n, int m1, int row, int axis,
             int lim_a, int lim_b, int nin, int nout, const FactorView<R>& fv = FactorView<R>{}) {
  constexpr bool REAL = KIND == FROM_REAL || KIND == TO_REAL;
  const Cx<R>* tw = nullptr;
  int rc = twiddle_table<R>(ctx, n, &tw);
  if (rc) return rc;
  const std::vector<int> f = factorize(n);
  QM_REQUIRE(ctx, (int)f.size() <= kMaxStages, QM_ELIMIT, "fft: too many stages for length %d", n);
  const AxisPlan plan = make_plan(n, f);
  const AxisPlan back = make_plan(n, std::vector<int>(f.rbegin(), f.rend()));
  const int64_t st[3] = {(int64_t)m1 * row, (int64_t)row, 1};
  AxisLines ln{};
  ln.stride = st[axis];
  const int oa = axis == 0 ? 1 : 0, ob = axis == 2 ? 1 : 2;   // other axes, oa < ob
  ln.nl0 = lim_a;
  ln.nl1 = REAL ? (lim_b + 1) / 2 : lim_b;
  ln.s0 = st[oa];
  ln.s1 = st[ob];
  ln.nin = nin;
  ln.nout = nout;
  ln.nr1 = lim_b;
  ln.nr2 = KIND == TO_REAL ? nout : nin;
  ln.hdiv = FastDiv::of(n / 2 + 1);
  QM_REQUIRE(ctx, nin >= 1 && nin <= n && nout >= 1 && nout <= n && (axis == 2 || !REAL), QM_EINVAL, "fft: bad pass");
  bool radix = f.size() >= 2;
  for (int r : f) radix = radix && r <= 10;
  const int planes = radix ? 1 : 2;
  const bool pow2 = radix && (n & (n - 1)) == 0;
  // B lines of n points per workgroup: B * n <= kMax (the register bound of a stage), whole cache lines
  // of adjacent lines where that allows it
  const int kMaxPts = pow2 ? FftPts<R, true>::kMax : FftPts<R, false>::kMax;
  // complex128: LDS would hold slightly longer lines than these, which callers have been refused
  const bool smooth = std::all_of(f.begin(), f.end(), [](int r) { return r <= 10; });
  const int limit = sizeof(R) == 4 ? 4096 : smooth ? 3855 : 2560;
  QM_REQUIRE(ctx, n <= limit, QM_ELIMIT, "fft: length %d exceeds %d", n, limit);
  int B = std::max(1, std::min(16, kMaxPts / n));
  if (!radix) B = std::max(1, std::min(B, 2048 / n));
  if (axis != 2 && B > 8) B = B / 8 * 8;
  B = std::max(1, std::min(B, ln.nl1));
  if (pow2)
    while (B & (B - 1)) B &= B - 1;   // the power-of-two kernel splits indices by shifts
  ln.B = B;
  ln.bdiv = FastDiv::of(B);
  const int lines_per_row = (ln.nl1 + B - 1) / B;
  const int64_t nwg = (int64_t)ln.nl0 * lines_per_row;
  const size_t shmem = sizeof(Cx<R>) * ((size_t)table_slots(n) + (size_t)planes * B * line_slots(n));
  QM_REQUIRE(ctx, shmem <= (size_t)128 * 1024, QM_ELIMIT, "fft: length %d needs %zu bytes of LDS per workgroup", n,
             shmem);
  QM_REQUIRE(ctx, nwg <= 0x7fffffff, QM_ELIMIT, "fft: too many lines");
  if (nwg == 0) return QM_OK;
  static bool attr_set = false;
  if (!attr_set) {
    const void* fns[3] = {(const void*)k_fft_axis<R, TO, KIND, POW2>, (const void*)k_fft_axis<R, TO, KIND, RADIX>,
                          (const void*)k_fft_axis<R, TO, KIND, GENERIC>};
    for (const void* f : fns)
      QM_CHECK_HIP(ctx, hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024));
    attr_set = true;
  }
  ProfScope ps(ctx, s, QM_K_FFT_AXIS);
  const dim3 grid((unsigned)nwg), thr(kFftThreads);
  if (pow2)
    hipLaunchKernelGGL((k_fft_axis<R, TO, KIND, POW2>), grid, thr, shmem, s, data, rin, rout, tw, plan, back, ln, fv);
  else if (radix)
    hipLaunchKernelGGL((k_fft_axis<R, TO, KIND, RADIX>), grid, thr, shmem, s, data, rin, rout, tw, plan, back, ln, fv);
  else
    hipLaunchKernelGGL((k_fft_axis<R, TO, KIND, GENERIC>), grid, thr, shmem, s, data, rin, rout, tw, plan, back, ln,
                       fv);
  QM_CHECK_LAUNCH(ctx);
  return QM_OK;
}

template <typename R>
int green_hat(qm_ctx* ctx, hipStream_t s, const int m[3], const R** out) {
  if (!ctx->fft) ctx->fft = new FftPlanCache();
  FftPlanCache& fc = *ctx->fft;
  for (auto& gr : fc.greens)
    if (gr.m0 == m[0] && gr.m1 == m[1] && gr.m2 == m[2] && gr.rbytes == (int)sizeof(R)) {
      gr.used = ++fc.clock;
      *out = (const R*)gr.gh;
      return QM_OK;
    }
  const int64_t M = (int64_t)m[0] * m[1] * m[2];
  Cx<R>* work = nullptr;
  int rc = qm_ws(ctx, s, WS_FFT_A, sizeof(Cx<R>) * (size_t)M, (void**)&work);
  if (rc) return rc;
  hipLaunchKernelGGL(k_green<R>, dim3((unsigned)((M + 255) / 256)), dim3(256), 0, s, work, m[0], m[1], m[2]);
  QM_CHECK_LAUNCH(ctx);
  R* const none = nullptr;
  if ((rc = fft_pass<R, R, FORWARD>(ctx, s, work, none, none, m[2], m[1], m[2], 2, m[0], m[1], m[2], m[2]))) return rc;
  if ((rc = fft_pass<R, R, FORWARD>(ctx, s, work, none, none, m[1], m[1], m[2], 1, m[0], m[2], m[1], m[1]))) return rc;
  if ((rc = fft_pass<R, R, FORWARD>(ctx, s, work, none, none, m[0], m[1], m[2], 0, m[1], m[2], m[0], m[0]))) return rc;
  const int o[3] = {m[0] / 2 + 1, m[1] / 2 + 1, m[2] / 2 + 1};
  const int64_t O = (int64_t)o[0] * o[1] * o[2];
  // make room: release the least recently used transforms (work queued earlier on s still reads them)
  const size_t bytes = sizeof(R) * (size_t)O;
  while (!fc.greens.empty() && fc.green_bytes + bytes > kGreenCacheBytes) {
    size_t lru = 0;
    for (size_t i = 1; i < fc.greens.size(); ++i)
      if (fc.greens[i].used < fc.greens[lru].used) lru = i;
    QM_CHECK_HIP(ctx, hipFreeAsync(fc.greens[lru].gh, s));
    fc.green_bytes -= fc.greens[lru].bytes;
    fc.greens.erase(fc.greens.begin() + lru);
  }
  void* gh = nullptr;
  QM_CHECK_HIP(ctx, hipMallocAsync(&gh, bytes, s));
  // V = -(h^3 / 4 pi) IFFT(rhs^ g^) / M   (rhs = -rho/eps0, g = 1/r); the step enters as h^2 at use
  const double scale = -1.0 / (4.0 * M_PI) / (double)M;
  hipLaunchKernelGGL(k_green_store<R>, dim3((unsigned)((O + 255) / 256)), dim3(256), 0, s, (const Cx<R>*)work,
                     (R*)gh, m[1], m[2], o[0], o[1], o[2], scale);
  QM_CHECK_LAUNCH(ctx);
  fc.greens.push_back({m[0], m[1], m[2], (int)sizeof(R), gh, bytes, ++fc.clock});
  fc.green_bytes += bytes;
  *out = (const R*)gh;
  return QM_OK;
}

template <typename R, typename TIO>
int hartree_fft(qm_ctx* ctx, qm_mol* mol, hipStream_t s, const qm_geom* g, const TIO* q, double sigma,
                double cutoff, int mode, TIO* out) {
  const bool fs = mode == QM_FFT_FREESPACE;
  const int n[3] = {g->nx, g->ny, g->nz};
  const int m[3] = {fs ? freespace_len(n[0]) : n[0], fs ? freespace_len(n[1]) : n[1],
                    fs ? freespace_len(n[2]) : n[2]};
  int rc;
  FactorView<R> fv{};
  fv.m0 = m[0];
  fv.m1 = m[1];
  fv.m2 = m[2];
  fv.step = g->step / kAng2Bor;
  if (fs) {
    if ((rc = green_hat<R>(ctx, s, m, &fv.g))) return rc;
    fv.o1 = m[1] / 2 + 1;
    fv.o2 = m[2] / 2 + 1;
    fv.scale = (R)(fv.step * fv.step);
  } else {
    fv.norm = 1.0 / (double)((int64_t)m[0] * m[1] * m[2]);
  }
  // half spectrum [n0][m1][hs] and the real right-hand side [n0][n1][n2]
  const int h2 = m[2] / 2 + 1, al = (int)(128 / sizeof(Cx<R>));
  const int hs = h2 >= 4 * al ? (h2 + al - 1) / al * al : h2;
  const size_t W = (size_t)n[0] * m[1] * hs, N = (size_t)n[0] * n[1] * n[2];
  Cx<R>* work = nullptr;
  if ((rc = qm_ws(ctx, s, WS_FFT_A, sizeof(Cx<R>) * W + sizeof(R) * N, (void**)&work))) return rc;
  R* rhs = (R*)(work + W);
  R* const none = nullptr;
  const GeomView gview = geom_view(g);
  const double cut2 = (cutoff * sigma) * (cutoff * sigma);
  hipLaunchKernelGGL((k_rhs<R, TIO>), dim3((n[0] + 31) / 32, n[1], (n[2] + 31) / 32), dim3(kThreads), 0, s, q,
                     (const double4*)mol->atoms, mol->natoms, gview, sigma, cut2, rhs);
  QM_CHECK_LAUNCH(ctx);
  if ((rc = fft_pass<R, R, FROM_REAL>(ctx, s, work, rhs, none, m[2], m[1], hs, 2, n[0], n[1], n[2], h2))) return rc;
  if ((rc = fft_pass<R, R, FORWARD>(ctx, s, work, none, none, m[1], m[1], hs, 1, n[0], h2, n[1], m[1]))) return rc;
  if (fs)
    rc = fft_pass<R, R, TURN_FREE>(ctx, s, work, none, none, m[0], m[1], hs, 0, m[1], h2, n[0], n[0], fv);
  else
    rc = fft_pass<R, R, TURN_PERIODIC>(ctx, s, work, none, none, m[0], m[1], hs, 0, m[1], h2, n[0], n[0], fv);
  if (rc) return rc;
  if ((rc = fft_pass<R, R, INVERSE>(ctx, s, work, none, none, m[1], m[1], hs, 1, n[0], h2, m[1], n[1]))) return rc;
  return fft_pass<R, TIO, TO_REAL>(ctx, s, work, none, out, m[2], m[1], hs, 2, n[0], n[1], h2, n[2]);
}

}  // namespace

extern "C" int qm_hartree_fft(qm_ctx* ctx, qm_mol* mol, void* stream, const qm_geom* g, int precision, int dtype,
                              const void* q, double sigma, double cutoff, int mode, void* out) {
  int rc = qm_enter(ctx);
  if (rc) return rc;
  if ((rc = qm_check_geom(ctx, g))) return rc;
  QM_REQUIRE(ctx, mol && q && out, QM_EINVAL, "fft: null argument");
  QM_REQUIRE(ctx, std::isfinite(sigma) && sigma > 0 && std::isfinite(cutoff) && cutoff > 0, QM_EINVAL,
             "fft: sigma and cutoff must be positive");
  QM_REQUIRE(ctx, mode == QM_FFT_PERIODIC || mode == QM_FFT_FREESPACE, QM_EINVAL, "fft: bad mode");
  QM_REQUIRE(ctx, g->nx >= 2 && g->ny >= 2 && g->nz >= 2, QM_EINVAL, "fft: grid too small");
  hipStream_t s = (hipStream_t)stream;
  if (precision == QM_PREC_FP64) {
    if (dtype == QM_F64)
      return hartree_fft<double, double>(ctx, mol, s, g, (const double*)q, sigma, cutoff, mode, (double*)out);
    if (dtype == QM_F32)
      return hartree_fft<double, float>(ctx, mol, s, g, (const float*)q, sigma, cutoff, mode, (float*)out);
  } else if (precision == QM_PREC_FP32) {
    if (dtype == QM_F64)
      return hartree_fft<float, double>(ctx, mol, s, g, (const double*)q, sigma, cutoff, mode, (double*)out);
    if (dtype == QM_F32)
      return hartree_fft<float, float>(ctx, mol, s, g, (const float*)q, sigma, cutoff, mode, (float*)out);
  } else {
    return qm_fail(ctx, QM_EINVAL, "fft: bad precision %d", precision);
  }
  return qm_fail(ctx, QM_EINVAL, "fft: bad dtype");
}
