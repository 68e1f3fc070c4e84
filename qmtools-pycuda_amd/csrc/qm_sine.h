// Sine transforms of a grid's interior (sine.hip), used by the relaxations' closed forms.
#pragma once

#include <functional>

#include "qm_internal.h"

struct SinePlan {
  int nx, ny;               // grid row and plane sizes
  int m[3], ld[3];          // interior points per axis, row length of the tables
  const double* S[3];       // S_kn = sqrt(2 / (m + 1)) sin(pi k n / (m + 1)), n <= (m + 1) / 2: odd k,
  const double* So[3];      // even k (1-based), zero padded
  const double* s2[3];      // sin^2(pi k / (2 (m + 1))), k = 1 .. m
  double* part;             // partial sums of an x pass
  double* red;              // block partials of their reduction
  double* sum;              // their sum
  int* flag;                // set when a residual is not finite or near the end of the range
  unsigned long long* ctl;  // of qm_sine_sweeps_if: workgroups so far, arrivals at its barriers, workgroups that take part
};

enum { SINE_JACOBI = 0, SINE_VNE = 1 };     // which sweep's eigenvalue a
enum { SINE_SUM = 0, SINE_POWER = 1 };      // (1 - a^n) / (1 - a), a^n

struct SineFactor {
  int sweep, kind;
  double n;                 // whole number below 2^53
  int odd;                  // n is odd
  double w0, w1, w2, w3;    // SINE_VNE: 1 - a = w0 + w1 sum (1 - c) + w2 sum (1 - c c') + w3 (1 - c c' c''), c = cos theta
};

// A tolerance below 1e-12 of the field's size is decided by the rounding of the sweeps, about 1e-16 of it: total is
// sum |V| (per point where delta is), delta the change that the closed form found.
__host__ __device__ inline bool sine_undecided(double total, double tol, double delta) {
  const double floor = 1e-12 * total;
  return !(floor < INFINITY) || (tol < floor && delta < floor);
}

// Held by a closed form from before its plan to its last launch.  The sweeps work in the caller's buffers
// alone, so calls on several streams of one context may be in flight together; the closed forms share the
// context's tables and work grid, and are ordered one after the other by an event.  (Nothing else uses these
// workspaces: the reductions have their own partials, red, instead of WS_RED.)  A call that has waited for its
// stream leaves nothing in flight and says so with waited() instead of recording the event (V_ne of 120 x 120 x 64:
// 377 -> 365 us).
struct SineUse {
  qm_ctx* ctx;
  hipStream_t s;
  bool held = false;
  SineUse(qm_ctx* c, hipStream_t st) : ctx(c), s(st) {}
  int begin();
  void waited() {
    held = false;
    ctx->sine_pending = false;
  }
  ~SineUse() {
    if (!held) return;
    ctx->sine_pending = hipEventRecord(ctx->sine_done, s) == hipSuccess;
    if (!ctx->sine_pending) (void)hipStreamSynchronize(s);
  }
};

bool qm_sine_fits(const qm_geom* g);   // every axis has 1 .. 1024 interior points
// tables in the context's workspace, valid on s until the next plan; clears the flag and ctl
int qm_sine_plan(qm_ctx* ctx, hipStream_t s, const qm_geom* g, SinePlan* p);
// The passes read and write interior points only and work in place where one buffer is given.
// x and y transforms of (one Jacobi sweep of v) - v; sets the plan's flag if that is not finite, or 1e290 and more, somewhere
int qm_sine_residual_xy(qm_ctx* ctx, hipStream_t s, const SinePlan& p, const double* rho, const double* v, double h,
                        double* out);
int qm_sine_xy(qm_ctx* ctx, hipStream_t s, const SinePlan& p, double* a);
int qm_sine_z(qm_ctx* ctx, hipStream_t s, const SinePlan& p, double* a);
// z transform, factor, z and y transforms
int qm_sine_z_scale_zy(qm_ctx* ctx, hipStream_t s, const SinePlan& p, const SineFactor& f, double* a);
// factor times a spectrum, z and y transforms (the same bits as qm_sine_z and then this, or the call above)
int qm_sine_scale_zy(qm_ctx* ctx, hipStream_t s, const SinePlan& p, const SineFactor& f, const double* spectrum,
                     double* out);
int qm_sine_x(qm_ctx* ctx, hipStream_t s, const SinePlan& p, double* a);
int qm_sine_x_add(qm_ctx* ctx, hipStream_t s, const SinePlan& p, const double* a, double* v);   // v += x transform of a, unless the flag is set
// the same, unless sine_undecided(sum, tol, delta) with the sum of the last qm_sine_x_sum
int qm_sine_x_add_decided(qm_ctx* ctx, hipStream_t s, const SinePlan& p, const double* a, double* v, double tol,
                          double delta);
// `sweeps` Jacobi sweeps of v (tmp: work space) if the flag is set, else nothing
int qm_sine_sweeps_if(qm_ctx* ctx, hipStream_t s, const SinePlan& p, const qm_geom* g, const double* rho, double* v,
                      double* tmp, int64_t sweeps);
// sum over the interior of |x transform of a| (v null) or |v + x transform of a|, on the device; qm_sine_sum waits for s
// and returns it
int qm_sine_x_sum(qm_ctx* ctx, hipStream_t s, const SinePlan& p, const double* a, const double* v);
int qm_sine_sum(qm_ctx* ctx, hipStream_t s, const SinePlan& p, double* host_sum);
// First check 1 .. n whose delta is at most tol, given that delta does not grow and delta(n) = dn <= tol, by
// bisection in the logarithm of delta.
int qm_sine_first_below(int64_t n, double dn, double tol, const std::function<int(int64_t, double*)>& delta_at,
                        int64_t* at, double* delta);
// Sweep counts from which a closed form is taken.  It costs what 5 to 11 sweeps do (us, closed form and one sweep: 16^3 31
// and 7.0, 64^3 52 and 9.0, 128^3 114 and 12.3, 256^3 850 and 83; its 6 n flops a point grow with the axis, a sweep's
// 24 bytes do not).  The line lies well above that crossing: short counts keep the bits of the sweeps, so that calls
// of up to 32 sweeps, one after the other, add up to the bits of the loop.
inline int64_t qm_sine_sweeps(const qm_geom* g) {
  const int n = g->nx > g->ny ? g->nx : g->ny;
  return 32 + (n > g->nz ? n : g->nz) / 16;
}
