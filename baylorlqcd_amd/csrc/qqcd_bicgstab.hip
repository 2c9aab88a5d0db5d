// qqcd_bicgstab.hip -- see qqcd_bicgstab.h.
//
// Bound on small lattices by launches and by the dependences between them, on
// large ones by the passes over memory.  An iteration takes five passes beside
// the two operator applications (nine with one operation each): p; <rhat, v>;
// r -= alpha v; <t, r> and <t, t>; x, r, ||r||^2 and the next <rhat, r>.  The
// last workgroup of a reduction sums the others' partials in a fixed order and
// forms the scalars, so no launch and no host round trip lies between a sum
// and its use.  8^3x16: 140 us an iteration with one operation a launch and
// four host round trips.
#include "qqcd_bicgstab.h"

#include <algorithm>
#include <cmath>
#include <stdexcept>

#include "qqcd_pool.h"

namespace qqcd {

static constexpr int TB = 256;
static constexpr int GMAX = 1024;

struct BState {
  double rho[2], alpha[2], omega[2], beta[2];  // beta and alpha of the coming / running iteration
  double goal;
  int it, itermin, maxiter, done;
  unsigned arrived[4];  // workgroups of each reduction that have left their partials
};

// a / b with b brought to order one by a power of two first: |b|^2 for rho (a
// squared norm) would leave the range of FP64 at sources of 1e-75 or 1e+80
__device__ __forceinline__ double2 cdiv(double2 a, double2 b) {
  const int e = -__builtin_amdgcn_frexp_exp(fmax(fabs(b.x), fabs(b.y)));
  b = make_double2(ldexp(b.x, e), ldexp(b.y, e));
  const double d = 1.0 / (b.x * b.x + b.y * b.y);
  return make_double2(ldexp((a.x * b.x + a.y * b.y) * d, e), ldexp((a.y * b.x - a.x * b.y) * d, e));
}
__device__ __forceinline__ double2 cmulz(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// The workgroup's totals of v[NV] into its row of part; true in the workgroup
// that arrives last, whose thread 0 then has the totals over all rows (summed
// in a fixed order) in v.  The rows are written and read past the L2s of the
// XCDs (agent scope).
template <int NV>
__device__ __forceinline__ bool sum_all(double (&v)[NV], double *part, unsigned *arrived) {
  __shared__ double sm[TB / 64][NV];
  __shared__ bool last;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  auto block = [&]() {
#pragma unroll
    for (int k = 0; k < NV; k++) {
      double s = v[k];
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
      if (lane == 0) sm[w][k] = s;
    }
    __syncthreads();
  };
  block();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < NV; k++) {
      double s = 0;
#pragma unroll
      for (int q = 0; q < TB / 64; q++) s += sm[q][k];
      __hip_atomic_store(part + (long)blockIdx.x * NV + k, s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    last = __hip_atomic_fetch_add(arrived, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
  }
  __syncthreads();
  if (!last) return false;
#pragma unroll
  for (int k = 0; k < NV; k++) v[k] = 0;
  for (unsigned b = threadIdx.x; b < gridDim.x; b += TB)
#pragma unroll
    for (int k = 0; k < NV; k++)
      v[k] += __hip_atomic_load(part + (long)b * NV + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  block();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < NV; k++) {
      v[k] = 0;
#pragma unroll
      for (int q = 0; q < TB / 64; q++) v[k] += sm[q][k];
    }
    *arrived = 0;  // for the next launch of this reduction
  }
  return true;
}

__global__ void __launch_bounds__(TB) k_bi_reset(long n, const double2 *r, double2 *rhat, double2 *p, double2 *v) {
#pragma unroll 4
  for (long i = blockIdx.x * (long)TB + threadIdx.x; i < n; i += (long)gridDim.x * TB) {
    rhat[i] = r[i];
    p[i] = v[i] = make_double2(0, 0);
  }
}

__global__ void k_bi_state(BState *s, BState a) {
  if (threadIdx.x == 0) *s = a;
}

// p = r + beta (p - omega v)
__global__ void __launch_bounds__(TB) k_bi_p(long n, const BState *s, const double2 *r, const double2 *v, double2 *p) {
  if (s->done) return;
  const double2 beta = make_double2(s->beta[0], s->beta[1]), om = make_double2(s->omega[0], s->omega[1]);
#pragma unroll 4
  for (long i = blockIdx.x * (long)TB + threadIdx.x; i < n; i += (long)gridDim.x * TB) {
    const double2 a = p[i], b = cmulz(om, v[i]), c = cmulz(beta, make_double2(a.x - b.x, a.y - b.y)), d = r[i];
    p[i] = make_double2(d.x + c.x, d.y + c.y);
  }
}

// alpha = rho / <rhat, v>
__global__ void __launch_bounds__(TB) k_bi_alpha(long n, BState *s, const double2 *rhat, const double2 *v, double *part) {
  if (s->done) return;
  double a[2] = {0, 0};
#pragma unroll 4
  for (long i = blockIdx.x * (long)TB + threadIdx.x; i < n; i += (long)gridDim.x * TB) {
    const double2 x = rhat[i], y = v[i];
    a[0] += x.x * y.x + x.y * y.y;
    a[1] += x.x * y.y - x.y * y.x;
  }
  if (sum_all<2>(a, part, &s->arrived[0]) && threadIdx.x == 0) {
    const double2 q = cdiv(make_double2(s->rho[0], s->rho[1]), make_double2(a[0], a[1]));
    s->alpha[0] = q.x;
    s->alpha[1] = q.y;
  }
}

// r -= alpha v
__global__ void __launch_bounds__(TB) k_bi_r(long n, const BState *s, const double2 *v, double2 *r) {
  if (s->done) return;
  const double2 al = make_double2(s->alpha[0], s->alpha[1]);
#pragma unroll 4
  for (long i = blockIdx.x * (long)TB + threadIdx.x; i < n; i += (long)gridDim.x * TB) {
    const double2 x = cmulz(al, v[i]), y = r[i];
    r[i] = make_double2(y.x - x.x, y.y - x.y);
  }
}

// omega = <t, r> / <t, t>
__global__ void __launch_bounds__(TB) k_bi_omega(long n, BState *s, const double2 *t, const double2 *r, double *part) {
  if (s->done) return;
  double a[3] = {0, 0, 0};
#pragma unroll 4
  for (long i = blockIdx.x * (long)TB + threadIdx.x; i < n; i += (long)gridDim.x * TB) {
    const double2 x = t[i], y = r[i];
    a[0] += x.x * y.x + x.y * y.y;
    a[1] += x.x * y.y - x.y * y.x;
    a[2] += x.x * x.x + x.y * x.y;
  }
  if (sum_all<3>(a, part, &s->arrived[1]) && threadIdx.x == 0) {
    s->omega[0] = a[0] / a[2];
    s->omega[1] = a[1] / a[2];
  }
}

// x += omega r + alpha p, r -= omega t, ||r||, the next rho = <rhat, r> and beta
__global__ void __launch_bounds__(TB) k_bi_x(long n, BState *s, const double2 *rhat, const double2 *p, const double2 *t,
                                             double2 *r, double2 *x, double *part, double *hist) {
  if (s->done) return;
  const double2 om = make_double2(s->omega[0], s->omega[1]), al = make_double2(s->alpha[0], s->alpha[1]);
  double a[3] = {0, 0, 0};
#pragma unroll 4
  for (long i = blockIdx.x * (long)TB + threadIdx.x; i < n; i += (long)gridDim.x * TB) {
    const double2 q = r[i], u = cmulz(om, q), w = cmulz(al, p[i]), z = x[i], m = cmulz(om, t[i]), h = rhat[i];
    x[i] = make_double2(z.x + u.x + w.x, z.y + u.y + w.y);
    const double2 e = make_double2(q.x - m.x, q.y - m.y);
    r[i] = e;
    a[0] += e.x * e.x + e.y * e.y;
    a[1] += h.x * e.x + h.y * e.y;
    a[2] += h.x * e.y - h.y * e.x;
  }
  if (sum_all<3>(a, part, &s->arrived[2]) && threadIdx.x == 0) {
    const double rr = sqrt(a[0]);
    const double2 rho = make_double2(a[1], a[2]);
    const double2 b = cmulz(cdiv(rho, make_double2(s->rho[0], s->rho[1])), cdiv(al, om));
    s->beta[0] = b.x;
    s->beta[1] = b.y;
    s->rho[0] = rho.x;
    s->rho[1] = rho.y;
    hist[s->it % BiCGStabDev::AHEAD] = rr;
    s->it++;
    if ((rr < s->goal && s->it >= s->itermin) || s->it >= s->maxiter || !isfinite(rr)) s->done = 1;
    hist[BiCGStabDev::AHEAD] = s->it;
    hist[BiCGStabDev::AHEAD + 1] = s->done;
  }
}

// ===================================================================== //

BiCGStabDev::BiCGStabDev(hipStream_t s, long n_) : stream(s), n(n_) {
  if (n < 1) throw std::runtime_error("bicgstab: empty vectors");
  bufs.get(&part, sizeof(double) * 3 * GMAX);
  bufs.get(&state, sizeof(BState));
  bufs.get_host(&hist, sizeof(double) * (AHEAD + 2));
}

static void check(const Vec &v, long n) {
  if (v.prec != PREC_DOUBLE || v.n != n) throw std::runtime_error("bicgstab: FP64 vectors of one length");
}
// four elements a lane where the vector is short: every workgroup of a
// reduction adds to one counter
#define BGRID dim3((unsigned)std::min((n + 4 * TB - 1) / (4 * TB), (long)GMAX)), dim3(TB), 0, stream

void BiCGStabDev::reset(const Vec &r, Vec &rhat, Vec &p, Vec &v, double rn, double goal, int taken, int itermin,
                        int maxiter) {
  for (const Vec *q : {&r, (const Vec *)&rhat, (const Vec *)&p, (const Vec *)&v}) check(*q, n);
  BState a{};
  a.rho[0] = rn * rn;
  a.omega[0] = a.alpha[0] = 1.0;
  a.goal = goal;
  a.it = taken;
  a.itermin = itermin;
  a.maxiter = maxiter;
  a.done = (rn < goal && taken >= itermin) || taken >= maxiter || !std::isfinite(rn);
  hist[AHEAD] = taken;
  hist[AHEAD + 1] = a.done;
  hipLaunchKernelGGL(k_bi_state, dim3(1), dim3(64), 0, stream, (BState *)state, a);
  hipLaunchKernelGGL(k_bi_reset, BGRID, n, (const double2 *)r.data, (double2 *)rhat.data, (double2 *)p.data,
                     (double2 *)v.data);
  QQCD_HIP(hipGetLastError());
}

void BiCGStabDev::start(const Vec &r, const Vec &v, Vec &p) {
  hipLaunchKernelGGL(k_bi_p, BGRID, n, (const BState *)state, (const double2 *)r.data, (const double2 *)v.data,
                     (double2 *)p.data);
  QQCD_HIP(hipGetLastError());
}

void BiCGStabDev::middle(const Vec &rhat, const Vec &v, Vec &r) {
  hipLaunchKernelGGL(k_bi_alpha, BGRID, n, (BState *)state, (const double2 *)rhat.data, (const double2 *)v.data, part);
  hipLaunchKernelGGL(k_bi_r, BGRID, n, (const BState *)state, (const double2 *)v.data, (double2 *)r.data);
  QQCD_HIP(hipGetLastError());
}

void BiCGStabDev::finish(const Vec &rhat, const Vec &p, const Vec &t, Vec &r, Vec &x) {
  check(t, n);
  check(x, n);
  hipLaunchKernelGGL(k_bi_omega, BGRID, n, (BState *)state, (const double2 *)t.data, (const double2 *)r.data, part);
  hipLaunchKernelGGL(k_bi_x, BGRID, n, (BState *)state, (const double2 *)rhat.data, (const double2 *)p.data,
                     (const double2 *)t.data, (double2 *)r.data, (double2 *)x.data, part, hist);
  QQCD_HIP(hipGetLastError());
}

int BiCGStabDev::fetch(int from, double *rr, bool *ended) const {
  const int it = (int)hist[AHEAD];
  for (int k = from; k < it; k++) rr[k - from] = hist[k % AHEAD];
  *ended = hist[AHEAD + 1] != 0;
  return it - from;
}

}  // namespace qqcd
