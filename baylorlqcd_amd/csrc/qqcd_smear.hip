// qqcd_smear.hip -- Gaussian smearing of a quark field.
//
// smear (qqcd-test/cfgsprops/quark/diracops.f90:712-856), equation (23) of
// Trottier, Phys. Rev. D55, 6844 (1997): nsmear times
//   h(x) <- b h(x) + a sum_{mu=1..3} [U_mu(x) h(x+mu) + U_mu(x-mu)^dag h(x-mu)],
// b = 1 - 6a, on both checkerboards from the previous iterate of both (the
// increments of the even and the odd sites are formed before either is
// updated), spin-diagonal, the fermion boundary condition bc(mu) on a hop
// across the spatial edge.  The increment of a direction is summed as the
// reference sums it: (acc + forward) + backward, mu = 1, 2, 3.
//
// FP64 throughout.  Per site and iteration: the spinor at x and at its 6
// spatial neighbours (7 x 192 B), 6 links (6 x 144 B) and the result (192 B):
// 2400 B, 816 B of them (a link and both spinors once) from memory.  Bound by
// latency where there are few sites and by the caches otherwise, so both
// checkerboards run in one launch, 64 sites of each in turn: a link read as
// the forward one of a site is the backward one of the other checkerboard's
// neighbour, on the same XCD and soon after.  An iteration on 16^3x32 takes 24
// us (50 with a launch per checkerboard and all spins of a site in one lane),
// 24^3x48 136 (184), 8^3x16 4.8 (18.4).
#include <stdexcept>

#include "qqcd_context.h"

namespace qqcd {

struct SmArgs {
  int n[4];
  int bc[3];
  long Vh, stride, ustride;
  double a, b;
};

__device__ __forceinline__ double2 sm_ld(const double2 *p, long stride, int k, long i) { return p[k * stride + i]; }

// w[d] = s * M v[d] (M row-major 3x3 in m), or M^dag v[d]
template <bool DAG, int SP>
__device__ __forceinline__ void sm_mv(const double2 (&m)[9], const double2 (&v)[SP][3], double s, double2 (&acc)[SP][3]) {
#pragma unroll
  for (int d = 0; d < SP; d++)
#pragma unroll
    for (int r = 0; r < 3; r++) {
      double re = 0, im = 0;
#pragma unroll
      for (int c = 0; c < 3; c++) {
        const double2 e = DAG ? make_double2(m[3 * c + r].x, -m[3 * c + r].y) : m[3 * r + c];
        re += e.x * v[d][c].x - e.y * v[d][c].y;
        im += e.x * v[d][c].y + e.y * v[d][c].x;
      }
      acc[d][r] = make_double2(acc[d][r].x + s * re, acc[d][r].y + s * im);
    }
}

struct SmField {
  const double2 *h[2];
  double2 *out[2];
};

template <int SP>
__global__ void __launch_bounds__(64 * 4 / SP) k_smear(SmArgs a, const double2 *U, SmField f) {
  const int nb = gridDim.x, per = (nb + 7) / 8;
  const int xcd = blockIdx.x & 7, kb = blockIdx.x >> 3;
  const int full = nb - 8 * (per - 1);  // XCDs that get `per` workgroups
  const int blk = xcd < full ? xcd * per + kb : full * per + (xcd - full) * (per - 1) + kb;
  const int par = blk & 1, opar = par ^ 1;
  const long i = (long)(blk >> 1) * 64 + (threadIdx.x & 63);
  const int s0 = SP * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (i >= a.Vh) return;
  const int *n = a.n;
  int x[4];
  {
    const unsigned r = 2u * (unsigned)i;
    const unsigned x0 = r % n[0];
    unsigned q = r / n[0];
    x[1] = q % n[1];
    q /= n[1];
    x[2] = q % n[2];
    x[3] = q / n[2];
    x[0] = x0 + ((par + x[1] + x[2] + x[3]) & 1);
  }
  const double2 *other = f.h[opar] + (long)(3 * s0) * a.stride;
  double2 acc[SP][3];
#pragma unroll
  for (int d = 0; d < SP; d++)
#pragma unroll
    for (int c = 0; c < 3; c++) acc[d][c] = make_double2(0.0, 0.0);
#pragma unroll
  for (int mu = 0; mu < 3; mu++) {
    int xf[4] = {x[0], x[1], x[2], x[3]}, xb[4] = {x[0], x[1], x[2], x[3]};
    const bool wf = x[mu] + 1 == n[mu], wb = x[mu] == 0;
    xf[mu] = wf ? 0 : x[mu] + 1;
    xb[mu] = wb ? n[mu] - 1 : x[mu] - 1;
    const long jf = (xf[0] + (long)n[0] * (xf[1] + (long)n[1] * (xf[2] + (long)n[2] * xf[3]))) >> 1;
    const long jb = (xb[0] + (long)n[0] * (xb[1] + (long)n[1] * (xb[2] + (long)n[2] * xb[3]))) >> 1;
    const double sf = wf ? (double)a.bc[mu] : 1.0, sb = wb ? (double)a.bc[mu] : 1.0;
    const double2 *uf = U + (long)((par * 4 + mu) * 9) * a.ustride + i;
    const double2 *ub = U + (long)((opar * 4 + mu) * 9) * a.ustride + jb;
    double2 m[9], mb[9], v[SP][3], vb[SP][3];
#pragma unroll
    for (int k = 0; k < 9; k++) m[k] = uf[(long)k * a.ustride];
#pragma unroll
    for (int d = 0; d < SP; d++)
#pragma unroll
      for (int c = 0; c < 3; c++) v[d][c] = sm_ld(other, a.stride, 3 * d + c, jf);
#pragma unroll
    for (int k = 0; k < 9; k++) mb[k] = ub[(long)k * a.ustride];
#pragma unroll
    for (int d = 0; d < SP; d++)
#pragma unroll
      for (int c = 0; c < 3; c++) vb[d][c] = sm_ld(other, a.stride, 3 * d + c, jb);
    sm_mv<false, SP>(m, v, sf, acc);
    sm_mv<true, SP>(mb, vb, sb, acc);
  }
  const double2 *same = f.h[par] + (long)(3 * s0) * a.stride;
  double2 *out = f.out[par] + (long)(3 * s0) * a.stride;
#pragma unroll
  for (int d = 0; d < SP; d++)
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const double2 h = sm_ld(same, a.stride, 3 * d + c, i);
      out[(3 * d + c) * a.stride + i] = make_double2(a.b * h.x + a.a * acc[d][c].x, a.b * h.y + a.a * acc[d][c].y);
    }
}

// nsmear iterations on h[0], h[1] (FP64, both checkerboards) in place; t[0], t[1] scratch
void smear(Context &c, Spinor h[2], Spinor t[2], double asmear, int nsmear) {
  const Geom &g = c.g;
  if (nsmear < 0) throw std::runtime_error("smear: nsmear >= 0 expected");
  for (int p = 0; p < 2; p++)
    if (h[p].prec != PREC_DOUBLE || t[p].prec != PREC_DOUBLE) throw std::runtime_error("smear: FP64 fields expected");
  SmArgs a{};
  for (int m = 0; m < 4; m++) a.n[m] = g.n[m];
  for (int m = 0; m < 3; m++) a.bc[m] = g.bc[m];
  a.Vh = g.Vh;
  a.stride = h[0].stride;
  a.ustride = c.U64.stride;
  a.a = asmear;
  a.b = 1.0 - 6.0 * asmear;
  const int nb = 2 * (int)((g.Vh + 63) / 64);
  Spinor *cur = h, *nxt = t;
  // one spin a lane fills the chip where there are few sites (a site's links then come from the L1 for three of its
  // four lanes); all four where the links no longer stay in the last-level cache and each is to be read once.
  // us an iteration, one | four: 8^3x16 4.8 | 7.2, 16^3x32 24.1 | 31.1, 16^3x48 34.8 | 37.8, 20^3x32 46.0 | 44.6,
  // 20^3x40 65.2 | 56.4, 24^3x48 178 | 136
  const bool wide = g.Vh > 110000;
  for (int it = 0; it < nsmear; it++) {
    SmField f;
    for (int p = 0; p < 2; p++) {
      f.h[p] = (const double2 *)cur[p].data;
      f.out[p] = (double2 *)nxt[p].data;
    }
    if (wide) hipLaunchKernelGGL(k_smear<4>, dim3(nb), dim3(64), 0, c.stream, a, (const double2 *)c.U64.data, f);
    else hipLaunchKernelGGL(k_smear<1>, dim3(nb), dim3(256), 0, c.stream, a, (const double2 *)c.U64.data, f);
    QQCD_HIP(hipGetLastError());
    std::swap(cur, nxt);
  }
  if (cur != h)
    for (int p = 0; p < 2; p++)
      QQCD_HIP(hipMemcpyAsync(h[p].data, cur[p].data, h[p].bytes(), hipMemcpyDeviceToDevice, c.stream));
}

// kernel time (ms) of one smearing iteration (both checkerboards) on the
// resident links, averaged over niter iterations after nwarm
double bench_smear(Context &c, int nwarm, int niter) {
  Spinor h[2], t[2];
  for (int p = 0; p < 2; p++) {
    h[p] = alloc_spinor(c.g, PREC_DOUBLE);
    t[p] = alloc_spinor(c.g, PREC_DOUBLE);
    QQCD_HIP(hipMemsetAsync(h[p].data, 0, h[p].bytes(), c.stream));
  }
  hipEvent_t e0, e1;
  QQCD_HIP(hipEventCreate(&e0));
  QQCD_HIP(hipEventCreate(&e1));
  smear(c, h, t, 0.25, 2 * nwarm);
  QQCD_HIP(hipEventRecord(e0, c.stream));
  smear(c, h, t, 0.25, 2 * niter);  // an even count: no copy back
  QQCD_HIP(hipEventRecord(e1, c.stream));
  QQCD_HIP(hipEventSynchronize(e1));
  float ms = 0;
  QQCD_HIP(hipEventElapsedTime(&ms, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  for (int p = 0; p < 2; p++) {
    free_spinor(h[p]);
    free_spinor(t[p]);
  }
  return ms / (2.0 * niter);
}

}  // namespace qqcd
