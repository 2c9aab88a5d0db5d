// qqcd_bicgstab.h -- the vector passes of BiCGStab with their scalars on the device.
#pragma once
#include "qqcd_blas.h"
#include "qqcd_pool.h"

namespace qqcd {

// One iteration is start(); v = A p; middle(); t = A r; finish(): p, r, v, t
// and x are FP64 vectors of one length.  Nothing is read back: rho, alpha,
// omega and the end of the solve are decided on the device, and after the
// end the passes leave everything as it is, so iterations can be queued
// ahead of the host.
class BiCGStabDev {
 public:
  static constexpr int AHEAD = 32;  // iterations queued between two reads of the history at most
  BiCGStabDev(hipStream_t s, long n);
  BiCGStabDev(const BiCGStabDev &) = delete;
  BiCGStabDev &operator=(const BiCGStabDev &) = delete;

  // a fresh start from r = rhat, p = v = 0 (written by reset): ||r|| = rn,
  // `taken` iterations done; ends at ||r|| < goal with itermin iterations, at
  // maxiter iterations, or at a residual that is not finite
  void reset(const Vec &r, Vec &rhat, Vec &p, Vec &v, double rn, double goal, int taken, int itermin, int maxiter);
  void start(const Vec &r, const Vec &v, Vec &p);                         // p = r + beta (p - omega v)
  void middle(const Vec &rhat, const Vec &v, Vec &r);                     // alpha = rho / <rhat, v>, r -= alpha v
  void finish(const Vec &rhat, const Vec &p, const Vec &t, Vec &r, Vec &x);  // omega, x, r, ||r||, rho, beta
  // after the stream has been waited for: residual norms of the iterations
  // since `from` (at most AHEAD), and whether the solve has ended
  int fetch(int from, double *rr, bool *ended) const;

 private:
  hipStream_t stream;
  long n;
  PoolSet bufs;
  double *part = nullptr;
  void *state = nullptr;     // device scalars
  double *hist = nullptr;    // pinned: AHEAD residual norms, iterations done, ended
};

}  // namespace qqcd
