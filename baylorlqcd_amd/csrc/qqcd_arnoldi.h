// qqcd_arnoldi.h -- Arnoldi steps in blocks of s over an FP64, FP32 or FP16 basis.
//
// With B = A - sigma (the operator without its identity part, the same Krylov
// space) and u_i = B^i v_j, i = 1..s, one pass over the basis forms the
// projections P = V^H [u_1..u_s] and the Gram matrix G = U^H U, and one more
// writes the s new basis vectors Q = (U - V P) R^-1 with R the Cholesky factor
// of G - P^H P: two reads of the basis for s steps.  The columns of the
// Hessenberg matrix follow from u_{i+1} = B u_i:
//   B q_i = (coef(u_{i+1}) - sum_{k<=j} P_ki H_k - sum_{l<i} R_li H_{j+l}) / R_ii,
// coef(u_i) = (P_i; R_i) in the basis (V, Q).
#pragma once
#include <complex>
#include <vector>

#include "qqcd_blas.h"
#include "qqcd_pool.h"

namespace qqcd {

class BlockArnoldi {
 public:
  static constexpr int SMAX = 4;
  static constexpr int NMAX = 128;  // vectors of a basis
  BlockArnoldi(hipStream_t s, int m);  // cycles of at most m steps
  BlockArnoldi(const BlockArnoldi &) = delete;
  BlockArnoldi &operator=(const BlockArnoldi &) = delete;

  // columns [0, n) of the Hessenberg matrix of A (rows 0..n) for the vectors
  // already in the basis; the device holds that of B = A - sigma
  void load(const std::complex<double> *h, int ldh, int n, double sigma);
  // column j of H (of A) on the device: rows 0..j+1
  void put(const std::complex<double> *h, int j, double sigma);
  // queue block `slot` (0..): V[j+1..j+s] hold B^i V[j] and become the next s
  // basis vectors.  No synchronisation.
  void queue(const Vec *V, int j, int s, int slot);
  // the same over an FP16 basis with per-site norms; the B^i V[j] are the FP32 U[0..s-1]
  void queue_half(const Vec *V, const Vec *U, int j, int s, int slot);
  // waits; the sums of the queue_half before: rows <V_q, u_c> of nv vectors, then <u_r, u_c>
  void half_sums(int nv, int s, std::complex<double> *out) const;
  // the first s of the same block's vectors orthogonalised once more, the
  // columns corrected
  void queue_again(const Vec *V, int j, int s, int slot);
  // after the stream has been waited for: columns j.. of H (of A) from block
  // `slot`; returns how many of the s steps are sound (a vector of whose squared
  // norm the span of the ones before it leaves less than 1e-6 -- FP32 basis:
  // 1e-10 -- ends the block)
  int fetch(int slot, int j, int s, double sigma, std::complex<double> *H, int ldh) const;
  // ||V^H V - 1|| (Frobenius) of n FP64 vectors
  double loss_of(const Vec *V, int n);
  // ||P R^-1|| (Frobenius) and smallest R_ii^2 / G_ii of that block: what the
  // loss of orthogonality of V is multiplied by in Q, and the cancellation
  double growth(int slot) const;
  double pivot(int slot) const;

 private:
  void run(const Vec *V, int j, int s, int slot, bool again);
  hipStream_t stream;
  int m, ld;
  PoolSet bufs;
  double *hd = nullptr;    // H of B on the device: ld rows, m columns, complex
  double *part = nullptr;  // partial sums
  double *sums = nullptr;  // their totals: left vectors x s, complex
  double *pr = nullptr;    // P and R of the last block (for queue_again)
  double *coef = nullptr;  // update coefficients: C (NMAX x SMAX), D (SMAX x SMAX), complex
  float *coef32 = nullptr;  // the same in FP32
  double *hh = nullptr;    // pinned: slots of SMAX columns of ld, then 4 numbers
  long slot_len() const { return 2L * SMAX * ld + 4; }
};

}  // namespace qqcd
