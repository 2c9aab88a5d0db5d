// qqcd_blockalg.h -- the small dense algebra of a block of Arnoldi steps, shared by
// the single- and the multi-right-hand-side kernels (qqcd_arnoldi.h has the
// recurrences).
#pragma once
#include <hip/hip_runtime.h>

namespace qqcd {

__device__ __forceinline__ double2 zmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 zsub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 zcmul(double2 a, double2 b) {  // conj(a) b
  return make_double2(a.x * b.x + a.y * b.y, a.x * b.y - a.y * b.x);
}

// a of the lanes whose bit is clear and b of those whose bit is set stay; the
// other halves change places: afterwards a + b is, in a lane, the sum of a (bit
// clear) or of b (bit set) over the lane and the one that differs in the bit.
template <int BIT> __device__ __forceinline__ void swap_halves(unsigned &a, unsigned &b, int lane) {
  if constexpr (BIT >= 16) {
    const auto r = BIT == 32 ? __builtin_amdgcn_permlane32_swap(a, b, false, false)
                             : __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
  } else {
    const bool hi = lane & BIT;
    const unsigned got = __shfl_xor(hi ? a : b, BIT, 64);
    a = hi ? got : a;
    b = hi ? b : got;
  }
}
template <int BIT> __device__ __forceinline__ void swap_halves(float &a, float &b, int lane) {
  unsigned x = __float_as_uint(a), y = __float_as_uint(b);
  swap_halves<BIT>(x, y, lane);
  a = __uint_as_float(x);
  b = __uint_as_float(y);
}
template <int BIT> __device__ __forceinline__ void swap_halves(double &a, double &b, int lane) {
  unsigned x0 = __double2loint(a), x1 = __double2hiint(a), y0 = __double2loint(b), y1 = __double2hiint(b);
  swap_halves<BIT>(x0, y0, lane);
  swap_halves<BIT>(x1, y1, lane);
  a = __hiloint2double(x1, x0);
  b = __hiloint2double(y1, y0);
}

// FP32 sums of a run of products, kept in FP64 across runs.  A wavefront's lanes
// hold N sums each; the H halvings below add them (in FP64) over the lanes that
// differ in their H highest bits and leave a lane with N >> H of them: those from
// `first` on.  About N lane swaps, and 2 (N >> H) registers between runs instead
// of 2 N.
template <int N, int H> struct Runs {
  static_assert(N % (1 << H) == 0, "halvings");
  static constexpr int M = N >> H;
  double tot[M];
  __device__ Runs() {
#pragma unroll
    for (int k = 0; k < M; k++) tot[k] = 0;
  }
  // adds af and clears it
  __device__ __forceinline__ void add(float (&af)[N], int lane) {
    if constexpr (H == 0) {
#pragma unroll
      for (int k = 0; k < N; k++) tot[k] += (double)af[k];
    } else {
      double d[N / 2];
#pragma unroll
      for (int k = 0; k < N / 2; k++) {
        swap_halves<32>(af[k], af[k + N / 2], lane);
        d[k] = (double)af[k] + (double)af[k + N / 2];
      }
      halve<1>(d, lane);
    }
#pragma unroll
    for (int k = 0; k < N; k++) af[k] = 0.f;
  }
  static __device__ __forceinline__ int first(int lane) {
    int f = 0;
#pragma unroll
    for (int h = 0; h < H; h++)
      if (lane & (32 >> h)) f += N >> (h + 1);
    return f;
  }

 private:
  template <int D, int C> __device__ __forceinline__ void halve(double (&d)[C], int lane) {
    if constexpr (D == H) {
#pragma unroll
      for (int k = 0; k < C; k++) tot[k] += d[k];
    } else {
      double e[C / 2];
#pragma unroll
      for (int k = 0; k < C / 2; k++) {
        swap_halves<(32 >> D)>(d[k], d[k + C / 2], lane);
        e[k] = d[k] + d[k + C / 2];
      }
      halve<D + 1>(e, lane);
    }
  }
};

// One workgroup of 256 threads per right-hand side, a basis of at most 128
// vectors (j + S < ld <= 128): from the sums P (rows 0..j) and G the factor R,
// the update coefficients C = -P R^-1 and D = R^-1, and the columns j..j+S-1 of
// H.  again: the vectors are the Q of this block, io.p1 / io.r1 the P and R of
// the first pass; the total projections are P + P2 R and the total factor R2 R.
// A vector is taken while more than `least` of its squared norm is left.  The
// column of the first that is not is written all the same: A times the last
// vector taken has all of it but that rest in the basis, whose norm is the
// column's last entry though no vector stands for it.  The columns after it are
// zero, and so are the new vectors from there on.
template <int S, typename IO>
__device__ __forceinline__ void block_columns(IO io, int j, int ld, int again, double least) {
  constexpr int NM = 128;
  __shared__ double2 P[NM][S], C[NM][S], G[S][S], R[S][S], D[S][S], Pt[NM][S], Rt[S][S], col[S][NM + S];
  __shared__ double red[2][S];
  __shared__ int good;
  __shared__ double worst;
  const int t = threadIdx.x, nv = j + 1;
  for (int i = t; i < nv * S; i += 256) P[i / S][i % S] = io.p(i / S, i % S);
  for (int i = t; i < S * S; i += 256) G[i / S][i % S] = io.g(i / S, i % S);
  __syncthreads();
  // G - P^H P, one entry per 16 threads
  for (int e0 = 0; e0 < S * S; e0 += 16) {
    const int e = e0 + (t >> 4), r = e / S, c = e % S;
    double2 a = make_double2(0, 0);
    if (e < S * S)
      for (int k = t & 15; k < nv; k += 16) {
        const double2 p = zcmul(P[k][r], P[k][c]);
        a.x += p.x;
        a.y += p.y;
      }
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) {
      a.x += __shfl_xor(a.x, o, 64);
      a.y += __shfl_xor(a.y, o, 64);
    }
    if (e < S * S && (t & 15) == 0) R[r][c] = zsub(G[r][c], a);
  }
  __syncthreads();
  if (t == 0) {
    // Cholesky R^H R of the upper triangle, in place; D = R^-1 (upper)
    double2 r[S][S], d[S][S];
    double least_seen = 1.0;
    int n = 0;
#pragma unroll
    for (int i = 0; i < S; i++)
#pragma unroll
      for (int k = 0; k < S; k++) {
        r[i][k] = k >= i ? R[i][k] : make_double2(0, 0);
        d[i][k] = make_double2(0, 0);
      }
    bool ok = true;
#pragma unroll
    for (int i = 0; i < S; i++) {
      double p = r[i][i].x;
#pragma unroll
      for (int l = 0; l < i; l++) p -= r[l][i].x * r[l][i].x + r[l][i].y * r[l][i].y;
      const double g = G[i][i].x;
      ok = ok && p > least * g && p > 0;
      const double h = ok ? sqrt(p) : 0.0, inv = ok ? 1.0 / h : 0.0;
      r[i][i] = make_double2(h, 0);
      if (ok) {
        least_seen = fmin(least_seen, p / g);
        n++;
      } else if (n == i && p > 0) {
        r[i][i].x = sqrt(p);  // of the first not taken: the last row of its column of H
      }
#pragma unroll
      for (int k = i + 1; k < S; k++) {
        double2 x = r[i][k];
#pragma unroll
        for (int l = 0; l < i; l++) x = zsub(x, zcmul(r[l][i], r[l][k]));
        r[i][k] = make_double2(x.x * inv, x.y * inv);
      }
      // column i of the inverse
      d[i][i] = make_double2(inv, 0);
#pragma unroll
      for (int l = i - 1; l >= 0; l--) {
        double2 x = make_double2(0, 0);
#pragma unroll
        for (int q = l + 1; q <= i; q++) {
          const double2 y = zmul(r[l][q], d[q][i]);
          x.x += y.x;
          x.y += y.y;
        }
        const double f = ok ? -d[l][l].x : 0.0;
        d[l][i] = make_double2(x.x * f, x.y * f);
      }
    }
#pragma unroll
    for (int i = 0; i < S; i++)
#pragma unroll
      for (int k = 0; k < S; k++) {
        R[i][k] = r[i][k];
        D[i][k] = d[i][k];
      }
    good = n;
    worst = least_seen;
  }
  __syncthreads();
  // C = -P D, row by row; with `again` the totals P + P2 R, R2 R
  double grow[S];
#pragma unroll
  for (int c = 0; c < S; c++) grow[c] = 0;
  if (t < nv) {
    const int k = t;
#pragma unroll
    for (int c = 0; c < S; c++) {
      double2 a = make_double2(0, 0);
      for (int l = 0; l <= c; l++) {
        const double2 x = zmul(P[k][l], D[l][c]);
        a.x -= x.x;
        a.y -= x.y;
      }
      C[k][c] = a;
      grow[c] += a.x * a.x + a.y * a.y;
      double2 p = P[k][c];
      if (again) {
        p = io.p1(k, c);
        for (int l = 0; l <= c; l++) {
          const double2 x = zmul(P[k][l], io.r1(l, c));
          p.x += x.x;
          p.y += x.y;
        }
      }
      Pt[k][c] = p;
    }
  }
  if (t < S * S) {
    const int r = t / S, c = t % S;
    double2 x = R[r][c];
    if (again) {
      x = make_double2(0, 0);
      for (int l = r; l <= c; l++) {
        const double2 y = zmul(R[r][l], io.r1(l, c));
        x.x += y.x;
        x.y += y.y;
      }
    }
    Rt[r][c] = x;
  }
  __syncthreads();
  // rows of C sit in the first NMAX = 128 threads: two wavefronts
#pragma unroll
  for (int c = 0; c < S; c++) {
    double s = grow[c];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (t < 128 && (t & 63) == 0) red[t >> 6][c] = s;
  }
  __syncthreads();
  double most = 0;
#pragma unroll
  for (int c = 0; c < S; c++) most += red[0][c] + red[1][c];
  for (int i = t; i < nv * S; i += 256) io.coef(i / S, i % S, C[i / S][i % S], Pt[i / S][i % S]);
  if (t < S * S) io.factor(t / S, t % S, D[t / S][t % S], Rt[t / S][t % S]);
  // the columns, one after the other: row t of column j + i.  What the old
  // columns contribute to all of them first (H_k has no rows past k + 1 <= j).
  double2 old[S];
#pragma unroll
  for (int i = 0; i < S; i++) old[i] = make_double2(0, 0);
  if (S > 1 && t <= j) {
#pragma unroll 4
    for (int k = 0; k < j; k++) {
      const double2 h = io.h(t, k);
#pragma unroll
      for (int i = 1; i < S; i++) {
        const double2 x = zmul(Pt[k][i - 1], h);
        old[i].x += x.x;
        old[i].y += x.y;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < S; i++) {
    const int rows = j + i + 2;
    if (t < ld) {
      double2 h = make_double2(0, 0);
      if (i <= good && t < rows) {
        // coef(u_{i+1}), u_1 first
        if (t <= j) h = Pt[t][i];
        else if (t - nv <= i) h = Rt[t - nv][i];
        if (i > 0) {
          // B q_i: less what u_i's other components contribute
          h = zsub(zsub(h, old[i]), zmul(Pt[j][i - 1], col[0][t]));
#pragma unroll
          for (int l = 1; l < i; l++) h = zsub(h, zmul(Rt[l - 1][i - 1], col[l][t]));
          const double inv = 1.0 / Rt[i - 1][i - 1].x;
          h.x *= inv;
          h.y *= inv;
        }
      }
      col[i][t] = h;  // read by this thread only
    }
  }
  if (t < ld)
#pragma unroll
    for (int i = 0; i < S; i++) io.put(t, j + i, i, col[i][t]);
  if (t == 0) io.info(good, sqrt(most), worst);
}

}  // namespace qqcd
