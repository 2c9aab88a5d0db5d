// qqcd_arnoldi.hip -- see qqcd_arnoldi.h.
#include "qqcd_arnoldi.h"

#include <algorithm>
#include <stdexcept>

#include "qqcd_blockalg.h"
#include "qqcd_pool.h"

namespace qqcd {

typedef std::complex<double> zd;

static constexpr int KV = 4;        // left vectors of a wavefront in the pass of dots
static constexpr int DW = 8;        // wavefronts of its workgroups at most
static constexpr int DGRID = 512;   // workgroups along the vector at most
static constexpr int UB = 256;      // threads of an update workgroup

struct VTab {
  void *p[BlockArnoldi::NMAX];
};

// One lane moves 16 bytes of every vector: E complex numbers.
template <typename T> struct Lane;
template <> struct Lane<double> {
  static constexpr int E = 1;
  typedef double2 Raw;
  static __device__ __forceinline__ void split(Raw v, double2 (&e)[1]) { e[0] = v; }
  static __device__ __forceinline__ void ld(const void *p, long i, double2 (&e)[1]) { e[0] = ((const double2 *)p)[i]; }
  static __device__ __forceinline__ void st(void *p, long i, const double2 (&e)[1]) { ((double2 *)p)[i] = e[0]; }
};
template <> struct Lane<float> {
  static constexpr int E = 2;
  typedef float4 Raw;
  static __device__ __forceinline__ void split(Raw v, double2 (&e)[2]) {
    e[0] = make_double2(v.x, v.y);
    e[1] = make_double2(v.z, v.w);
  }
  static __device__ __forceinline__ void ld(const void *p, long i, double2 (&e)[2]) {
    const float4 v = ((const float4 *)p)[i];
    e[0] = make_double2(v.x, v.y);
    e[1] = make_double2(v.z, v.w);
  }
  static __device__ __forceinline__ void st(void *p, long i, const double2 (&e)[2]) {
    ((float4 *)p)[i] = make_float4((float)e[0].x, (float)e[0].y, (float)e[1].x, (float)e[1].y);
  }
};

// part[(chunk * gridDim.x + block) * 2 KV S + 2 (q S + c) + {0, 1}] = <v_{KV chunk + q}, u_c>
// over the block's lanes, u_c the last S of the nleft vectors.
//
// Bound by reading the basis once.  The wavefronts of a workgroup take KV
// vectors each and the same stretch of the u_c, which so come from memory once
// per workgroup (up to 32 vectors) and from the L1 for its other wavefronts;
// KV S = 16 complex FP64 accumulators leave three wavefronts per SIMD.
// The next stretch is loaded ahead of a stretch's arithmetic (FP32 vectors, whose
// products are formed in FP64, 16^3x32: 83.6 -> 44.2 us; FP64 3%).  24^3x48, FP64,
// S = 4 over 31 vectors on average: 358 us, 5.5 TB/s.
template <typename T, int S>
__global__ void __launch_bounds__(64 * DW) k_bdot(long nu, VTab v, int nleft, double *part) {
  constexpr int E = Lane<T>::E;
  const int lane = threadIdx.x & 63;
  const int chunk = blockIdx.y * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int k0 = __builtin_amdgcn_readfirstlane(chunk * KV);
  if (k0 >= nleft) return;
  const void *a[KV], *u[S];
#pragma unroll
  for (int q = 0; q < KV; q++) a[q] = v.p[k0 + q < nleft ? k0 + q : nleft - 1];
#pragma unroll
  for (int c = 0; c < S; c++) u[c] = v.p[nleft - S + c];
  double acc[2 * KV * S];
#pragma unroll
  for (int k = 0; k < 2 * KV * S; k++) acc[k] = 0;
  typedef typename Lane<T>::Raw Raw;
  const long step = gridDim.x * 64L;
  Raw rb[S], re[KV];
  auto fetch = [&](long i) {
#pragma unroll
    for (int c = 0; c < S; c++) rb[c] = ((const Raw *)u[c])[i];
#pragma unroll
    for (int q = 0; q < KV; q++) re[q] = ((const Raw *)a[q])[i];
  };
  long i = blockIdx.x * 64L + lane;
  if (i < nu) fetch(i);
  for (; i < nu; i += step) {
    double2 b[S][E], e[KV][E];
#pragma unroll
    for (int c = 0; c < S; c++) Lane<T>::split(rb[c], b[c]);
#pragma unroll
    for (int q = 0; q < KV; q++) Lane<T>::split(re[q], e[q]);
    if (i + step < nu) fetch(i + step);  // ahead of this stretch's arithmetic
#pragma unroll
    for (int q = 0; q < KV; q++)
#pragma unroll
      for (int c = 0; c < S; c++)
#pragma unroll
        for (int x = 0; x < E; x++) {
          acc[2 * (q * S + c)] += e[q][x].x * b[c][x].x + e[q][x].y * b[c][x].y;
          acc[2 * (q * S + c) + 1] += e[q][x].x * b[c][x].y - e[q][x].y * b[c][x].x;
        }
  }
  double mine = 0;
#pragma unroll
  for (int k = 0; k < 2 * KV * S; k++) {
    double s = acc[k];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (lane == k) mine = s;
  }
  if (lane < 2 * KV * S) part[((long)chunk * gridDim.x + blockIdx.x) * (2 * KV * S) + lane] = mine;
}

// sums[chunk * nq + q] = sum over the nb blocks, in a fixed order; one workgroup per chunk
__global__ void __launch_bounds__(1024) k_bsum(int nb, int nq, const double *part, double *sums) {
  __shared__ double sm[32][33];
  const int q = threadIdx.x & 31, g = threadIdx.x >> 5;
  const double *p = part + (long)blockIdx.x * nb * nq + q;
  double s = 0;
  if (q < nq) {
#pragma unroll 4
    for (int b = g; b < nb; b += 32) s += p[(long)b * nq];
  }
  sm[g][q] = s;
  __syncthreads();
  // row g now sums column g
  double c = sm[q][g];
#pragma unroll
  for (int o = 16; o > 0; o >>= 1) c += __shfl_xor(c, o, 32);
  if (q == 0 && g < nq) sums[(long)blockIdx.x * nq + g] = c;
}

// what block_columns reads and writes for one right-hand side
template <int S> struct BlockIO {
  const double2 *sums;
  double2 *hd, *pr, *c;
  float2 *c32;
  double2 *hout;
  double *inf;
  int ld, g0, nv;
  static constexpr int SM = BlockArnoldi::SMAX, NM = BlockArnoldi::NMAX;
  __device__ double2 p(int k, int c_) const { return sums[k * S + c_]; }
  __device__ double2 g(int r, int c_) const { return sums[(long)(g0 + r) * S + c_]; }
  // (rows of SM: a second pass may take fewer vectors than the first)
  __device__ double2 p1(int k, int c_) const { return pr[k * SM + c_]; }
  __device__ double2 r1(int l, int c_) const { return pr[(nv + l) * SM + c_]; }
  __device__ void coef(int k, int c_, double2 x, double2 pt) {
    const int i = k * S + c_;
    c[i] = x;
    c32[i] = make_float2((float)x.x, (float)x.y);
    pr[k * SM + c_] = pt;
    // the update walks the vectors four at a time
    if (k == nv - 1)
      for (int q = nv; q < (nv + 3) / 4 * 4; q++) {
        c[q * S + c_] = make_double2(0, 0);
        c32[q * S + c_] = make_float2(0, 0);
      }
  }
  __device__ void factor(int r, int c_, double2 d, double2 rt) {
    c[NM * SM + r * S + c_] = d;
    c32[NM * SM + r * S + c_] = make_float2((float)d.x, (float)d.y);
    pr[(nv + r) * SM + c_] = rt;
  }
  __device__ double2 h(int row, int col) const { return hd[row + (long)ld * col]; }
  __device__ void put(int row, int col, int i, double2 x) {
    hd[row + (long)ld * col] = x;
    hout[row + (long)ld * i] = x;
  }
  __device__ void info(int good, double growth, double pivot) {
    inf[0] = good;
    inf[1] = growth;
    inf[2] = pivot;
  }
};

template <int S>
__global__ void __launch_bounds__(256) k_bcols(int j, int ld, int again, int g0, double least, const double2 *sums,
                                               double2 *hd, double2 *pr, double2 *coef, float2 *coef32, double2 *hout,
                                               double *info) {
  block_columns<S>(BlockIO<S>{sums, hd, pr, coef, coef32, hout, info, ld, g0, j + 1}, j, ld, again, least);
}

// v_{nv+c} <- sum_l u_l D_lc + sum_k v_k C_kc, u_l = v_{nv+l} before: Q in place
// of U.  Bound by reading the basis and U once and writing Q once (a lane's S
// sums stay in registers over all nv vectors, four vectors' loads ahead); the
// coefficients are wavefront-uniform and come through scalar loads.  24^3x48,
// FP64, S = 4: 448 us, 5.1 TB/s.
template <typename T, int S>
__global__ void __launch_bounds__(UB) k_bupdate(long nu, VTab v, int nv, const double *__restrict__ coef) {
  constexpr int E = Lane<T>::E;
  const double *D = coef + 2 * BlockArnoldi::NMAX * BlockArnoldi::SMAX;
  for (long i = blockIdx.x * (long)UB + threadIdx.x; i < nu; i += (long)gridDim.x * UB) {
    double2 u[S][E], s[S][E];
#pragma unroll
    for (int c = 0; c < S; c++) Lane<T>::ld(v.p[nv + c], i, u[c]);
#pragma unroll
    for (int c = 0; c < S; c++)
#pragma unroll
      for (int x = 0; x < E; x++) {
        s[c][x] = make_double2(0, 0);
#pragma unroll
        for (int l = 0; l <= c; l++) {
          const double dr = D[2 * (l * S + c)], di = D[2 * (l * S + c) + 1];
          s[c][x].x += dr * u[l][x].x - di * u[l][x].y;
          s[c][x].y += dr * u[l][x].y + di * u[l][x].x;
        }
      }
    for (int k = 0; k < nv; k += 4) {
      double2 e[4][E];
#pragma unroll
      for (int q = 0; q < 4; q++) Lane<T>::ld(v.p[k + q < nv ? k + q : nv - 1], i, e[q]);
#pragma unroll
      for (int q = 0; q < 4; q++)
#pragma unroll
        for (int c = 0; c < S; c++) {
          const double cr = coef[2 * ((k + q) * S + c)], ci = coef[2 * ((k + q) * S + c) + 1];
#pragma unroll
          for (int x = 0; x < E; x++) {
            s[c][x].x += cr * e[q][x].x - ci * e[q][x].y;
            s[c][x].y += cr * e[q][x].y + ci * e[q][x].x;
          }
        }
    }
#pragma unroll
    for (int c = 0; c < S; c++) Lane<T>::st(v.p[nv + c], i, s[c]);
  }
}

// ---- an FP16 basis with per-site norms, the block's u_c in FP32 ----------

struct NTab {
  float *n[BlockArnoldi::NMAX];
};
struct UTab {
  const void *p[BlockArnoldi::SMAX];
};
typedef f16 h2v __attribute__((ext_vector_type(2)));
typedef f16 h8v __attribute__((ext_vector_type(8)));

__device__ __forceinline__ void ld4(const void *p, long i, float2 (&e)[4]) {
  const float4 a = ((const float4 *)p)[2 * i], b = ((const float4 *)p)[2 * i + 1];
  e[0] = make_float2(a.x, a.y);
  e[1] = make_float2(a.z, a.w);
  e[2] = make_float2(b.x, b.y);
  e[3] = make_float2(b.z, b.w);
}
// k_bdot for an FP16 basis: the chunks of KV basis vectors, and after them one
// of the u_c themselves (G).  A lane takes four consecutive sites and walks
// their 12 component runs (nq = stride / 4 site quads), so each vector's norms
// are read once; 16 bytes of a vector a lane.  Sums in FP32 over the 48 products
// of a lane's quad (the basis carries 11 bits), in FP64 beyond.
template <int S>
__global__ void __launch_bounds__(64 * DW) k_bdot_h(long nq, VTab v, NTab vn, UTab ut, int nv, double *part) {
  const int lane = threadIdx.x & 63, cv = (nv + KV - 1) / KV;
  const int chunk = __builtin_amdgcn_readfirstlane(blockIdx.y * (blockDim.x >> 6) + (threadIdx.x >> 6));
  if (chunk > cv) return;
  constexpr int HV = S % 4 == 0 ? 5 : S % 2 == 0 ? 4 : 3;  // 2 KV S is a multiple of 2^HV
  Runs<2 * KV * S, HV> runs;
  float af[2 * KV * S];
#pragma unroll
  for (int k = 0; k < 2 * KV * S; k++) af[k] = 0.f;
  auto add = [&](const float2(&e)[4], const float2(&b)[S][4], int q) {
#pragma unroll
    for (int c = 0; c < S; c++)
#pragma unroll
      for (int x = 0; x < 4; x++) {
        af[2 * (q * S + c)] += e[x].x * b[c][x].x + e[x].y * b[c][x].y;
        af[2 * (q * S + c) + 1] += e[x].x * b[c][x].y - e[x].y * b[c][x].x;
      }
  };
  if (chunk < cv) {
    const int k0 = chunk * KV;
    const void *pv[KV];
#pragma unroll
    for (int k = 0; k < KV; k++) pv[k] = v.p[k0 + k < nv ? k0 + k : nv - 1];
    for (long q0 = blockIdx.x * 64L; q0 < nq; q0 += gridDim.x * 64L) {
      const long q = q0 + lane < nq ? q0 + lane : nq - 1;  // lanes past the end repeat the last quad for nothing
      float4 m[KV], ub[2 * S];
      h8v vb[KV];
      auto fetch = [&](long i) {
#pragma unroll
        for (int k = 0; k < KV; k++) vb[k] = ((const h8v *)pv[k])[i];
#pragma unroll
        for (int c = 0; c < S; c++) {
          ub[2 * c] = ((const float4 *)ut.p[c])[2 * i];
          ub[2 * c + 1] = ((const float4 *)ut.p[c])[2 * i + 1];
        }
      };
      fetch(q);
#pragma unroll
      for (int k = 0; k < KV; k++) {
        m[k] = *(const float4 *)(vn.n[k0 + k < nv ? k0 + k : nv - 1] + 4 * q);
        if (q0 + lane >= nq) m[k] = make_float4(0.f, 0.f, 0.f, 0.f);
      }
      for (int r = 0; r < 12; r++) {
        float2 b[S][4];
        h8v vc[KV];
#pragma unroll
        for (int c = 0; c < S; c++) {
          b[c][0] = make_float2(ub[2 * c].x, ub[2 * c].y);
          b[c][1] = make_float2(ub[2 * c].z, ub[2 * c].w);
          b[c][2] = make_float2(ub[2 * c + 1].x, ub[2 * c + 1].y);
          b[c][3] = make_float2(ub[2 * c + 1].z, ub[2 * c + 1].w);
        }
#pragma unroll
        for (int k = 0; k < KV; k++) vc[k] = vb[k];
        if (r < 11) fetch((r + 1) * nq + q);  // ahead of this run's arithmetic
#pragma unroll
        for (int k = 0; k < KV; k++) {
          float2 e[4];
          e[0] = make_float2(m[k].x * (float)vc[k][0], m[k].x * (float)vc[k][1]);
          e[1] = make_float2(m[k].y * (float)vc[k][2], m[k].y * (float)vc[k][3]);
          e[2] = make_float2(m[k].z * (float)vc[k][4], m[k].z * (float)vc[k][5]);
          e[3] = make_float2(m[k].w * (float)vc[k][6], m[k].w * (float)vc[k][7]);
          add(e, b, k);
        }
      }
      runs.add(af, lane);
    }
  } else {
    for (long q0 = blockIdx.x * 64L; q0 < nq; q0 += gridDim.x * 64L) {
      const long q = q0 + lane;
      for (int r = 0; r < 12 && q < nq; r++) {
        float2 b[S][4];
#pragma unroll
        for (int c = 0; c < S; c++) ld4(ut.p[c], r * nq + q, b[c]);
#pragma unroll
        for (int k = 0; k < S; k++) add(b[k], b, k);
      }
      runs.add(af, lane);
    }
  }
  // a lane is left with M totals (2 KV S / 32 where that is whole), over the lanes of its lower bits
  constexpr int M = decltype(runs)::M;
#pragma unroll
  for (int q = 0; q < M; q++) {
    double s = runs.tot[q];
#pragma unroll
    for (int o = (64 >> HV) / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((lane & ((64 >> HV) - 1)) == 0)
      part[((long)chunk * gridDim.x + blockIdx.x) * (2 * KV * S) + runs.first(lane) + q] = s;
  }
}

// k_bupdate for an FP16 basis, one lane per site: the S new vectors of a site
// in registers (24 S floats), rounded to the basis's format at the end (the
// site's 24 reals over their largest magnitude, that magnitude as its norm).
// Reads the basis and the u_c once, writes the new vectors once: 244 us at
// 32^3x64 and 14.5 vectors, 5.7 TB/s.
template <int S>
__global__ void __launch_bounds__(UB) k_bupdate_h(long stride, VTab v, NTab vn, UTab ut, int nv,
                                                  const float *__restrict__ coef) {
  const float *D = coef + 2 * BlockArnoldi::NMAX * BlockArnoldi::SMAX;
  const long i = blockIdx.x * (long)UB + threadIdx.x;
  if (i >= stride) return;
  float2 s[S][12];
#pragma unroll
  for (int r = 0; r < 12; r++) {
    float2 u[S];
#pragma unroll
    for (int c = 0; c < S; c++) u[c] = ((const float2 *)ut.p[c])[r * stride + i];
#pragma unroll
    for (int c = 0; c < S; c++) {
      s[c][r] = make_float2(0, 0);
#pragma unroll
      for (int l = 0; l <= c; l++) {
        const float dr = D[2 * (l * S + c)], di = D[2 * (l * S + c) + 1];
        s[c][r].x += dr * u[l].x - di * u[l].y;
        s[c][r].y += dr * u[l].y + di * u[l].x;
      }
    }
  }
  for (int k = 0; k < nv; k++) {
    const float m = vn.n[k][i];
    const h2v *p = (const h2v *)v.p[k] + i;
    h2v h[12];
#pragma unroll
    for (int r = 0; r < 12; r++) h[r] = p[r * stride];
    float cr[S], ci[S];
#pragma unroll
    for (int c = 0; c < S; c++) {
      cr[c] = m * coef[2 * (k * S + c)];
      ci[c] = m * coef[2 * (k * S + c) + 1];
    }
#pragma unroll
    for (int r = 0; r < 12; r++) {
      const float x = (float)h[r].x, y = (float)h[r].y;
#pragma unroll
      for (int c = 0; c < S; c++) {
        s[c][r].x += cr[c] * x - ci[c] * y;
        s[c][r].y += cr[c] * y + ci[c] * x;
      }
    }
  }
#pragma unroll
  for (int c = 0; c < S; c++) {
    float m = 0.f;
#pragma unroll
    for (int r = 0; r < 12; r++) m = fmaxf(m, fmaxf(fabsf(s[c][r].x), fabsf(s[c][r].y)));
    const float f = m > 0.f ? 1.f / m : 0.f;
    h2v *o = (h2v *)v.p[nv + c] + i;
#pragma unroll
    for (int r = 0; r < 12; r++) {
      h2v h;
      h.x = (f16)(s[c][r].x * f);
      h.y = (f16)(s[c][r].y * f);
      o[r * stride] = h;
    }
    vn.n[nv + c][i] = m;
  }
}

// ===================================================================== //

static constexpr int CHUNKS = BlockArnoldi::NMAX / KV + 1;

BlockArnoldi::BlockArnoldi(hipStream_t s, int m_) : stream(s), m(m_), ld(m_ + 1) {
  if (m < 1 || m + 1 > NMAX) throw std::runtime_error("BlockArnoldi: at most 127 steps");
  const int slots = m;  // one per block at least
  bufs.get(&hd, sizeof(double) * 2 * ld * m);
  bufs.get(&part, sizeof(double) * 2 * KV * SMAX * DGRID * CHUNKS);
  bufs.get(&sums, sizeof(double) * 2 * KV * SMAX * CHUNKS);
  bufs.get(&pr, sizeof(double) * 2 * SMAX * (NMAX + SMAX));
  bufs.get(&coef, sizeof(double) * 2 * SMAX * (NMAX + SMAX));
  bufs.get(&coef32, sizeof(float) * 2 * SMAX * (NMAX + SMAX));
  bufs.get_host(&hh, sizeof(double) * slot_len() * slots);
}

void BlockArnoldi::load(const zd *h, int ldh, int n, double sigma) {
  if (n < 0 || n > m) throw std::runtime_error("BlockArnoldi: too many columns");
  if (n == 0) return;
  std::vector<zd> a((size_t)ld * n, 0.0);
  for (int q = 0; q < n; q++)
    for (int i = 0; i <= n; i++) a[i + (size_t)ld * q] = h[i + (size_t)ldh * q] - (i == q ? sigma : 0.0);
  QQCD_HIP(hipMemcpyAsync(hd, a.data(), sizeof(zd) * a.size(), hipMemcpyHostToDevice, stream));
  QQCD_HIP(hipStreamSynchronize(stream));
}

void BlockArnoldi::put(const zd *h, int j, double sigma) {
  if (j < 0 || j >= m) throw std::runtime_error("BlockArnoldi: no such column");
  std::vector<zd> a(ld, 0.0);
  for (int i = 0; i <= j + 1; i++) a[i] = h[i] - (i == j ? sigma : 0.0);
  QQCD_HIP(hipMemcpyAsync(hd + 2L * ld * j, a.data(), sizeof(zd) * ld, hipMemcpyHostToDevice, stream));
  QQCD_HIP(hipStreamSynchronize(stream));
}

template <typename F> static void with_s(int s, F &&f) {
  switch (s) {
    case 1: f(std::integral_constant<int, 1>()); break;
    case 2: f(std::integral_constant<int, 2>()); break;
    case 3: f(std::integral_constant<int, 3>()); break;
    case 4: f(std::integral_constant<int, 4>()); break;
    default: throw std::runtime_error("BlockArnoldi: 1..4 steps a block");
  }
}

void BlockArnoldi::run(const Vec *V, int j, int s, int slot, bool again) {
  if (j < 0 || s < 1 || s > SMAX || j + s > m || slot < 0 || slot >= m) throw std::runtime_error("BlockArnoldi: bad block");
  const int nleft = j + 1 + s;
  VTab tab{};
  for (int q = 0; q < nleft; q++) {
    if (V[q].prec != V[0].prec || V[q].n != V[0].n) throw std::runtime_error("BlockArnoldi: mixed vectors");
    tab.p[q] = V[q].data;
  }
  const long n = V[0].n;
  double *slot_h = hh + slot_len() * slot;
  auto go = [&](auto tag) {
    typedef decltype(tag) T;
    constexpr int E = Lane<T>::E;
    if (n % E) throw std::runtime_error("BlockArnoldi: odd vector length");
    const long nu = n / E;
    const int chunks = (nleft + KV - 1) / KV, ny = (chunks + DW - 1) / DW, w = (chunks + ny - 1) / ny;
    // about 3000 wavefronts in flight; no more workgroups than 64-lane stretches
    const int gx = (int)std::max(1L, std::min({(nu + 63) / 64, (long)DGRID, 3072L / (long)(w * ny) + 1}));
    const int gu = (int)std::min((nu + UB - 1) / UB, 2048L);
    with_s(s, [&](auto SS) {
      constexpr int S = decltype(SS)::value;
      hipLaunchKernelGGL((k_bdot<T, S>), dim3(gx, ny), dim3(64 * w), 0, stream, nu, tab, nleft, part);
      hipLaunchKernelGGL(k_bsum, dim3(chunks), dim3(1024), 0, stream, gx, 2 * KV * S, part, sums);
      // a vector is taken while at least 1e-6 (FP64: the Arnoldi relation then holds to 1e-13, the rounding over the
      // square root of this; FP32: 1e-10, its rounding squared being 4e-15) of its squared norm is left
      hipLaunchKernelGGL((k_bcols<S>), dim3(1), dim3(256), 0, stream, j, ld, again ? 1 : 0, j + 1,
                         sizeof(T) == 8 ? 1e-6 : 1e-10, (const double2 *)sums, (double2 *)hd, (double2 *)pr,
                         (double2 *)coef, (float2 *)coef32, (double2 *)slot_h, slot_h + 2L * SMAX * ld);
      hipLaunchKernelGGL((k_bupdate<T, S>), dim3(gu), dim3(UB), 0, stream, nu, tab, j + 1, coef);
    });
    QQCD_HIP(hipGetLastError());
  };
  if (V[0].prec == PREC_DOUBLE) go(double());
  else if (V[0].prec == PREC_SINGLE) go(float());
  else throw std::runtime_error("BlockArnoldi: FP64 or FP32 vectors");
}

void BlockArnoldi::queue_half(const Vec *V, const Vec *U, int j, int s, int slot) {
  if (j < 0 || s < 1 || s > SMAX || j + s > m || slot < 0 || slot >= m) throw std::runtime_error("BlockArnoldi: bad block");
  VTab tab{};
  NTab nt{};
  UTab ut{};
  for (int q = 0; q <= j + s; q++) {
    if (V[q].prec != PREC_HALF || !V[q].norm || V[q].n != V[0].n) throw std::runtime_error("BlockArnoldi: FP16 basis");
    tab.p[q] = V[q].data;
    nt.n[q] = const_cast<float *>(V[q].norm);
  }
  for (int c = 0; c < s; c++) {
    if (U[c].prec != PREC_SINGLE || U[c].n != V[0].n) throw std::runtime_error("BlockArnoldi: FP32 work vectors");
    ut.p[c] = U[c].data;
  }
  const long stride = V[0].n / 12, nq = stride / 4;
  if (V[0].n % 48) throw std::runtime_error("BlockArnoldi: not a checkerboard field");
  const int nv = j + 1, cv = (nv + KV - 1) / KV, chunks = cv + 1, ny = (chunks + DW - 1) / DW, w = (chunks + ny - 1) / ny;
  const int gx = (int)std::max(1L, std::min({(nq + 63) / 64, (long)DGRID, 3072L / (long)(w * ny) + 1}));
  double *slot_h = hh + slot_len() * slot;
  with_s(s, [&](auto SS) {
    constexpr int S = decltype(SS)::value;
    hipLaunchKernelGGL((k_bdot_h<S>), dim3(gx, ny), dim3(64 * w), 0, stream, nq, tab, nt, ut, nv, part);
    hipLaunchKernelGGL(k_bsum, dim3(chunks), dim3(1024), 0, stream, gx, 2 * KV * S, part, sums);
    // FP32 sums over vectors of an FP16 operator: below 1e-6 of its squared norm a vector is their rounding
    hipLaunchKernelGGL((k_bcols<S>), dim3(1), dim3(256), 0, stream, j, ld, 0, cv * KV, 1e-6, (const double2 *)sums,
                       (double2 *)hd, (double2 *)pr, (double2 *)coef, (float2 *)coef32, (double2 *)slot_h,
                       slot_h + 2L * SMAX * ld);
    hipLaunchKernelGGL((k_bupdate_h<S>), dim3((unsigned)((stride + UB - 1) / UB)), dim3(UB), 0, stream, stride, tab, nt,
                       ut, nv, coef32);
  });
  QQCD_HIP(hipGetLastError());
}

void BlockArnoldi::half_sums(int nv, int s, zd *out) const {
  const int cv = (nv + KV - 1) / KV;
  QQCD_HIP(hipMemcpyAsync(out, sums, sizeof(zd) * nv * s, hipMemcpyDeviceToHost, stream));
  QQCD_HIP(hipMemcpyAsync(out + (size_t)nv * s, sums + 2L * cv * KV * s, sizeof(zd) * s * s, hipMemcpyDeviceToHost,
                          stream));
  QQCD_HIP(hipStreamSynchronize(stream));
}

void BlockArnoldi::queue(const Vec *V, int j, int s, int slot) { run(V, j, s, slot, false); }
void BlockArnoldi::queue_again(const Vec *V, int j, int s, int slot) { run(V, j, s, slot, true); }

double BlockArnoldi::loss_of(const Vec *V, int n) {
  if (n < 1 || n > NMAX || V[0].prec != PREC_DOUBLE) throw std::runtime_error("BlockArnoldi: FP64 vectors");
  VTab tab{};
  for (int q = 0; q < n; q++) tab.p[q] = V[q].data;
  std::vector<zd> g((size_t)KV * SMAX * CHUNKS);
  double f = 0;
  // the upper triangle, SMAX columns at a time (the last columns again where n is not a multiple)
  for (int c0 = 0; c0 < n; c0 += SMAX) {
    const int nleft = std::min(n, c0 + SMAX), first = std::max(0, nleft - SMAX);
    const int chunks = (nleft + KV - 1) / KV, ny = (chunks + DW - 1) / DW, w = (chunks + ny - 1) / ny;
    const int s = nleft - first, gx = (int)std::min({(V[0].n + 63) / 64, (long)DGRID, 3072L / (w * ny) + 1});
    with_s(s, [&](auto SS) {
      constexpr int S = decltype(SS)::value;
      hipLaunchKernelGGL((k_bdot<double, S>), dim3(gx, ny), dim3(64 * w), 0, stream, V[0].n, tab, nleft, part);
      hipLaunchKernelGGL(k_bsum, dim3(chunks), dim3(1024), 0, stream, gx, 2 * KV * S, part, sums);
    });
    QQCD_HIP(hipGetLastError());
    QQCD_HIP(hipMemcpyAsync(g.data(), sums, sizeof(zd) * nleft * s, hipMemcpyDeviceToHost, stream));
    QQCD_HIP(hipStreamSynchronize(stream));
    for (int q = 0; q < nleft; q++)
      for (int c = std::max(c0, q); c < nleft; c++) {
        const zd e = g[(size_t)q * s + c - first] - (q == c ? 1.0 : 0.0);
        f += (q == c ? 1.0 : 2.0) * std::norm(e);
      }
  }
  return std::sqrt(f);
}

int BlockArnoldi::fetch(int slot, int j, int s, double sigma, zd *H, int ldh) const {
  const double *a = hh + slot_len() * slot, *info = a + 2L * SMAX * ld;
  const int good = std::min(s, (int)info[0]);
  for (int i = 0; i < good; i++)
    for (int r = 0; r <= j + i + 1; r++)
      H[r + (size_t)ldh * (j + i)] =
          zd(a[2 * (r + (size_t)ld * i)], a[2 * (r + (size_t)ld * i) + 1]) + (r == j + i ? sigma : 0.0);
  return good;
}

double BlockArnoldi::growth(int slot) const { return hh[slot_len() * slot + 2L * SMAX * ld + 1]; }
double BlockArnoldi::pivot(int slot) const { return hh[slot_len() * slot + 2L * SMAX * ld + 2]; }

}  // namespace qqcd
