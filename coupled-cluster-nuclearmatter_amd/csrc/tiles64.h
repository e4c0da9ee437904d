// FP64 contraction tiles shared by the launches of contract.hip and the merged launches of
// small batches (kernels.hip).  Complex products take three real MFMAs (Gauss: ar br, ai
// bi, (ar+ai)(br+bi)).  A 16-wide k chunk is four 16x16x4 steps; lane group g = lane / 16
// of step q takes k0 + 4 q + g, so each operand load reads 64 contiguous bytes of a row.
#pragma once
#include "device.h"

namespace ccgpu {

typedef double cd4 __attribute__((ext_vector_type(4)));
typedef double cd2 __attribute__((ext_vector_type(2)));

// element e of a block whose base is the same for the whole wave (a scalar
// base and a 32-bit offset per lane; a channel's block is far below 4 GB)
__device__ __forceinline__ double2 gl(const double2 *base, unsigned e) {
  const __attribute__((address_space(1))) char *p = (const __attribute__((address_space(1))) char *)base;
  const cd2 v = *(const __attribute__((address_space(1))) cd2 *)(p + (e << 4));
  return make_double2(v.x, v.y);
}
// The elements of a lane for the Q steps from k0 of a row of length K that
// starts at element `row`, clamped to the row (the other operand, or zero_past,
// is zero past it).
template <int Q>
__device__ __forceinline__ void row_chunk(double2 (&a)[Q], const double2 *base, unsigned row, int K, int k0, int lg) {
#pragma unroll
  for (int q = 0; q < Q; ++q) a[q] = gl(base, row + min(k0 + 4 * q + lg, K - 1));
}
__device__ __forceinline__ void zero_past(double2 (&a)[4], int K, int k0, int lg) {
  if (k0 + 16 > K)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (k0 + 4 * q + lg >= K) a[q] = make_double2(0.0, 0.0);
}
// The same k of one column: row length N, column c < N
__device__ __forceinline__ void column_chunk(double2 (&b)[4], const double2 *base, unsigned c, int N, int K, int k0,
                                             int lg) {
#pragma unroll
  for (int q = 0; q < 4; ++q) b[q] = gl(base, (unsigned)min(k0 + 4 * q + lg, K - 1) * N + c);
}
__device__ __forceinline__ double2 zero_unless(bool ok, double2 v) {
  return make_double2(ok ? v.x : 0.0, ok ? v.y : 0.0);
}

// accumulators of one 16 x 16 block, and its value in register r
struct CAcc {
  cd4 re, im, s;
  __device__ __forceinline__ void clear() { re = im = s = (cd4){0.0, 0.0, 0.0, 0.0}; }
  __device__ __forceinline__ void mac(double2 a, double2 b) {
    re = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.x, re, 0, 0, 0);
    im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b.y, im, 0, 0, 0);
    s = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x + a.y, b.x + b.y, s, 0, 0, 0);
  }
  __device__ __forceinline__ double2 at(int r) const { return make_double2(re[r] - im[r], s[r] - (re[r] + im[r])); }
};

// ---------------------------------------------------------------------------
// X and I9.  K is the long side (particle pairs, up to thousands) and M = N the
// short one (hole pairs of a channel): a tile is 16 rows by up to 32 columns, its
// four waves take every fourth 16-wide chunk of k and add their partials in
// LDS in wave order.  Bound by the k chain of a tile; one block per 64 x 16
// tile over the whole k range, in a launch per width class, took 128 us of an
// iteration of PNM A=66 |n_i|<=4 (seven launches), this one 27 us, I9 included.
// ---------------------------------------------------------------------------
template <int NB>
__device__ __forceinline__ void x64_tile(const ZTile &t, double2 *red0, double2 *red1) {
  double2 *const red[2] = {red0, red1};   // of a column block each: 4 waves x 4 registers x 64 lanes
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, li = lane & 15, lg = lane >> 4;
  CAcc acc[NB];
#pragma unroll
  for (int y = 0; y < NB; ++y) acc[y].clear();
  // rows and columns past the matrix are copies of the last one and never stored
  const unsigned row = (unsigned)min(t.m0 + li, t.M - 1) * t.K;
  unsigned col[NB];
#pragma unroll
  for (int y = 0; y < NB; ++y) col[y] = min(t.n0 + 16 * y + li, t.N - 1);
  double2 a0[4], b0[NB][4], a1[4], b1[NB][4];
  auto load = [&](double2 (&a)[4], double2 (&b)[NB][4], int k0) {
    row_chunk(a, t.A, row, t.K, k0, lg);
#pragma unroll
    for (int y = 0; y < NB; ++y) column_chunk(b[y], t.B, col[y], t.N, t.K, k0, lg);
    zero_past(a, t.K, k0, lg);
  };
  auto compute = [&](const double2 (&a)[4], const double2 (&b)[NB][4]) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int y = 0; y < NB; ++y) acc[y].mac(a[q], b[y][q]);
  };
  int k0 = 16 * w;
  if (k0 < t.K) {
    load(a0, b0, k0);
    for (; k0 < t.K; k0 += 128) {
      if (k0 + 64 < t.K) load(a1, b1, k0 + 64);
      compute(a0, b0);
      if (k0 + 64 >= t.K) break;
      if (k0 + 128 < t.K) load(a0, b0, k0 + 128);
      compute(a1, b1);
    }
  }
#pragma unroll
  for (int y = 0; y < NB; ++y)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[y][(w * 4 + r) * 64 + lane] = acc[y].at(r);
  __syncthreads();
  // register r of lane l: row (l >> 4) + 4 r, column l & 15 of its block
  for (int i = w; i < 4 * NB; i += 4) {
    const int y = i >> 2, r = i & 3;
    double2 v = red[y][r * 64 + lane];
#pragma unroll
    for (int p = 1; p < 4; ++p) {
      const double2 x = red[y][(p * 4 + r) * 64 + lane];
      v.x += x.x;
      v.y += x.y;
    }
    const int mm = t.m0 + lg + 4 * r, n = t.n0 + 16 * y + li;
    if (mm < t.M && n < t.N) {
      const int64_t e = (int64_t)mm * t.N + n;
      const double2 c = t.C0[e];
      t.C[e] = v;
      t.C2[e] = make_double2(v.x + c.x, v.y + c.y);
    }
  }
}

// ---------------------------------------------------------------------------
// hh ladder: M = particle pairs, N = K = hole pairs.  64 rows by up to 32
// columns, a wave per 16 rows; I9 comes through the L1.  24 us on the same
// lattice; a launch per width class took 68 us in four.
// ---------------------------------------------------------------------------
template <int NB>
__device__ __forceinline__ void hh64_tile(const ZTile &t) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, li = lane & 15, lg = lane >> 4;
  const int mw = t.m0 + 16 * w;
  if (mw >= t.M) return;
  CAcc acc[NB];
#pragma unroll
  for (int y = 0; y < NB; ++y) acc[y].clear();
  const unsigned row = (unsigned)min(mw + li, t.M - 1) * t.K;
  unsigned col[NB];
#pragma unroll
  for (int y = 0; y < NB; ++y) col[y] = min(t.n0 + 16 * y + li, t.N - 1);
  double2 a0[4], b0[NB][4], a1[4], b1[NB][4];
  auto load = [&](double2 (&a)[4], double2 (&b)[NB][4], int k0) {
    row_chunk(a, t.A, row, t.K, k0, lg);
#pragma unroll
    for (int y = 0; y < NB; ++y) column_chunk(b[y], t.B, col[y], t.N, t.K, k0, lg);
    zero_past(a, t.K, k0, lg);
  };
  auto compute = [&](const double2 (&a)[4], const double2 (&b)[NB][4]) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int y = 0; y < NB; ++y) acc[y].mac(a[q], b[y][q]);
  };
  load(a0, b0, 0);
  for (int k0 = 0; k0 < t.K; k0 += 32) {
    if (k0 + 16 < t.K) load(a1, b1, k0 + 16);
    compute(a0, b0);
    if (k0 + 16 >= t.K) break;
    if (k0 + 32 < t.K) load(a0, b0, k0 + 32);
    compute(a1, b1);
  }
#pragma unroll
  for (int y = 0; y < NB; ++y)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int mm = mw + lg + 4 * r, n = t.n0 + 16 * y + li;
      if (mm < t.M && n < t.N) t.C[(int64_t)mm * t.N + n] = acc[y].at(r);
    }
}

}  // namespace ccgpu
