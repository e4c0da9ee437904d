// FP64 contractions of the CCD residual outside the pp ladder, one launch each
// (the ring one per channel size class), every channel and solve of a batch in
// it: X = V_hhpp T with I9 = V_hhhh + X (ccm_t2_eqn.f90:431-464, 558-560), the
// hh ladder T I9 (:614-647), and the ring of a channel pair, R~ = T~ (W0 + V~ T~) +
// W1 T~ (:657-780, 995-1026; Plan::ph_pair).
//
// Complex products take three real MFMAs (Gauss: ar br, ai bi, (ar+ai)(br+bi)).
// A 16-wide k chunk is four 16x16x4 steps; lane group g = lane / 16 of step q
// takes k0 + 4 q + g, so each operand load reads 64 contiguous bytes of a row.
// Operands that one wave alone needs go straight to its registers: a 16x16x4
// FP64 MFMA takes 64 clocks of its SIMD, so even 16 columns per row need
// only 21 bytes a clock and CU.
#include "bf3.h"
#include "device.h"
#include "tiles64.h"

#include <algorithm>

namespace ccgpu {

__global__ __launch_bounds__(256, 2) void k_x64(const ZTile *__restrict__ tiles, const SolveDesc *__restrict__ descs) {
  __shared__ double2 red[2][4 * 4 * 64];
  const ZTile t = tiles[blockIdx.x];
  if (!descs[t.solve].active) return;
  if (t.nb == 1) x64_tile<1>(t, red[0], red[1]);
  else x64_tile<2>(t, red[0], red[1]);
}

__global__ __launch_bounds__(256, 2) void k_hh64(const ZTile *__restrict__ tiles, const SolveDesc *__restrict__ descs) {
  const ZTile t = tiles[blockIdx.x];
  if (!descs[t.solve].active) return;
  if (t.nb == 1) hh64_tile<1>(t);
  else hh64_tile<2>(t);
}

// ---------------------------------------------------------------------------
// Ring of a channel pair: column block n0 of R~ = W1 T~ + T~ (W0 + V~ T~)
// needs the T~ columns n0 and that block of I4 = W0 + V~ T~ only, so one block does all
// three products, with the T~ columns and then the I4 columns in LDS (I4 never goes
// to memory).  Eight waves: WR along the rows, RB 16-row blocks each, by WC of 16
// columns.  V~, W1 and T~ rows go straight to the wave that owns them.  Column
// blocks of a channel run on one XCD, whose L2 holds the operands for them.
//
// 16 WR RB covers the channel's larger side: 64 (WR 4, WC 2) and 128 (WR 8) in one
// launch, 32 KB of LDS and two workgroups per CU, 256 (WR 8, RB 2) in another.
// Bound by FP64 MFMA: PNM A=66 |n_i|<=4 takes 190 us alone on the device, MFMA alone
// 114.  Both channels of a pair contracted on their own (four products instead of
// three, T~ and R~ of both) took 272 us; launches of their own for up to 64, 96 (six
// waves) and 128 rows 224, 32 columns per wave 216.
// ---------------------------------------------------------------------------
template <int WR, int WC, int RB>
__device__ __forceinline__ void ring64_tile(const RingTile &t, double2 *Bs) {
  constexpr int BC = 16 * WC, NT = 512;
  const int lane = threadIdx.x & 63, w = (threadIdx.x >> 6) % WR, li = lane & 15, lg = lane >> 4;
  const int cw = 16 * ((threadIdx.x >> 6) / WR);   // first column of the wave in LDS
  const int c = t.n0 + cw + li;
  CAcc acc[RB];
  // two MFMA steps (8 k) ahead: with four waves on a SIMD the loads have the
  // other waves' 3 x 768 clocks, and 16 registers less keep 128 without spills
  double2 a0[RB][2], a1[RB][2];
  // steps from k0 of this wave's rows (blocks w and w + WR) of A, M x K.  Rows
  // past M are copies of the last and never used; k past K meets zeros in LDS.
  auto load = [&](double2 (&a)[RB][2], const double2 *A, int M, int K, int k0) {
#pragma unroll
    for (int x = 0; x < RB; ++x) row_chunk(a[x], A, (unsigned)min(16 * (w + WR * x) + li, M - 1) * K, K, k0, lg);
  };
  auto compute = [&](const double2 (&a)[RB][2], int k0) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const double2 bv = Bs[(k0 + 4 * q + lg) * BC + cw + li];
#pragma unroll
      for (int x = 0; x < RB; ++x) acc[x].mac(a[x][q], bv);
    }
  };
  auto clear = [&] {
#pragma unroll
    for (int x = 0; x < RB; ++x) acc[x].clear();
  };
  // plus the rows times the columns in LDS; the first two steps are in a0 already
  auto product = [&](const double2 *A, int M, int K) {
    if (16 * w >= M || t.n0 + cw >= t.nhp) return;
    for (int k0 = 0; k0 < K; k0 += 16) {   // whole chunks of 16: LDS is zero past K
      load(a1, A, M, K, k0 + 8);
      compute(a0, k0);
      load(a0, A, M, K, k0 + 16);
      compute(a1, k0 + 8);
    }
  };
  load(a0, t.Vt, t.nhp, t.nph, 0);
  // T~ columns, zero past the matrix (up to the last whole chunk of k); eight
  // loads per thread in flight
  {
    const int n = ((t.nph + 15) & ~15) * BC;
    for (int e0 = threadIdx.x; e0 < n; e0 += 8 * NT) {
      double2 v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int e = e0 + j * NT, k = e / BC, x = t.n0 + e % BC;
        v[j] = zero_unless(k < t.nph && x < t.nhp, gl(t.Tt, (unsigned)min(k, t.nph - 1) * t.nhp + min(x, t.nhp - 1)));
      }
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (e0 + j * NT < n) Bs[e0 + j * NT] = v[j];
    }
  }
  __syncthreads();
  clear();
  product(t.Vt, t.nhp, t.nph);
  load(a0, t.W1, t.nph, t.nph, 0);
  // I4 = W0 + V~ T~ in registers; rows past nhp in a wave's block are zero
  double2 i4[RB][4];
#pragma unroll
  for (int x = 0; x < RB; ++x)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = 16 * (w + WR * x) + lg + 4 * r;
      const double2 s = acc[x].at(r);
      const double2 c0 = gl(t.W0, (unsigned)min(m, t.nhp - 1) * t.nhp + min(c, t.nhp - 1));
      i4[x][r] = zero_unless(m < t.nhp && c < t.nhp, make_double2(s.x + c0.x, s.y + c0.y));
    }
  clear();
  product(t.W1, t.nph, t.nph);
  load(a0, t.Tt, t.nph, t.nhp, 0);
  __syncthreads();   // every wave has read the T~ columns
#pragma unroll
  for (int x = 0; x < RB; ++x) {
    if (16 * (w + WR * x) >= t.nhp) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) Bs[(16 * (w + WR * x) + lg + 4 * r) * BC + cw + li] = i4[x][r];
  }
  __syncthreads();
  product(t.Tt, t.nph, t.nhp);
#pragma unroll
  for (int x = 0; x < RB; ++x)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = 16 * (w + WR * x) + lg + 4 * r;
      if (m < t.nph && c < t.nhp) t.Rt[(int64_t)m * t.nhp + c] = acc[x].at(r);
    }
}

// channels of up to 128 (RB 1) or 256 (RB 2) rows
template <int RB>
__global__ __launch_bounds__(512, RB == 1 ? 4 : 2) void k_ring64(const RingTile *__restrict__ tiles,
                                                                 const SolveDesc *__restrict__ descs) {
  __shared__ double2 Bs[128 * RB * 16];
  const RingTile t = tiles[blockIdx.x];
  if (!descs[t.solve].active) return;
  if (RB == 1 && max(t.nph, t.nhp) <= 64) ring64_tile<4, 2, 1>(t, Bs);
  else ring64_tile<8, 1, RB>(t, Bs);
}

int ring64_class(int nph, int nhp) {   // launch of a channel, -1: too large for the fused kernel
  const int d = std::max(nph, nhp);
  return d <= 128 ? 0 : d <= 256 ? 1 : -1;
}
int ring64_columns(int nph, int nhp) { return std::max(nph, nhp) <= 64 ? 32 : 16; }

void launch_ring64(const RingTile *tiles, int ntiles, int cls, const SolveDesc *dd, hipStream_t st) {
  if (ntiles <= 0) return;
  if (cls == 0) hipLaunchKernelGGL(k_ring64<1>, dim3(ntiles), dim3(512), 0, st, tiles, dd);
  else hipLaunchKernelGGL(k_ring64<2>, dim3(ntiles), dim3(512), 0, st, tiles, dd);
}

// ---------------------------------------------------------------------------
// The same ring under BF16x3, on the FP32 blocks: the T~ columns, then the I4 columns
// (rounded to FP32 first), stand in LDS split once, (re, -im) as bf16 pairs in MFMA
// lane order; the rows of V~, W1 and T~ are split by the wave that owns them.  Same
// products and sums as k_zgemm_bf3.  Eight waves of RB 16-row blocks by NC
// 16-column blocks, WR along the rows by WC along the columns.
//
// Channels of up to 64 rows (WR 4, WC 2, NC 2), 128 (WR 8, NC 4) and 256 (RB 2, NC 1)
// in one launch, 64 KB of LDS, two workgroups per CU.  Channels with at most 4 pairs on
// either side stay in FP64 (ringbf_thin, ringbf_flat).  Bound by the L2 reads of the rows:
// four densities of PNM A=66 |n_i|<=4 take 313 us, as I4 and R~ with a launch per width
// class 561 in twelve.
// ---------------------------------------------------------------------------
typedef float cf4 __attribute__((ext_vector_type(4), aligned(8)));   // two float2

template <int WR, int WC, int RB, int NC>
__device__ __forceinline__ void ringbf_tile(const RingTile32 &t, unsigned *S) {
  constexpr int KS = 16 * WR * RB, BC = 16 * NC * WC, NT = 512;
  unsigned *Sl = S + BC * KS;
  const int lane = threadIdx.x & 63, w = (threadIdx.x >> 6) % WR, li = lane & 15, lg = lane >> 4;
  const int cw = 16 * NC * ((threadIdx.x >> 6) / WR);   // first column of the wave
  // four consecutive k, from 4 q, of column c: one 16-byte word, spread over the banks
  auto at = [](int c, int q) { return c * KS + ((q ^ (c & 15)) << 2); };
  f4 cre[RB][NC], cim[RB][NC];
  auto clear = [&] {
#pragma unroll
    for (int x = 0; x < RB; ++x)
#pragma unroll
      for (int y = 0; y < NC; ++y) cre[x][y] = cim[x][y] = (f4){0.f, 0.f, 0.f, 0.f};
  };
  // chunk k0 of the wave's rows: lane group lg takes k0 + 4 lg ..  Rows past M are copies
  // of the last one and never used; a last word reaches up to three elements past its
  // row, into the next or the padding behind the blocks, and is cut in compute.
  auto load = [&](cf4 (&a)[RB][2], const float2 *A, int M, int K, int k0) {
    const int k = min(k0 + 4 * lg, (K - 1) & ~3);
#pragma unroll
    for (int x = 0; x < RB; ++x) {
      const float2 *p = A + (unsigned)min(16 * (w + WR * x) + li, M - 1) * K + k;
      a[x][0] = *(const cf4 *)p;
      a[x][1] = *(const cf4 *)(p + 2);
    }
  };
  auto compute = [&](const cf4 (&a)[RB][2], int K, int k0) {
    u32x4 ah[RB], al[RB];
#pragma unroll
    for (int x = 0; x < RB; ++x)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool ok = k0 + 4 * lg + j < K;
        unsigned h, l;
        bf3_split(ok ? a[x][j >> 1][2 * (j & 1)] : 0.f, ok ? a[x][j >> 1][2 * (j & 1) + 1] : 0.f, h, l);
        ah[x][j] = h;
        al[x][j] = l;
      }
#pragma unroll
    for (int y = 0; y < NC; ++y) {
      const int o = at(cw + 16 * y + li, (k0 >> 2) + lg);
      const u32x4 brh = *(const u32x4 *)(S + o), brl = *(const u32x4 *)(Sl + o);
      const u32x4 bih = bf3_im_pairs(brh), bil = bf3_im_pairs(brl);
#pragma unroll
      for (int x = 0; x < RB; ++x) {
        const bf16x8 xh = __builtin_bit_cast(bf16x8, ah[x]), xl = __builtin_bit_cast(bf16x8, al[x]);
        cre[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xl, __builtin_bit_cast(bf16x8, brh), cre[x][y], 0, 0, 0);
        cre[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xh, __builtin_bit_cast(bf16x8, brl), cre[x][y], 0, 0, 0);
        cre[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xh, __builtin_bit_cast(bf16x8, brh), cre[x][y], 0, 0, 0);
        cim[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xl, __builtin_bit_cast(bf16x8, bih), cim[x][y], 0, 0, 0);
        cim[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xh, __builtin_bit_cast(bf16x8, bil), cim[x][y], 0, 0, 0);
        cim[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xh, __builtin_bit_cast(bf16x8, bih), cim[x][y], 0, 0, 0);
      }
    }
  };
  cf4 a0[RB][2], a1[RB][2];
  // plus the rows times the columns in LDS; the first chunk is in a0 already
  auto product = [&](const float2 *A, int M, int K) {
    if (16 * w >= M || t.n0 + cw >= t.nhp) return;
    for (int k0 = 0; k0 < K; k0 += 32) {
      load(a1, A, M, K, k0 + 16);
      compute(a0, K, k0);
      if (k0 + 16 >= K) break;
      load(a0, A, M, K, k0 + 32);
      compute(a1, K, k0 + 16);
    }
  };
  load(a0, t.Vt, t.nhp, t.nph, 0);
  // T~ columns, zero past the matrix (up to the last whole chunk of k)
  {
    const int n = ((t.nph + 15) >> 4) * 4 * BC;
    for (int e = threadIdx.x; e < n; e += NT) {
      const int c = e % BC, q = e / BC, x = t.n0 + c;
      u32x4 h, l;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = 4 * q + j;
        const float2 v = t.Tt[(unsigned)min(k, t.nph - 1) * t.nhp + min(x, t.nhp - 1)];
        const bool ok = k < t.nph && x < t.nhp;
        unsigned hj, lj;
        bf3_split(ok ? v.x : 0.f, ok ? -v.y : 0.f, hj, lj);
        h[j] = hj;
        l[j] = lj;
      }
      *(u32x4 *)(S + at(c, q)) = h;
      *(u32x4 *)(Sl + at(c, q)) = l;
    }
  }
  __syncthreads();
  clear();
  product(t.Vt, t.nhp, t.nph);
  load(a0, t.W1, t.nph, t.nph, 0);
  // I4 = W0 + V~ T~, split, in registers (register r of a lane: row 4 lg + r, column
  // li); zero past the matrix
  u32x4 ih[RB][NC], il[RB][NC];
#pragma unroll
  for (int x = 0; x < RB; ++x)
#pragma unroll
    for (int y = 0; y < NC; ++y)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = 16 * (w + WR * x) + 4 * lg + r, c = t.n0 + cw + 16 * y + li;
        const float2 v = t.W0[(unsigned)min(m, t.nhp - 1) * t.nhp + min(c, t.nhp - 1)];
        const bool ok = m < t.nhp && c < t.nhp;
        unsigned h, l;
        bf3_split(ok ? cre[x][y][r] + v.x : 0.f, ok ? -(cim[x][y][r] + v.y) : 0.f, h, l);
        ih[x][y][r] = h;
        il[x][y][r] = l;
      }
  clear();
  product(t.W1, t.nph, t.nph);
  load(a0, t.Tt, t.nph, t.nhp, 0);
  __syncthreads();   // every wave has read the T~ columns
#pragma unroll
  for (int x = 0; x < RB; ++x) {
    if (16 * (w + WR * x) >= t.nhp) continue;
#pragma unroll
    for (int y = 0; y < NC; ++y) {
      const int o = at(cw + 16 * y + li, 4 * (w + WR * x) + lg);
      *(u32x4 *)(S + o) = ih[x][y];
      *(u32x4 *)(Sl + o) = il[x][y];
    }
  }
  __syncthreads();
  product(t.Tt, t.nph, t.nhp);
#pragma unroll
  for (int x = 0; x < RB; ++x)
#pragma unroll
    for (int y = 0; y < NC; ++y)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = 16 * (w + WR * x) + 4 * lg + r, c = t.n0 + cw + 16 * y + li;
        if (m < t.nph && c < t.nhp) t.Rt[(unsigned)m * t.nhp + c] = make_float2(cre[x][y][r], cim[x][y][r]);
      }
}

__device__ __forceinline__ void mac(double2 &s, float2 x, float2 y) {
  s.x += (double)x.x * y.x - (double)x.y * y.y;
  s.y += (double)x.x * y.y + (double)x.y * y.x;
}
// at most 4 hp pairs: a thread per element, products and sums in FP64
__device__ __forceinline__ void ringbf_thin(const RingTile32 &t, float2 *i4) {
  auto row = [](double2 s, const float2 *a, const float2 *b, int K, int N) {   // s + a . column of b
    for (int k = 0; k < K; ++k) mac(s, a[k], b[k * N]);
    return s;
  };
  const int N = t.nhp;
  for (int e = threadIdx.x; e < N * N; e += 512) {
    const float2 c = t.W0[e];
    const double2 s = row(make_double2(c.x, c.y), t.Vt + e / N * t.nph, t.Tt + e % N, t.nph, N);
    i4[e] = make_float2((float)s.x, (float)s.y);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < t.nph * N; e += 512) {
    double2 s = row(make_double2(0.0, 0.0), t.W1 + (unsigned)(e / N) * t.nph, t.Tt + e % N, t.nph, N);
    s = row(s, t.Tt + (unsigned)(e / N) * N, i4 + e % N, N, N);
    t.Rt[e] = make_float2((float)s.x, (float)s.y);
  }
}

// at most 4 ph pairs: R~ = T~ W0 + (W1 + T~ V~) T~, the bracket of up to 4 x 4 elements
// first, 32 lanes to each
__device__ __forceinline__ void ringbf_flat(const RingTile32 &t, double2 *b) {
  const int M = t.nph, N = t.nhp;
  const int x = threadIdx.x >> 5, l = threadIdx.x & 31;
  if (x < M * M) {
    const int r = x / M, s = x % M;
    double2 v = make_double2(0.0, 0.0);
    for (int k = l; k < N; k += 32) mac(v, t.Tt[r * N + k], t.Vt[k * M + s]);
    for (int off = 16; off > 0; off >>= 1) {
      v.x += __shfl_xor(v.x, off);
      v.y += __shfl_xor(v.y, off);
    }
    if (l == 0) b[x] = make_double2(v.x + t.W1[x].x, v.y + t.W1[x].y);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < M * N; e += 512) {
    const int r = e / N, c = e % N;
    double2 v = make_double2(0.0, 0.0);
    for (int k = 0; k < N; ++k) mac(v, t.Tt[r * N + k], t.W0[(unsigned)k * N + c]);
    for (int k = 0; k < M; ++k) {
      const double2 q = b[r * M + k];
      const float2 y = t.Tt[k * N + c];
      v.x += q.x * y.x - q.y * y.y;
      v.y += q.x * y.y + q.y * y.x;
    }
    t.Rt[e] = make_float2((float)v.x, (float)v.y);
  }
}

__global__ __launch_bounds__(512, 4) void k_ringbf(const RingTile32 *__restrict__ tiles,
                                                   const SolveDesc *__restrict__ descs) {
  __shared__ __align__(16) unsigned S[2 * 128 * 64];
  const RingTile32 t = tiles[blockIdx.x];
  if (!descs[t.solve].active) return;
  const int d = max(t.nph, t.nhp);
  if (t.nhp <= 4) ringbf_thin(t, (float2 *)S);
  else if (t.nph <= 4) ringbf_flat(t, (double2 *)S);
  else if (d <= 64) ringbf_tile<4, 2, 1, 2>(t, S);
  else if (d <= 128) ringbf_tile<8, 1, 1, 4>(t, S);
  else ringbf_tile<8, 1, 2, 1>(t, S);
}

int ringbf_columns(int nph, int nhp) {   // columns of a tile, 0: channel too large for the kernel
  const int d = std::max(nph, nhp);
  if (nph <= 4 || nhp <= 4) return nhp;
  return d <= 128 ? 64 : d <= 256 ? 16 : 0;
}
void launch_ringbf(const RingTile32 *tiles, int ntiles, const SolveDesc *dd, hipStream_t st) {
  if (ntiles > 0) hipLaunchKernelGGL(k_ringbf, dim3(ntiles), dim3(512), 0, st, tiles, dd);
}
void launch_x64(const ZTile *tiles, int ntiles, const SolveDesc *dd, hipStream_t st) {
  if (ntiles > 0) hipLaunchKernelGGL(k_x64, dim3(ntiles), dim3(256), 0, st, tiles, dd);
}
void launch_hh64(const ZTile *tiles, int ntiles, const SolveDesc *dd, hipStream_t st) {
  if (ntiles > 0) hipLaunchKernelGGL(k_hh64, dim3(ntiles), dim3(256), 0, st, tiles, dd);
}

}  // namespace ccgpu
