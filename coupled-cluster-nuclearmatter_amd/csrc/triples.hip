// Perturbative triples (T) on the GPU: pert_triples2 (ccm_triples.f90:528-735)
// with three_body_oneparticle_1 / three_body_onehole_1 (ccm_triples.f90:174-294)
// and the (K3, Tz3) channels of setup_t3_channel_structures
// (ccm_t3full_channels.f90:4-284).
//
// E(T) = sum over channels, a<b<c and i<j<k of conj(W) W / D with
//   D = f_ii + f_jj + f_kk - f_aa - f_bb - f_cc            (diagonal Fock)
//   W = sum of 9 signed F terms - sum of 9 signed H terms
//   F(a,b,c,i,j,k) = sum_d conj(<cb||kd>) t(ad,ij),  n_d = n_i + n_j - n_a
//   H(a,b,c,i,j,k) = sum_l conj(<jk||lc>) t(ab,il),  n_l = n_k + n_j - n_c
// (d runs over the particle spin states of its momentum, l over the holes).
// The interaction elements are evaluated in place by the same generator that
// filled the V blocks, or, for handed-over interactions, read from a device
// hash table of the <cb||kd> (vnn_hppp) and <jk||lc> (vnn_hhhp) blocks.
//
// Work decomposition: one thread per particle triple (a<b<c): block x = the
// particle pair (a,b), threads stride over c.  A thread whose (K3,Tz3) has hole
// triples walks that channel's hole-triple list and accumulates its own sum in
// fixed order; blocks reduce with a fixed tree and a final pass adds the block
// partials in order, so the result is deterministic.
#include "device.h"
#include "interaction.h"

#include <algorithm>
#include <cstdlib>

namespace ccgpu {


__device__ __forceinline__ double minnesota_direct_t(const SolveDesc &d, double volume, int p, int q, int r, int s) {
  Orb o;
  o.kx = d.kx; o.ky = d.ky; o.kz = d.kz; o.sz = d.sz; o.tz = d.tz; o.volume = volume;
  return minnesota_direct(o, p, q, r, s);
}

__device__ __forceinline__ double2 tcmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

__device__ __forceinline__ int orb_lookup(const TriplesDesc &td, int nx, int ny, int nz, int sz, int tz) {
  const int n = 2 * td.nmax + 1;
  if (nx < -td.nmax || nx > td.nmax || ny < -td.nmax || ny > td.nmax || nz < -td.nmax || nz > td.nmax) return -1;
  if (tz < -1 || tz > 1 || (tz & 1) == 0) return -1;
  int idx = (((nx + td.nmax) * n + (ny + td.nmax)) * n + (nz + td.nmax)) * 4 + ((sz + 1) / 2) * 2 + (tz + 1) / 2;
  return td.orbitof[idx];
}

// amplitude t(ab,ij) for any ordering, 0 when absent
__device__ __forceinline__ double2 t_of(const SolveDesc &d, int a, int b, int i, int j) {
  if (a == b || i == j) return make_double2(0.0, 0.0);
  DPair p = d.ppref[(size_t)(a - d.A) * d.np + (b - d.A)];
  DPair h = d.hhref[(size_t)i * d.A + j];
  if (p.ch < 0 || p.ch != h.ch) return make_double2(0.0, 0.0);
  double2 t = d.T[d.off_t[p.ch] + (int64_t)(p.v >> 1) * d.nhh[p.ch] + (h.v >> 1)];
  double sg = (((p.v ^ h.v) & 1) ? -1.0 : 1.0);
  return make_double2(sg * t.x, sg * t.y);
}

// antisymmetrized element <pq||rs>: from the table of handed-over elements,
// else from the built-in generator (chiral, or Minnesota which is real)
__device__ __forceinline__ double2 vas_t(const SolveDesc &d, const TriplesDesc &td, double volume, int p, int q,
                                         int r, int s) {
  if (td.vkeys) {
    const unsigned long long n = (unsigned long long)d.nsp;
    const unsigned long long key = (((unsigned long long)p * n + q) * n + r) * n + s;
    unsigned long long h = key;
    h ^= h >> 33;
    h *= 0xff51afd7ed558ccdull;
    h ^= h >> 33;
    h &= td.vmask;
    // the table is at most half full, so an empty slot ends every probe
    for (;;) {
      const unsigned long long k = td.vkeys[h];
      if (k == key) return td.vvals[h];
      if (k == ~0ull) return make_double2(0.0, 0.0);
      h = (h + 1) & td.vmask;
    }
  }
  if (td.chiral) {
    const double2 a = chiral_direct(td.ch, d.nx, d.ny, d.nz, d.sz, d.tz, p, q, r, s);
    const double2 b = chiral_direct(td.ch, d.nx, d.ny, d.nz, d.sz, d.tz, p, q, s, r);
    return make_double2(a.x - b.x, a.y - b.y);
  }
  if (td.mtab) {
    const int ax = d.nx[p] - d.nx[q], ay = d.ny[p] - d.ny[q], az = d.nz[p] - d.nz[q];
    const int dx1 = ax - d.nx[r] + d.nx[s], dy1 = ay - d.ny[r] + d.ny[s], dz1 = az - d.nz[r] + d.nz[s];
    const int dx2 = ax - d.nx[s] + d.nx[r], dy2 = ay - d.ny[s] + d.ny[r], dz2 = az - d.nz[s] + d.nz[r];
    const int m1 = dx1 * dx1 + dy1 * dy1 + dz1 * dz1, m2 = dx2 * dx2 + dy2 * dy2 + dz2 * dz2;
    const int sp = d.sz[p], sq = d.sz[q], sr = d.sz[r], ss = d.sz[s];
    const int tp = d.tz[p], tq = d.tz[q], tr = d.tz[r], ts = d.tz[s];
    const double v = minnesota_direct_tab(td.mtab + 3 * m1, sp, sq, sr, ss, tp, tq, tr, ts, volume) -
                     minnesota_direct_tab(td.mtab + 3 * m2, sp, sq, ss, sr, tp, tq, ts, tr, volume);
    return make_double2(v, 0.0);
  }
  return make_double2(minnesota_direct_t(d, volume, p, q, r, s) - minnesota_direct_t(d, volume, p, q, s, r), 0.0);
}

// F(a,b,c,i,j,k) = sum_d conj(<cb||kd>) t(ad,ij)  (three_body_oneparticle_1);
// TAB: elements from the dense tables, else evaluated in place
template <bool TAB>
__device__ double2 f_term(const SolveDesc &d, const TriplesDesc &td, double vol, int a, int b, int c, int i, int j,
                          int k) {
  double2 s = make_double2(0.0, 0.0);
  const int nx = d.nx[i] + d.nx[j] - d.nx[a], ny = d.ny[i] + d.ny[j] - d.ny[a], nz = d.nz[i] + d.nz[j] - d.nz[a];
  const int tz = d.tz[i] + d.tz[j] - d.tz[a];
  const int64_t row = TAB ? ((int64_t)(c - d.A) * d.np + (b - d.A)) * d.A + k : 0;
  for (int sz = -1; sz <= 1; sz += 2) {
    int dd = orb_lookup(td, nx, ny, nz, sz, tz);
    if (dd < d.A) continue;
    const double2 t = t_of(d, a, dd, i, j);
    double2 v;   // conj(v) t
    if constexpr (TAB) v = td.vhppp[2 * row + (sz + 1) / 2];
    else v = vas_t(d, td, vol, c, b, k, dd);
    s.x += v.x * t.x + v.y * t.y;
    s.y += v.x * t.y - v.y * t.x;
  }
  return s;
}

// H(a,b,c,i,j,k) = sum_l conj(<jk||lc>) t(ab,il)  (three_body_onehole_1)
template <bool TAB>
__device__ double2 h_term(const SolveDesc &d, const TriplesDesc &td, double vol, int a, int b, int c, int i, int j,
                          int k) {
  double2 s = make_double2(0.0, 0.0);
  const int nx = d.nx[k] + d.nx[j] - d.nx[c], ny = d.ny[k] + d.ny[j] - d.ny[c], nz = d.nz[k] + d.nz[j] - d.nz[c];
  const int tz = d.tz[k] + d.tz[j] - d.tz[c];
  const int64_t row = TAB ? ((int64_t)j * d.A + k) * d.np + (c - d.A) : 0;
  for (int sz = -1; sz <= 1; sz += 2) {
    int l = orb_lookup(td, nx, ny, nz, sz, tz);
    if (l < 0 || l >= d.A) continue;
    const double2 t = t_of(d, a, b, i, l);
    double2 v;   // conj(v) t
    if constexpr (TAB) v = td.vhhhp[2 * row + (sz + 1) / 2];
    else v = vas_t(d, td, vol, j, k, l, c);
    s.x += v.x * t.x + v.y * t.y;
    s.y += v.x * t.y - v.y * t.x;
  }
  return s;
}

// Dense element tables for (T): every <cb||kd> (particles c, b, hole k, the
// particle d of either spin that conserves momentum and isospin) and every
// <jk||lc>, evaluated once by the same element source as the in-place path.
// <cb||kd> = -<bc||kd> (the NN element and the normal-ordered 3NF sum are
// both antisymmetric in the bra): the fill evaluates c < b and writes both
// entries, c = b is zero.  Grid stride over the half (c < b) only.
template <bool ONE>
__global__ __launch_bounds__(256) void k_t3_fill_hppp(SolveDesc d, TriplesDesc td, double vol, double2 *out) {
  const int np = d.np;
  const int64_t npair = (int64_t)np * (np - 1) / 2;   // c < b, in the order of pairs (b, c) with c < b
  const int64_t per = (int64_t)d.A * 2;
  const int64_t n = npair * per;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t q = e / per;
    const int rem = (int)(e - q * per);
    const int sd = (rem & 1) * 2 - 1, k = rem >> 1;
    // pair index q -> (c < b): b - A = largest x with x (x - 1) / 2 <= q
    int bx = (int)((1.0 + sqrt(1.0 + 8.0 * (double)q)) * 0.5);
    while ((int64_t)bx * (bx - 1) / 2 > q) --bx;
    while ((int64_t)(bx + 1) * bx / 2 <= q) ++bx;
    const int cx = (int)(q - (int64_t)bx * (bx - 1) / 2);
    const int b = bx + d.A, c = cx + d.A;
    // parity image (Pc, Pb, Pk): the element with the smaller (pair, k) key of
    // the two is evaluated and written to both places
    int pbx = -1, pcx = -1, pk = -1;
    if (td.parity) {
      const int ib = orb_lookup(td, -d.nx[b], -d.ny[b], -d.nz[b], d.sz[b], d.tz[b]) - d.A;
      const int ic = orb_lookup(td, -d.nx[c], -d.ny[c], -d.nz[c], d.sz[c], d.tz[c]) - d.A;
      pk = orb_lookup(td, -d.nx[k], -d.ny[k], -d.nz[k], d.sz[k], d.tz[k]);
      const int hi = max(ib, ic), lo = min(ib, ic);
      const int64_t qi = (int64_t)hi * (hi - 1) / 2 + lo;
      if (qi < q || (qi == q && pk < k)) continue;
      if (qi != q || pk != k) {
        pbx = ib;
        pcx = ic;
      }
    }
    const int dd = orb_lookup(td, d.nx[c] + d.nx[b] - d.nx[k], d.ny[c] + d.ny[b] - d.ny[k],
                              d.nz[c] + d.nz[b] - d.nz[k], sd, d.tz[c] + d.tz[b] - d.tz[k]);
    double2 v = make_double2(0.0, 0.0);
    if (dd >= d.A) {
      v = vas_t(d, td, vol, c, b, k, dd);
      if (td.tnf) {
        const double2 w = no2b_sum<ONE>(td.c3, d.A, c, b, k, dd);
        v.x += w.x;
        v.y += w.y;
      }
    }
    const int64_t tail = (int64_t)k * 2 + (sd + 1) / 2;
    out[((int64_t)cx * np + bx) * per + tail] = v;
    out[((int64_t)bx * np + cx) * per + tail] = make_double2(-v.x, -v.y);
    if (pbx >= 0) {
      const int64_t ptail = (int64_t)pk * 2 + (sd + 1) / 2;
      out[((int64_t)pcx * np + pbx) * per + ptail] = v;
      out[((int64_t)pbx * np + pcx) * per + ptail] = make_double2(-v.x, -v.y);
    }
  }
  // the diagonal c = b
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < (int64_t)np * per;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t x = e / per;
    out[(x * np + x) * per + (e - x * per)] = make_double2(0.0, 0.0);
  }
}

__global__ __launch_bounds__(256) void k_t3_fill_hhhp(SolveDesc d, TriplesDesc td, double vol, double2 *out) {
  const int64_t n = (int64_t)d.A * d.A * d.np * 2;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
    const int sl = (int)(e & 1) * 2 - 1;
    const int64_t r = e >> 1;
    const int c = (int)(r % d.np) + d.A;
    const int64_t jk = r / d.np;
    const int k = (int)(jk % d.A), j = (int)(jk / d.A);
    const int l = orb_lookup(td, d.nx[j] + d.nx[k] - d.nx[c], d.ny[j] + d.ny[k] - d.ny[c],
                             d.nz[j] + d.nz[k] - d.nz[c], sl, d.tz[j] + d.tz[k] - d.tz[c]);
    out[e] = (l >= 0 && l < d.A) ? vas_t(d, td, vol, j, k, l, c) : make_double2(0.0, 0.0);
  }
}

// The 18 signed terms of W (pert_triples2, ccm_triples.f90:611-700): kind
// (0 F, 1 H), sign, the particle order as indices into (a, b, c) and the hole
// order as indices into (i, j, k).
struct TermCode {
  signed char kind, sign, p0, p1, p2, h0, h1, h2;
};
__constant__ TermCode kTerms[18] = {
    {0, 1, 0, 1, 2, 0, 1, 2},  {0, -1, 1, 0, 2, 0, 1, 2}, {0, -1, 2, 1, 0, 0, 1, 2}, {0, -1, 0, 1, 2, 2, 1, 0},
    {0, -1, 0, 1, 2, 0, 2, 1}, {0, 1, 2, 1, 0, 0, 2, 1},  {0, 1, 2, 1, 0, 2, 1, 0},  {0, 1, 1, 0, 2, 0, 2, 1},
    {0, 1, 1, 0, 2, 2, 1, 0},  {1, -1, 0, 1, 2, 0, 1, 2}, {1, 1, 0, 2, 1, 0, 1, 2},  {1, 1, 2, 1, 0, 0, 1, 2},
    {1, 1, 0, 1, 2, 2, 1, 0},  {1, 1, 0, 1, 2, 1, 0, 2},  {1, -1, 2, 1, 0, 1, 0, 2}, {1, -1, 2, 1, 0, 2, 1, 0},
    {1, -1, 0, 2, 1, 1, 0, 2}, {1, -1, 0, 2, 1, 2, 1, 0}};

__device__ __forceinline__ int sel3(int s, int x0, int x1, int x2) { return s == 0 ? x0 : (s == 1 ? x1 : x2); }

__global__ __launch_bounds__(256) void k_triples(SolveDesc d, TriplesDesc td, double volume, double2 *partial,
                                                 unsigned long long *count) {
  __shared__ double sre[256], sim[256];
  __shared__ unsigned long long scnt[256];
  double re = 0.0, im = 0.0;
  unsigned long long nel = 0;
  for (int64_t pr = blockIdx.x; pr < td.npairs; pr += gridDim.x) {
    const int a = td.pair_a[pr], b = td.pair_b[pr];
    for (int c = b + 1 + threadIdx.x; c < d.nsp; c += blockDim.x) {
      const int kx = d.nx[a] + d.nx[b] + d.nx[c], ky = d.ny[a] + d.ny[b] + d.ny[c], kz = d.nz[a] + d.nz[b] + d.nz[c];
      const int tz = d.tz[a] + d.tz[b] + d.tz[c];
      const int ix = kx - td.k0, iy = ky - td.k0, iz = kz - td.k0, it = tz - td.tz0;
      if (ix < 0 || iy < 0 || iz < 0 || ix >= td.nk || iy >= td.nk || iz >= td.nk || it < 0 || it >= td.ntz) continue;
      const int ch = td.chan[((it * td.nk + ix) * td.nk + iy) * td.nk + iz];
      if (ch < 0) continue;
      const double fa = d.fdiag[a].x, fb = d.fdiag[b].x, fc = d.fdiag[c].x;
      const double fai = d.fdiag[a].y, fbi = d.fdiag[b].y, fci = d.fdiag[c].y;
      nel += (unsigned long long)(td.hptr[ch + 1] - td.hptr[ch]);
      for (int h = td.hptr[ch]; h < td.hptr[ch + 1]; ++h) {
        const int i = td.hijk[3 * h], j = td.hijk[3 * h + 1], k = td.hijk[3 * h + 2];
        double2 w = make_double2(0.0, 0.0);
        auto add = [&](double sg, double2 v) { w.x += sg * v.x; w.y += sg * v.y; };
        add(1, f_term<false>(d, td, volume, a, b, c, i, j, k));
        add(-1, f_term<false>(d, td, volume, b, a, c, i, j, k));
        add(-1, f_term<false>(d, td, volume, c, b, a, i, j, k));
        add(-1, f_term<false>(d, td, volume, a, b, c, k, j, i));
        add(-1, f_term<false>(d, td, volume, a, b, c, i, k, j));
        add(1, f_term<false>(d, td, volume, c, b, a, i, k, j));
        add(1, f_term<false>(d, td, volume, c, b, a, k, j, i));
        add(1, f_term<false>(d, td, volume, b, a, c, i, k, j));
        add(1, f_term<false>(d, td, volume, b, a, c, k, j, i));
        add(-1, h_term<false>(d, td, volume, a, b, c, i, j, k));
        add(1, h_term<false>(d, td, volume, a, c, b, i, j, k));
        add(1, h_term<false>(d, td, volume, c, b, a, i, j, k));
        add(1, h_term<false>(d, td, volume, a, b, c, k, j, i));
        add(1, h_term<false>(d, td, volume, a, b, c, j, i, k));
        add(-1, h_term<false>(d, td, volume, c, b, a, j, i, k));
        add(-1, h_term<false>(d, td, volume, c, b, a, k, j, i));
        add(-1, h_term<false>(d, td, volume, a, c, b, j, i, k));
        add(-1, h_term<false>(d, td, volume, a, c, b, k, j, i));
        // conj(W) W / D with complex D
        const double dre = d.fdiag[i].x + d.fdiag[j].x + d.fdiag[k].x - fa - fb - fc;
        const double dim = d.fdiag[i].y + d.fdiag[j].y + d.fdiag[k].y - fai - fbi - fci;
        const double ww = w.x * w.x + w.y * w.y;
        const double den = dre * dre + dim * dim;
        re += ww * dre / den;
        im += -ww * dim / den;
      }
    }
  }
  sre[threadIdx.x] = re;
  sim[threadIdx.x] = im;
  scnt[threadIdx.x] = nel;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) {
      sre[threadIdx.x] += sre[threadIdx.x + s];
      sim[threadIdx.x] += sim[threadIdx.x + s];
      scnt[threadIdx.x] += scnt[threadIdx.x + s];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    partial[blockIdx.x] = make_double2(sre[0], sim[0]);
    count[blockIdx.x] = scnt[0];
  }
}

// Table mode, one wave per particle triple: a block takes particle pairs
// (a,b), its four waves take c = b+1+wave, b+5+wave, ..., and the 64 lanes of
// a wave stride over the hole triples of that (K3,Tz3) channel.  Every lane of
// a wave reads the same <c.||..> and <..||.c> table rows (cache-friendly), and
// no lane waits for a longer hole-triple list than its wave's.  MODE as in
// k_triples_g.
template <int MODE, bool ONE>
__global__ __launch_bounds__(256) void k_triples_w(SolveDesc d, TriplesDesc td, double volume, double2 *partial,
                                                   unsigned long long *count) {
  __shared__ double sre[256], sim[256];
  __shared__ unsigned long long scnt[256];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double re = 0.0, im = 0.0;
  unsigned long long nel = 0;
  for (int64_t pr = blockIdx.x; pr < td.npairs; pr += gridDim.x) {
    const int a = td.pair_a[pr], b = td.pair_b[pr];
    for (int c = b + 1 + wave; c < d.nsp; c += 4) {
      const int kx = d.nx[a] + d.nx[b] + d.nx[c], ky = d.ny[a] + d.ny[b] + d.ny[c], kz = d.nz[a] + d.nz[b] + d.nz[c];
      const int tz = d.tz[a] + d.tz[b] + d.tz[c];
      const int ix = kx - td.k0, iy = ky - td.k0, iz = kz - td.k0, it = tz - td.tz0;
      if (ix < 0 || iy < 0 || iz < 0 || ix >= td.nk || iy >= td.nk || iz >= td.nk || it < 0 || it >= td.ntz) continue;
      const int ch = td.chan[((it * td.nk + ix) * td.nk + iy) * td.nk + iz];
      if (ch < 0) continue;
      const double fa = d.fdiag[a].x, fb = d.fdiag[b].x, fc = d.fdiag[c].x;
      const double fai = d.fdiag[a].y, fbi = d.fdiag[b].y, fci = d.fdiag[c].y;
      const int h0 = td.hptr[ch], h1 = td.hptr[ch + 1];
      if (lane == 0) nel += (unsigned long long)(h1 - h0);
      Nucleon na, nb, nc;
      double reg = 0.0;
      if constexpr (MODE != 0) {
        na = nucleon_of(td.c3w, a);
        nb = nucleon_of(td.c3w, b);
        nc = nucleon_of(td.c3w, c);
        reg = freg3(td.c3w, na.k, nb.k, nc.k);
      }
      for (int h = h0 + lane; h < h1; h += 64) {
        const int i = td.hijk[3 * h], j = td.hijk[3 * h + 1], k = td.hijk[3 * h + 2];
        double2 w = make_double2(0.0, 0.0);
#pragma unroll 1
        for (int t = 0; t < (MODE == 2 ? 0 : 18); ++t) {
          const TermCode tc = kTerms[t];
          const int x = sel3(tc.p0, a, b, c), y = sel3(tc.p1, a, b, c), z = sel3(tc.p2, a, b, c);
          const int u = sel3(tc.h0, i, j, k), v = sel3(tc.h1, i, j, k), q = sel3(tc.h2, i, j, k);
          const double2 f = tc.kind == 0 ? f_term<true>(d, td, volume, x, y, z, u, v, q)
                                         : h_term<true>(d, td, volume, x, y, z, u, v, q);
          w.x += (double)tc.sign * f.x;
          w.y += (double)tc.sign * f.y;
        }
        const double dre = d.fdiag[i].x + d.fdiag[j].x + d.fdiag[k].x - fa - fb - fc;
        const double dim = d.fdiag[i].y + d.fdiag[j].y + d.fdiag[k].y - fai - fbi - fci;
        const double den = dre * dre + dim * dim;
        double nre = w.x * w.x + w.y * w.y, nim = 0.0;
        if constexpr (MODE != 0) {
          const double2 w3 = chiral3_asym<ONE>(td.c3w, reg, na, nb, nc, nucleon_of(td.c3w, i), nucleon_of(td.c3w, j),
                                               nucleon_of(td.c3w, k));
          const double xr = w3.x + w.x, xi = w3.y + w.y;
          nre = MODE == 3 ? xr * xr + xi * xi : xr * w3.x + xi * w3.y;
          if constexpr (MODE == 1) nim = xi * w3.x - xr * w3.y;
        }
        re += (nre * dre + nim * dim) / den;
        im += (nim * dre - nre * dim) / den;
      }
    }
  }
  sre[threadIdx.x] = re;
  sim[threadIdx.x] = im;
  scnt[threadIdx.x] = nel;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) {
      sre[threadIdx.x] += sre[threadIdx.x + s];
      sim[threadIdx.x] += sim[threadIdx.x + s];
      scnt[threadIdx.x] += scnt[threadIdx.x + s];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    partial[blockIdx.x] = make_double2(sre[0], sim[0]);
    count[blockIdx.x] = scnt[0];
  }
}

// Amplitude factor of every F term, t(x d, u v) for each particle x, ordered
// hole pair (u, v) and both spins of the particle d that conserves momentum
// and isospin (zero where d is a hole or absent): out[((x - A) A + u) A + v]
// holds the two spins side by side.  Rebuilt from T for every (T) sum.
__global__ __launch_bounds__(256) void k_t3_fill_td(SolveDesc d, TriplesDesc td, double2 *out) {
  const int64_t n = (int64_t)d.np * d.A * d.A * 2;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
    const int sd = (int)(e & 1) * 2 - 1;
    const int64_t r = e >> 1;
    const int v = (int)(r % d.A), u = (int)((r / d.A) % d.A);
    const int x = (int)(r / ((int64_t)d.A * d.A)) + d.A;
    const int dd = orb_lookup(td, d.nx[u] + d.nx[v] - d.nx[x], d.ny[u] + d.ny[v] - d.ny[x],
                              d.nz[u] + d.nz[v] - d.nz[x], sd, d.tz[u] + d.tz[v] - d.tz[x]);
    out[e] = dd >= d.A ? t_of(d, x, dd, u, v) : make_double2(0.0, 0.0);
  }
}

// (T) from the element tables with the amplitudes staged: the same sum, terms
// and order as k_triples_w<0> (the same bits), with fewer gathers per
// element.  A wave's particle triple (a,b,c) fixes the three particle pairs
// (a,b), (a,c), (c,b) of the H terms: their rows of T (one per pair, the hole
// pairs of its channel) are copied into the wave's slice of LDS, and an H term
// reads t(xy, u l) there at the column of the hole pair (u, l).  The F terms
// read t(x d, u v) for both spins of d from the table above (one 32-byte
// load instead of the momentum lookup and three index loads per spin).
__device__ __forceinline__ void t3_wave_sync() {
  __builtin_amdgcn_s_waitcnt((15) | (3 << 14) | (7 << 4) | (0 << 8));   // lgkmcnt(0)
  __builtin_amdgcn_wave_barrier();
}

__global__ __launch_bounds__(256) void k_triples_s(SolveDesc d, TriplesDesc td, const double2 *__restrict__ tdt,
                                                   int maxnhh, double2 *partial, unsigned long long *count) {
  extern __shared__ double2 t3rows[];   // 4 waves x 3 pairs x maxnhh
  __shared__ double sre[256], sim[256];
  __shared__ unsigned long long scnt[256];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double2 *rows = t3rows + (int64_t)wave * 3 * maxnhh;
  const int A = d.A, np = d.np;
  double re = 0.0, im = 0.0;
  unsigned long long nel = 0;
  for (int64_t pr = blockIdx.x; pr < td.npairs; pr += gridDim.x) {
    const int a = td.pair_a[pr], b = td.pair_b[pr];
    for (int c = b + 1 + wave; c < d.nsp; c += 4) {
      const int kx = d.nx[a] + d.nx[b] + d.nx[c], ky = d.ny[a] + d.ny[b] + d.ny[c], kz = d.nz[a] + d.nz[b] + d.nz[c];
      const int tz = d.tz[a] + d.tz[b] + d.tz[c];
      const int ix = kx - td.k0, iy = ky - td.k0, iz = kz - td.k0, it = tz - td.tz0;
      if (ix < 0 || iy < 0 || iz < 0 || ix >= td.nk || iy >= td.nk || iz >= td.nk || it < 0 || it >= td.ntz) continue;
      const int ch = td.chan[((it * td.nk + ix) * td.nk + iy) * td.nk + iz];
      if (ch < 0) continue;
      const int h0 = td.hptr[ch], h1 = td.hptr[ch + 1];
      if (lane == 0) nel += (unsigned long long)(h1 - h0);
      // the pairs (a,b), (a,c), (c,b): channel, row, orientation; their rows
      int pch[3], psg[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        const int x = p == 2 ? c : a, y = p == 0 ? b : (p == 1 ? c : b);
        const DPair q = d.ppref[(size_t)(x - A) * np + (y - A)];
        pch[p] = q.ch;
        psg[p] = q.v & 1;
        if (q.ch >= 0) {
          const int nh = d.nhh[q.ch];
          const double2 *src = d.T + d.off_t[q.ch] + (int64_t)(q.v >> 1) * nh;
          for (int col = lane; col < nh; col += 64) rows[p * maxnhh + col] = src[col];
        }
      }
      t3_wave_sync();
      const double fa = d.fdiag[a].x, fb = d.fdiag[b].x, fc = d.fdiag[c].x;
      const double fai = d.fdiag[a].y, fbi = d.fdiag[b].y, fci = d.fdiag[c].y;
      for (int h = h0 + lane; h < h1; h += 64) {
        const int i = td.hijk[3 * h], j = td.hijk[3 * h + 1], k = td.hijk[3 * h + 2];
        double2 w = make_double2(0.0, 0.0);
#pragma unroll 1
        for (int t = 0; t < 18; ++t) {
          const TermCode tc = kTerms[t];
          const int x = sel3(tc.p0, a, b, c), y = sel3(tc.p1, a, b, c), z = sel3(tc.p2, a, b, c);
          const int u = sel3(tc.h0, i, j, k), v = sel3(tc.h1, i, j, k), q = sel3(tc.h2, i, j, k);
          double2 f = make_double2(0.0, 0.0);
          if (tc.kind == 0) {
            // F = sum_d conj(<zy||qd>) t(x d, u v)
            const double2 *vv = td.vhppp + 2 * (((int64_t)(z - A) * np + (y - A)) * A + q);
            const double2 *tt = tdt + 2 * (((int64_t)(x - A) * A + u) * A + v);
#pragma unroll
            for (int sd = 0; sd < 2; ++sd) {
              const double2 vx = vv[sd], tx = tt[sd];
              f.x += vx.x * tx.x + vx.y * tx.y;
              f.y += vx.x * tx.y - vx.y * tx.x;
            }
          } else {
            // H = sum_l conj(<vq||lz>) t(xy, u l)
            const int slot = tc.p0 == 2 ? 2 : (tc.p1 == 1 ? 0 : 1);
            const int nx = d.nx[q] + d.nx[v] - d.nx[z], ny = d.ny[q] + d.ny[v] - d.ny[z];
            const int nz = d.nz[q] + d.nz[v] - d.nz[z], tl = d.tz[q] + d.tz[v] - d.tz[z];
            const double2 *vv = td.vhhhp + 2 * (((int64_t)v * A + q) * np + (z - A));
#pragma unroll
            for (int sd = 0; sd < 2; ++sd) {
              const int l = orb_lookup(td, nx, ny, nz, 2 * sd - 1, tl);
              if (l < 0 || l >= A) continue;
              double2 tx = make_double2(0.0, 0.0);
              const DPair hr = d.hhref[(size_t)u * A + l];
              if (pch[slot] >= 0 && hr.ch == pch[slot]) {
                tx = rows[slot * maxnhh + (hr.v >> 1)];
                if ((psg[slot] ^ hr.v) & 1) tx = make_double2(-tx.x, -tx.y);
              }
              const double2 vx = vv[sd];
              f.x += vx.x * tx.x + vx.y * tx.y;
              f.y += vx.x * tx.y - vx.y * tx.x;
            }
          }
          w.x += (double)tc.sign * f.x;
          w.y += (double)tc.sign * f.y;
        }
        const double dre = d.fdiag[i].x + d.fdiag[j].x + d.fdiag[k].x - fa - fb - fc;
        const double dim = d.fdiag[i].y + d.fdiag[j].y + d.fdiag[k].y - fai - fbi - fci;
        const double den = dre * dre + dim * dim;
        const double nre = w.x * w.x + w.y * w.y, nim = 0.0;
        re += (nre * dre + nim * dim) / den;
        im += (nim * dre - nre * dim) / den;
      }
      // the rows are overwritten for the next triple only after every lane read them
      t3_wave_sync();
    }
  }
  sre[threadIdx.x] = re;
  sim[threadIdx.x] = im;
  scnt[threadIdx.x] = nel;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) {
      sre[threadIdx.x] += sre[threadIdx.x + s];
      sim[threadIdx.x] += sim[threadIdx.x + s];
      scnt[threadIdx.x] += scnt[threadIdx.x + s];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    partial[blockIdx.x] = make_double2(sre[0], sim[0]);
    count[blockIdx.x] = scnt[0];
  }
}

// ---------------------------------------------------------------------------
// The group kernel: (T) and the CCDT-1 sums over spin groups.
//
// Momentum conservation acts on groups (the two spin states of one momentum and
// isospin), so a particle group triple and a hole group triple that conserve
// it are 8 x 8 elements (abc, ijk) that share every index.  The F and the H
// term of a particle x and a hole pair uv sum over the states d and l of the
// same momentum n_u + n_v - n_x: w, a particle in the F term and a hole in the H
// term.  With
//   E_a[s](w) = conj <cb||s w> (particle) or t(cb, s w) (hole); E_b, E_c likewise
//               with the pairs (c, a) and (b, a),
//   D_x[uv](w) = t(x w, u v) or conj <uv||w x>
// the 18 signed F and H terms (pert_triples2, ccm_triples.f90:611-700) are
//   W = sum over the splits (ij|k) - (ik|j) + (jk|i) of the three holes into
//       pair uv and single s of  E_a[s].D_a[uv] - E_b[s].D_b[uv] + E_c[s].D_c[uv],
// nine products of length two.  A lane takes one w and, for one hole group
// triple and one (as, bs), all 16 (cs, is, js, ks): per split 26 loads of 16
// bytes, two lanes to a record, for 192 FMAs, no index arithmetic per element.
// The two lanes then add up (each keeps eight elements).  A block takes a pair
// of particle groups (a, b) and lists the (c, hole group triple) items of its
// channels in LDS, eight items to a wave at a time, so no lane idles on a short
// channel.
//
// Bound: the L1's request rate (275 requests per 64 elements at 0.7 a clock and
// CU, most for 32 bytes), then FP64 issue (6 of 16.7 ms).  The kernel before
// gathered 36 x 16 bytes per element with a lookup for each: PNM A=66 |n_i|<=3
// (1.62e9 elements) 181 to 16.7 ms; with the d and l terms kept apart (64-byte
// records, one wave per particle group triple) it took 66 ms.
//
// With W3 = <abc||ijk> the antisymmetrized three-nucleon element
// (chiral_3nf_asym) and D = f_i + f_j + f_k - f_a - f_b - f_c, the sum over
// a<b<c, i<j<k is
//   MODE 0: |W|^2 / D                 (T), et_4
//   MODE 1: (W3 + W) conj(W3) / D     CCDT-1 energy of T3 = (W3 + W)/D
//           (t3_intermediate, ccm_t3_eqn.f90:1-192; t3_energy,
//           ccm_t3full_channels.f90:570-667)
//   MODE 2: |W3|^2 / D                CCDT-1 energy of the start T3 = W3/D
//           (setup_t3, ccm_t3full_channels.f90:291-567)
//   MODE 3: |W + W3|^2 / D            (T) at tnf_approx 3, et_5 (:656-722)
// The eight elements a lane keeps differ in is, js and ks only, so W3 takes its
// geometry once for them.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int slot_of(int2 g, int s) { return s ? g.y : g.x; }

// pair index t = y (y + 1) / 2 + z, z <= y
__device__ __forceinline__ void tri_yz(int64_t t, int &y, int &z) {
  int64_t x = (int64_t)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
  while (x * (x + 1) / 2 > t) --x;
  while ((x + 1) * (x + 2) / 2 <= t) ++x;
  y = (int)x;
  z = (int)(t - x * (x + 1) / 2);
}
__device__ __forceinline__ int64_t tri_at(int64_t y, int64_t z) { return y * (y + 1) / 2 + z; }

// an entry of gE: the orbitals of its record and the w of spin sd
struct T3E {
  int y, z, s, ys, zs, ss, S, d;
  int64_t gp;
};
__device__ __forceinline__ T3E t3_e_entry(const SolveDesc &d, const TriplesDesc &td, int64_t rec, int sd) {
  T3E e;
  e.ss = (int)(rec & 1);
  int64_t r = rec >> 1;
  e.S = (int)(r % td.nhg);
  r /= td.nhg;
  e.zs = (int)(r & 1);
  e.ys = (int)((r >> 1) & 1);
  e.gp = r >> 2;
  int gy, gz;
  tri_yz(e.gp, gy, gz);
  e.y = slot_of(td.pg[gy], e.ys);
  e.z = slot_of(td.pg[gz], e.zs);
  e.s = slot_of(td.hg[e.S], e.ss);
  e.d = -1;
  if (e.y >= 0 && e.z >= 0 && e.s >= 0 && e.y != e.z)
    e.d = orb_lookup(td, d.nx[e.y] + d.nx[e.z] - d.nx[e.s], d.ny[e.y] + d.ny[e.z] - d.ny[e.s],
                     d.nz[e.y] + d.nz[e.z] - d.nz[e.s], 2 * sd - 1, d.tz[e.y] + d.tz[e.z] - d.tz[e.s]);
  return e;
}

// conj <yz||s w> of every record and particle w: once per interaction.  The
// element is evaluated for the ascending orbital order of (y, z) and signed.
// With no twist one of each parity pair (n -> -n) is evaluated and written to
// both places.  A block lists the entries of its chunk that need evaluating
// (half or more conserve momentum with no particle w) and evaluates the list
// with full waves.
template <bool ONE>
__global__ __launch_bounds__(256) void k_t3_fill_ev(SolveDesc d, TriplesDesc td, double vol, int64_t nrec) {
  constexpr int kChunk = 4096;
  __shared__ int list[kChunk];
  __shared__ int cnt;
  const int64_t n = 2 * nrec;
  auto image = [&](const T3E &e, int64_t &rec, double &sg) {   // record of the parity image, its sign
    auto img = [&](int x) { return td.og[orb_lookup(td, -d.nx[x], -d.ny[x], -d.nz[x], d.sz[x], d.tz[x])]; };
    const int oy = img(e.y), oz = img(e.z), os = img(e.s);
    const bool keep = (oy >> 1) >= (oz >> 1);
    const int o1 = keep ? oy : oz, o2 = keep ? oz : oy;
    sg = keep ? 1.0 : -1.0;
    rec = ((tri_at(o1 >> 1, o2 >> 1) * 4 + 2 * (o1 & 1) + (o2 & 1)) * td.nhg + (os >> 1)) * 2 + (os & 1);
  };
  for (int64_t base = (int64_t)blockIdx.x * kChunk; base < n; base += (int64_t)gridDim.x * kChunk) {
    if (threadIdx.x == 0) cnt = 0;
    __syncthreads();
    for (int t = threadIdx.x; t < kChunk && base + t < n; t += 256) {
      const int64_t rec = (base + t) >> 1;
      const int sd = t & 1;
      const T3E e = t3_e_entry(d, td, rec, sd);
      if (e.d < d.A) {   // a hole's entry is the amplitude's
        if (e.d < 0) td.gE[2 * rec + sd] = make_double2(0.0, 0.0);
        continue;
      }
      if (td.parity) {
        int64_t ir;
        double sg;
        image(e, ir, sg);
        const int64_t igp = ir / ((int64_t)8 * td.nhg);
        const int iS = (int)((ir >> 1) % td.nhg);
        if (igp < e.gp || (igp == e.gp && iS < e.S)) continue;
      }
      list[atomicAdd(&cnt, 1)] = t;
    }
    __syncthreads();
    const int m = cnt;
    for (int q = threadIdx.x; q < m; q += 256) {
      const int64_t rec = (base + list[q]) >> 1;
      const int sd = list[q] & 1;
      const T3E e = t3_e_entry(d, td, rec, sd);
      const int lo = min(e.y, e.z), hi = max(e.y, e.z);
      double2 v = vas_t(d, td, vol, lo, hi, e.s, e.d);
      if (td.tnf) {
        const double2 w = no2b_sum<ONE>(td.c3, d.A, lo, hi, e.s, e.d);
        v.x += w.x;
        v.y += w.y;
      }
      const double s1 = e.y < e.z ? 1.0 : -1.0;
      v = make_double2(s1 * v.x, -s1 * v.y);   // conjugated
      td.gE[2 * rec + sd] = v;
      if (td.parity) {
        int64_t ir;
        double sg;
        image(e, ir, sg);
        const int64_t igp = ir / ((int64_t)8 * td.nhg);
        const int iS = (int)((ir >> 1) % td.nhg);
        if (igp != e.gp || iS != e.S) td.gE[2 * ir + sd] = make_double2(sg * v.x, sg * v.y);
      }
    }
    __syncthreads();
  }
}

// t(yz, s w) of every record and hole w
__global__ __launch_bounds__(256) void k_t3_fill_et(SolveDesc d, TriplesDesc td, int64_t nrec) {
  for (int64_t rec = (int64_t)blockIdx.x * 256 + threadIdx.x; rec < nrec; rec += (int64_t)gridDim.x * 256) {
#pragma unroll
    for (int sl = 0; sl < 2; ++sl) {
      const T3E e = t3_e_entry(d, td, rec, sl);
      if (e.d >= 0 && e.d < d.A) td.gE[2 * rec + sl] = t_of(d, e.y, e.z, e.s, e.d);
    }
  }
}

// gD: T false conj <uv||w x> of the holes w (once per interaction; zero where
// there is no w), true t(x w, u v) of the particles w
template <bool T>
__global__ __launch_bounds__(256) void k_t3_fill_d(SolveDesc d, TriplesDesc td, double vol, int64_t nrec) {
  for (int64_t rec = (int64_t)blockIdx.x * 256 + threadIdx.x; rec < nrec; rec += (int64_t)gridDim.x * 256) {
    const int vs = (int)(rec & 1), us = (int)((rec >> 1) & 1);
    const int64_t r = rec >> 2;
    const int gx = (int)(r / td.nhp);
    int gu, gv;
    tri_yz(r - (int64_t)gx * td.nhp, gv, gu);
    const int x = slot_of(td.pg[gx >> 1], gx & 1), u = slot_of(td.hg[gu], us), v = slot_of(td.hg[gv], vs);
#pragma unroll
    for (int sp = 0; sp < 2; ++sp) {
      int w = -1;
      if (x >= 0 && u >= 0 && v >= 0 && u != v)
        w = orb_lookup(td, d.nx[u] + d.nx[v] - d.nx[x], d.ny[u] + d.ny[v] - d.ny[x],
                       d.nz[u] + d.nz[v] - d.nz[x], 2 * sp - 1, d.tz[u] + d.tz[v] - d.tz[x]);
      if (T) {
        if (w >= d.A) td.gD[2 * rec + sp] = t_of(d, x, w, u, v);
      } else if (w < d.A) {
        double2 o = make_double2(0.0, 0.0);
        if (w >= 0) {
          o = vas_t(d, td, vol, u, v, w, x);
          o.y = -o.y;
        }
        td.gD[2 * rec + sp] = o;
      }
    }
  }
}

// f_i + f_j + f_k of the hole group triples' states
__global__ __launch_bounds__(256) void k_t3_fill_gf(SolveDesc d, TriplesDesc td) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e >= 8 * td.ngtrip) return;
  const T3Hole t = td.gtrip[e >> 3];
  double2 f = make_double2(0.0, 0.0);
  if ((t.mask >> (e & 7)) & 1) {
    const int i = slot_of(td.hg[t.I], (e >> 2) & 1), j = slot_of(td.hg[t.J], (e >> 1) & 1),
              k = slot_of(td.hg[t.K], e & 1);
    f = make_double2(d.fdiag[i].x + d.fdiag[j].x + d.fdiag[k].x, d.fdiag[i].y + d.fdiag[j].y + d.fdiag[k].y);
  }
  td.gf[e] = f;
}

__device__ __forceinline__ void cmac(double2 &a, const double2 &e, const double2 &x) {
  a.x = fma(e.x, x.x, a.x);
  a.x = fma(-e.y, x.y, a.x);
  a.y = fma(e.x, x.y, a.y);
  a.y = fma(e.y, x.x, a.y);
}
__device__ __forceinline__ void cmac_neg(double2 &a, const double2 &e, const double2 &x) {
  a.x = fma(-e.x, x.x, a.x);
  a.x = fma(e.y, x.y, a.x);
  a.y = fma(-e.x, x.y, a.y);
  a.y = fma(-e.y, x.x, a.y);
}
// One split of the hole triple: SP 0 (ij|k), 1 (ik|j) with the minus sign, 2
// (jk|i).  acc[8 cs + 4 is + 2 js + ks]; pointers at the lane's component.
template <int SP>
__device__ __forceinline__ void t3_split(double2 (&acc)[16], const double2 *Da, const double2 *Db, const double2 *Dc0,
                                         const double2 *Dc1, const double2 *Ea0, const double2 *Ea1,
                                         const double2 *Eb0, const double2 *Eb1, const double2 *Ec) {
  double2 da[4], db[4], dc[2][4], ea[2][2], eb[2][2], ec[2];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    da[q] = Da[2 * q];
    db[q] = Db[2 * q];
    dc[0][q] = Dc0[2 * q];
    dc[1][q] = Dc1[2 * q];
  }
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    ea[0][s] = Ea0[2 * s];
    ea[1][s] = Ea1[2 * s];
    eb[0][s] = Eb0[2 * s];
    eb[1][s] = Eb1[2 * s];
    ec[s] = Ec[2 * s];
  }
#pragma unroll
  for (int cs = 0; cs < 2; ++cs)
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int v = 0; v < 2; ++v)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const int o = 8 * cs + (SP == 0 ? 4 * u + 2 * v + s : SP == 1 ? 4 * u + 2 * s + v : 4 * s + 2 * u + v);
          const int q = 2 * u + v;
          if (SP != 1) {
            cmac(acc[o], ea[cs][s], da[q]);
            cmac_neg(acc[o], eb[cs][s], db[q]);
            cmac(acc[o], ec[s], dc[cs][q]);
          } else {
            cmac_neg(acc[o], ea[cs][s], da[q]);
            cmac(acc[o], eb[cs][s], db[q]);
            cmac_neg(acc[o], ec[s], dc[cs][q]);
          }
        }
}

// value of the neighbouring lane (lane ^ 1)
__device__ __forceinline__ double pair_swap(double x) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_mov_dpp((int)b, 0xB1, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), 0xB1, 0xF, 0xF, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

constexpr int kT3Items = 2048;

// Order of the pairs (a, b) of particle groups, a <= b: tiles of 2 a by 4 b, a
// tile at a time to the blocks that an XCD runs together (workgroup i runs on
// XCD i mod 8), so that they share rows of the tables: (T) of PNM A=66
// |n_i|<=3 25.6 to 16.7 ms (tiles of 4 x 8 the same, 8 x 16 18.0 ms and slower on
// smaller lattices).  Tile t holds b in [4 tb, 4 tb + 4) and a in [2 ta, 2 ta +
// 2), t = tb (tb + 1) + ta.
constexpr int kTileA = 2, kTileB = 4, kTile = kTileA * kTileB;
__host__ __device__ inline int64_t t3_tile_ids(int npg) {   // virtual block indices, a multiple of 8
  const int64_t nb = (npg + kTileB - 1) / kTileB;
  return (nb * (nb + 1) + 7) / 8 * 8 * kTile;
}
__device__ __forceinline__ bool t3_tile_pair(int64_t v, int npg, int &ga, int &gb) {
  const int64_t s = v >> 3;
  const int64_t t = s / kTile * 8 + (v & 7);
  const int p = (int)(s % kTile);
  int64_t tb = (int64_t)((sqrt(4.0 * (double)t + 1.0) - 1.0) * 0.5);
  while (tb * (tb + 1) > t) --tb;
  while ((tb + 1) * (tb + 2) <= t) ++tb;
  gb = (int)tb * kTileB + p / kTileA;
  ga = (int)(t - tb * (tb + 1)) * kTileA + p % kTileA;
  return gb < npg && ga <= gb;
}
constexpr int t3_threads(int mode) { return mode == 0 ? 512 : 256; }   // W3 takes twice the registers

template <int MODE, bool ONE>
__global__ __launch_bounds__(t3_threads(MODE), 2) void k_triples_g(SolveDesc d, TriplesDesc td, double2 *partial,
                                                          unsigned long long *count) {
  constexpr int kT3Threads = t3_threads(MODE), kT3Waves = kT3Threads / 64;
  __shared__ int ic[kT3Items], ig[kT3Items];   // items: particle group c, hole group triple
  __shared__ int wsum[kT3Waves];
  __shared__ double sre[kT3Waves], sim[kT3Waves];
  __shared__ unsigned long long scnt[kT3Waves];
  __shared__ double2 stash[MODE == 0 || MODE == 2 ? 1 : 8][MODE == 0 || MODE == 2 ? 1 : kT3Threads];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int kk = lane & 1, as = (lane >> 1) & 1, bs = (lane >> 2) & 1, hq = lane >> 3;
  double re = 0.0, im = 0.0;
  unsigned long long nel = 0;
  const int64_t nid = t3_tile_ids(td.npg);
  const int64_t erow = (int64_t)td.nhg * 4, drow = (int64_t)td.nhp * 8;   // double2 per (pair, ys, zs) and per x
  for (int64_t id = blockIdx.x; id < nid; id += gridDim.x) {
    int gb, ga;
    if (!t3_tile_pair(id, td.npg, ga, gb)) continue;
    const int a = slot_of(td.pg[ga], as), b = slot_of(td.pg[gb], bs);
    const int4 ma = td.pgn[ga], mb_ = td.pgn[gb];
    const bool ab_ok = a >= 0 && b >= 0 && (ga != gb || (as == 0 && bs == 1));
    const double2 *Ec = nullptr, *Da = nullptr, *Db = nullptr;
    if constexpr (MODE != 2) {
      Ec = td.gE + (tri_at(gb, ga) * 4 + 2 * bs + as) * erow + kk;
      Da = td.gD + (int64_t)(2 * ga + as) * drow + kk;
      Db = td.gD + (int64_t)(2 * gb + bs) * drow + kk;
    }
    for (int c0 = gb; c0 < td.npg; c0 += kT3Threads) {
      // items of this thread's c: the hole group triples of its channel
      int n = 0, g0 = 0;
      const int myc = c0 + tid;
      if (myc < td.npg && myc != ga) {   // three particles do not fit in two states
        const int4 mc = td.pgn[myc];
        const int ix = ma.x + mb_.x + mc.x - td.k0, iy = ma.y + mb_.y + mc.y - td.k0, iz = ma.z + mb_.z + mc.z - td.k0;
        const int it = ma.w + mb_.w + mc.w - td.tz0;
        if (ix >= 0 && iy >= 0 && iz >= 0 && ix < td.nk && iy < td.nk && iz < td.nk && it >= 0 && it < td.ntz) {
          const int ch = td.chan[((it * td.nk + ix) * td.nk + iy) * td.nk + iz];
          if (ch >= 0) {
            g0 = td.gptr[ch];
            n = td.gptr[ch + 1] - g0;
          }
        }
      }
      int pos = n;   // inclusive scan over the block
      for (int off = 1; off < 64; off <<= 1) {
        const int x = __shfl_up(pos, off);
        if (lane >= off) pos += x;
      }
      if (lane == 63) wsum[wave] = pos;
      __syncthreads();
      int total = 0;
      for (int w = 0; w < kT3Waves; ++w) {
        if (w < wave) pos += wsum[w];
        total += wsum[w];
      }
      pos -= n;
      for (int i0 = 0; i0 < total; i0 += kT3Items) {
        __syncthreads();   // the items before are done
        for (int q = max(0, i0 - pos); q < n && pos + q < i0 + kT3Items; ++q) {
          ic[pos + q - i0] = myc;
          ig[pos + q - i0] = g0 + q;
        }
        __syncthreads();
        const int m = min(kT3Items, total - i0);
        for (int q0 = 8 * wave; q0 < m; q0 += 8 * kT3Waves) {
          const int q = min(q0 + hq, m - 1);
          const int gc = ic[q], g = ig[q];
          const T3Hole t = td.gtrip[g];
          const int2 pc = td.pg[gc];
          // this lane finishes cs = kk
          const int c = kk ? pc.y : pc.x;
          const bool ok = q0 + hq < m && ab_ok && c >= 0 && (gb != gc || (kk == 1 && bs == 0));
          double2 w[8];
          if constexpr (MODE != 2) {
            const double2 *Ea0 = td.gE + (tri_at(gc, gb) * 4 + bs) * erow + kk, *Ea1 = Ea0 + 2 * erow;
            const double2 *Eb0 = td.gE + (tri_at(gc, ga) * 4 + as) * erow + kk, *Eb1 = Eb0 + 2 * erow;
            const double2 *Dc0 = td.gD + (int64_t)(2 * gc) * drow + kk, *Dc1 = Dc0 + drow;
            double2 acc[16];
#pragma unroll
            for (int o = 0; o < 16; ++o) acc[o] = make_double2(0.0, 0.0);
            t3_split<0>(acc, Da + 8 * t.hij, Db + 8 * t.hij, Dc0 + 8 * t.hij, Dc1 + 8 * t.hij, Ea0 + 4 * t.K,
                        Ea1 + 4 * t.K, Eb0 + 4 * t.K, Eb1 + 4 * t.K, Ec + 4 * t.K);
            t3_split<1>(acc, Da + 8 * t.hik, Db + 8 * t.hik, Dc0 + 8 * t.hik, Dc1 + 8 * t.hik, Ea0 + 4 * t.J,
                        Ea1 + 4 * t.J, Eb0 + 4 * t.J, Eb1 + 4 * t.J, Ec + 4 * t.J);
            t3_split<2>(acc, Da + 8 * t.hjk, Db + 8 * t.hjk, Dc0 + 8 * t.hjk, Dc1 + 8 * t.hjk, Ea0 + 4 * t.I,
                        Ea1 + 4 * t.I, Eb0 + 4 * t.I, Eb1 + 4 * t.I, Ec + 4 * t.I);
            // sum over the two w: lane kk keeps cs = kk
#pragma unroll
            for (int o = 0; o < 8; ++o) {
              const double2 x = kk ? acc[o] : acc[8 + o], y = kk ? acc[8 + o] : acc[o];
              w[o] = make_double2(y.x + pair_swap(x.x), y.y + pair_swap(x.y));
              if constexpr (MODE != 0) stash[o][tid] = w[o];
            }
          }
          if (!ok) continue;
          nel += (unsigned long long)__popc(t.mask);
          const double2 fabc = make_double2(d.fdiag[a].x + d.fdiag[b].x + d.fdiag[c].x,
                                            d.fdiag[a].y + d.fdiag[b].y + d.fdiag[c].y);
          auto finish = [&](int o, double nre, double nim) {
            const double2 fh = td.gf[8 * (int64_t)g + o];
            const double dre = fh.x - fabc.x, dim = fh.y - fabc.y;
            const double inv = 1.0 / (dre * dre + dim * dim);
            re += (nre * dre + nim * dim) * inv;
            im += (nim * dre - nre * dim) * inv;
          };
          if constexpr (MODE == 0) {
#pragma unroll
            for (int o = 0; o < 8; ++o)
              if ((t.mask >> o) & 1) finish(o, w[o].x * w[o].x + w[o].y * w[o].y, 0.0);
          } else {
            auto rep = [&](int2 s) { return nucleon_of(td.c3w, s.x >= 0 ? s.x : s.y); };
            const int2 hi = td.hg[t.I], hj = td.hg[t.J], hk = td.hg[t.K];
            const Nucleon ni = rep(hi), nj = rep(hj), nk = rep(hk);
            const Nucleon na = nucleon_of(td.c3w, a), nb = nucleon_of(td.c3w, b), nc = nucleon_of(td.c3w, c);
            Geo3 geo;
            geo3_transfer<0, 0>(td.c3w, geo, na, ni);
            geo3_transfer<0, 1>(td.c3w, geo, na, nj);
            geo3_transfer<0, 2>(td.c3w, geo, na, nk);
            geo3_transfer<1, 0>(td.c3w, geo, nb, ni);
            geo3_transfer<1, 1>(td.c3w, geo, nb, nj);
            geo3_transfer<1, 2>(td.c3w, geo, nb, nk);
            geo3_transfer<2, 0>(td.c3w, geo, nc, ni);
            geo3_transfer<2, 1>(td.c3w, geo, nc, nj);
            geo3_transfer<2, 2>(td.c3w, geo, nc, nk);
            const double f = freg3(td.c3w, na.k, nb.k, nc.k) * td.c3w.scale;
            geo.f[0] = f * freg3(td.c3w, nj.k, nk.k, ni.k);
            geo.f[1] = f * freg3(td.c3w, ni.k, nk.k, nj.k);
            geo.f[2] = f * freg3(td.c3w, ni.k, nj.k, nk.k);
            auto up = [&](int2 s) {   // bit s: the state's spin is up
              return (s.x >= 0 && d.sz[s.x] > 0 ? 1 : 0) | (s.y >= 0 && d.sz[s.y] > 0 ? 2 : 0);
            };
            const int ui = up(hi), uj = up(hj), uk = up(hk);
            const int mb[3] = {na.sz, nb.sz, nc.sz}, tb[3] = {na.tz, nb.tz, nc.tz}, tk[3] = {ni.tz, nj.tz, nk.tz};
#pragma unroll 1
            for (int o = 0; o < 8; ++o) {
              if (!((t.mask >> o) & 1)) continue;
              // the geometry changes for all the compiler knows: what asym3
              // derives from it stays inside the loop (hoisted, it spills)
#pragma unroll
              for (int x = 0; x < 3; ++x)
#pragma unroll
                for (int y = 0; y < 3; ++y) {
                  asm volatile("" : "+v"(geo.w[x][y]));
#pragma unroll
                  for (int z = 0; z < 3; ++z) asm volatile("" : "+v"(geo.q[x][y][z]));
                }
              const int mk[3] = {2 * ((ui >> (o >> 2)) & 1) - 1, 2 * ((uj >> ((o >> 1) & 1)) & 1) - 1,
                                 2 * ((uk >> (o & 1)) & 1) - 1};
              const double2 w3 = asym3<ONE, false>(td.c3w, geo, mb, mk, tb, tk);
              if constexpr (MODE == 2) {
                finish(o, w3.x * w3.x + w3.y * w3.y, 0.0);
              } else {
                const double2 wo = stash[o][tid];
                const double xr = w3.x + wo.x, xi = w3.y + wo.y;
                if constexpr (MODE == 1) finish(o, xr * w3.x + xi * w3.y, xi * w3.x - xr * w3.y);
                else finish(o, xr * xr + xi * xi, 0.0);
              }
            }
          }
        }
      }
      __syncthreads();   // wsum and the items
    }
  }
  // fixed-order sums: butterfly in the wave, then the waves
  for (int off = 32; off > 0; off >>= 1) {
    re += __shfl_xor(re, off);
    im += __shfl_xor(im, off);
    nel += __shfl_xor(nel, off);
  }
  if (lane == 0) {
    sre[wave] = re;
    sim[wave] = im;
    scnt[wave] = nel;
  }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < kT3Waves; ++w) {
      sre[0] += sre[w];
      sim[0] += sim[w];
      scnt[0] += scnt[w];
    }
    partial[blockIdx.x] = make_double2(sre[0], sim[0]);
    count[blockIdx.x] = scnt[0];
  }
}

// Sums of the blocks' partials and element counts
__global__ __launch_bounds__(256) void k_triples_final(const double2 *partial, const unsigned long long *count, int n,
                                                       double2 *out, unsigned long long *count_out) {
  __shared__ double sre[256], sim[256];
  __shared__ unsigned long long scnt[256];
  double re = 0.0, im = 0.0;
  unsigned long long c = 0;
  for (int p = threadIdx.x; p < n; p += 256) {
    re += partial[p].x;
    im += partial[p].y;
    c += count[p];
  }
  sre[threadIdx.x] = re;
  sim[threadIdx.x] = im;
  scnt[threadIdx.x] = c;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) {
      sre[threadIdx.x] += sre[threadIdx.x + s];
      sim[threadIdx.x] += sim[threadIdx.x + s];
      scnt[threadIdx.x] += scnt[threadIdx.x + s];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[0] = make_double2(sre[0], sim[0]);
    count_out[0] = scnt[0];
  }
}

void launch_t3_tables(const SolveDesc &d, const TriplesDesc &td, double volume, double2 *hppp, double2 *hhhp,
                      hipStream_t st) {
  if (td.tnf && !td.c3.one_species)
    hipLaunchKernelGGL(k_t3_fill_hppp<false>, dim3(8192), dim3(256), 0, st, d, td, volume, hppp);
  else
    hipLaunchKernelGGL(k_t3_fill_hppp<true>, dim3(8192), dim3(256), 0, st, d, td, volume, hppp);
  hipLaunchKernelGGL(k_t3_fill_hhhp, dim3(1024), dim3(256), 0, st, d, td, volume, hhhp);
}

void launch_t3_td(const SolveDesc &d, const TriplesDesc &td, double2 *tdt, hipStream_t st) {
  hipLaunchKernelGGL(k_t3_fill_td, dim3(4096), dim3(256), 0, st, d, td, tdt);
}

static int64_t t3_e_records(const TriplesDesc &td) {
  return (int64_t)td.npg * (td.npg + 1) / 2 * 4 * td.nhg * 2;
}
static int64_t t3_d_records(const TriplesDesc &td) { return (int64_t)td.npg * 2 * td.nhp * 4; }
static unsigned t3_grid(int64_t n, int64_t most) {
  return (unsigned)std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, most));
}

// The interaction halves of the group tables
void launch_t3_group_v(const SolveDesc &d, const TriplesDesc &td, double volume, hipStream_t st) {
  const int64_t ne = t3_e_records(td), nd = t3_d_records(td);
  const unsigned g = (unsigned)std::max<int64_t>(1, std::min<int64_t>((2 * ne + 4095) / 4096, 16384));
  if (td.tnf && !td.c3.one_species)
    hipLaunchKernelGGL(k_t3_fill_ev<false>, dim3(g), dim3(256), 0, st, d, td, volume, ne);
  else
    hipLaunchKernelGGL(k_t3_fill_ev<true>, dim3(g), dim3(256), 0, st, d, td, volume, ne);
  hipLaunchKernelGGL(k_t3_fill_d<false>, dim3(t3_grid(nd, 16384)), dim3(256), 0, st, d, td, volume, nd);
}

// Sum over the triples with the group kernel (modes above); the amplitude
// halves of the tables are refilled from the current T first.
void launch_triples_group(const SolveDesc &d, const TriplesDesc &td, double2 *partial, unsigned long long *count,
                          int nblocks, double2 *out, unsigned long long *count_out, hipStream_t st, int mode) {
  if (mode != 2) {
    const int64_t ne = t3_e_records(td), nd = t3_d_records(td);
    hipLaunchKernelGGL(k_t3_fill_et, dim3(t3_grid(ne, 16384)), dim3(256), 0, st, d, td, ne);
    hipLaunchKernelGGL(k_t3_fill_d<true>, dim3(t3_grid(nd, 16384)), dim3(256), 0, st, d, td, 0.0, nd);
  }
  if (td.ngtrip > 0)
    hipLaunchKernelGGL(k_t3_fill_gf, dim3((8 * td.ngtrip + 255) / 256), dim3(256), 0, st, d, td);
  const bool one = td.c3w.one_species != 0;
  // nblocks is a multiple of 8: a block's later pairs stay on its XCD
  const int nb = (int)std::max<int64_t>(1, std::min<int64_t>(t3_tile_ids(td.npg), nblocks));
  auto run = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(nb), dim3(t3_threads(mode)), 0, st, d, td, partial, count);
  };
  if (mode == 0) run(k_triples_g<0, true>);
  else if (mode == 1) run(one ? k_triples_g<1, true> : k_triples_g<1, false>);
  else if (mode == 2) run(one ? k_triples_g<2, true> : k_triples_g<2, false>);
  else run(one ? k_triples_g<3, true> : k_triples_g<3, false>);
  hipLaunchKernelGGL(k_triples_final, dim3(1), dim3(256), 0, st, partial, count, nb, out, count_out);
}

// The sum by one of the element-by-element kernels: 0 in place (no tables, mode 0
// alone), 1 the staged kernel (mode 0 alone), 3 the kernel that gathers every amplitude
void launch_triples(const SolveDesc &d, const TriplesDesc &td, double volume, double2 *partial,
                    unsigned long long *count, int nblocks, double2 *out, unsigned long long *count_out,
                    hipStream_t st, int variant, int mode, const double2 *tdt, int maxnhh) {
  const bool one = td.c3w.one_species != 0;
  auto run = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(nblocks), dim3(256), 0, st, d, td, volume, partial, count);
  };
  if (variant == 1) {
    const size_t lds = (size_t)4 * 3 * maxnhh * sizeof(double2);
    hipLaunchKernelGGL(k_triples_s, dim3(nblocks), dim3(256), lds, st, d, td, tdt, maxnhh, partial, count);
  } else if (variant == 0) {
    run(k_triples);
  } else if (mode == 0) {
    run(k_triples_w<0, true>);
  } else if (mode == 1) {
    run(one ? k_triples_w<1, true> : k_triples_w<1, false>);
  } else if (mode == 2) {
    run(one ? k_triples_w<2, true> : k_triples_w<2, false>);
  } else {
    run(one ? k_triples_w<3, true> : k_triples_w<3, false>);
  }
  hipLaunchKernelGGL(k_triples_final, dim3(1), dim3(256), 0, st, partial, count, nblocks, out, count_out);
}

}  // namespace ccgpu
