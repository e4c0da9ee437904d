// Device-side descriptors shared by the kernels and the host runtime.
#pragma once
#include "interaction.h"
#include <hip/hip_runtime.h>
#include <cstdint>

namespace ccgpu {

// Ordered pair reference packed for the device: ch = channel (-1 absent),
// v = idx * 2 + (sign < 0).
struct DPair {
  int ch;
  int v;
};

// Up to four pairs of one list whose states differ in spin only: a state of each, and
// the places at[2 s + t] of the pairs with spins s, t (0 down, 1 up), -1 absent.
struct PairGroup {
  int a, b, at[4];
};
// the pair groups of a list, channel by channel
struct PairGroups {
  const PairGroup *g;
  const int64_t *off;   // channels + 1
  int max;              // most groups of a channel
};

// Everything one solve's kernels read or write.  All pointers are device
// pointers; arrays indexed by unique amplitude u have length nT.
struct SolveDesc {
  int A, nsp, np, nch, nphc;
  int64_t nT;
  int active;  // 0: converged, kernels skip this solve
  // orbitals
  const double *kx, *ky, *kz, *e;
  const int *nx, *ny, *nz, *sz, *tz, *partner;
  // channels
  const int *t_ch, *npp, *nhh;
  const int64_t *off_t, *off_pp, *off_hh, *off_vpp, *off_vhh;
  const int *pp_a, *pp_b, *hh_i, *hh_j;
  PairGroups gpp, ghh, ghp, gph;   // of the lists above and below, (hole, particle) in the last two
  // per unique amplitude its orbitals a | b << 16 | i << 32 | j << 48
  const uint64_t *lab;
  const int *ob_rowB, *ob_rowA, *ob_colJ, *ob_colI;
  // I6 by rows: channel of each unique pp row, CSR lists of partials per particle
  int64_t nrows;
  const int *row_ch;
  const int *i6_dptr, *i6_didx, *i6_optr, *i6_oidx;
  double2 *p6;
  const DPair *ppref, *hhref;
  // parity image of each orbital, n -> -n (null unless the lattice maps onto
  // itself with k -> -k bit for bit and holes onto holes): the 3NF fill of
  // V_pppp evaluates one element of each parity pair
  const int *pimg;
  // Pandya
  const int *nph, *nhp;
  const int64_t *off_ph, *off_hp, *off_i4, *off_vt, *off_w1;
  const int *ph_a, *ph_i, *hp_j, *hp_b;
  // two ring positions per unique amplitude, and their second ones in channels that
  // pair with themselves (-1 elsewhere; null: no such channel)
  const int *ring2, *ring2b;
  // amplitudes and blocks
  double2 *T, *R, *R0, *Vhhpp, *Vhhhh, *X, *Vpppp;
  double2 *Rh;   // hh ladder T I9 of the residual, added to R by its closing pass
  float2 *Vpppp32;
  double2 *Tt, *Rt, *I4, *W0, *W1, *Vt;
  // FP32 ring blocks of the BF16x3 residual (null until the FP32 copies are
  // made): T~, R~, I4 per iteration, V~, W0 and W1 copied from the FP64 blocks
  float2 *Tt32, *Rt32, *I4_32, *W0_32, *W1_32, *Vt32;
  // T as the BF16x3 pp ladder's B operand, split once per residual: per
  // amplitude the bf16 hi and lo pairs of (re, -im) and of (im, re)
  uint4 *Tbf;
  // one-body
  double2 *fdiag, *fpart;   // f(p,p) and f(p,partner(p))
  double2 *dh, *I7off, *dp, *I6off;
  double2 *e0;              // device E0
  // DIIS history (depth x nT) and reductions.  With the Anderson update hist
  // holds the mixed iterates y_j = T_j + beta f_j and histf the residual
  // vectors f_j = R_j/D_j - T_j in FP32 (for the Gram matrix only).
  double2 *hist;
  float2 *histf;
  double2 *red;             // reduction partials
};

// What one iteration of the solve loop tells the kernels about one solve,
// uploaded once per iteration.
struct IterCtrl {
  // T = sum_j c[j] hist[from[j]] over np columns opens the iteration; np = 0: T as it is
  int np, from[8];
  int fresh;          // the history column the update writes
  int m, held[8];     // Anderson: columns of the held vectors, oldest first
  double c[8], beta;
};

// One member of a grouped complex GEMM: C = alpha * A * B + beta * C0.
// With nsplit > 1 the K range is split over tiles that write raw partial
// products to P (nsplit blocks of M x N); k_splitk_reduce then forms C.
struct GemmGroup {
  const void *A;
  const double2 *B;
  double2 *C;
  const double2 *C0;
  double2 *P;
  int M, N, K;
  int lda, ldb, ldc, ldc0;
  int nsplit;
  int thin;   // runs the thin FP64 kernel in every precision
  double alpha, beta;
};

struct GemmTile {
  int g, m0, n0, ks;   // group, tile origin, split index
  int kb, ke, pad0, pad1;  // k range of this tile
};

// One tile of the FP64 X or hh-ladder contraction (contract.hip): 16 (X) or 64
// (hh) rows from m0 by nb <= 2 blocks of 16 columns from n0 of C = A B.  X also
// writes C2 = C + C0 (I9).
struct ZTile {
  const double2 *A, *B, *C0;
  double2 *C, *C2;
  int M, N, K, m0, n0, nb, solve, g;
  float cost;
};

constexpr int kRingClasses = 2;   // launches of the fused ring (ring64_class)

// Columns n0 .. of one Pandya channel pair's ring contractions (contract.hip)
template <class T>   // double2, or float2 for the FP32 blocks
struct RingTileOf {
  const T *Vt, *Tt, *W0, *W1;
  T *Rt;
  int nhp, nph, n0, solve, g;
  float cost;
};
typedef RingTileOf<double2> RingTile;
typedef RingTileOf<float2> RingTile32;

// A triple of hole groups I <= J <= K (a group: the up to two spin states of one
// momentum and isospin, in orbital order) of one (K3, Tz3) channel: its pair
// indices into the tables below and the spin combinations 4 is + 2 js + ks that
// are distinct states in canonical order.
struct T3Hole {
  int I, J, K, hij, hik, hjk, mask, pad;
};

// (T) channel tables and, for handed-over interactions, the open-addressing
// table of the <cb||kd> and <jk||lc> elements (key ((p*nsp+q)*nsp+r)*nsp+s,
// empty slots ~0, capacity a power of two at least twice the entries).
struct TriplesDesc {
  // channel lookup over (Tz3, K3): index = ((tz - tz0) * nk + (kx - k0)) * nk^2 + ...
  int k0, nk, tz0, ntz;
  const int *chan;        // dense table -> channel or -1
  const int *hptr;        // CSR over channels of hole triples
  const int *hijk;        // 3 ints per hole triple
  const int *orbitof;     // dense (n, sz, tz) -> orbital, -1 absent
  int nmax;
  const int *pair_a, *pair_b;  // every particle pair a<b (all momenta)
  int64_t npairs;
  const unsigned long long *vkeys;  // null: elements from the built-in generator
  const double2 *vvals;
  unsigned long long vmask;
  // built-in generator: radial factors of the three Minnesota Gaussians for
  // q^2 = (pi/L)^2 m, m = |n_p - n_q - n_r + n_s|^2 (twists cancel), 3 per m
  const double *mtab;
  int mmax;
  // built-in chiral NN (used when chiral != 0)
  int chiral;
  ChiralDev ch;
  // dense element tables (null: elements evaluated in place): vhppp holds
  // <cb||kd> at ((c-A) np + (b-A)) A + k, times 2 for the spin of d (d's
  // momentum and isospin follow from conservation); vhhhp holds <jk||lc> at
  // (j A + k) np + (c-A), times 2 for the spin of l
  const double2 *vhppp, *vhhhp;
  // Groups (k_triples_g): the two states of every particle and hole group
  // (orbital or -1), a particle group's momentum and isospin, and per orbital
  // 2 group + state.  Group triples of a channel: [gptr[ch], gptr[ch + 1]), with
  // f_i + f_j + f_k of their eight spin combinations in gf.
  int npg, nhg, nhp, ngtrip;     // groups, hole group pairs U <= V, group triples
  const int2 *pg, *hg;
  const int4 *pgn;
  const int *og;
  const int *gptr;
  const T3Hole *gtrip;
  double2 *gf;
  // Tables of the group kernel, 32-byte records of two elements, one per spin
  // state w of the group whose momentum and isospin conservation leaves:
  //   gE[((pair(y, z) 4 + 2 ys + zs) nhg + S) 2 + ss]: conj <yz||s w> where w is a
  //     particle, t(yz, s w) where it is a hole; pair(y, z) = y (y + 1) / 2 + z over
  //     particle groups y >= z, S the hole group of s
  //   gD[((x 2 + xs) nhp + pair(v, u)) 4 + 2 us + vs]: t(x w, u v) where w is a
  //     particle, conj <uv||w x> where it is a hole
  // The amplitude entries are refilled for every sum.
  double2 *gE, *gD;
  // 1: the lattice maps onto itself under n -> -n with k -> -k exactly (no
  // twist) and holes onto holes, so <cb||kd> = <Pc Pb||Pk Pd> (the NN and 3NF
  // elements are even under parity) and the table fill evaluates one of each
  // parity pair
  int parity;
  // normal-ordered 3NF in <cb||kd> (the reference adds it to vnn_hppp, not to
  // vnn_hhhp: ccm_iter.f90:1641-1690)
  int tnf;
  Chiral3Dev c3;
  // the antisymmetrized three-body element W3 = <abc||ijk> (chiral_3nf_asym)
  // of the CCDT-1 triples and of (T) at tnf_approx 3
  Chiral3Dev c3w;
};

// Warm-start network: number of parameters (flat FP32 vector, layout in
// mlp.hip) and the buffers of one training step: activations and pre-activation
// gradients of the minibatch in blocks of 64 samples (B samples, a multiple of 64).
constexpr int kMlpParamCount = 9473;
struct MlpTrainBufs {
  uint16_t *x1t, *h1t, *h2t, *h3t;   // 16 B, 64 B x 3
  uint16_t *dz1t, *dz2t, *dz3t;      // 64 B x 3
  float *g;                          // B: dL/dy
  float *loss_part;                  // [gridDim.x of the pass]
};

}  // namespace ccgpu
