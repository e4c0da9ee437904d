// The built-in interaction generator shared by the block-fill kernels and the
// (T) kernel: the Minnesota potential in momentum space.
#pragma once
#include <hip/hip_runtime.h>

namespace ccgpu {

// ---------------------------------------------------------------------------
// Interaction: Minnesota potential in momentum space, vmom_minnesota
// (chiral_module_andreas_with_delta.f90:8980-9111).  The reference's
// default-real literals are reproduced as their float32 values.
// ---------------------------------------------------------------------------
struct Orb {
  const double *kx, *ky, *kz;
  const int *sz, *tz;
  double volume;
};

static __device__ __forceinline__ double sig_dot_sig(int m1, int m2, int m3, int m4) {
  // <m1 m2| s1.s2 |m3 m4> for m = +-1: m1*m2 on the diagonal, 2 for a spin exchange
  double r = 0.0;
  if (m1 == m3 && m2 == m4) r += (double)(m1 * m2);
  if (m1 == m4 && m2 == m3 && m1 != m2) r += 2.0;
  return r;
}

static __device__ __forceinline__ double minnesota_direct(const Orb &o, int p, int q, int r, int s) {
  const double PI = 3.14159265358979;
  const double v0r = 200.0, v0t = 178.0, v0s = (double)91.85f;
  const double kr = (double)1.487f, kt = (double)0.639f, ks = (double)0.465f;
  double qx = 0.5 * (o.kx[p] - o.kx[q]) - 0.5 * (o.kx[r] - o.kx[s]);
  double qy = 0.5 * (o.ky[p] - o.ky[q]) - 0.5 * (o.ky[r] - o.ky[s]);
  double qz = 0.5 * (o.kz[p] - o.kz[q]) - 0.5 * (o.kz[r] - o.kz[s]);
  double q2 = qx * qx + qy * qy + qz * qz;
  double pi15 = pow(PI, 1.5);
  double vr = v0r * pi15 * exp(-q2 / (4.0 * kr)) / pow(kr, 1.5);
  double vt = -v0t * pi15 * exp(-q2 / (4.0 * kt)) / pow(kt, 1.5);
  double vs = -v0s * pi15 * exp(-q2 / (4.0 * ks)) / pow(ks, 1.5);
  int m1 = o.sz[p], m2 = o.sz[q], m3 = o.sz[r], m4 = o.sz[s];
  int t1 = o.tz[p], t2 = o.tz[q], t3 = o.tz[r], t4 = o.tz[s];
  if (t1 + t2 != t3 + t4) return 0.0;
  double ds = (m1 == m3 && m2 == m4) ? 1.0 : 0.0;
  double dt = (t1 == t3 && t2 == t4) ? 1.0 : 0.0;
  double ss = sig_dot_sig(m1, m2, m3, m4);
  double tt = sig_dot_sig(t1, t2, t3, t4);
  vr = vr * (3.0 * ds * dt - tt * ds - ss * dt - tt * ss) / 8.0;
  vs = vs * (3.0 * ds * dt + tt * ds - 3.0 * ss * dt - tt * ss) / 16.0;
  vt = vt * (3.0 * ds * dt - 3.0 * tt * ds + ss * dt - tt * ss) / 16.0;
  return (vs + vr + vt) / o.volume;
}

// The same element with the radial factors read from a table over the integer
// momentum transfer m = |n_p - n_q - n_r + n_s|^2 (q = (pi/L) dn for every
// twist): rad[0..2] = v0 pi^1.5 exp(-q^2/(4 kappa)) / kappa^1.5 for the R, T
// and S Gaussians (the last two carry their minus sign).
static __device__ __forceinline__ double minnesota_direct_tab(const double *rad, int m1, int m2, int m3, int m4,
                                                              int t1, int t2, int t3, int t4, double volume) {
  if (t1 + t2 != t3 + t4) return 0.0;
  const double ds = (m1 == m3 && m2 == m4) ? 1.0 : 0.0;
  const double dt = (t1 == t3 && t2 == t4) ? 1.0 : 0.0;
  const double ss = sig_dot_sig(m1, m2, m3, m4);
  const double tt = sig_dot_sig(t1, t2, t3, t4);
  const double vr = rad[0] * (3.0 * ds * dt - tt * ds - ss * dt - tt * ss) / 8.0;
  const double vs = rad[2] * (3.0 * ds * dt + tt * ds - 3.0 * ss * dt - tt * ss) / 16.0;
  const double vt = rad[1] * (3.0 * ds * dt - 3.0 * tt * ds + ss * dt - tt * ss) / 16.0;
  return (vs + vr + vt) / volume;
}

// ---------------------------------------------------------------------------
// Interaction: the Delta-full chiral NN, chiral_NN_with_delta
// (chiral_module_andreas_with_delta.f90:6304-6668).  Every radial function
// depends on the momentum transfer only, q = (pi/L) dn with the integer
// dn = (n_p - n_q) - (n_r - n_s) (twists cancel), so the host tabulates them
// over m = |dn|^2; the regulator and the relativity factor split into one
// factor per side, tabulated over j = |n_p - n_q|^2.  The element is then a
// few table reads and the spin-isospin algebra.
// ---------------------------------------------------------------------------
constexpr int kChiralRad = 13;
enum ChiralSlot {
  kOpe0 = 0,  // one-pion exchange, neutral pion        (:1110-1124)
  kOpe1,      // charged pion
  kOpe2,      // average pion mass (LO)
  kWc,        // NLO 2PE + leading Delta: W_C, V_S, V_T, V_C, W_T, W_S (:6553-6598)
  kVs,
  kVt,
  kVc,
  kWt,
  kWs,
  kVc3,       // NNLO 2PE + Delta triangles: V_C, W_T, W_S (:6620-6658)
  kWt3,
  kWs3,
  kQ2         // q^2 as the contacts see it (1e-16 at q = 0 from NLO on)
};

struct ChiralDev {
  const double *rad;      // kChiralRad per m
  const double *side;     // 3 pair charges (pp, np, nn) x (jmax + 1)
  int jmax, order;
  double qunit;           // pi hbarc / L, MeV per unit of dn
  double scale;           // hbarc^3 / volume
  double cs[3], ct[3];    // LO contacts per pair charge
  double cnlo[7];         // NLO contacts
  double cg0[2], cg1[2];  // np isospin CG for T = 0, 1, index (1 - tz) / 2
};

// <mo| sigma.v |mi> for spin projections +-1
static __device__ __forceinline__ double2 pauli_dot(int mo, int mi, double vx, double vy, double vz) {
  if (mo == mi) return make_double2(mo > 0 ? vz : -vz, 0.0);
  return mo > 0 ? make_double2(vx, -vy) : make_double2(vx, vy);
}

static __device__ __forceinline__ double2 cmul_i(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// v(p,q,r,s) of the chiral NN in MeV, complex (the spin-orbit and tensor
// operators carry sigma_y); zero unless momentum and isospin are conserved.
static __device__ __forceinline__ double2 chiral_direct(const ChiralDev &c, const int *nx, const int *ny,
                                                       const int *nz, const int *sz, const int *tz, int p, int q,
                                                       int r, int s) {
  const int t1 = tz[p], t2 = tz[q], t3 = tz[r], t4 = tz[s];
  const int ax = nx[p] - nx[q], ay = ny[p] - ny[q], az = nz[p] - nz[q];
  const int bx = nx[r] - nx[s], by = ny[r] - ny[s], bz = nz[r] - nz[s];
  if (t1 + t2 != t3 + t4 || nx[p] + nx[q] != nx[r] + nx[s] || ny[p] + ny[q] != ny[r] + ny[s] ||
      nz[p] + nz[q] != nz[r] + nz[s])
    return make_double2(0.0, 0.0);
  const int dx = ax - bx, dy = ay - by, dz = az - bz;
  const double *R = c.rad + kChiralRad * (dx * dx + dy * dy + dz * dz);
  const int ch = (t1 + t2) / 2 + 1;
  const double f = c.side[ch * (c.jmax + 1) + ax * ax + ay * ay + az * az] *
                   c.side[ch * (c.jmax + 1) + bx * bx + by * by + bz * bz];
  const int m1 = sz[p], m2 = sz[q], m3 = sz[r], m4 = sz[s];
  const double dm = (m1 == m3 && m2 == m4) ? 1.0 : 0.0;
  const double dt = (t1 == t3 && t2 == t4) ? 1.0 : 0.0;
  const double ss = sig_dot_sig(m1, m2, m3, m4);
  const double tt = sig_dot_sig(t1, t2, t3, t4);
  const double u = c.qunit;
  const double qx = u * dx, qy = u * dy, qz = u * dz;
  const double2 sq = cmul_i(pauli_dot(m1, m3, qx, qy, qz), pauli_dot(m2, m4, qx, qy, qz));
  double2 v;
  if (c.order == 0) {
    // LO: (sigma1.q)(sigma2.q) OPE tau.tau + CS + CT sigma.sigma (np contacts)
    const double a = R[kOpe2] * tt;
    v = make_double2(sq.x * a + c.cs[1] * dm * dt + c.ct[1] * ss * dt, sq.y * a);
  } else {
    double wt1;
    if (t1 + t2 == 0) {
      const double a = c.cg0[(1 - t1) / 2] * c.cg0[(1 - t3) / 2], b = c.cg1[(1 - t1) / 2] * c.cg1[(1 - t3) / 2];
      wt1 = a * (-R[kOpe0] - 2.0 * R[kOpe1]) + b * (-R[kOpe0] + 2.0 * R[kOpe1]);
    } else {
      wt1 = R[kOpe0];
    }
    const double q2 = R[kQ2];
    const double kx = 0.5 * u * (ax + bx), ky = 0.5 * u * (ay + by), kz = 0.5 * u * (az + bz);
    const double k2 = kx * kx + ky * ky + kz * kz;
    // coefficients of the operator structures
    const double a_sq = wt1 + R[kVt] * dt + R[kWt] * tt + c.cnlo[5] * dt + R[kWt3] * tt;
    const double a_1 = c.cs[ch] * dm * dt + R[kVc] * dm * dt + R[kWc] * tt * dm +
                       (c.cnlo[0] * q2 + c.cnlo[1] * k2) * dm * dt + R[kVc3] * dm * dt;
    const double a_ss = (c.ct[ch] + R[kVs] + c.cnlo[2] * q2 + c.cnlo[3] * k2) * dt + (R[kWs] + R[kWs3]) * tt;
    v = make_double2(a_sq * sq.x + a_1 + a_ss * ss, a_sq * sq.y);
    if (dt != 0.0) {
      // C5 i/2 (sigma1 + sigma2).(k x q) and C7 (sigma1.k)(sigma2.k)
      const double wx = qy * kz - qz * ky, wy = qz * kx - qx * kz, wz = qx * ky - qy * kx;
      double2 so = make_double2(0.0, 0.0);
      if (m2 == m4) {
        const double2 e = pauli_dot(m1, m3, wx, wy, wz);
        so.x += e.x; so.y += e.y;
      }
      if (m1 == m3) {
        const double2 e = pauli_dot(m2, m4, wx, wy, wz);
        so.x += e.x; so.y += e.y;
      }
      // -i/2 so
      v.x += c.cnlo[4] * 0.5 * so.y;
      v.y -= c.cnlo[4] * 0.5 * so.x;
      const double2 kk = cmul_i(pauli_dot(m1, m3, kx, ky, kz), pauli_dot(m2, m4, kx, ky, kz));
      v.x += c.cnlo[6] * kk.x;
      v.y += c.cnlo[6] * kk.y;
    }
  }
  const double g = c.scale * f;
  return make_double2(g * v.x, g * v.y);
}

// What chiral_direct takes from the momenta and isospins of its four states alone, shared
// by the sixteen spin combinations (dt: isospins unchanged).
struct ChiralGeo {
  double asq, a1, ass, g;
  double qx, qy, qz, kx, ky, kz, wx, wy, wz;
  bool spin_orbit;
};

// a = n_p - n_q, b = n_r - n_s of a combination that conserves momentum and isospin
static __device__ __forceinline__ ChiralGeo chiral_geo(const ChiralDev &c, int ax, int ay, int az, int bx, int by,
                                                       int bz, int t1, int t2, int t3, int t4) {
  ChiralGeo o;
  const int dx = ax - bx, dy = ay - by, dz = az - bz;
  const double *R = c.rad + kChiralRad * (dx * dx + dy * dy + dz * dz);
  const int ch = (t1 + t2) / 2 + 1;
  const double f = c.side[ch * (c.jmax + 1) + ax * ax + ay * ay + az * az] *
                   c.side[ch * (c.jmax + 1) + bx * bx + by * by + bz * bz];
  const double dt = (t1 == t3 && t2 == t4) ? 1.0 : 0.0;
  const double tt = sig_dot_sig(t1, t2, t3, t4);
  const double u = c.qunit;
  o.qx = u * dx; o.qy = u * dy; o.qz = u * dz;
  o.g = c.scale * f;
  o.spin_orbit = false;
  o.kx = o.ky = o.kz = o.wx = o.wy = o.wz = 0.0;
  if (c.order == 0) {
    o.asq = R[kOpe2] * tt;
    o.a1 = c.cs[1] * dt;
    o.ass = c.ct[1] * dt;
    return o;
  }
  double wt1;
  if (t1 + t2 == 0) {
    const double a = c.cg0[(1 - t1) / 2] * c.cg0[(1 - t3) / 2], b = c.cg1[(1 - t1) / 2] * c.cg1[(1 - t3) / 2];
    wt1 = a * (-R[kOpe0] - 2.0 * R[kOpe1]) + b * (-R[kOpe0] + 2.0 * R[kOpe1]);
  } else {
    wt1 = R[kOpe0];
  }
  const double q2 = R[kQ2];
  o.kx = 0.5 * u * (ax + bx); o.ky = 0.5 * u * (ay + by); o.kz = 0.5 * u * (az + bz);
  const double k2 = o.kx * o.kx + o.ky * o.ky + o.kz * o.kz;
  o.asq = wt1 + R[kVt] * dt + R[kWt] * tt + c.cnlo[5] * dt + R[kWt3] * tt;
  o.a1 = c.cs[ch] * dt + R[kVc] * dt + R[kWc] * tt + (c.cnlo[0] * q2 + c.cnlo[1] * k2) * dt + R[kVc3] * dt;
  o.ass = (c.ct[ch] + R[kVs] + c.cnlo[2] * q2 + c.cnlo[3] * k2) * dt + (R[kWs] + R[kWs3]) * tt;
  o.spin_orbit = dt != 0.0;
  o.wx = o.qy * o.kz - o.qz * o.ky; o.wy = o.qz * o.kx - o.qx * o.kz; o.wz = o.qx * o.ky - o.qy * o.kx;
  return o;
}

// (sigma1.v)(sigma2.v) between spins that are constants after unrolling: the diagonal
// elements of sigma.v are real
static __device__ __forceinline__ double2 pauli_pair(int m1, int m2, int m3, int m4, double x, double y, double z) {
  const double2 a = pauli_dot(m1, m3, x, y, z), b = pauli_dot(m2, m4, x, y, z);
  if (m1 == m3 && m2 == m4) return make_double2(a.x * b.x, 0.0);
  if (m1 == m3) return make_double2(a.x * b.x, a.x * b.y);
  if (m2 == m4) return make_double2(a.x * b.x, a.y * b.x);
  return cmul_i(a, b);
}

// chiral_direct for spins m1 m2 | m3 m4
static __device__ __forceinline__ double2 chiral_spin(const ChiralDev &c, const ChiralGeo &o, int m1, int m2, int m3,
                                                      int m4) {
  const double2 sq = pauli_pair(m1, m2, m3, m4, o.qx, o.qy, o.qz);
  const double a1 = (m1 == m3 && m2 == m4) ? o.a1 : 0.0;
  double2 v = make_double2(o.asq * sq.x + a1 + o.ass * sig_dot_sig(m1, m2, m3, m4), o.asq * sq.y);
  if (o.spin_orbit) {
    double2 so = make_double2(0.0, 0.0);
    if (m2 == m4) {
      const double2 e = pauli_dot(m1, m3, o.wx, o.wy, o.wz);
      so.x += e.x; so.y += e.y;
    }
    if (m1 == m3) {
      const double2 e = pauli_dot(m2, m4, o.wx, o.wy, o.wz);
      so.x += e.x; so.y += e.y;
    }
    v.x += c.cnlo[4] * 0.5 * so.y;
    v.y -= c.cnlo[4] * 0.5 * so.x;
    const double2 kk = pauli_pair(m1, m2, m3, m4, o.kx, o.ky, o.kz);
    v.x += c.cnlo[6] * kk.x;
    v.y += c.cnlo[6] * kk.y;
  }
  return make_double2(o.g * v.x, o.g * v.y);
}

// ---------------------------------------------------------------------------
// The NNLO three-nucleon force, chiral_3nf_with_delta
// (chiral_module_andreas_with_delta.f90:6670-6902): cD and cE contacts,
// two-pion exchange with c1, c3, c4 shifted by the Delta (c3 - 4hA^2/9Delta,
// c4 + 2hA^2/9Delta), summed over the three choices of the middle nucleon, with
// the nonlocal regulator freg_3nfnonlocal (:3400-3423) on both sides.  The
// reference's default-real (2./3.) in the regulator is kept (float32 value).
// ---------------------------------------------------------------------------
struct Chiral3Dev {
  double econst, dconst;     // cE / (fpi^4 Lambda_chi), cD / (fpi^2 Lambda_chi)
  double k21;                // gA / (8 fpi^2)
  double c1t, c3f, c4f;      // -c1 gA^2/(4fpi^2) 4mpi^2/fpi^2, c3 gA^2/(4fpi^2) 2/fpi^2, c4 gA^2/(4fpi^2) 1/(2fpi^2)
  double mpi2;               // average pion mass squared
  double llambda;            // 4 cutoff^2
  double two_thirds;         // float32(2/3)
  double scale;              // hbarc^6 / volume^2
  int nexp;                  // regulator power
  int one_species;           // every orbital has the same tz (neutron matter)
  const double *kx, *ky, *kz;   // single-particle momenta, fm^-1
  const int *nx, *ny, *nz, *sz, *tz;
};

static __device__ __forceinline__ double freg3(const Chiral3Dev &c, const double *k1, const double *k2,
                                               const double *k3) {
  double q2 = 0.0;
  double pp = 0.0, qq = 0.0;
  for (int x = 0; x < 3; ++x) {
    const double p = 0.5 * (k1[x] - k2[x]);
    const double q = c.two_thirds * (k3[x] - 0.5 * (k1[x] + k2[x]));
    pp += p * p;
    qq += q * q;
  }
  q2 = 4.0 * pp + 3.0 * qq;
  const double r = q2 / c.llambda;
  double e = 1.0;
  for (int i = 0; i < c.nexp; ++i) e *= r;
  return exp(-e);
}

// ---------------------------------------------------------------------------
// The antisymmetrized element <abc||def> = sum over the six ket permutations
// (chiral_3nf_with_delta_asym, :6904-6917) of the direct element
// (chiral_3nf_with_delta, :6670-6902), in two parts.
//
// Geo3, what the momenta decide: the nine transfers q[x][y] from bra nucleon x
// to ket nucleon y, their pion propagators, and per choice z of the third
// nucleon's ket the regulators of both sides (the regulator is symmetric in
// its first two nucleons, so the six permutations need three).  asym3 then
// runs the spin-isospin algebra of the 18 (permutation, pair) terms.  Every
// quantity of the direct element thus is evaluated once per element instead of
// once per permutation, and the holes of one momentum share the geometry.
//
// Isospin: <ta|tau|td>.(<tb|tau|te> x <tc|tau|tf>) (chp_tau1_dot_tauXtau,
// :3544-3602) is imaginary and antisymmetric in its nucleons, so the difference
// that multiplies c4 is twice one of them; it vanishes unless exactly two
// nucleons exchange charge, and with one species (N1) always.
//
// FP64 issue bounds every kernel that sums these.  Against the six direct
// elements each evaluated in full (six regulators, 18 divisions, 36 general
// isospin products), SNM A=28 |n_i|<=2: V_pppp 10.2 to 1.54 ms, W0 4.75 to 0.63
// ms, V_hhpp 1.02 to 0.27 ms, the <cb||kd> table of (T) 15.2 to 4.7 ms.
// ---------------------------------------------------------------------------
struct Nucleon {
  double k[3];   // MeV
  int sz, tz;
};
static __device__ __forceinline__ Nucleon nucleon_of(const Chiral3Dev &c, int p) {
  const double hbarc = 197.326968;
  Nucleon o;
  o.k[0] = c.kx[p] * hbarc;
  o.k[1] = c.ky[p] * hbarc;
  o.k[2] = c.kz[p] * hbarc;
  o.sz = c.sz[p];
  o.tz = c.tz[p];
  return o;
}
// total momentum and isospin conserved
static __device__ __forceinline__ bool conserves3(const Chiral3Dev &c, int p, int q, int r, int s, int t, int u) {
  return c.tz[p] + c.tz[q] + c.tz[r] == c.tz[s] + c.tz[t] + c.tz[u] &&
         c.nx[p] + c.nx[q] + c.nx[r] == c.nx[s] + c.nx[t] + c.nx[u] &&
         c.ny[p] + c.ny[q] + c.ny[r] == c.ny[s] + c.ny[t] + c.ny[u] &&
         c.nz[p] + c.nz[q] + c.nz[r] == c.nz[s] + c.nz[t] + c.nz[u];
}

struct Geo3 {
  double q[3][3][3];
  double w[3][3];
  double f[3];   // bra regulator x ket regulator x scale; the caller multiplies the bra's in
};
template <int X, int Y>
static __device__ __forceinline__ void geo3_transfer(const Chiral3Dev &c, Geo3 &g, const Nucleon &bra,
                                                     const Nucleon &ket) {
  double q2 = 0.0;
#pragma unroll
  for (int x = 0; x < 3; ++x) {
    const double v = ket.k[x] - bra.k[x];
    g.q[X][Y][x] = v;
    q2 += v * v;
  }
  g.w[X][Y] = 1.0 / (q2 + c.mpi2);
}

// <mo| sigma.v |mi>, v in an array
static __device__ __forceinline__ double2 pauli_of(int mo, int mi, const double *v) {
  return pauli_dot(mo, mi, v[0], v[1], v[2]);
}

// ONE: one species; HH: the third nucleons of bra and ket are the same state
// (q[2][2] = 0, the normal-ordering sum), so terms in its one-pion exchange drop
template <bool ONE, bool HH>
static __device__ __forceinline__ double2 asym3(const Chiral3Dev &c, const Geo3 &g, const int (&mb)[3],
                                                const int (&mk)[3], const int (&tb)[3], const int (&tk)[3]) {
  double2 ope[3][3];
#pragma unroll
  for (int x = 0; x < 3; ++x)
#pragma unroll
    for (int y = 0; y < 3; ++y) {
      if (HH && x == 2 && y == 2) continue;
      const double2 s = pauli_of(mb[x], mk[y], g.q[x][y]);
      ope[x][y] = make_double2(g.w[x][y] * s.x, g.w[x][y] * s.y);
    }
  // the term of nucleons A -> a and B -> b with C -> cc as the spectator (or
  // the middle nucleon of the c4 part)
  auto pair = [&](int A, int a, int B, int b, int C, int cc) -> double2 {
    const bool za = HH && A == 2 && a == 2, zb = HH && B == 2 && b == 2;   // no pion at A (B)
    double2 r = make_double2(0.0, 0.0);
    double wt;
    if (ONE) wt = mb[C] == mk[cc] ? 1.0 : 0.0;
    else wt = mb[C] == mk[cc] && tb[C] == tk[cc] ? sig_dot_sig(tb[A], tb[B], tk[a], tk[b]) : 0.0;
    // 4 t_Z t_X: Z the nucleon that keeps its charge, X the next one
    int td = 0;
    if (!ONE && !za && !zb) {
      const bool fa = tb[A] != tk[a], fb = tb[B] != tk[b], fc = tb[C] != tk[cc];
      if (fa && fb && !fc) td = 4 * tb[C] * tb[A];
      else if (fb && fc && !fa) td = 4 * tb[A] * tb[B];
      else if (fa && fc && !fb) td = 4 * tb[B] * tb[C];
    }
    double2 oo = make_double2(0.0, 0.0);
    if (!za && !zb) oo = cmul_i(ope[A][a], ope[B][b]);
    if (wt != 0.0) {
      double2 in = make_double2(mb[A] == mk[a] && mb[B] == mk[b] ? c.econst : 0.0, 0.0);
      const double dk = c.dconst * c.k21;
      if (!zb) {
        const double2 d = cmul_i(ope[B][b], pauli_of(mb[A], mk[a], g.q[B][b]));
        in.x -= dk * d.x;
        in.y -= dk * d.y;
      }
      if (!za) {
        const double2 d = cmul_i(ope[A][a], pauli_of(mb[B], mk[b], g.q[A][a]));
        in.x -= dk * d.x;
        in.y -= dk * d.y;
      }
      if (!za && !zb) {
        const double *p = g.q[A][a], *q = g.q[B][b];
        const double cc3 = c.c1t + c.c3f * (p[0] * q[0] + p[1] * q[1] + p[2] * q[2]);
        in.x += cc3 * oo.x;
        in.y += cc3 * oo.y;
      }
      r.x += wt * in.x;
      r.y += wt * in.y;
    }
    if (!ONE && !za && !zb && td != 0) {
      const double *p = g.q[A][a], *q = g.q[B][b];
      const double x[3] = {p[1] * q[2] - p[2] * q[1], p[2] * q[0] - p[0] * q[2], p[0] * q[1] - p[1] * q[0]};
      const double2 s = cmul_i(oo, pauli_of(mb[C], mk[cc], x));
      const double f = c.c4f * (double)td;
      r.x -= f * s.y;
      r.y += f * s.x;
    }
    return r;
  };
  auto direct = [&](int x, int y, int z) -> double2 {   // nucleons 0, 1, 2 to kets x, y, z
    const double2 u = pair(0, x, 1, y, 2, z), v = pair(0, x, 2, z, 1, y), t = pair(1, y, 2, z, 0, x);
    return make_double2(u.x + v.x + t.x, u.y + v.y + t.y);
  };
  double2 r = make_double2(0.0, 0.0);
  auto both = [&](int x, int y, int z, double f) {   // + (x, y, z) - (y, x, z)
    const double2 u = direct(x, y, z), v = direct(y, x, z);
    r.x += f * (u.x - v.x);
    r.y += f * (u.y - v.y);
  };
  both(0, 1, 2, g.f[2]);
  both(1, 2, 0, g.f[0]);
  both(2, 0, 1, g.f[1]);
  return r;
}

// <abc||def> of three bra and three ket nucleons (momentum and isospin
// conserved); fb the bra regulator
template <bool ONE>
static __device__ __forceinline__ double2 chiral3_asym(const Chiral3Dev &c, double fb, const Nucleon &a,
                                                       const Nucleon &b, const Nucleon &e, const Nucleon &k,
                                                       const Nucleon &l, const Nucleon &m) {
  Geo3 g;
  geo3_transfer<0, 0>(c, g, a, k);
  geo3_transfer<0, 1>(c, g, a, l);
  geo3_transfer<0, 2>(c, g, a, m);
  geo3_transfer<1, 0>(c, g, b, k);
  geo3_transfer<1, 1>(c, g, b, l);
  geo3_transfer<1, 2>(c, g, b, m);
  geo3_transfer<2, 0>(c, g, e, k);
  geo3_transfer<2, 1>(c, g, e, l);
  geo3_transfer<2, 2>(c, g, e, m);
  const double f = fb * c.scale;
  g.f[0] = f * freg3(c, l.k, m.k, k.k);
  g.f[1] = f * freg3(c, k.k, m.k, l.k);
  g.f[2] = f * freg3(c, k.k, l.k, m.k);
  const int mb[3] = {a.sz, b.sz, e.sz}, mk[3] = {k.sz, l.sz, m.sz};
  const int tb[3] = {a.tz, b.tz, e.tz}, tk[3] = {k.tz, l.tz, m.tz};
  return asym3<ONE, false>(c, g, mb, mk, tb, tk);
}

// sum over the holes h of <pqh||rsh> (the normal-ordered two-body part); the
// geometry is that of h's momentum, kept over its spin and isospin states
template <bool ONE>
static __device__ __forceinline__ double2 no2b_sum(const Chiral3Dev &c, int A, int p, int q, int r, int s) {
  double2 acc = make_double2(0.0, 0.0);
  if (!conserves3(c, p, q, 0, r, s, 0)) return acc;
  const Nucleon a = nucleon_of(c, p), b = nucleon_of(c, q), k = nucleon_of(c, r), l = nucleon_of(c, s);
  Geo3 g;
  geo3_transfer<0, 0>(c, g, a, k);
  geo3_transfer<0, 1>(c, g, a, l);
  geo3_transfer<1, 0>(c, g, b, k);
  geo3_transfer<1, 1>(c, g, b, l);
#pragma unroll 1
  for (int h = 0; h < A; ++h) {
    const Nucleon n = nucleon_of(c, h);
    if (h == 0 || c.nx[h] != c.nx[h - 1] || c.ny[h] != c.ny[h - 1] || c.nz[h] != c.nz[h - 1]) {
      geo3_transfer<0, 2>(c, g, a, n);
      geo3_transfer<1, 2>(c, g, b, n);
      geo3_transfer<2, 0>(c, g, n, k);
      geo3_transfer<2, 1>(c, g, n, l);
      const double f = freg3(c, a.k, b.k, n.k) * c.scale;
      g.f[0] = f * freg3(c, l.k, n.k, k.k);
      g.f[1] = f * freg3(c, k.k, n.k, l.k);
      g.f[2] = f * freg3(c, k.k, l.k, n.k);
    }
    const int mb[3] = {a.sz, b.sz, n.sz}, mk[3] = {k.sz, l.sz, n.sz};
    const int tb[3] = {a.tz, b.tz, n.tz}, tk[3] = {k.tz, l.tz, n.tz};
    const double2 v = asym3<ONE, true>(c, g, mb, mk, tb, tk);
    acc.x += v.x;
    acc.y += v.y;
  }
  return acc;
}

}  // namespace ccgpu
