// membrane.hip -- the reference's FP64 capsule membrane law on gfx950, three kernels over
// batches of capsules (libmemb.so, C ABI in include/memb.h).
//
// Per capsule (forcing.f90:11-114 with the force grid equal to the harmonic grid):
//   1. shape coefficients: longitude DFT per latitude, then Gauss-Legendre quadrature
//      (the SPHEREPACK analysis of sph1.f90:29-79);
//   2. on the 2x (dealias) grid, latitude ring by ring: x and all its derivatives up to 4th
//      order (sph3.f90:9-182), then per node the geometry (normal, metrics, curvature,
//      Christoffel symbols and their derivatives) and the load q1 a1 + q2 a2 + q3 n of the
//      neo-Hookean tension and the bending moment (sph.f90:1523-1700);
//   3. the dealias filter: analysis of the 2x-grid load and normal, synthesis of degrees
//      <= L on the force grid (sph1.f90:723-951, 1378-1406), and the point area from the
//      surface metric (sph3.f90:186-260; forcing.f90:91).
// Everything is FP64.  Tables (Gauss nodes, Legendre functions and their theta-derivatives,
// the unit-sphere reference state) are built once per degree by memb_plan_create.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/memb.h"

namespace memb {

constexpr int NQ = 15;        // derivatives of total order <= 4
constexpr int NREF = 32;      // reference-state doubles per fine node
constexpr int LMAX = 23;
constexpr int ND_THREADS = 128;  // per workgroup of the node kernel (two wavefronts)
constexpr int SH_THREADS = 256;  // per workgroup of the shape and filter kernels
constexpr int AB_SLOTS = 4;   // rings whose coefficients are in LDS
constexpr int F_SLOTS = 3;    // rings whose outputs are in LDS

__host__ __device__ constexpr int qidx(int kt, int kp) {
  return (kt + kp) * (kt + kp + 1) / 2 + kp;
}
// Harmonics (m, n = m + d) packed with m fastest: for one d, neighbouring m are neighbours, in
// the tables as in the coefficients, so that threads that own an m each read them coalesced
// and without bank conflicts while they walk d.
__host__ __device__ constexpr int tidx(int N, int d, int m) { return d * N - d * (d - 1) / 2 + m; }

// Colatitudes come in pairs (theta, pi - theta): P_n^m(pi - theta) = (-1)^(n + m) P_n^m(theta),
// and each theta-derivative adds a sign, so tables hold the northern ring of a pair only.
struct Tables {
  // lanes of a ring in the node kernel: its quads are phi_j, -phi_j and both plus pi, j <= N
  __host__ __device__ int slots() const { return 4 * (N + 1); }
  int L, N, np2, nt, np, NT;   // N = L+1 coarse latitudes; nt = 2N, np = 2 np2; NT harmonics
  const double* w2;            // [N] coarse Gauss weights
  const double* s2;            // [N] sin(theta) coarse
  const double* WPc;           // [N][NT] w2 Pbar, coarse (analysis of the shape)
  const double* Pc;            // [(N+1)/2][NT] coarse Pbar, northern rings
  const double* Pcd;           // [(N+1)/2][NT] coarse dPbar/dtheta, northern rings
  const double* Pfd;           // [N][5][NT] fine theta-derivatives 0..4, northern rings
  const double* WPf;           // [N][NT] w Pbar, fine northern rings (the filter's quadrature)
  const double2* e2;           // [np2] cos, sin(2 pi q / np2)
  const double2* ef;           // [np] cos, sin(2 pi q / np)
  const double* ref;           // [NREF][nt*slots] unit-sphere state (the law reads it)
};

__device__ inline double dot3(const double* u, const double* v) {
  return u[0] * v[0] + u[1] * v[1] + u[2] * v[2];
}
__device__ inline void cross3(const double* u, const double* v, double* r) {
  r[0] = u[1] * v[2] - u[2] * v[1];
  r[1] = u[2] * v[0] - u[0] * v[2];
  r[2] = u[0] * v[1] - u[1] * v[0];
}

// v of another lane of the quad, the DPP quad_perm CTRL on the two halves: a VALU move instead of
// an LDS-crossbar permute; the lanes of a quad must be active
template <int CTRL>
__device__ __forceinline__ double quad_perm(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)b, CTRL, 0xF, 0xF, false);
  const unsigned hi = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)(b >> 32), CTRL, 0xF, 0xF, false);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ double swap_pair(double v) { return quad_perm<0xB1>(v); }  // lane ^ 1
__device__ __forceinline__ double swap_half(double v) { return quad_perm<0x4E>(v); }  // lane ^ 2

// ---- per-node geometry and law -----------------------------------------------------------------
// Tensors that are symmetric in a pair of indices keep one value per sum of the pair: a metric
// g[a + b], its derivatives gd[c][a + b] and gdd[c + d][a + b].  Everything past the surface's
// own derivatives is scalar: with D21[s][b] = x_,s . x_,b (s the number of phi-derivatives of
// the second derivative) and so on, the Christoffel symbols are Gam[l][s] = G[l][p] D21[s][p],
// n_,c = -b_cl a^l turns the derivatives of the curvature into products of b, Gam and
// H[l][s] = x_,s(third) . a^l, and no contravariant vector or derivative of the normal is formed:
// less than half of the products a node, with 32 instead of 56 values of reference state (the
// reference's mixed curvature and its derivatives as products).
struct Geom {
  double n[3], x1[2][3];
  double g[3], gd[2][3], G[3], Gd[2][3], Gdd[3][3];
  double b[3], bd[2][3], bdd[3][3];
  double Gam[2][3], Gamd[2][2][3];  // [l][s], [derivative][l][s]
};

// the entries of R = X S (S symmetric, X full) that a symmetric result needs: (0,0), (0,1), (1,1)
__device__ __forceinline__ void mul_fs(const double X[2][2], const double S[3], double R[2][2]) {
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) R[i][j] = X[i][0] * S[j] + X[i][1] * S[1 + j];
}

// P^pa Q_cp and its first and second derivatives (P symmetric contravariant, Q covariant), the
// mixed curvature of the current and of the reference state
__device__ __forceinline__ double mixed(const double P[3], const double Q[3], int c, int a) {
  return P[a] * Q[c] + P[1 + a] * Q[c + 1];
}
__device__ __forceinline__ double mixed_d(const double P[3], const double Pl[3], const double Q[3],
                                          const double Ql[3], int c, int a) {
  return Pl[a] * Q[c] + Pl[1 + a] * Q[c + 1] + P[a] * Ql[c] + P[1 + a] * Ql[c + 1];
}
__device__ __forceinline__ double mixed_dd(const double P[3], const double (&Pd)[2][3],
                                           const double Plk[3], const double Q[3],
                                           const double (&Qd)[2][3], const double Qlk[3], int l,
                                           int k, int c, int a) {
  double v = 0.0;
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    v += Plk[p + a] * Q[c + p] + P[p + a] * Qlk[c + p];
    if (l == k)
      v += 2.0 * (Pd[l][p + a] * Qd[l][c + p]);
    else
      v += Pd[k][p + a] * Qd[l][c + p] + Pd[l][p + a] * Qd[k][c + p];
  }
  return v;
}
// field of the reference's second derivative e of K^a_c: (a, b) with a + b = e only is read
__host__ __device__ constexpr int ref_dd(int e, int c, int a) {
  return e == 1 ? 26 + 2 * c + a : (e == 0 ? 24 : 30) + c;
}

// X[c][q]: derivatives of coordinate c.  BEND: the second derivatives of metric and curvature
// too, which only the bending moment needs (they are what reads the third and fourth
// derivatives of the surface).
template <bool BEND>
__device__ __forceinline__ void geometry(const double (&X)[3][BEND ? NQ : 6], Geom& o) {
  double x2[3][3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    o.x1[0][k] = X[k][qidx(1, 0)], o.x1[1][k] = X[k][qidx(0, 1)];
#pragma unroll
    for (int s = 0; s < 3; ++s) x2[s][k] = X[k][qidx(2 - s, s)];
  }
  double cv[3];
  cross3(o.x1[0], o.x1[1], cv);
  const double rJ = 1.0 / sqrt(dot3(cv, cv));
#pragma unroll
  for (int k = 0; k < 3; ++k) o.n[k] = cv[k] * rJ;
  double D21[3][2];
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    o.b[s] = dot3(x2[s], o.n);
#pragma unroll
    for (int p = 0; p < 2; ++p) D21[s][p] = dot3(x2[s], o.x1[p]);
  }
  o.g[0] = dot3(o.x1[0], o.x1[0]), o.g[1] = dot3(o.x1[0], o.x1[1]), o.g[2] = dot3(o.x1[1], o.x1[1]);
  const double rdet = 1.0 / (o.g[0] * o.g[2] - o.g[1] * o.g[1]);
  o.G[0] = o.g[2] * rdet, o.G[1] = -o.g[1] * rdet, o.G[2] = o.g[0] * rdet;
  double U[2][2][2];  // U[c] = G g_,c
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    o.gd[c][0] = 2.0 * D21[c][0];
    o.gd[c][1] = D21[c][1] + D21[1 + c][0];
    o.gd[c][2] = 2.0 * D21[1 + c][1];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) U[c][i][j] = o.G[i] * o.gd[c][j] + o.G[1 + i] * o.gd[c][1 + j];
    o.Gd[c][0] = -(U[c][0][0] * o.G[0] + U[c][0][1] * o.G[1]);
    o.Gd[c][1] = -(U[c][0][0] * o.G[1] + U[c][0][1] * o.G[2]);
    o.Gd[c][2] = -(U[c][1][0] * o.G[1] + U[c][1][1] * o.G[2]);
  }
#pragma unroll
  for (int l = 0; l < 2; ++l)
#pragma unroll
    for (int s = 0; s < 3; ++s) o.Gam[l][s] = o.G[l] * D21[s][0] + o.G[1 + l] * D21[s][1];
  if (!BEND) return;
  double D31[4][2], D22[3][3], N3[4], N4[5], H[2][4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    double v[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) v[k] = X[k][BEND ? qidx(3 - s, s) : 0];
    N3[s] = dot3(v, o.n);
#pragma unroll
    for (int p = 0; p < 2; ++p) D31[s][p] = dot3(v, o.x1[p]);
#pragma unroll
    for (int l = 0; l < 2; ++l) H[l][s] = o.G[l] * D31[s][0] + o.G[1 + l] * D31[s][1];
  }
#pragma unroll
  for (int s = 0; s < 5; ++s) {
    double v[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) v[k] = X[k][BEND ? qidx(4 - s, s) : 0];
    N4[s] = dot3(v, o.n);
  }
#pragma unroll
  for (int s = 0; s < 3; ++s)
#pragma unroll
    for (int t = s; t < 3; ++t) D22[s][t] = D22[t][s] = dot3(x2[s], x2[t]);
#pragma unroll
  for (int e = 0; e < 3; ++e) {  // (c, d) = (0, 0), (0, 1), (1, 1)
    const int c = e >> 1, d = (e + 1) >> 1;
    const double gdd[3] = {2.0 * (D31[e][0] + D22[c][d]),
                           (D31[e][1] + D31[1 + e][0]) + (D22[c][1 + d] + D22[d][1 + c]),
                           2.0 * (D31[1 + e][1] + D22[1 + c][1 + d])};
    double V[2][2], M[2][2], Y[2][2], Z[2][2];  // M = U_d U_c G, Z = G g_,cd G
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        V[i][j] = U[d][i][0] * U[c][0][j] + U[d][i][1] * U[c][1][j];
        Y[i][j] = o.G[i] * gdd[j] + o.G[1 + i] * gdd[1 + j];
      }
    mul_fs(V, o.G, M);
    mul_fs(Y, o.G, Z);
    o.Gdd[e][0] = 2.0 * M[0][0] - Z[0][0];
    o.Gdd[e][1] = (M[0][1] + M[1][0]) - Z[0][1];
    o.Gdd[e][2] = 2.0 * M[1][1] - Z[1][1];
  }
  double W[2][2][3];  // W[d][l][s] = x_,s . (a^l)_,d
#pragma unroll
  for (int d = 0; d < 2; ++d)
#pragma unroll
    for (int l = 0; l < 2; ++l)
#pragma unroll
      for (int s = 0; s < 3; ++s) {
        W[d][l][s] = (o.Gd[d][l] * D21[s][0] + o.Gd[d][1 + l] * D21[s][1]) +
                     (o.G[l] * D22[s][d] + o.G[1 + l] * D22[s][1 + d]);
        o.Gamd[d][l][s] = H[l][s + d] + W[d][l][s];
      }
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int s = 0; s < 3; ++s)
      o.bd[c][s] = N3[s + c] - (o.b[c] * o.Gam[0][s] + o.b[c + 1] * o.Gam[1][s]);
#pragma unroll
  for (int e = 0; e < 3; ++e) {
    const int c = e >> 1, d = (e + 1) >> 1;
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      double t = N4[s + e];
#pragma unroll
      for (int l = 0; l < 2; ++l) {
        t -= o.b[d + l] * H[l][s + c] + o.b[c + l] * H[l][s + d];
        t -= o.bd[d][c + l] * o.Gam[l][s] + o.b[c + l] * W[d][l][s];
      }
      o.bdd[e][s] = t;
    }
  }
}

// load q1 a1 + q2 a2 + q3 n at one node (sph.f90:1615-1700; membmodel.c:60-79); R: the node's
// reference state, field q at R[q * rs]
template <bool BEND>
__device__ __forceinline__ void law(const Geom& o, const double* __restrict__ R, long long rs,
                                    double gs, double eb, double f[3]) {
  double A[3], Ad[2][3];
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    A[s] = R[s * rs];
#pragma unroll
    for (int c = 0; c < 2; ++c) Ad[c][s] = R[(3 + 3 * c + s) * rs];
  }
  const double detA = R[9 * rs];
  const double deta = o.g[0] * o.g[2] - o.g[1] * o.g[1];
  const double I2 = detA * deta - 1.0;
  const double Js = sqrt(1.0 + I2);
  const double rJs = 1.0 / Js, rI = 1.0 / (I2 + 1.0);  // one division each
  const double w1 = 0.5 * gs;
  const double w2 = -0.5 * gs * (rI * rI);
  const double tA = 2.0 * rJs * w1, tG = 2.0 * Js * w2;  // T = tA A + tG G
  double T[3], Td[2][3];
#pragma unroll
  for (int s = 0; s < 3; ++s) T[s] = tA * A[s] + tG * o.G[s];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const double dA = R[(10 + c) * rs];
    const double da = o.gd[c][0] * o.g[2] + o.g[0] * o.gd[c][2] - 2.0 * o.g[1] * o.gd[c][1];
    const double I2d = dA * deta + da * detA;
    const double Jsd = 0.5 * rJs * I2d;
    const double w2d = gs * (rI * rI * rI) * I2d;
    const double uA = -2.0 * (rJs * rJs) * Jsd * w1, uG = 2.0 * Jsd * w2 + 2.0 * Js * w2d;
#pragma unroll
    for (int s = 0; s < 3; ++s)
      Td[c][s] = (uA * A[s] + tA * Ad[c][s]) + (uG * o.G[s] + tG * o.Gd[c][s]);
  }
  double tr[2];  // Gam^a_al
#pragma unroll
  for (int l = 0; l < 2; ++l) tr[l] = o.Gam[0][l] + o.Gam[1][1 + l];
  double q[2];
#pragma unroll
  for (int b = 0; b < 2; ++b)
    q[b] = (Td[0][b] + Td[1][1 + b]) + (tr[0] * T[b] + tr[1] * T[1 + b]) +
           (o.Gam[b][0] * T[0] + 2.0 * o.Gam[b][1] * T[1] + o.Gam[b][2] * T[2]);
  double q3 = T[0] * o.b[0] + 2.0 * T[1] * o.b[1] + T[2] * o.b[2];
  if (BEND) {
    // K^a_c = A^pa B_cp - G^pa b_cp, its first derivatives, and in dds the contraction of
    // (G^bc K^a_c),ab; K[c][a], Kd[l][c][a]
    double K[2][2], Kd[2][2][2];
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        K[c][a] = R[(12 + 2 * c + a) * rs] - mixed(o.G, o.b, c, a);
#pragma unroll
        for (int l = 0; l < 2; ++l)
          Kd[l][c][a] = R[(16 + 4 * l + 2 * c + a) * rs] - mixed_d(o.G, o.Gd[l], o.b, o.bd[l], c, a);
      }
    double dds = 0.0;
#pragma unroll
    for (int e = 0; e < 3; ++e) {  // derivatives l, k with l + k = e
      const int l = e >> 1, k = (e + 1) >> 1;
      // (a, b) with a + b = e: once for a = b, both orders for e = 1
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const int b = e - a;
        if (b < 0 || b > 1) continue;
#pragma unroll
        for (int c = 0; c < 2; ++c)
          dds += (o.Gdd[e][b + c] * K[c][a] +
                  o.G[b + c] * (R[ref_dd(e, c, a) * rs] -
                                mixed_dd(o.G, o.Gd, o.Gdd[e], o.b, o.bd, o.bdd[e], l, k, c, a))) +
                 (o.Gd[a][b + c] * Kd[b][c][a] + o.Gd[b][b + c] * Kd[a][c][a]);
      }
    }
    double M[3], Md[2][3];  // (a, b) = (0, 0), (0, 1), (1, 1); the moment is symmetric
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      const int a = s >> 1, b = (s + 1) >> 1;
      M[s] = eb * (o.G[b] * K[0][a] + o.G[b + 1] * K[1][a]);
#pragma unroll
      for (int l = 0; l < 2; ++l)
        Md[l][s] = eb * ((o.Gd[l][b] * K[0][a] + o.Gd[l][b + 1] * K[1][a]) +
                         (o.G[b] * Kd[l][0][a] + o.G[b + 1] * Kd[l][1][a]));
    }
    double Q[2], Qc = eb * dds;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      Q[b] = (Md[0][b] + Md[1][1 + b]) + (tr[0] * M[b] + tr[1] * M[1 + b]) +
             (o.Gam[b][0] * M[0] + 2.0 * o.Gam[b][1] * M[1] + o.Gam[b][2] * M[2]);
      Qc += (o.Gam[b][0] * Md[b][0] + 2.0 * o.Gam[b][1] * Md[b][1] + o.Gam[b][2] * Md[b][2]);
      // Gam^a_al,b M^lb
#pragma unroll
      for (int l = 0; l < 2; ++l)
        Qc += (o.Gamd[b][0][l] + o.Gamd[b][1][1 + l]) * M[l + b];
    }
#pragma unroll
    for (int l = 0; l < 2; ++l)  // Gam^a_al (M^lb_,b + Q^l)
      Qc += tr[l] * ((Md[0][l] + Md[1][1 + l]) + Q[l]);
#pragma unroll
    for (int s = 0; s < 3; ++s)  // Gam^b_al,b M^al
      Qc += (s == 1 ? 2.0 : 1.0) * (o.Gamd[0][0][s] + o.Gamd[1][1][s]) * M[s];
    double bm[2][2];
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int a = 0; a < 2; ++a) bm[b][a] = o.G[a] * o.b[b] + o.G[1 + a] * o.b[b + 1];
    q[0] -= bm[0][0] * Q[0] + bm[1][0] * Q[1];
    q[1] -= bm[0][1] * Q[0] + bm[1][1] * Q[1];
    q3 += Qc;
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) f[k] = q[0] * o.x1[0][k] + q[1] * o.x1[1][k] + q3 * o.n[k];
}

// ---- the kernels ---------------------------------------------------------------------------------
// The law of a batch is three kernels: shape (k_shape: coefficients and areas), nodes (k_nodes:
// the doubled grid's load and its longitude DFT) and filter (k_filter).  Their data per capsule
// slot: the coefficients [3][NT] (a, b) and the DFT rows [nt][N][6] (cos, sin sums).
// As one kernel a capsule was one chain of 19 node chunks on one CU (478 us at degree 16,
// whether 1 capsule or 1000 ran), with the registers of the node phase (256, 42 spilled) held
// through the transforms.  Apart, the node phase spreads a few capsules over the chip (8
// capsules: 55 us in all) and holds 220 registers, none spilled; the transforms run 16 wavefronts
// a CU on tables read coalesced.  8000 capsules of degree 16: 4.74 -> 2.8 ms (shape 0.25, nodes
// 2.14, filter 0.39); 301 of degree 23 without bending: 1053 -> 252 us.
// Capsules: slot q holds capsule list[q], q < *cnt (list null: capsule c0 + q, q < n).
struct Work {
  int n;              // slots (list null), or the most there can be
  const int* list;
  const int* cnt;
  long long c0;       // list null: slot q holds capsule c0 + q
  double2* coef;      // [slot][3][NT]
  double2* rows;      // [slot][nt][N][6]
};
__device__ __forceinline__ int work_n(const Work& w) { return w.list ? *w.cnt : w.n; }
__device__ __forceinline__ long long work_cap(const Work& w, int q) { return w.list ? w.list[q] : w.c0 + q; }

enum Shape {
  SHAPE_LAW = 0,     // coefficients into the slot, areas
  SHAPE_COEFFS = 1,  // coefficients packed into `out`
  SHAPE_GEOM = 2,    // areas and unit normals of the force grid
  SHAPE_REF = 3,     // coefficients into the slot only
};

// Coefficients of the three coordinates (the SPHEREPACK analysis of sph1.f90:29-79) and, from
// them, x_theta and x_phi on the force grid: area |x_theta x x_phi| w / sin(theta) dphi
// (sph3.f90:186-260; forcing.f90:91) and, for SHAPE_GEOM, the unit normal.
// The raw coordinates carry the capsule's position, whose rounding lands in the near-zero high-m
// coefficients and comes out of the fourth derivatives multiplied by m^4: the law sums every
// point in order, as the reference does, so that it rounds there as the reference does.  The
// geometry alone reads first derivatives: it takes the coordinates relative to the capsule's
// first point and pairs points j and j + np2/2 (factors equal up to (-1)^m).
template <int MODE>
__global__ void __launch_bounds__(SH_THREADS)
    k_shape(Tables T, Work wk, const double* __restrict__ x, const double* __restrict__ y,
            const double* __restrict__ z, double* __restrict__ nx, double* __restrict__ ny,
            double* __restrict__ nz, double* __restrict__ area, double* __restrict__ out,
            const int* __restrict__ skip) {
  extern __shared__ double lds[];
  constexpr bool REL = MODE == SHAPE_GEOM;
  const int tid = threadIdx.x;
  const int N = T.N, NN = N * N, np2 = T.np2, nc = N * np2, NT = T.NT, hp = N;
  double2* te = reinterpret_cast<double2*>(lds);  // [np2]
  double2* cf = te + np2;                         // [3][NT] coefficients (a, b)
  double2* tmp = cf + 3 * NT;  // [6][N][N] partial sums of x_theta (0..2), x_phi (3..5); before:
  double* pts = reinterpret_cast<double*>(tmp);   // [3][nc] the points and
  double2* U = tmp + (3 * nc + 1) / 2;            // [3][N][N] their longitude DFT
  for (int q = tid; q < np2; q += SH_THREADS) te[q] = T.e2[q];
  const int n = work_n(wk);
  for (int slot = blockIdx.x; slot < n; slot += gridDim.x) {
    const long long cap = work_cap(wk, slot);
    if (skip && skip[cap]) continue;  // uniform over the workgroup
    for (int t = tid; t < 3 * nc; t += SH_THREADS) {
      const int c = t / nc, q = t - c * nc;
      const double* p = (c == 0 ? x : (c == 1 ? y : z)) + cap * nc;
      pts[t] = REL ? p[q] - p[0] : p[q];
    }
    __syncthreads();
    // longitude DFT, one thread per (i, m) for the three coordinates
    for (int t = tid; t < NN; t += SH_THREADS) {
      const int i = t / N, m = t % N;
      double cs[3] = {0.0, 0.0, 0.0}, sn[3] = {0.0, 0.0, 0.0};
      const double sg = (m & 1) ? -1.0 : 1.0;
      int q = 0;  // (m j) mod np2
      #pragma unroll 4
      for (int j = 0; j < (REL ? hp : np2); ++j) {
        const double2 e = te[q];
        q += m;
        if (q >= np2) q -= np2;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const double* p = pts + k * nc + i * np2 + j;
          const double v = REL ? p[0] + sg * p[hp] : p[0];
          cs[k] += v * e.x;
          sn[k] += v * e.y;
        }
      }
#pragma unroll
      for (int k = 0; k < 3; ++k) U[k * NN + t] = make_double2(cs[k], sn[k]);
    }
    __syncthreads();
    // quadrature, one thread per harmonic for the three coordinates
    for (int t = tid; t < NT; t += SH_THREADS) {
      int d = 0, m = t;
      while (m >= N - d) m -= N - d, ++d;
      double sa[3] = {0.0, 0.0, 0.0}, sb[3] = {0.0, 0.0, 0.0};
      #pragma unroll 4
      for (int i = 0; i < N; ++i) {
        const double p = T.WPc[i * NT + t];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const double2 u = U[(k * N + i) * N + m];
          sa[k] += p * u.x;
          sb[k] += p * u.y;
        }
      }
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const double a = 2.0 / np2 * sa[k], b = -2.0 / np2 * sb[k];
        if (MODE == SHAPE_COEFFS) {
          // packed: a(m, n >= m) then b(m >= 1, n >= m), per coordinate
          double* o = out + (cap * 3 + k) * NN;
          o[m * N - m * (m - 1) / 2 + d] = a;
          if (m >= 1) o[NT + (m - 1) * N - (m - 1) * (m - 2) / 2 - (m - 1) + d] = b;
        } else {
          cf[k * NT + t] = make_double2(a, b);
          if (MODE != SHAPE_GEOM)
            wk.coef[((size_t)slot * 3 + k) * NT + t] = make_double2(a, b);
        }
      }
    }
    __syncthreads();
    if (MODE == SHAPE_LAW || MODE == SHAPE_GEOM) {
      // x_theta and x_phi of coordinate c per (c, ring pair, m): the sums over even and odd d
      // give the northern ring as E + O and the southern one as +-(E - O)
      const int nh = (N + 1) / 2;
      for (int t = tid; t < 3 * nh * N; t += SH_THREADS) {
        const int c = t / (nh * N), u = t % (nh * N), i = u / N, m = u % N;
        const double* Pt = T.Pcd + i * NT;
        const double* Pp = T.Pc + i * NT;
        double2 st[2] = {{0.0, 0.0}, {0.0, 0.0}}, sp[2] = {{0.0, 0.0}, {0.0, 0.0}};
        int q = m;  // tidx(N, d, m)
        for (int d = 0; d < N - m; d += 2) {
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const bool on = d + e < N - m;
            const int qq = on ? q : m;
            const double2 v = cf[c * NT + qq];
            const double a = on ? Pt[qq] : 0.0, b = on ? Pp[qq] : 0.0;
            st[e].x += a * v.x, st[e].y += a * v.y;
            sp[e].x += b * v.x, sp[e].y += b * v.y;
            q += N - (d + e);
          }
        }
        const double h = m == 0 ? 0.5 : 1.0;
        double2* tt = tmp + c * NN + m;
        double2* tp = tmp + (3 + c) * NN + m;
        tt[i * N] = make_double2(h * (st[0].x + st[1].x), h * (st[0].y + st[1].y));
        tp[i * N] = make_double2(h * (sp[0].x + sp[1].x), h * (sp[0].y + sp[1].y));
        if (N - 1 - i > i) {
          const int k = (N - 1 - i) * N;
          tt[k] = make_double2(h * (st[1].x - st[0].x), h * (st[1].y - st[0].y));
          tp[k] = make_double2(h * (sp[0].x - sp[1].x), h * (sp[0].y - sp[1].y));
        }
      }
      __syncthreads();
      // node sums, one thread per (i, j < np2/2) and its partner j + np2/2: the even-m terms E
      // and the odd-m terms O give E + O and E - O
      for (int t = tid; t < N * hp; t += SH_THREADS) {
        const int i = t / hp, j = t % hp;
        double s[2][6];
#pragma unroll
        for (int f = 0; f < 6; ++f) s[0][f] = 0.0, s[1][f] = 0.0;
        int q = 0;  // (m j) mod np2
        for (int m = 0; m < N; m += 2) {
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            if (m + e >= N) break;
            const double2 w = te[q];
            q += j;
            if (q >= np2) q -= np2;
#pragma unroll
            for (int f = 0; f < 6; ++f) {
              const double2 v = tmp[f * NN + i * N + m + e];
              s[e][f] += f < 3 ? v.x * w.x - v.y * w.y : (double)(m + e) * (-v.x * w.y - v.y * w.x);
            }
          }
        }
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          double v[6], cr[3];
#pragma unroll
          for (int f = 0; f < 6; ++f) v[f] = e ? s[0][f] - s[1][f] : s[0][f] + s[1][f];
          cross3(&v[0], &v[3], cr);
          const double J = sqrt(dot3(cr, cr));
          const size_t o = (size_t)cap * nc + i * np2 + j + e * hp;
          if (MODE == SHAPE_GEOM) nx[o] = cr[0] / J, ny[o] = cr[1] / J, nz[o] = cr[2] / J;
          area[o] = J * T.w2[i] / T.s2[i] * (2.0 * M_PI / np2);
        }
      }
      __syncthreads();
    }
  }
}

// The doubled grid: x and its derivatives up to 4th order (sph3.f90:9-182; to 2nd order without
// bending, where nothing reads the others), per node the geometry and the load q1 a1 + q2 a2 +
// q3 n (sph.f90:1523-1700), and the longitude DFT of load and normal, degrees <= L.
// REF: the unit sphere's state of slot 0 into `refout` instead.
//
// A unit of work is a run of rings of one capsule; rings go in the order north, south, north
// ... (ring 0, nt - 1, 1, nt - 2, ...).  A few capsules are cut into so many runs that the
// workgroups in flight are all used (8 capsules of degree 16: one ring each), many are one run
// each: a ring's sums do not depend on the cut.  Within a run, chunks of W consecutive lanes' nodes.
// A chunk of W <= 2 rings touches at most three; ring r's coefficients live in slot
// r % AB_SLOTS and are summed (with those of its pair) before the first chunk that touches it, its
// outputs live in slot r % F_SLOTS until the DFT after the chunk that completes it.
//
// Lanes 4j .. 4j + 3 of a ring are the nodes phi_j, phi_j + pi, -phi_j, -phi_j + pi (j <= N; the
// quads j = 0 and j = N hold two nodes twice).  With (A, B)_m the ring's coefficients the four
// are the same sums up to signs: A cos and B sin over even and over odd m.  Each lane takes one of
// the four sums and two exchanges give every lane its node's values.
// A lane that reads A or B reads half of the LDS that one which needs both does and multiplies
// half as much, and the DFT of the quads' sums and differences runs over N + 1 instead of 2 N
// points: 3250 -> 2340 vector instructions a node with the reference's products taken from the
// table.  8000 capsules of degree 16: 2.40 -> 2.14 ms; 301 of degree 23 without bending
// 316 -> 275 us in all, 252 with the runs cut for the workgroups that fit.  What is left waits half
// its time at two wavefronts per SIMD (the vector units are busy 63 %, LDS 29 %), in no one place:
// without the coefficients' sums, the DFT, the reference loads or the rest of the law it takes
// 0.34, 0.24, 0.26, 0.08 ms less; reading the tables ten at a time in the sums changes nothing.
// Registers: two wavefronts per SIMD.
template <bool REF, bool BEND>
__global__ void __launch_bounds__(ND_THREADS, 2)
    k_nodes(Tables T, Work wk, int most, double gs, double eb, double* __restrict__ refout) {
  extern __shared__ double lds[];
  constexpr int NK = BEND ? 5 : 3, NX = BEND ? NQ : 6;  // theta-derivatives, derivatives
  constexpr int NKG = (NK + 1) / 2;
  const int tid = threadIdx.x;
  const int N = T.N, nt = T.nt, np = T.np, NT = T.NT;
  const int RS = T.slots();
  double2* te = reinterpret_cast<double2*>(lds);   // [np]
  double2* cf = te + np;                           // [3][NT]
  double* AB = reinterpret_cast<double*>(cf + 3 * NT);  // [AB_SLOTS][N][A, B][3][NK]
  double* F = AB + AB_SLOTS * 6 * NK * N;          // [F_SLOTS][N + 1][even, odd m][cos, sin][6]
  for (int q = tid; q < np; q += ND_THREADS) te[q] = T.ef[q];
  // runs of rp rings (an even number, so that pairs stay together, or single rings)
  const int n = work_n(wk);
  if (n == 0) return;
  const int want = min(nt, max(1, most / n));
  int rp = (nt + want - 1) / want;
  if (rp > 1) rp += rp & 1;
  const int parts = (nt + rp - 1) / rp;
  const int W = min(ND_THREADS, 2 * RS);  // a multiple of 4: quads stay in one chunk
  for (int u = blockIdx.x; u < n * parts; u += gridDim.x) {
    const int slot = u / parts, s0 = (u - slot * parts) * rp, s1 = min(s0 + rp, nt);
    __syncthreads();
    for (int t = tid; t < 3 * NT; t += ND_THREADS) cf[t] = wk.coef[(size_t)slot * 3 * NT + t];
    __syncthreads();
    const int node0 = s0 * RS, node1 = s1 * RS;
    int rnext = s0, rdone = s0;  // first ring without coefficients / without its DFT
    for (int n0 = node0; n0 < node1; n0 += W) {
      const int n1 = min(n0 + W, node1);
      const int rhi = (n1 - 1) / RS;  // last ring of the chunk
      if (rhi >= rnext) {
        // one thread per (ring pair, two k, m) for the three coordinates: a coefficient read feeds
        // two FMAs, a table load three and both rings of the pair, north E + O, south
        // (-1)^k (E - O) of the sums over even and odd n - m
        const int p0 = rnext >> 1, p1 = rhi >> 1;
        for (int t = tid; t < (p1 - p0 + 1) * NKG * N; t += ND_THREADS) {
          const int p = p0 + t / (NKG * N), k0 = 2 * ((t / N) % NKG), m = t % N;
          const bool both = k0 + 1 < NK;
          const double* P = T.Pfd + ((size_t)p * 5 + k0) * NT;
          const int kp = both ? NT : 0;
          double2 s[2][2][3];  // [k - k0][n - m even, odd][coordinate]
#pragma unroll
          for (int c = 0; c < 12; ++c) (&s[0][0][0])[c] = make_double2(0.0, 0.0);
          int q = m;  // tidx(N, d, m)
          for (int d = 0; d < N - m; d += 2) {
            const bool two = d + 1 < N - m;
            const int q1 = two ? q + N - d : q;
            double e[2][2] = {{P[q], P[q1]}, {P[kp + q], P[kp + q1]}};
            if (!two) e[0][1] = e[1][1] = 0.0;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
              const double2 v0 = cf[c * NT + q], v1 = cf[c * NT + q1];
#pragma unroll
              for (int i = 0; i < 2; ++i) {
                s[i][0][c].x += e[i][0] * v0.x, s[i][0][c].y += e[i][0] * v0.y;
                s[i][1][c].x += e[i][1] * v1.x, s[i][1][c].y += e[i][1] * v1.y;
              }
            }
            q += 2 * (N - d) - 1;
          }
          const double h = m == 0 ? 0.5 : 1.0;
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            if (i && !both) break;
            const double hs = i ? -h : h;  // k0 is even
            double* north = AB + (((2 * p) % AB_SLOTS) * N + m) * 6 * NK + k0 + i;
            double* south = AB + (((2 * p + 1) % AB_SLOTS) * N + m) * 6 * NK + k0 + i;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
              const double2 E = s[i][0][c], O = s[i][1][c];
              north[c * NK] = h * (E.x + O.x), north[c * NK + 3 * NK] = h * (E.y + O.y);
              south[c * NK] = hs * (E.x - O.x), south[c * NK + 3 * NK] = hs * (E.y - O.y);
            }
          }
        }
        rnext = 2 * p1 + 2;
      }
      __syncthreads();
      // lane bits: par, the parity of the m it sums and phi + pi; neg, B's sums and -phi
      if (n0 + tid < n1) {
        const int pn = n0 + tid;
        const int ring = pn / RS, jq = (pn - ring * RS) >> 2;
        const int par = pn & 1;
        const bool neg = pn & 2, twice = jq == 0 || jq == N;
        const double sp = par ? -1.0 : 1.0, sn = neg ? -1.0 : 1.0;
        double X[3][NX];
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
          for (int q = 0; q < NX; ++q) X[c][q] = 0.0;
        int q = par * jq;  // (m jq) mod np
        const int dq = 2 * jq;
        const double* ab = AB + ((ring % AB_SLOTS) * N + par) * 6 * NK + (neg ? 3 * NK : 0);
        for (int m = par; m < N; m += 2, ab += 12 * NK) {
          const double2 w = te[q];
          q += dq;
          if (q >= np) q -= np;
          // phi-derivatives of A cos, or of -B sin
          const double m1 = (double)m, m2 = -(m1 * m1);
          const double w0 = neg ? -w.y : w.x, w1 = m1 * (neg ? -w.x : -w.y);
          const double w2 = m2 * w0, w3 = m2 * w1, w4 = m2 * w2;
#pragma unroll
          for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int kt = 0; kt < NK; ++kt) {
              const double v = ab[c * NK + kt];
              X[c][qidx(kt, 0)] += v * w0;
              if (kt <= NK - 2) X[c][qidx(kt, 1)] += v * w1;
              if (kt <= NK - 3) X[c][qidx(kt, 2)] += v * w2;
              if (BEND && kt <= 1) X[c][BEND ? qidx(kt, 3) : 0] += v * w3;
              if (BEND && kt == 0) X[c][BEND ? qidx(0, 4) : 0] += v * w4;
            }
        }
        // even + odd m, minus at phi + pi; then A's + B's: at -phi what holds a sine changes its
        // sign (B's in an even phi-derivative, A's in an odd one)
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
          for (int kt = 0; kt < NK; ++kt)
#pragma unroll
            for (int kp = 0; kp < NK - kt; ++kp) {
              double& v = X[c][qidx(kt, kp)];
              double other = swap_pair(v);
              v = sp * v + other;
              other = swap_half(v);
              v = kp & 1 ? sn * other + v : sn * v + other;
            }
        Geom o;
        geometry<BEND>(X, o);
        const long long nodes = (long long)nt * RS;
        if (REF) {
          double* R = refout + pn;
          for (int s = 0; s < 3; ++s) {
            R[s * nodes] = o.G[s];
#pragma unroll
            for (int c = 0; c < 2; ++c) R[(3 + 3 * c + s) * nodes] = o.Gd[c][s];
          }
          R[9 * nodes] = o.G[0] * o.G[2] - o.G[1] * o.G[1];
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            R[(10 + c) * nodes] =
                o.Gd[c][0] * o.G[2] + o.G[0] * o.Gd[c][2] - 2.0 * o.G[1] * o.Gd[c][1];
#pragma unroll
            for (int a = 0; a < 2; ++a) {
              R[(12 + 2 * c + a) * nodes] = mixed(o.G, o.b, c, a);
#pragma unroll
              for (int l = 0; l < 2; ++l)
                R[(16 + 4 * l + 2 * c + a) * nodes] = mixed_d(o.G, o.Gd[l], o.b, o.bd[l], c, a);
#pragma unroll
              for (int b = 0; b < 2; ++b) {
                const int e = a + b;
                R[ref_dd(e, c, a) * nodes] = mixed_dd(o.G, o.Gd, o.Gdd[e], o.b, o.bd, o.bdd[e],
                                                      e >> 1, (e + 1) >> 1, c, a);
              }
            }
          }
        } else {
          double f[6];
          law<BEND>(o, T.ref + pn, nodes, gs, eb, f);
#pragma unroll
          for (int k = 0; k < 3; ++k) f[3 + k] = o.n[k];
          // the DFT needs v(phi) + v(phi + pi) for even and the difference for odd m, and of these
          // the sum over phi and -phi for cos and the difference for sin
          double* Fo = F + (((size_t)(ring % F_SLOTS) * (N + 1) + jq) * 4 + par * 2 + neg) * 6;
#pragma unroll
          for (int k = 0; k < 6; ++k) {
            double v = f[k], other = swap_pair(v);
            v = sp * v + other;
            other = swap_half(v);
            Fo[k] = twice ? (neg ? other : v) : sn * v + other;
          }
        }
      }
      __syncthreads();
      if (!REF && n1 / RS > rdone) {
        // rings rdone .. n1 / RS - 1 are complete: longitude DFT of their six outputs, a thread
        // for the cos or the sin sums of one (ring, m); from the last thread on, since the first
        // ones go on to the next coefficients without a barrier
        for (int t = ND_THREADS - 1 - tid; t < (n1 / RS - rdone) * 2 * N; t += ND_THREADS) {
          const int ring = rdone + t / (2 * N), m = (t >> 1) % N, sc = t & 1;
          const double2* v = reinterpret_cast<const double2*>(
              F + ((size_t)(ring % F_SLOTS) * (N + 1) * 4 + (m & 1) * 2 + sc) * 6);
          const double* e = reinterpret_cast<const double*>(te) + sc;
          double2 sum[3] = {{0.0, 0.0}, {0.0, 0.0}, {0.0, 0.0}};
          int q = 0;  // (m j) mod np
          #pragma unroll 3
          for (int j = 0; j <= N; ++j, v += 12) {
            const double ev = e[2 * q];
            q += m;
            if (q >= np) q -= np;
#pragma unroll
            for (int g = 0; g < 3; ++g) sum[g].x += v[g].x * ev, sum[g].y += v[g].y * ev;
          }
          double* r =
              reinterpret_cast<double*>(wk.rows + (((size_t)slot * nt + ring) * N + m) * 6) + sc;
#pragma unroll
          for (int g = 0; g < 3; ++g) r[4 * g] = sum[g].x, r[4 * g + 2] = sum[g].y;
        }
        rdone = n1 / RS;
      }
    }
  }
}

// The dealias filter: quadrature of the doubled grid's load and normal (degrees <= L), synthesis
// on the force grid (sph1.f90:723-951), unit normal (cal_unitO_filter, sph1.f90:1378-1406).  A
// unit is one capsule, or with parts = 2 its load (0) or its normal (1).
// The DFT rows come nq ring pairs at a time through LDS as the sum and the difference of the
// pair's rings, which is what the harmonics of even and of odd n - m integrate.
constexpr int FL_STAGE = 4;  // ring pairs per staged chunk
__global__ void __launch_bounds__(SH_THREADS)
    k_filter(Tables T, Work wk, int most, double* __restrict__ fx, double* __restrict__ fy,
             double* __restrict__ fz, double* __restrict__ nx, double* __restrict__ ny,
             double* __restrict__ nz) {
  extern __shared__ double lds[];
  const int tid = threadIdx.x;
  const int N = T.N, NN = N * N, np2 = T.np2, nt = T.nt, nc = N * np2, NT = T.NT, hp = N;
  const int nh = (N + 1) / 2;
  double2* te = reinterpret_cast<double2*>(lds);  // [np2]
  double2* fc = te + np2;                         // [3][NT] coefficients of the three fields
  double2* stg = fc + 3 * NT;                     // [FL_STAGE][2][N][3] staged rows, then
  double2* tmp = stg;                             // [3][N][N] partial sums
  for (int q = tid; q < np2; q += SH_THREADS) te[q] = T.e2[q];
  const int n = work_n(wk);
  const int parts = 2 * n <= most ? 2 : 1;
  for (int u = blockIdx.x; u < n * parts; u += gridDim.x) {
    const int slot = u / parts;
    const long long cap = work_cap(wk, slot);
    for (int g = parts == 2 ? u - slot * 2 : 0; g < (parts == 2 ? u - slot * 2 + 1 : 2); ++g) {
      const double2* rows = wk.rows + (size_t)slot * nt * N * 6 + 3 * g;
      // quadrature, one thread per harmonic and field; up to 4 items a thread (NT <= 300)
      double2 acc[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) acc[k] = make_double2(0.0, 0.0);
      for (int c0 = 0; c0 < N; c0 += FL_STAGE) {
        const int cr = min(FL_STAGE, N - c0);
        __syncthreads();  // the previous chunk (and unit) is consumed
        for (int e = tid; e < cr * 3 * N; e += SH_THREADS) {
          const int r = e / (3 * N), k = e - r * 3 * N;  // k = 3 m + field
          const size_t a = (size_t)(2 * (c0 + r)) * N * 6 + (k / 3) * 6 + k % 3;
          const double2 v = rows[a], w = rows[a + (size_t)N * 6];
          stg[(r * 2) * 3 * N + k] = make_double2(v.x + w.x, v.y + w.y);
          stg[(r * 2 + 1) * 3 * N + k] = make_double2(v.x - w.x, v.y - w.y);
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int it = tid + k * SH_THREADS;
          if (it >= 3 * NT) break;
          const int f = it / NT, t = it - f * NT;
          int d = 0, m = t;
          while (m >= N - d) m -= N - d, ++d;
          const double2* s = stg + (d & 1) * 3 * N + 3 * m + f;
          for (int r = 0; r < cr; ++r) {
            const double p = T.WPf[(c0 + r) * NT + t];
            const double2 v = s[r * 6 * N];
            acc[k].x += p * v.x;
            acc[k].y += p * v.y;
          }
        }
      }
      __syncthreads();
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int it = tid + k * SH_THREADS;
        if (it < 3 * NT) fc[it] = make_double2(2.0 / T.np * acc[k].x, -2.0 / T.np * acc[k].y);
      }
      __syncthreads();
      // partial sums per (field, ring pair, m): northern ring E + O, southern ring E - O
      for (int t = tid; t < 3 * nh * N; t += SH_THREADS) {
        const int f = t / (nh * N), w = t % (nh * N), i = w / N, m = w % N;
        const double* P = T.Pc + i * NT;
        double2 s[2] = {{0.0, 0.0}, {0.0, 0.0}};
        int q = m;  // tidx(N, d, m)
        #pragma unroll 2
        for (int d = 0; d < N - m; d += 2) {
          const bool two = d + 1 < N - m;
          const int q1 = two ? q + N - d : q;
          const double a = P[q], b = two ? P[q1] : 0.0;
          const double2 v0 = fc[f * NT + q], v1 = fc[f * NT + q1];
          s[0].x += a * v0.x, s[0].y += a * v0.y;
          s[1].x += b * v1.x, s[1].y += b * v1.y;
          q += 2 * (N - d) - 1;
        }
        const double h = m == 0 ? 0.5 : 1.0;
        double2* o = tmp + f * NN + m;
        o[i * N] = make_double2(h * (s[0].x + s[1].x), h * (s[0].y + s[1].y));
        if (N - 1 - i > i)
          o[(N - 1 - i) * N] = make_double2(h * (s[0].x - s[1].x), h * (s[0].y - s[1].y));
      }
      __syncthreads();
      // node sums of the three fields, one thread per (i, j < np2/2) and its partner j + np2/2
      for (int t = tid; t < N * hp; t += SH_THREADS) {
        const int i = t / hp, j = t % hp;
        double s[2][3] = {{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}};
        int q = 0;  // (m j) mod np2
        for (int m = 0; m < N; m += 2) {
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            if (m + e >= N) break;
            const double2 w = te[q];
            q += j;
            if (q >= np2) q -= np2;
#pragma unroll
            for (int f = 0; f < 3; ++f) {
              const double2 v = tmp[f * NN + i * N + m + e];
              s[e][f] += v.x * w.x - v.y * w.y;
            }
          }
        }
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          double v[3];
#pragma unroll
          for (int f = 0; f < 3; ++f) v[f] = e ? s[0][f] - s[1][f] : s[0][f] + s[1][f];
          const size_t o = (size_t)cap * nc + i * np2 + j + e * hp;
          if (g == 0) {
            fx[o] = v[0], fy[o] = v[1], fz[o] = v[2];
          } else {
            const double r = sqrt(dot3(v, v));
            nx[o] = v[0] / r, ny[o] = v[1] / r, nz[o] = v[2] / r;
          }
        }
      }
    }
  }
}

// list[0 .. *cnt): the capsules of sel[0 .. n) that are set, in order.  One workgroup.
constexpr int SL_THREADS = 1024;
__global__ void __launch_bounds__(SL_THREADS)
    k_select(int n, const int* __restrict__ sel, long long c0, int* __restrict__ list,
             int* __restrict__ cnt) {
  __shared__ int wsum[SL_THREADS / 64];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  int base = 0;
  for (int b = 0; b < n; b += SL_THREADS) {
    const bool on = b + tid < n && sel[c0 + b + tid] != 0;
    const unsigned long long bal = __ballot(on);
    if (lane == 0) wsum[wv] = __popcll(bal);
    __syncthreads();
    int before = 0, total = 0;
    for (int w = 0; w < SL_THREADS / 64; ++w) {
      before += w < wv ? wsum[w] : 0;
      total += wsum[w];
    }
    if (on) list[base + before + __popcll(bal & __lanemask_lt())] = (int)(c0 + b + tid);
    base += total;
    __syncthreads();
  }
  if (tid == 0) *cnt = base;
}

}  // namespace memb

#include "law_ordered.hpp"

namespace memb {

// ---- host tables ------------------------------------------------------------------------
void gauss(int n, double* theta, double* w) {
  for (int i = 0; i < n; ++i) {
    double x = std::cos(M_PI * (i + 0.75) / (n + 0.5)), dp = 1.0;
    for (int it = 0; it < 100; ++it) {
      double p0 = 1.0, p1 = x;
      for (int k = 2; k <= n; ++k) {
        const double p2 = ((2.0 * k - 1.0) * x * p1 - (k - 1.0) * p0) / k;
        p0 = p1, p1 = p2;
      }
      const double pn = n == 1 ? x : p1, pm = n == 1 ? 1.0 : p0;
      dp = n * (x * pn - pm) / (x * x - 1.0);
      const double dx = pn / dp;
      x -= dx;
      if (std::fabs(dx) < 1e-16) {
        p0 = 1.0, p1 = x;
        for (int k = 2; k <= n; ++k) {
          const double p2 = ((2.0 * k - 1.0) * x * p1 - (k - 1.0) * p0) / k;
          p0 = p1, p1 = p2;
        }
        const double qn = n == 1 ? x : p1, qm = n == 1 ? 1.0 : p0;
        dp = n * (x * qn - qm) / (x * x - 1.0);
        break;
      }
    }
    theta[i] = std::acos(x);
    w[i] = 2.0 / ((1.0 - x * x) * dp * dp);
  }
}

// Pbar_n^m(cos t), m <= n < nmax: P[m * nmax + n]
void legendre(int nmax, double t, double* P) {
  const double c = std::cos(t), s = std::sin(t);
  std::fill(P, P + nmax * nmax, 0.0);
  double pmm = std::sqrt(0.5);
  for (int m = 0; m < nmax; ++m) {
    if (m > 0) pmm *= std::sqrt((2.0 * m + 1.0) / (2.0 * m)) * s;
    P[m * nmax + m] = pmm;
    if (m + 1 < nmax) P[m * nmax + m + 1] = std::sqrt(2.0 * m + 3.0) * c * pmm;
    for (int n = m + 2; n < nmax; ++n) {
      const double a = std::sqrt((4.0 * n * n - 1.0) / ((double)n * n - (double)m * m));
      const double a1 =
          std::sqrt((4.0 * (n - 1.0) * (n - 1.0) - 1.0) / ((n - 1.0) * (n - 1.0) - (double)m * m));
      P[m * nmax + n] = a * (c * P[m * nmax + n - 1] - P[m * nmax + n - 2] / a1);
    }
  }
}

// theta-derivatives 0..4 by the ladder d/dt Pbar^m = (c-_m Pbar^{m-1} - c+_m Pbar^{m+1}) / 2
void legendre_derivs(int nmax, double t, double* D /* [5][nmax][nmax] */) {
  std::vector<double> P(nmax * nmax);
  legendre(nmax, t, P.data());
  std::fill(D, D + 5 * nmax * nmax, 0.0);
  std::vector<double> v(5 * (2 * nmax + 3));
  for (int n = 0; n < nmax; ++n) {
    const int off = n + 1, W = 2 * nmax + 3;
    std::fill(v.begin(), v.end(), 0.0);
    for (int m = -n; m <= n; ++m) {
      const int am = m < 0 ? -m : m;
      v[m + off] = ((m < 0 && (am & 1)) ? -1.0 : 1.0) * P[am * nmax + n];
    }
    for (int k = 1; k < 5; ++k)
      for (int m = -n; m <= n; ++m) {
        const double cm = std::sqrt((double)(n + m) * (double)(n - m + 1));
        const double cp = std::sqrt((double)(n + m + 1) * (double)(n - m));
        v[k * W + m + off] = 0.5 * (cm * v[(k - 1) * W + m - 1 + off] - cp * v[(k - 1) * W + m + 1 + off]);
      }
    for (int k = 0; k < 5; ++k)
      for (int m = 0; m <= n; ++m) D[(k * nmax + m) * nmax + n] = v[k * W + m + off];
  }
}

// unit-sphere points of the force grid, x block, y block, z block (sph.f90:84-86)
void sphere(int N, int np2, const double* theta, double* xyz) {
  for (int i = 0; i < N; ++i)
    for (int j = 0; j < np2; ++j) {
      const double ph = 2.0 * M_PI * j / np2;
      xyz[i * np2 + j] = std::sin(theta[i]) * std::sin(ph);
      xyz[N * np2 + i * np2 + j] = std::sin(theta[i]) * std::cos(ph);
      xyz[2 * N * np2 + i * np2 + j] = std::cos(theta[i]);
    }
}

}  // namespace memb

using namespace memb;

struct memb_plan {
  int device = 0, L = 0;
  hipStream_t own = nullptr, stream = nullptr;
  std::string err;
  Tables T{};
  std::vector<void*> bufs;  // device allocations of the tables
  double* ref = nullptr;
  // work of the law: capsule slots with their coefficients and DFT rows, and the list of the
  // selected capsules of a batch with its length behind it
  double2* coef = nullptr;
  double2* rows = nullptr;
  int* list = nullptr;
  int slots = 0;
  int num_wg = 0;         // shape and filter workgroups in flight, about
  int nodes_wg[2] = {};   // node workgroups that fit the device, without and with bending
  ordered::OrderedTables O{};  // built at the first use of the ordered law
};

namespace {
int fail(memb_plan* p, int code, const std::string& m) {
  if (p) p->err = m;
  return code;
}
#define MCHK(p, call)                                                                      \
  do {                                                                                     \
    hipError_t e_ = (call);                                                                \
    if (e_ != hipSuccess)                                                                  \
      return fail((p), MEMB_E_HIP, std::string(#call) + ": " + hipGetErrorString(e_));     \
  } while (0)

int upload(memb_plan* p, const std::vector<double>& h, const double** dst) {
  void* d = nullptr;
  MCHK(p, hipMalloc(&d, h.size() * sizeof(double)));
  p->bufs.push_back(d);
  MCHK(p, hipMemcpy(d, h.data(), h.size() * sizeof(double), hipMemcpyHostToDevice));
  *dst = (const double*)d;
  return MEMB_OK;
}

// ---- co-rotated frame of the surrogate ---------------------------------------------------------
// The law is invariant under translation and covariant under rotation of the current shape
// (f(R x + c) = R f(x)): its load depends on the capsule's deformation only.  One workgroup
// per capsule: centroid c, the cross-covariance H = sum (x_p - c) X_p^T against the
// stress-free points X, the rotation R = the orthogonal polar factor of H (the rotation that
// brings X closest to the shape, Kabsch), the displacement delta_p = R^T (x_p - c) - X_p, its
// RMS amplitude s and the direction delta / s.
constexpr int CR_THREADS = 256;

__device__ inline void inv3t(const double A[3][3], double B[3][3], double& det) {
  // B = inverse(A)^T
  const double c00 = A[1][1] * A[2][2] - A[1][2] * A[2][1];
  const double c01 = A[1][2] * A[2][0] - A[1][0] * A[2][2];
  const double c02 = A[1][0] * A[2][1] - A[1][1] * A[2][0];
  det = A[0][0] * c00 + A[0][1] * c01 + A[0][2] * c02;
  const double id = 1.0 / det;
  B[0][0] = c00 * id, B[0][1] = c01 * id, B[0][2] = c02 * id;
  B[1][0] = (A[0][2] * A[2][1] - A[0][1] * A[2][2]) * id;
  B[1][1] = (A[0][0] * A[2][2] - A[0][2] * A[2][0]) * id;
  B[1][2] = (A[0][1] * A[2][0] - A[0][0] * A[2][1]) * id;
  B[2][0] = (A[0][1] * A[1][2] - A[0][2] * A[1][1]) * id;
  B[2][1] = (A[0][2] * A[1][0] - A[0][0] * A[1][2]) * id;
  B[2][2] = (A[0][0] * A[1][1] - A[0][1] * A[1][0]) * id;
}

__global__ void __launch_bounds__(CR_THREADS)
    k_corot(int n, const double* __restrict__ X, const double* __restrict__ x,
            const double* __restrict__ y, const double* __restrict__ z,
            double* __restrict__ delta, double* __restrict__ dhx, double* __restrict__ dhy,
            double* __restrict__ dhz, double* __restrict__ rot, double* __restrict__ amp) {
  __shared__ double red[12][CR_THREADS / 64];
  __shared__ double sh[12];
  const long long cap = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const double* px = x + cap * n;
  const double* py = y + cap * n;
  const double* pz = z + cap * n;
  auto block_sum = [&](double* v, int k) {  // sums v[0..k) over the workgroup into sh
    for (int a = 0; a < k; ++a) {
      double t = v[a];
      for (int o = 32; o > 0; o >>= 1) t += __shfl_down(t, o);
      if (lane == 0) red[a][wv] = t;
    }
    __syncthreads();
    if (tid < k) {
      double t = 0.0;
      for (int w = 0; w < CR_THREADS / 64; ++w) t += red[tid][w];
      sh[tid] = t;
    }
    __syncthreads();
  };
  double v[12];
  v[0] = v[1] = v[2] = 0.0;
  for (int p = tid; p < n; p += CR_THREADS) v[0] += px[p], v[1] += py[p], v[2] += pz[p];
  block_sum(v, 3);
  const double c[3] = {sh[0] / n, sh[1] / n, sh[2] / n};
  __syncthreads();
  for (int a = 0; a < 9; ++a) v[a] = 0.0;
  for (int p = tid; p < n; p += CR_THREADS) {
    const double d[3] = {px[p] - c[0], py[p] - c[1], pz[p] - c[2]};
    const double r[3] = {X[p], X[n + p], X[2 * n + p]};
    for (int a = 0; a < 3; ++a)
      for (int b = 0; b < 3; ++b) v[3 * a + b] += d[a] * r[b];
  }
  block_sum(v, 9);
  __shared__ double R[3][3];
  __shared__ int ok;
  if (tid == 0) {
    // polar factor by Newton's iteration Y <- (Y + Y^-T) / 2 from the scaled H
    double Y[3][3], Z[3][3], det = 0.0, nrm = 0.0;
    for (int a = 0; a < 9; ++a) nrm += sh[a] * sh[a];
    nrm = sqrt(nrm / 3.0);
    for (int a = 0; a < 3; ++a)
      for (int b = 0; b < 3; ++b) Y[a][b] = nrm > 0.0 ? sh[3 * a + b] / nrm : (a == b ? 1.0 : 0.0);
    for (int it = 0; it < 24; ++it) {
      inv3t(Y, Z, det);
      for (int a = 0; a < 3; ++a)
        for (int b = 0; b < 3; ++b) Y[a][b] = 0.5 * (Y[a][b] + Z[a][b]);
    }
    inv3t(Y, Z, det);
    ok = isfinite(det) && det > 0.5;
    for (int a = 0; a < 3; ++a)
      for (int b = 0; b < 3; ++b) R[a][b] = Y[a][b], rot[cap * 9 + 3 * a + b] = Y[a][b];
  }
  __syncthreads();
  // delta = R^T (x - c) - X, layout [cap][3][n]
  double ss = 0.0;
  for (int p = tid; p < n; p += CR_THREADS) {
    const double d[3] = {px[p] - c[0], py[p] - c[1], pz[p] - c[2]};
    for (int a = 0; a < 3; ++a) {
      const double q = R[0][a] * d[0] + R[1][a] * d[1] + R[2][a] * d[2] - X[a * n + p];
      delta[(cap * 3 + a) * n + p] = q;
      ss += q * q;
    }
  }
  v[0] = ss;
  block_sum(v, 1);
  const double s = sqrt(sh[0] / n);
  const double inv = s > 0.0 ? 1.0 / s : 0.0;
  for (int p = tid; p < n; p += CR_THREADS) {
    dhx[cap * n + p] = delta[(cap * 3 + 0) * n + p] * inv;
    dhy[cap * n + p] = delta[(cap * 3 + 1) * n + p] * inv;
    dhz[cap * n + p] = delta[(cap * 3 + 2) * n + p] * inv;
  }
  if (tid == 0) amp[cap] = ok ? s : __builtin_inf();
}

// f = R (flin + s^2 resid) per point, into the capsule-major traction arrays
__global__ void __launch_bounds__(256)
    k_corot_apply(long long ncap, int n, const double* __restrict__ flin,
                  const float* __restrict__ resid, const double* __restrict__ rot,
                  const double* __restrict__ amp, double* __restrict__ fx,
                  double* __restrict__ fy, double* __restrict__ fz) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= ncap * n) return;
  const long long cap = q / n;
  const int p = (int)(q - cap * n);
  const double s2 = amp[cap] * amp[cap];
  double g[3];
  for (int a = 0; a < 3; ++a) {
    const long long o = (cap * 3 + a) * n + p;
    g[a] = flin[o] + (resid ? s2 * (double)resid[o] : 0.0);
  }
  const double* R = rot + cap * 9;
  fx[q] = R[0] * g[0] + R[1] * g[1] + R[2] * g[2];
  fy[q] = R[3] * g[0] + R[4] * g[1] + R[5] * g[2];
  fz[q] = R[6] * g[0] + R[7] * g[1] + R[8] * g[2];
}

// The anchored surrogate's prediction and gate, one workgroup per capsule (rows of 3n values,
// component-major: [c][3][n]):
//   cc = <delta, delta0> / |delta0|^2 (0 when delta0 = 0), drift = sqrt(sum (delta - delta0)^2 / n),
//   f' = (lin + cc^2 m0) + b (m0 = NULL: f' = lin + b), f = R f' into fx, fy, fz,
//   sel = 1 unless beta drift <= tol and every f is finite; drift_out (optional).
// pre (optional): capsules with pre[c] != 0 (already rejected by the drift test, k_anch_gate)
// are left to the law: sel[c] = 1, nothing else written.  late (optional): 1 for the other
// capsules this kernel rejects (their prediction is not finite), else 0.
__global__ void __launch_bounds__(CR_THREADS)
    k_anch_predict(int n, const double* __restrict__ lin, const double* __restrict__ m0,
                   const double* __restrict__ b, const double* __restrict__ delta,
                   const double* __restrict__ delta0, const double* __restrict__ rot,
                   double beta, double tol, double* __restrict__ fx, double* __restrict__ fy,
                   double* __restrict__ fz, int* __restrict__ sel,
                   double* __restrict__ drift_out, const int* __restrict__ pre,
                   int* __restrict__ late) {
  __shared__ double red[3][CR_THREADS / 64];
  __shared__ int bad;
  const long long cap = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const long long r0 = cap * 3 * n;
  if (pre && pre[cap]) {
    if (tid == 0) {
      sel[cap] = 1;
      if (late) late[cap] = 0;
    }
    return;
  }
  if (tid == 0) bad = 0;
  double v[3] = {0.0, 0.0, 0.0};
  for (int q = tid; q < 3 * n; q += CR_THREADS) {
    const double d = delta[r0 + q], d0 = delta0[r0 + q], e = d - d0;
    v[0] += d * d0, v[1] += d0 * d0, v[2] += e * e;
  }
  for (int a = 0; a < 3; ++a) {
    double t = v[a];
    for (int o = 32; o > 0; o >>= 1) t += __shfl_down(t, o);
    if (lane == 0) red[a][wv] = t;
  }
  __syncthreads();
  double sdd0 = 0.0, s00 = 0.0, sdr = 0.0;
  for (int w = 0; w < CR_THREADS / 64; ++w) sdd0 += red[0][w], s00 += red[1][w], sdr += red[2][w];
  const double c = s00 > 0.0 ? sdd0 / s00 : 0.0, c2 = c * c;
  const double drift = sqrt(sdr / (double)n);
  const double* R = rot + cap * 9;
  int nonfinite = 0;
  for (int p = tid; p < n; p += CR_THREADS) {
    double g[3];
    for (int a = 0; a < 3; ++a) {
      const long long o = r0 + (long long)a * n + p;
      g[a] = (m0 ? lin[o] + c2 * m0[o] : lin[o]) + b[o];
    }
    const long long q = cap * n + p;
    const double ox = R[0] * g[0] + R[1] * g[1] + R[2] * g[2];
    const double oy = R[3] * g[0] + R[4] * g[1] + R[5] * g[2];
    const double oz = R[6] * g[0] + R[7] * g[1] + R[8] * g[2];
    fx[q] = ox, fy[q] = oy, fz[q] = oz;
    nonfinite |= !(isfinite(ox) && isfinite(oy) && isfinite(oz));
  }
  if (nonfinite) atomicOr(&bad, 1);
  __syncthreads();
  if (tid == 0) {
    sel[cap] = (beta * drift <= tol && !bad) ? 0 : 1;
    if (late) late[cap] = sel[cap];
    if (drift_out) drift_out[cap] = drift;
  }
}

// The drift test of k_anch_predict alone (the same sums in the same order, so the same
// drift): pre[c] = 1 unless beta rms(delta - delta0) <= tol.  The law can then start on these
// capsules while the linear response is computed for the others.
__global__ void __launch_bounds__(CR_THREADS)
    k_anch_gate(int n, const double* __restrict__ delta, const double* __restrict__ delta0,
                double beta, double tol, int* __restrict__ pre) {
  __shared__ double red[CR_THREADS / 64];
  const long long cap = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const long long r0 = cap * 3 * n;
  double v = 0.0;
  for (int q = tid; q < 3 * n; q += CR_THREADS) {
    const double e = delta[r0 + q] - delta0[r0 + q];
    v += e * e;
  }
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o);
  if (lane == 0) red[wv] = v;
  __syncthreads();
  if (tid == 0) {
    double sdr = 0.0;
    for (int w = 0; w < CR_THREADS / 64; ++w) sdr += red[w];
    const double drift = sqrt(sdr / (double)n);
    pre[cap] = beta * drift <= tol ? 0 : 1;
  }
}

// New anchors for the capsules with sel != 0 (the law has just written their traction):
//   b = R^T f - lin (- m_now), delta0 = delta, m0 = m_now, s0 = amp, refreshed += 1.
// slot (optional): m_now holds rows only for the capsules with slot[c] >= 0 (row slot[c]); a
// selected capsule without a row keeps its old anchor (its traction this step is the law's
// all the same, and it is selected again at the next step).
__global__ void __launch_bounds__(CR_THREADS)
    k_anch_update(int n, const int* __restrict__ sel, const int* __restrict__ slot,
                  const double* __restrict__ rot, const double* __restrict__ fx,
                  const double* __restrict__ fy, const double* __restrict__ fz,
                  const double* __restrict__ lin, const double* __restrict__ m_now,
                  const double* __restrict__ delta, const double* __restrict__ amp,
                  double* __restrict__ b, double* __restrict__ delta0, double* __restrict__ m0,
                  double* __restrict__ s0, long long* __restrict__ refreshed) {
  const long long cap = blockIdx.x;
  if (sel[cap] == 0) return;
  const int tid = threadIdx.x;
  if (tid == 0) refreshed[cap] += 1;
  const long long row = slot ? (long long)slot[cap] : cap;
  if (row < 0) return;
  const long long r0 = cap * 3 * n, m_r0 = row * 3 * n;
  const double* R = rot + cap * 9;
  for (int p = tid; p < n; p += CR_THREADS) {
    const long long q = cap * n + p;
    const double f0 = fx[q], f1 = fy[q], f2 = fz[q];
    const double g[3] = {R[0] * f0 + R[3] * f1 + R[6] * f2, R[1] * f0 + R[4] * f1 + R[7] * f2,
                         R[2] * f0 + R[5] * f1 + R[8] * f2};
    for (int a = 0; a < 3; ++a) {
      const long long o = r0 + (long long)a * n + p;
      double bl = g[a] - lin[o];
      if (m_now) {
        const double mn = m_now[m_r0 + (long long)a * n + p];
        bl = bl - mn;
        m0[o] = mn;
      }
      b[o] = bl;
      delta0[o] = delta[o];
    }
  }
  if (tid == 0 && m_now && s0) s0[cap] = amp[cap];
}

// The first k capsules with sel != 0, in capsule order: idx[r] = c (padded with 0) and
// slot[c] = r, or -1 for the others and for selected capsules beyond k.  One workgroup.
constexpr int CS_THREADS = 1024;
__global__ void __launch_bounds__(CS_THREADS)
    k_compact_sel(long long ncap, const int* __restrict__ sel, int k, int* __restrict__ idx,
                  int* __restrict__ slot) {
  __shared__ int wsum[CS_THREADS / 64];
  __shared__ int base;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  if (tid == 0) base = 0;
  for (int r = tid; r < k; r += CS_THREADS) idx[r] = 0;
  __syncthreads();
  for (long long c0 = 0; c0 < ncap; c0 += CS_THREADS) {
    const long long c = c0 + tid;
    const bool on = c < ncap && sel[c] != 0;
    const unsigned long long bal = __ballot(on);
    if (lane == 0) wsum[wv] = __popcll(bal);
    __syncthreads();
    int before = 0, total = 0;
    for (int w = 0; w < CS_THREADS / 64; ++w) {
      before += w < wv ? wsum[w] : 0;
      total += wsum[w];
    }
    const int r = base + before + __popcll(bal & __lanemask_lt());
    if (c < ncap) {
      const bool kept = on && r < k;
      slot[c] = kept ? r : -1;
      if (kept) idx[r] = (int)c;
    }
    __syncthreads();
    if (tid == 0) base += total;
    __syncthreads();
  }
}

// LDS of the three kernels (bytes)
size_t lds_shape(const Tables& T) {
  const int NN = T.N * T.N;
  return (size_t)(T.np2 + 3 * T.NT + 6 * NN) * sizeof(double2);
}
size_t lds_nodes(const Tables& T, bool bend) {
  return (size_t)(T.np + 3 * T.NT + AB_SLOTS * 3 * (bend ? 5 : 3) * T.N) * sizeof(double2) +
         (size_t)F_SLOTS * T.slots() * 6 * sizeof(double);
}
size_t lds_filter(const Tables& T) {
  const int NN = T.N * T.N;
  return (size_t)(T.np2 + 3 * T.NT + std::max(FL_STAGE * 6 * T.N, 3 * NN)) * sizeof(double2);
}

// The law of ncap capsules (those with sel != 0), in batches of the plan's slots.
int run_law(memb_plan* p, long long ncap, double gs, double eb, const double* x, const double* y,
            const double* z, double* fx, double* fy, double* fz, double* nx, double* ny,
            double* nz, double* area, const int* sel) {
  const Tables& T = p->T;
  const int most = p->nodes_wg[eb != 0.0];
  for (long long c0 = 0; c0 < ncap; c0 += p->slots) {
    const int n = (int)std::min<long long>(p->slots, ncap - c0);
    Work w{};
    w.n = n, w.c0 = c0, w.coef = p->coef, w.rows = p->rows;
    if (sel) {
      w.list = p->list, w.cnt = p->list + p->slots;
      k_select<<<1, SL_THREADS, 0, p->stream>>>(n, sel, c0, p->list, p->list + p->slots);
    }
    k_shape<SHAPE_LAW><<<n, SH_THREADS, lds_shape(T), p->stream>>>(
        T, w, x, y, z, nullptr, nullptr, nullptr, area, nullptr, nullptr);
    const int gn = (int)std::min<long long>(most, (long long)n * T.nt);
    if (eb != 0.0)
      k_nodes<false, true><<<gn, ND_THREADS, lds_nodes(T, true), p->stream>>>(T, w, most, gs, eb,
                                                                             nullptr);
    else
      k_nodes<false, false><<<gn, ND_THREADS, lds_nodes(T, false), p->stream>>>(T, w, most, gs,
                                                                               eb, nullptr);
    k_filter<<<2 * n <= p->num_wg ? 2 * n : n, SH_THREADS, lds_filter(T), p->stream>>>(
        T, w, p->num_wg, fx, fy, fz, nx, ny, nz);
  }
  MCHK(p, hipGetLastError());
  return MEMB_OK;
}
}  // namespace

extern "C" {

int memb_plan_create(memb_plan** out, int L, int device) {
  if (!out || L < 2 || L > LMAX) return MEMB_E_ARG;
  *out = nullptr;
  memb_plan* p = new memb_plan();
  p->device = device, p->L = L;
  int rc;
  auto bail = [&](int code) {
    *out = p;  // keep the message readable through memb_last_error
    return code;
  };
  if (hipSetDevice(device) != hipSuccess) return bail(fail(p, MEMB_E_HIP, "hipSetDevice failed"));
  if (hipStreamCreate(&p->own) != hipSuccess)
    return bail(fail(p, MEMB_E_HIP, "hipStreamCreate failed"));
  p->stream = p->own;
  Tables& T = p->T;
  T.L = L, T.N = L + 1, T.np2 = 2 * (L + 1), T.nt = 2 * T.N, T.np = 2 * T.np2;
  T.NT = T.N * (T.N + 1) / 2;
  const int N = T.N, nt = T.nt, np = T.np, np2 = T.np2, NT = T.NT, nh = (N + 1) / 2;
  std::vector<double> th2(N), w2(N), th(nt), w(nt), s2(N);
  gauss(N, th2.data(), w2.data());
  gauss(nt, th.data(), w.data());
  for (int i = 0; i < N; ++i) s2[i] = std::sin(th2[i]);
  std::vector<double> WPc((size_t)N * NT), Pc((size_t)nh * NT), Pcd((size_t)nh * NT),
      Pfd((size_t)N * 5 * NT), WPf((size_t)N * NT), D(5 * N * N);
  auto each = [&](auto&& f) {  // f(packed index, index into D's [m][n])
    for (int d = 0; d < N; ++d)
      for (int m = 0; m < N - d; ++m) f(tidx(N, d, m), m * N + m + d);
  };
  for (int i = 0; i < N; ++i) {
    legendre_derivs(N, th2[i], D.data());
    each([&](int t, int q) {
      WPc[(size_t)i * NT + t] = w2[i] * D[q];
      if (i < nh) Pc[(size_t)i * NT + t] = D[q], Pcd[(size_t)i * NT + t] = D[N * N + q];
    });
    legendre_derivs(N, th[i], D.data());  // the northern half of the doubled grid
    each([&](int t, int q) {
      for (int k = 0; k < 5; ++k) Pfd[((size_t)i * 5 + k) * NT + t] = D[k * N * N + q];
      WPf[(size_t)i * NT + t] = w[i] * D[q];
    });
  }
  // cos / sin(m phi_j) is entry (m j) mod n of cos / sin(2 pi q / n): the angle is reduced first,
  // as the longitude FFT's twiddle factors are formed (hrfft.f:214-267): exact to the last bit
  // of cos / sin of an angle below 2 pi, where m phi_j itself (up to 2 pi L) carries 1e-14 of
  // rounding that the fourth phi derivatives multiply by m^4
  auto unit = [](int n) {
    std::vector<double> e(2 * (size_t)n);
    for (int q = 0; q < n; ++q) {
      const double a = 2.0 * M_PI * q / n;
      e[2 * q] = std::cos(a), e[2 * q + 1] = std::sin(a);
    }
    return e;
  };
  const double *e2 = nullptr, *ef = nullptr;
  if ((rc = upload(p, w2, &T.w2)) || (rc = upload(p, s2, &T.s2)) || (rc = upload(p, WPc, &T.WPc)) ||
      (rc = upload(p, Pc, &T.Pc)) || (rc = upload(p, Pcd, &T.Pcd)) ||
      (rc = upload(p, Pfd, &T.Pfd)) || (rc = upload(p, WPf, &T.WPf)) ||
      (rc = upload(p, unit(np2), &e2)) || (rc = upload(p, unit(np), &ef)))
    return bail(rc);
  T.e2 = reinterpret_cast<const double2*>(e2), T.ef = reinterpret_cast<const double2*>(ef);
  int cus = 256;
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device);
  p->num_wg = 4 * cus;
  // capsules per batch; half as many would halve the plan's 128 MB (degree 16), but 8000 capsules
  // then take 2866 us instead of 2811, a ragged end more often
  p->slots = 8 * cus;
  auto alloc = [&](auto** d, size_t bytes) {
    void* q = nullptr;
    if (hipMalloc(&q, bytes) != hipSuccess) return false;
    p->bufs.push_back(q);
    *d = reinterpret_cast<std::remove_reference_t<decltype(**d)>*>(q);
    return true;
  };
  if (!alloc(&p->coef, (size_t)p->slots * 3 * NT * sizeof(double2)) ||
      !alloc(&p->rows, (size_t)p->slots * nt * N * 6 * sizeof(double2)) ||
      !alloc(&p->list, (size_t)(p->slots + 1) * sizeof(int)) ||
      !alloc(&p->ref, (size_t)NREF * nt * T.slots() * sizeof(double)))
    return bail(fail(p, MEMB_E_HIP, "hipMalloc of the plan's work arrays failed"));
  // the reference state: the unit sphere through the same kernels (sph.f90:56-70, 152-161)
  std::vector<double> sx((size_t)N * np2 * 3);
  sphere(N, np2, th2.data(), sx.data());
  const double* dsx = nullptr;
  if ((rc = upload(p, sx, &dsx))) return bail(rc);
  auto big = [&](const void* f, size_t lds) {
    return hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess;
  };
  if (!big((const void*)k_shape<SHAPE_LAW>, lds_shape(T)) ||
      !big((const void*)k_shape<SHAPE_COEFFS>, lds_shape(T)) ||
      !big((const void*)k_shape<SHAPE_GEOM>, lds_shape(T)) ||
      !big((const void*)k_shape<SHAPE_REF>, lds_shape(T)) ||
      !big((const void*)k_nodes<true, true>, lds_nodes(T, true)) ||
      !big((const void*)k_nodes<false, true>, lds_nodes(T, true)) ||
      !big((const void*)k_nodes<false, false>, lds_nodes(T, false)) ||
      !big((const void*)k_filter, lds_filter(T)))
    return bail(fail(p, MEMB_E_HIP, "hipFuncSetAttribute failed"));
  // four per CU by the registers, three by the LDS from degree 19 on (without bending 22): cut for
  // four all the same, the runs of some hundred capsules made a thin second round (301 capsules of
  // degree 23: 425 us with bending and 278 without, 376 and 254 cut for three).  Low degrees without
  // bending have room for more, which is not always better: 301 capsules of degree 16 take
  // 109 us cut for four and 113 for five.
  for (int bend = 0; bend < 2; ++bend) {
    int per_cu = 0;
    const void* f = bend ? (const void*)k_nodes<false, true> : (const void*)k_nodes<false, false>;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, f, ND_THREADS,
                                                     lds_nodes(T, bend)) != hipSuccess)
      return bail(fail(p, MEMB_E_HIP, "occupancy of the node kernel failed"));
    p->nodes_wg[bend] = std::min(4, std::max(1, per_cu)) * cus;
  }
  T.ref = nullptr;
  Work wk{};
  wk.n = 1, wk.coef = p->coef, wk.rows = p->rows;
  k_shape<SHAPE_REF><<<1, SH_THREADS, lds_shape(T), p->stream>>>(
      T, wk, dsx, dsx + N * np2, dsx + 2 * N * np2, nullptr, nullptr, nullptr, nullptr, nullptr,
      nullptr);
  k_nodes<true, true><<<nt, ND_THREADS, lds_nodes(T, true), p->stream>>>(T, wk, nt, 0.0, 0.0,
                                                                        p->ref);
  if (hipGetLastError() != hipSuccess || hipStreamSynchronize(p->stream) != hipSuccess)
    return bail(fail(p, MEMB_E_HIP, "reference state failed"));
  T.ref = p->ref;
  *out = p;
  return MEMB_OK;
}

void memb_plan_destroy(memb_plan* p) {
  if (!p) return;
  (void)hipSetDevice(p->device);
  if (p->stream) (void)hipStreamSynchronize(p->stream);
  for (void* b : p->bufs) (void)hipFree(b);
  if (p->own) (void)hipStreamDestroy(p->own);
  delete p;
}

const char* memb_last_error(const memb_plan* p) { return p ? p->err.c_str() : "null plan"; }

int memb_set_stream(memb_plan* p, void* s) {
  if (!p) return MEMB_E_ARG;
  p->stream = s ? (hipStream_t)s : p->own;
  return MEMB_OK;
}

int memb_sync(memb_plan* p) {
  if (!p) return MEMB_E_ARG;
  MCHK(p, hipSetDevice(p->device));
  MCHK(p, hipStreamSynchronize(p->stream));
  return MEMB_OK;
}

int memb_npts(const memb_plan* p) { return p ? p->T.N * p->T.np2 : 0; }
int memb_ncoef(const memb_plan* p) { return p ? p->T.N * p->T.N : 0; }

int memb_traction_f64_dev(memb_plan* p, int64_t ncap, double gs, double eb, const double* x,
                          const double* y, const double* z, double* fx, double* fy, double* fz,
                          double* nx, double* ny, double* nz, double* area) {
  if (!p) return MEMB_E_ARG;
  if (!p->T.ref) return fail(p, MEMB_E_STATE, "plan not initialised");
  if (ncap < 0) return fail(p, MEMB_E_ARG, "ncap < 0");
  if (ncap > 0 && !(x && y && z && fx && fy && fz && nx && ny && nz && area))
    return fail(p, MEMB_E_ARG, "null pointer");
  MCHK(p, hipSetDevice(p->device));
  return run_law(p, ncap, gs, eb, x, y, z, fx, fy, fz, nx, ny, nz, area, nullptr);
}

// Tables and reference state of the ordered node phase, once per plan (waits).
static int ordered_tables(memb_plan* p) {
  if (p->O.ref) return MEMB_OK;
  const Tables& T = p->T;
  const int N = T.N, nt = T.nt, NT = T.NT, np2 = T.np2;
  std::vector<double> th(nt), w(nt), th2(N), w2(N), D(5 * N * N), Pfd((size_t)nt * 5 * NT);
  gauss(nt, th.data(), w.data());
  gauss(N, th2.data(), w2.data());
  for (int i = 0; i < nt; ++i) {
    legendre_derivs(N, th[i], D.data());
    for (int k = 0; k < 5; ++k)
      for (int d = 0; d < N; ++d)
        for (int m = 0; m < N - d; ++m)
          Pfd[((size_t)i * 5 + k) * NT + tidx(N, d, m)] = D[(k * N + m) * N + m + d];
  }
  int rc;
  if ((rc = upload(p, Pfd, &p->O.Pfd))) return rc;
  std::vector<double> sx((size_t)N * np2 * 3);
  sphere(N, np2, th2.data(), sx.data());
  const double* dsx = nullptr;
  if ((rc = upload(p, sx, &dsx))) return rc;
  void* ref = nullptr;
  MCHK(p, hipMalloc(&ref, (size_t)nt * T.np * ordered::NREF * sizeof(double)));
  p->bufs.push_back(ref);
  const int lds = (int)ordered::lds_bytes(T);
  MCHK(p, hipFuncSetAttribute((const void*)ordered::k_nodes_ordered<true>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, lds));
  MCHK(p, hipFuncSetAttribute((const void*)ordered::k_nodes_ordered<false>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, lds));
  Work wk{};
  wk.n = 1, wk.coef = p->coef, wk.rows = p->rows;
  k_shape<SHAPE_REF><<<1, SH_THREADS, lds_shape(T), p->stream>>>(
      T, wk, dsx, dsx + N * np2, dsx + 2 * N * np2, nullptr, nullptr, nullptr, nullptr, nullptr,
      nullptr);
  ordered::k_nodes_ordered<true><<<1, ordered::THREADS, lds, p->stream>>>(T, p->O, wk, 0.0, 0.0,
                                                                         (double*)ref);
  MCHK(p, hipGetLastError());
  MCHK(p, hipStreamSynchronize(p->stream));
  p->O.ref = (const double*)ref;
  return MEMB_OK;
}

int memb_traction_ordered_f64_dev(memb_plan* p, int64_t ncap, double gs, double eb,
                                  const double* x, const double* y, const double* z, double* fx,
                                  double* fy, double* fz, double* nx, double* ny, double* nz,
                                  double* area) {
  if (!p) return MEMB_E_ARG;
  if (!p->T.ref) return fail(p, MEMB_E_STATE, "plan not initialised");
  if (ncap < 0) return fail(p, MEMB_E_ARG, "ncap < 0");
  if (ncap > 0 && !(x && y && z && fx && fy && fz && nx && ny && nz && area))
    return fail(p, MEMB_E_ARG, "null pointer");
  MCHK(p, hipSetDevice(p->device));
  int rc = ordered_tables(p);
  if (rc) return rc;
  const Tables& T = p->T;
  for (long long c0 = 0; c0 < ncap; c0 += p->slots) {
    const int n = (int)std::min<long long>(p->slots, ncap - c0);
    Work w{};
    w.n = n, w.c0 = c0, w.coef = p->coef, w.rows = p->rows;
    k_shape<SHAPE_LAW><<<n, SH_THREADS, lds_shape(T), p->stream>>>(
        T, w, x, y, z, nullptr, nullptr, nullptr, area, nullptr, nullptr);
    ordered::k_nodes_ordered<false><<<n, ordered::THREADS, ordered::lds_bytes(T), p->stream>>>(
        T, p->O, w, gs, eb, nullptr);
    k_filter<<<2 * n <= p->num_wg ? 2 * n : n, SH_THREADS, lds_filter(T), p->stream>>>(
        T, w, p->num_wg, fx, fy, fz, nx, ny, nz);
  }
  MCHK(p, hipGetLastError());
  return MEMB_OK;
}

int memb_coeffs_f64_dev(memb_plan* p, int64_t ncap, const double* x, const double* y,
                        const double* z, double* coef) {
  if (!p) return MEMB_E_ARG;
  if (ncap < 0) return fail(p, MEMB_E_ARG, "ncap < 0");
  if (ncap > 0 && !(x && y && z && coef)) return fail(p, MEMB_E_ARG, "null pointer");
  MCHK(p, hipSetDevice(p->device));
  if (ncap == 0) return MEMB_OK;
  // (uses no slot: it may run beside the law on another stream)
  Work w{};
  w.n = (int)std::min<long long>(ncap, INT_MAX);
  if (ncap > w.n) return fail(p, MEMB_E_ARG, "more than 2^31 - 1 capsules");
  k_shape<SHAPE_COEFFS><<<(unsigned)std::min<long long>(ncap, p->num_wg), SH_THREADS,
                          lds_shape(p->T), p->stream>>>(p->T, w, x, y, z, nullptr, nullptr,
                                                        nullptr, nullptr, coef, nullptr);
  MCHK(p, hipGetLastError());
  return MEMB_OK;
}

int memb_geometry_f64_dev(memb_plan* p, int64_t ncap, const double* x, const double* y,
                          const double* z, double* nx, double* ny, double* nz, double* area,
                          const int* skip) {
  if (!p) return MEMB_E_ARG;
  if (ncap < 0) return fail(p, MEMB_E_ARG, "ncap < 0");
  if (ncap > 0 && !(x && y && z && nx && ny && nz && area))
    return fail(p, MEMB_E_ARG, "null pointer");
  MCHK(p, hipSetDevice(p->device));
  if (ncap == 0) return MEMB_OK;
  // (uses no slot: it may run beside the law on another stream)
  Work w{};
  w.n = (int)std::min<long long>(ncap, INT_MAX);
  if (ncap > w.n) return fail(p, MEMB_E_ARG, "more than 2^31 - 1 capsules");
  k_shape<SHAPE_GEOM><<<(unsigned)std::min<long long>(ncap, p->num_wg), SH_THREADS,
                        lds_shape(p->T), p->stream>>>(p->T, w, x, y, z, nx, ny, nz, area, nullptr,
                                                      skip);
  MCHK(p, hipGetLastError());
  return MEMB_OK;
}

int memb_traction_select_f64_dev(memb_plan* p, int64_t ncap, const int* sel, double gs,
                                 double eb, const double* x, const double* y, const double* z,
                                 double* fx, double* fy, double* fz, double* nx, double* ny,
                                 double* nz, double* area) {
  if (!p) return MEMB_E_ARG;
  if (!p->T.ref) return fail(p, MEMB_E_STATE, "plan not initialised");
  if (ncap < 0) return fail(p, MEMB_E_ARG, "ncap < 0");
  if (ncap > 0 && !(sel && x && y && z && fx && fy && fz && nx && ny && nz && area))
    return fail(p, MEMB_E_ARG, "null pointer");
  MCHK(p, hipSetDevice(p->device));
  return run_law(p, ncap, gs, eb, x, y, z, fx, fy, fz, nx, ny, nz, area, sel);
}

int memb_corot_f64_dev(memb_plan* p, int64_t ncap, const double* X, const double* x,
                       const double* y, const double* z, double* delta, double* dhx,
                       double* dhy, double* dhz, double* rot, double* amp) {
  if (!p) return MEMB_E_ARG;
  if (ncap < 0) return fail(p, MEMB_E_ARG, "ncap < 0");
  if (ncap > 0 && !(X && x && y && z && delta && dhx && dhy && dhz && rot && amp))
    return fail(p, MEMB_E_ARG, "null pointer");
  if (ncap == 0) return MEMB_OK;
  MCHK(p, hipSetDevice(p->device));
  k_corot<<<(unsigned)ncap, CR_THREADS, 0, p->stream>>>(p->T.N * p->T.np2, X, x, y, z, delta,
                                                         dhx, dhy, dhz, rot, amp);
  MCHK(p, hipGetLastError());
  return MEMB_OK;
}

int memb_anchored_predict_f64_dev(memb_plan* p, int64_t ncap, const double* lin,
                                  const double* m0, const double* b, const double* delta,
                                  const double* delta0, const double* rot, double beta,
                                  double tol, double* fx, double* fy, double* fz, int* sel,
                                  double* drift, const int* pre, int* late) {
  if (!p) return MEMB_E_ARG;
  if (ncap < 0) return fail(p, MEMB_E_ARG, "ncap < 0");
  if (ncap > 0 && !(lin && b && delta && delta0 && rot && fx && fy && fz && sel))
    return fail(p, MEMB_E_ARG, "null pointer");
  if (ncap == 0) return MEMB_OK;
  MCHK(p, hipSetDevice(p->device));
  const int n = p->T.N * p->T.np2;
  k_anch_predict<<<(unsigned)ncap, CR_THREADS, 0, p->stream>>>(n, lin, m0, b, delta, delta0, rot,
                                                              beta, tol, fx, fy, fz, sel, drift,
                                                              pre, late);
  MCHK(p, hipGetLastError());
  return MEMB_OK;
}

int memb_anchored_gate_f64_dev(memb_plan* p, int64_t ncap, const double* delta,
                               const double* delta0, double beta, double tol, int* pre) {
  if (!p) return MEMB_E_ARG;
  if (ncap < 0) return fail(p, MEMB_E_ARG, "ncap < 0");
  if (ncap > 0 && !(delta && delta0 && pre)) return fail(p, MEMB_E_ARG, "null pointer");
  if (ncap == 0) return MEMB_OK;
  MCHK(p, hipSetDevice(p->device));
  const int n = p->T.N * p->T.np2;
  k_anch_gate<<<(unsigned)ncap, CR_THREADS, 0, p->stream>>>(n, delta, delta0, beta, tol, pre);
  MCHK(p, hipGetLastError());
  return MEMB_OK;
}

int memb_anchored_update_f64_dev(memb_plan* p, int64_t ncap, const int* sel, const int* slot,
                                 const double* rot, const double* fx, const double* fy,
                                 const double* fz, const double* lin, const double* m_now,
                                 const double* delta, const double* amp, double* b,
                                 double* delta0, double* m0, double* s0, int64_t* refreshed) {
  if (!p) return MEMB_E_ARG;
  if (ncap < 0) return fail(p, MEMB_E_ARG, "ncap < 0");
  if (ncap > 0 && !(sel && rot && fx && fy && fz && lin && delta && amp && b && delta0 &&
                    refreshed))
    return fail(p, MEMB_E_ARG, "null pointer");
  if (m_now && !m0) return fail(p, MEMB_E_ARG, "m_now needs m0");
  if (ncap == 0) return MEMB_OK;
  MCHK(p, hipSetDevice(p->device));
  const int n = p->T.N * p->T.np2;
  k_anch_update<<<(unsigned)ncap, CR_THREADS, 0, p->stream>>>(n, sel, slot, rot, fx, fy, fz, lin,
                                                             m_now, delta, amp, b, delta0, m0,
                                                             s0, (long long*)refreshed);
  MCHK(p, hipGetLastError());
  return MEMB_OK;
}

int memb_compact_sel_dev(memb_plan* p, int64_t ncap, const int* sel, int k, int* idx,
                         int* slot) {
  if (!p) return MEMB_E_ARG;
  if (ncap < 0 || k < 1) return fail(p, MEMB_E_ARG, "ncap < 0 or k < 1");
  if (!(sel && idx && slot)) return fail(p, MEMB_E_ARG, "null pointer");
  if (ncap > 0x7fffffffLL) return fail(p, MEMB_E_ARG, "more than 2^31 - 1 capsules");
  MCHK(p, hipSetDevice(p->device));
  k_compact_sel<<<1, CS_THREADS, 0, p->stream>>>(ncap, sel, k, idx, slot);
  MCHK(p, hipGetLastError());
  return MEMB_OK;
}

int memb_corot_apply_f64_dev(memb_plan* p, int64_t ncap, const double* flin, const float* resid,
                             const double* rot, const double* amp, double* fx, double* fy,
                             double* fz) {
  if (!p) return MEMB_E_ARG;
  if (ncap < 0) return fail(p, MEMB_E_ARG, "ncap < 0");
  if (ncap > 0 && !(flin && rot && amp && fx && fy && fz))
    return fail(p, MEMB_E_ARG, "null pointer");
  if (ncap == 0) return MEMB_OK;
  MCHK(p, hipSetDevice(p->device));
  const int n = p->T.N * p->T.np2;
  const long long tot = ncap * n;
  k_corot_apply<<<(unsigned)((tot + 255) / 256), 256, 0, p->stream>>>(ncap, n, flin, resid, rot,
                                                                      amp, fx, fy, fz);
  MCHK(p, hipGetLastError());
  return MEMB_OK;
}

}  // extern "C"
