// law_ordered.hpp -- the node phase of the membrane law in the oracle's order of operations, for
// the Jacobian of the surrogate.
//
// The Jacobian's central differences divide differences of the law by 2e-6, so what limits
// them is the rounding of the law: 1e-7 of the second-order remainder that an anchor stores.
// Surrogates are saved with their Jacobian and calibrated gates, so the Jacobian is built with the
// arithmetic it has always been built with, and a rebuilt surrogate agrees with a saved one to
// 1e-12 instead of to that rounding: the Legendre sums of every ring in index order from the
// ring's own table, the geometry through contravariant vectors and the derivatives of the
// normal, every entry of a symmetric tensor by its own sum.  The law itself (k_nodes) does the
// same with fewer operations: 1734 capsules of degree 16 take 0.47 ms in its node phase, 1.10 ms
// in this one.
// Shape and filter round at the size of their results and are the law's own.
#pragma once

namespace memb {
namespace ordered {

constexpr int NREF = 56;      // reference-state doubles per fine node
constexpr int THREADS = 128;

// What the ordered node phase reads besides the law's tables
struct OrderedTables {
  const double* Pfd;           // [nt][5][NT] fine theta-derivatives 0..4 of every ring
  const double* ref;           // [nt * np][NREF] unit-sphere state
};

struct Geom {
  double a[2][3], n[3], J;
  double g[2][2], gd[2][2][2];
  double G[2][2], Gd[2][2][2], Gdd[2][2][2][2];
  double b[2][2], bd[2][2][2], bdd[2][2][2][2];
  double Gam[2][2][2], Gamd[2][2][2][2];
};

__device__ inline void mul2(const double X[2][2], const double Y[2][2], double R[2][2]) {
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) R[i][j] = X[i][0] * Y[0][j] + X[i][1] * Y[1][j];
}

// X[c][q]: derivatives of coordinate c; returns the node geometry
__device__ __forceinline__ void geometry(const double (*X)[NQ], Geom& o) {
  double x1[2][3], x2[2][2][3], x3[2][2][2][3], x4[2][2][2][2][3];
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      x1[a][k] = X[k][qidx(1 - a, a)];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        x2[a][b][k] = X[k][qidx(2 - a - b, a + b)];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          x3[a][b][c][k] = X[k][qidx(3 - a - b - c, a + b + c)];
#pragma unroll
          for (int d = 0; d < 2; ++d) x4[a][b][c][d][k] = X[k][qidx(4 - a - b - c - d, a + b + c + d)];
        }
      }
    }
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int k = 0; k < 3; ++k) o.a[a][k] = x1[a][k];
  double cv[3], nd[2][3];
  cross3(x1[0], x1[1], cv);
  o.J = sqrt(dot3(cv, cv));
  const double rJ = 1.0 / o.J;  // one division per node; the others multiply by it
#pragma unroll
  for (int k = 0; k < 3; ++k) o.n[k] = cv[k] * rJ;
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    double t1[3], t2[3], cd[3];
    cross3(x2[0][c], x1[1], t1);
    cross3(x1[0], x2[1][c], t2);
#pragma unroll
    for (int k = 0; k < 3; ++k) cd[k] = t1[k] + t2[k];
    const double Jd = dot3(o.n, cd);
#pragma unroll
    for (int k = 0; k < 3; ++k) nd[c][k] = (cd[k] - Jd * o.n[k]) * rJ;
  }
  double gdd[2][2][2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      o.g[a][b] = dot3(x1[a], x1[b]);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        o.gd[c][a][b] = dot3(x2[a][c], x1[b]) + dot3(x1[a], x2[b][c]);
#pragma unroll
        for (int d = 0; d < 2; ++d)
          gdd[c][d][a][b] = dot3(x3[a][c][d], x1[b]) + dot3(x2[a][c], x2[b][d]) +
                            dot3(x2[a][d], x2[b][c]) + dot3(x1[a], x3[b][c][d]);
      }
    }
  const double det = o.g[0][0] * o.g[1][1] - o.g[0][1] * o.g[1][0];
  const double rdet = 1.0 / det;
  o.G[0][0] = o.g[1][1] * rdet, o.G[1][1] = o.g[0][0] * rdet;
  o.G[0][1] = -o.g[0][1] * rdet, o.G[1][0] = -o.g[1][0] * rdet;
  double GdgG[2][2][2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    double t[2][2], u[2][2];
    mul2(o.G, o.gd[c], t);
    mul2(t, o.G, u);
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) GdgG[c][a][b] = u[a][b], o.Gd[c][a][b] = -u[a][b];
  }
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      double t1[2][2], t2[2][2], t3[2][2], t4[2][2], t5[2][2], gcd[2][2];
      mul2(GdgG[d], o.gd[c], t1);
      mul2(t1, o.G, t2);
      mul2(GdgG[c], o.gd[d], t3);
      mul2(t3, o.G, t4);
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) gcd[a][b] = gdd[c][d][a][b];
      mul2(o.G, gcd, t1);
      mul2(t1, o.G, t5);
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) o.Gdd[c][d][a][b] = t2[a][b] + t4[a][b] - t5[a][b];
    }
  double ac[2][3], acd[2][2][3];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      ac[a][k] = o.G[a][0] * x1[0][k] + o.G[a][1] * x1[1][k];
#pragma unroll
      for (int c = 0; c < 2; ++c)
        acd[c][a][k] = o.Gd[c][a][0] * x1[0][k] + o.Gd[c][a][1] * x1[1][k] +
                       o.G[a][0] * x2[0][c][k] + o.G[a][1] * x2[1][c][k];
    }
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      o.b[a][b] = dot3(x2[a][b], o.n);
#pragma unroll
      for (int c = 0; c < 2; ++c) o.bd[c][a][b] = dot3(x3[a][b][c], o.n) + dot3(x2[a][b], nd[c]);
    }
  double ndd[2][2][3];
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        double s = 0.0;
#pragma unroll
        for (int l = 0; l < 2; ++l) s += o.bd[d][c][l] * ac[l][k] + o.b[c][l] * acd[d][l][k];
        ndd[c][d][k] = -s;
      }
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
          o.bdd[c][d][a][b] = dot3(x4[a][b][c][d], o.n) + dot3(x3[a][b][c], nd[d]) +
                              dot3(x3[a][b][d], nd[c]) + dot3(x2[a][b], ndd[c][d]);
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        o.Gam[b][a][c] = dot3(x2[a][c], ac[b]);
#pragma unroll
        for (int l = 0; l < 2; ++l)
          o.Gamd[l][b][a][c] = dot3(x3[a][c][l], ac[b]) + dot3(x2[a][c], acd[l][b]);
      }
}

// load q1 a1 + q2 a2 + q3 n at one node (sph.f90:1615-1700; membmodel.c:60-79)
__device__ __forceinline__ void law(const Geom& o, const double* __restrict__ R, double gs, double eb,
                    double f[3]) {
  double A[2][2], Ad[2][2][2], Add[2][2][2][2], B[2][2], Bd[2][2][2], Bdd[2][2][2][2];
#pragma unroll
  for (int q = 0; q < 4; ++q) (&A[0][0])[q] = R[q], (&B[0][0])[q] = R[28 + q];
#pragma unroll
  for (int q = 0; q < 8; ++q) (&Ad[0][0][0])[q] = R[4 + q], (&Bd[0][0][0])[q] = R[32 + q];
#pragma unroll
  for (int q = 0; q < 16; ++q) (&Add[0][0][0][0])[q] = R[12 + q], (&Bdd[0][0][0][0])[q] = R[40 + q];
  const double detA = A[0][0] * A[1][1] - A[0][1] * A[0][1];
  const double deta = o.g[0][0] * o.g[1][1] - o.g[0][1] * o.g[0][1];
  const double I2 = detA * deta - 1.0;
  const double Js = sqrt(1.0 + I2);
  const double rJs = 1.0 / Js, rI = 1.0 / (I2 + 1.0);  // one division each
  double I2d[2], Jsd[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const double dA = Ad[c][0][0] * A[1][1] + A[0][0] * Ad[c][1][1] - 2.0 * A[0][1] * Ad[c][0][1];
    const double da = o.gd[c][0][0] * o.g[1][1] + o.g[0][0] * o.gd[c][1][1] -
                      2.0 * o.g[0][1] * o.gd[c][0][1];
    I2d[c] = dA * deta + da * detA;
    Jsd[c] = 0.5 * rJs * I2d[c];
  }
  const double w1 = 0.5 * gs;
  const double w2 = -0.5 * gs * (rI * rI);
  double w2d[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) w2d[c] = gs * (rI * rI * rI) * I2d[c];
  double T[2][2], Td[2][2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      T[a][b] = 2.0 * rJs * w1 * A[a][b] + 2.0 * Js * w2 * o.G[a][b];
#pragma unroll
      for (int c = 0; c < 2; ++c)
        Td[c][a][b] = -2.0 * (rJs * rJs) * Jsd[c] * w1 * A[a][b] + 2.0 * rJs * w1 * Ad[c][a][b] +
                      2.0 * Jsd[c] * w2 * o.G[a][b] + 2.0 * Js * w2d[c] * o.G[a][b] +
                      2.0 * Js * w2 * o.Gd[c][a][b];
    }
  double q[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    double s = Td[0][0][b] + Td[1][1][b];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int l = 0; l < 2; ++l) s += o.Gam[a][a][l] * T[l][b] + o.Gam[b][a][l] * T[a][l];
    q[b] = s;
  }
  double q3 = 0.0;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) q3 += T[a][b] * o.b[a][b];
  if (eb != 0.0) {
    double K[2][2], Kd[2][2][2], Kdd[2][2][2][2];
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        double s = 0.0;
#pragma unroll
        for (int cp = 0; cp < 2; ++cp) s += A[cp][a] * B[c][cp] - o.G[cp][a] * o.b[c][cp];
        K[c][a] = s;
#pragma unroll
        for (int l = 0; l < 2; ++l) {
          double t = 0.0;
#pragma unroll
          for (int cp = 0; cp < 2; ++cp)
            t += Ad[l][cp][a] * B[c][cp] + A[cp][a] * Bd[l][c][cp] - o.Gd[l][cp][a] * o.b[c][cp] -
                 o.G[cp][a] * o.bd[l][c][cp];
          Kd[l][c][a] = t;
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            double u = 0.0;
#pragma unroll
            for (int cp = 0; cp < 2; ++cp)
              u += Add[l][k][cp][a] * B[c][cp] + Ad[k][cp][a] * Bd[l][c][cp] +
                   Ad[l][cp][a] * Bd[k][c][cp] + A[cp][a] * Bdd[l][k][c][cp] -
                   o.Gdd[l][k][cp][a] * o.b[c][cp] - o.Gd[k][cp][a] * o.bd[l][c][cp] -
                   o.Gd[l][cp][a] * o.bd[k][c][cp] - o.G[cp][a] * o.bdd[l][k][c][cp];
            Kdd[l][k][c][a] = u;
          }
        }
      }
    double M[2][2], Md[2][2][2], dds = 0.0;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        double m = 0.0, md0 = 0.0, md1 = 0.0;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          m += o.G[b][c] * K[c][a];
          md0 += o.Gd[0][b][c] * K[c][a] + o.G[b][c] * Kd[0][c][a];
          md1 += o.Gd[1][b][c] * K[c][a] + o.G[b][c] * Kd[1][c][a];
          dds += o.Gdd[b][a][b][c] * K[c][a] + o.Gd[a][b][c] * Kd[b][c][a] +
                 o.Gd[b][b][c] * Kd[a][c][a] + o.G[b][c] * Kdd[b][a][c][a];
        }
        M[a][b] = m, Md[0][a][b] = md0, Md[1][a][b] = md1;
      }
    M[1][0] = M[0][1];
    Md[0][1][0] = Md[0][0][1], Md[1][1][0] = Md[1][0][1];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        M[a][b] *= eb;
        Md[0][a][b] *= eb, Md[1][a][b] *= eb;
      }
    dds *= eb;
    double Q[2], Qc = dds;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      double s = 0.0;
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        s += Md[a][a][b];
#pragma unroll
        for (int l = 0; l < 2; ++l) {
          s += o.Gam[a][a][l] * M[l][b] + o.Gam[b][a][l] * M[a][l];
          Qc += o.Gamd[b][a][a][l] * M[l][b] + o.Gam[a][a][l] * Md[b][l][b] +
                o.Gamd[b][b][a][l] * M[a][l] + o.Gam[b][a][l] * Md[b][a][l];
        }
      }
      Q[b] = s;
    }
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int l = 0; l < 2; ++l) Qc += Q[l] * o.Gam[b][b][l];
    double bm[2][2];
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int a = 0; a < 2; ++a) bm[b][a] = o.G[0][a] * o.b[b][0] + o.G[1][a] * o.b[b][1];
    q[0] -= bm[0][0] * Q[0] + bm[1][0] * Q[1];
    q[1] -= bm[0][1] * Q[0] + bm[1][1] * Q[1];
    q3 += Qc;
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) f[k] = q[0] * o.a[0][k] + q[1] * o.a[1][k] + q3 * o.n[k];
}

// One workgroup per capsule slot, ring by ring: coefficients, nodes (lane pairs split the sums by
// the parity of m, as in k_nodes), longitude DFT.  REF: the unit sphere's state into `refout`.
template <bool REF>
__global__ void __launch_bounds__(THREADS, 2)
    k_nodes_ordered(Tables T, OrderedTables O, Work wk, double gs, double eb,
                    double* __restrict__ refout) {
  extern __shared__ double lds[];
  const int tid = threadIdx.x;
  const int N = T.N, nt = T.nt, np = T.np, hp = np / 2, NT = T.NT;
  double2* te = reinterpret_cast<double2*>(lds);  // [np]
  double2* cf = te + np;                          // [3][NT]
  double2* AB = cf + 3 * NT;                      // [N][3][5]
  double* F = reinterpret_cast<double*>(AB + 15 * N);  // [hp][2][6]
  for (int q = tid; q < np; q += THREADS) te[q] = T.ef[q];
  for (int slot = blockIdx.x; slot < wk.n; slot += gridDim.x) {
    __syncthreads();
    for (int t = tid; t < 3 * NT; t += THREADS) cf[t] = wk.coef[(size_t)slot * 3 * NT + t];
    for (int ring = 0; ring < nt; ++ring) {
      // row of this ring in the DFT rows: north, south, north ... (k_nodes)
      const int row = ring < N ? 2 * ring : 2 * (nt - 1 - ring) + 1;
      __syncthreads();
      for (int t = tid; t < 5 * N; t += THREADS) {
        const int k = t / N, m = t % N;
        const double* P = O.Pfd + ((size_t)ring * 5 + k) * NT;
        const double h = m == 0 ? 0.5 : 1.0;
        double sa[3] = {0.0, 0.0, 0.0}, sb[3] = {0.0, 0.0, 0.0};
        int q = m;  // tidx(N, d, m)
        #pragma unroll 4
        for (int d = 0; d < N - m; ++d) {
          const double p = P[q];
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            const double2 v = cf[c * NT + q];
            sa[c] += p * v.x, sb[c] += p * v.y;
          }
          q += N - d;
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) AB[(m * 3 + c) * 5 + k] = make_double2(h * sa[c], h * sb[c]);
      }
      __syncthreads();
      if (tid < np) {
        const int par = tid & 1, jj = tid >> 1, node = ring * np + jj + par * hp;
        double X[3][NQ];
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
          for (int q = 0; q < NQ; ++q) X[c][q] = 0.0;
        int q = par * jj;  // (m jj) mod np
        int dq = 2 * jj;
        if (dq >= np) dq -= np;
        for (int m = par; m < N; m += 2) {
          const double cm = te[q].x, sm = te[q].y;
          q += dq;
          if (q >= np) q -= np;
          const double m1 = (double)m, m2 = m1 * m1, m3 = m2 * m1, m4 = m2 * m2;
#pragma unroll
          for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int kt = 0; kt <= 4; ++kt) {
              const double A = AB[(m * 3 + c) * 5 + kt].x, B = AB[(m * 3 + c) * 5 + kt].y;
              const double h0 = A * cm - B * sm, h1 = -A * sm - B * cm;
              X[c][qidx(kt, 0)] += h0;
              if (kt <= 3) X[c][qidx(kt, 1)] += m1 * h1;
              if (kt <= 2) X[c][qidx(kt, 2)] -= m2 * h0;
              if (kt <= 1) X[c][qidx(kt, 3)] -= m3 * h1;
              if (kt == 0) X[c][qidx(0, 4)] += m4 * h0;
            }
        }
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
          for (int qq = 0; qq < NQ; ++qq) {
            const double other = swap_pair(X[c][qq]);
            X[c][qq] = par ? other - X[c][qq] : X[c][qq] + other;
          }
        Geom o;
        geometry(X, o);
        if (REF) {
          double* R = refout + (size_t)node * NREF;
#pragma unroll
          for (int q = 0; q < 4; ++q) R[q] = (&o.G[0][0])[q], R[28 + q] = (&o.b[0][0])[q];
#pragma unroll
          for (int q = 0; q < 8; ++q) R[4 + q] = (&o.Gd[0][0][0])[q], R[32 + q] = (&o.bd[0][0][0])[q];
#pragma unroll
          for (int q = 0; q < 16; ++q)
            R[12 + q] = (&o.Gdd[0][0][0][0])[q], R[40 + q] = (&o.bdd[0][0][0][0])[q];
        } else {
          double f[6];
          law(o, O.ref + (size_t)node * NREF, gs, eb, f);
#pragma unroll
          for (int k = 0; k < 3; ++k) f[3 + k] = o.n[k];
#pragma unroll
          for (int k = 0; k < 6; ++k) {
            const double other = swap_pair(f[k]);
            F[(jj * 2 + par) * 6 + k] = par ? other - f[k] : f[k] + other;
          }
        }
      }
      __syncthreads();
      if (REF) continue;
      for (int t = tid; t < 3 * N; t += THREADS) {
        const int g = t / N, m = t % N;
        const double2* v = reinterpret_cast<const double2*>(F + (m & 1) * 6) + g;
        double2 s0 = {0.0, 0.0}, s1 = {0.0, 0.0};
        int q = 0;  // (m j) mod np
        #pragma unroll 4
        for (int j = 0; j < hp; ++j) {
          const double2 e = te[q], w = v[6 * j];
          q += m;
          if (q >= np) q -= np;
          s0.x += w.x * e.x, s0.y += w.x * e.y;
          s1.x += w.y * e.x, s1.y += w.y * e.y;
        }
        double2* r = wk.rows + (((size_t)slot * nt + row) * N + m) * 6 + 2 * g;
        r[0] = s0, r[1] = s1;
      }
    }
  }
}

inline size_t lds_bytes(const Tables& T) {
  return (size_t)(T.np + 3 * T.NT + 15 * T.N) * sizeof(double2) + (size_t)T.np * 6 * sizeof(double);
}

}  // namespace ordered
}  // namespace memb
