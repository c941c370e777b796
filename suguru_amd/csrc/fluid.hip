// fluid.hip -- libfluid: the FFT flow update of one rank on gfx950 (declarations and reference
// citations in include/fluid.h).
//
// Layout.  The caller's fields are Fortran (0:i1,0:j1,0:k1) arrays, i fastest.  The solves work
// in compact spectral arrays of itot x jtot x ktot doubles (i fastest), one per velocity
// component; the pressure solve reuses the first.  A solve is five passes:
//   1. x transform of every (j, k) line (k_x_fwd; lines contiguous),
//   2. y transform of every (i, k) line (k_y; two neighbouring columns per complex line, row
//      segments of 64 bytes and more per workgroup),
//   3. Gaussian elimination in k per (i, j) mode (k_tri_seg: one lane per mode, the k rows in
//      register-held segments joined through LDS, the per-mode reciprocal pivots read from a
//      table built once per context; k_tri, two passes through the array, above 257 planes),
//   4. y inverse, 5. x inverse (into the caller's field interior).
// Transforms.  A real line of length N = 2M is transformed as M complex values
// z_n = x_2n + i x_2n+1, then split into the half spectrum X_0 .. X_M; a pair of y lines as the
// real and imaginary part of one complex line.  Lines of 16 .. 2048 (x) and 8 .. 1024 values (y)
// go through registers (radix 8, fft_reg.hpp), the others through LDS (k_rfft: radix 4, input
// bit-reversed on load).  Packed real layout of a line: [X_0, X_M, Re X_1, Im X_1, ...,
// Re X_M-1, Im X_M-1]; position p carries wavenumber 0 (p = 0), M (p = 1) or p / 2.  The
// second-difference eigenvalue of a position depends only on its wavenumber, which is what the
// reference's xrt/yrt tables encode for VFFTPACK's layout (initsolver.f90:108-132).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/fluid.h"
#include "fft_reg.hpp"

#pragma clang fp contract(off)

namespace {

constexpr int FFT_THREADS = 256;
// loads each thread keeps in flight while a transform reads its lines (8 for the forward
// transforms; 4 for the inverse ones, whose four loads per value would cost occupancy at 8)
constexpr int FFT_LB_FWD = 8;
constexpr int FFT_LB_INV = 4;
constexpr int TRI_MODES = 64;        // modes (lanes) per elimination workgroup
constexpr int Y_LINES_FWD = 8;       // columns per forward y-transform workgroup
constexpr int Y_LINES_INV = 8;       // columns per inverse y-transform workgroup
constexpr size_t LDS_MAX = 160 * 1024;

struct FGrid {
  int itot, jtot, ktot;
  long long sy, sz;  // Fortran field pitches: row itot+2, plane (itot+2)(jtot+2)
  double dxi, dyi, dzi;
};

__device__ __forceinline__ long long fidx(const FGrid& g, int i, int j, int k) {
  return (long long)i + g.sy * j + g.sz * k;
}

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// ---- transforms ---------------------------------------------------------------------------
// One workgroup transforms `nl` lines of length N = 2M of one k plane; element e of line l
// lives at base + l * ls + e * es (source and destination each have their own geometry), the
// workgroup's base being plane * (block / groups_per_plane) + gstride * (block % groups).
// tw[k] = exp(-2 pi i k / N), k < M.  x lines: nl consecutive rows; y lines: nl consecutive
// columns.

// radix-2 decimation in time over nl lines of M complex values (input in bit-reversed order)
// Line l starts at l * (M + 1) complex values in LDS: the pad of one keeps the lines of a
// workgroup in different banks when neighbouring threads work on neighbouring lines.
// Decimation in time over nl lines of M complex values (input in bit-reversed order): one
// radix-2 stage when log2 M is odd, then radix-4 passes, each the two radix-2 stages of spans
// h and 2h on four values held in registers (half the LDS round trips and barriers).
template <bool INV>
__device__ void fft_stages(double2* s, int nl, int M, int logm, int logn,
                           const double2* __restrict__ tw) {
  int h = 1, lg = 0;
  if (logm & 1) {
    __syncthreads();
    const int half_m = M >> 1;
    for (int b = threadIdx.x; b < nl * half_m; b += blockDim.x) {
      const int line = b >> (logm - 1), r = b & (half_m - 1);
      const int i0 = line * (M + 1) + 2 * r, i1 = i0 + 1;
      const double2 a = s[i0], t = s[i1];  // twiddle W^0 = 1
      s[i0] = make_double2(a.x + t.x, a.y + t.y);
      s[i1] = make_double2(a.x - t.x, a.y - t.y);
    }
    h = 2, lg = 1;
  }
  const int quarter = M >> 2;
  for (; h < M; h <<= 2, lg += 2) {
    __syncthreads();
    const int ts1 = logn - 1 - lg, ts2 = logn - 2 - lg;  // N / (2h), N / (4h)
    for (int b = threadIdx.x; b < nl * quarter; b += blockDim.x) {
      const int line = b >> (logm - 2), r = b & (quarter - 1);
      const int pos = r & (h - 1), grp = r >> lg;
      const int base = line * (M + 1) + (grp << (lg + 2)) + pos;
      double2 w1 = tw[pos << ts1], w2 = tw[pos << ts2], w3 = tw[(pos + h) << ts2];
      if (INV) w1.y = -w1.y, w2.y = -w2.y, w3.y = -w3.y;
      const double2 a0 = s[base], a1 = s[base + h], a2 = s[base + 2 * h], a3 = s[base + 3 * h];
      const double2 t1 = cmul(w1, a1), t3 = cmul(w1, a3);
      const double2 b0 = make_double2(a0.x + t1.x, a0.y + t1.y);
      const double2 b1 = make_double2(a0.x - t1.x, a0.y - t1.y);
      const double2 b2 = make_double2(a2.x + t3.x, a2.y + t3.y);
      const double2 b3 = make_double2(a2.x - t3.x, a2.y - t3.y);
      const double2 u2 = cmul(w2, b2), u3 = cmul(w3, b3);
      s[base] = make_double2(b0.x + u2.x, b0.y + u2.y);
      s[base + 2 * h] = make_double2(b0.x - u2.x, b0.y - u2.y);
      s[base + h] = make_double2(b1.x + u3.x, b1.y + u3.y);
      s[base + 3 * h] = make_double2(b1.x - u3.x, b1.y - u3.y);
    }
  }
  __syncthreads();
}

// Workgroup b runs on XCD b % 8 (round-robin dispatch).  With a grid of a multiple of 8
// workgroups, the y transforms take logical block (b % 8) (grid / 8) + b / 8, so that each XCD
// works through one contiguous eighth of the lines: neighbouring groups of y lines share their
// 128-byte rows, and these are then fetched once, into one L2 (k_y: a step at 1024 x 512 x 256
// 15.79 -> 14.36 ms, 512 x 512 x 250 7.63 -> 6.93).  The x lines are whole rows and keep the dispatch
// order.
template <bool XMAJOR>
__device__ __forceinline__ int xcd_logical_block() {
  const unsigned nb = gridDim.x;
  if (XMAJOR || (nb & 7u)) return (int)blockIdx.x;
  return (int)((blockIdx.x & 7u) * (nb >> 3) + (blockIdx.x >> 3));
}

// The same for any number nb of workgroups: the blockIdx-th of the launch, which the hardware
// deals out over the eight XCDs in turn, as its place in eight contiguous ranges.
__device__ __forceinline__ unsigned xcd_contiguous(unsigned id, unsigned nb) {
  const unsigned x = id & 7u, q = nb >> 3, r = nb & 7u;
  return x * q + min(x, r) + (id >> 3);
}

__device__ __forceinline__ int brev(int n, int logm) {
  return logm ? (int)(__brev((unsigned)n) >> (32 - logm)) : 0;
}

// The velocity divergence of fillps.f90:8-47 as the source of an x transform: the value of
// compact cell (i, j, k) is computed from the fields while the lines are loaded, with
// k_fillps's expression (cz = dzi / dt, cy = dyi / dt, cx = dxi / dt as k_fillps forms them).
// It reads the interior alone: below the first cell of a line or row lies the last one (periodic),
// and w is 0 on both wall faces (bound.f90:38-56), so the halos need not be set first.
struct FillSrc {
  const double* u;
  const double* v;
  const double* w;
  double cx, cy, cz;
  long long sy, sz;
  int itot, jtot, ktot;
  // from cell (., j, .) to the one below it in y
  __device__ __forceinline__ long long below(int j) const { return j ? -sy : (jtot - 1) * sy; }
};

// The arrays of one launch: workgroup row blockIdx.y transforms src[y] into dst[y].  The three
// momentum solves share their launches: at 64^3 cells a launch is 5 us of latency whatever it
// holds (26 launches -> 15; with fewer planes per momentum workgroup as well, a step there takes
// 104 us instead of 211; 512 x 512 x 250 cells 8.09 instead of 8.27 ms, from the eliminations).
struct Arrays {
  const double* src[3];
  double* dst[3];
};

// Forward: real lines -> packed half spectra.  XMAJOR: element index fastest across threads
// (x lines); otherwise line index fastest (y lines).  src and dst may be the same array (the
// workgroup reads all of its lines before the first barrier and writes them after the last).
// FILL (x lines of a compact array only): the lines are fillps's divergence (fs), not src.
template <bool XMAJOR, bool FILL = false>
__global__ void __launch_bounds__(FFT_THREADS)
    k_rfft_fwd(Arrays arr, int N, int logm,
               int nl, int groups_per_plane, long long plane_src, long long plane_dst,
               long long gstride_src, long long gstride_dst, long long es_src, long long ls_src,
               long long es_dst, long long ls_dst, long long off_src,
               const double2* __restrict__ tw, FillSrc fs) {
  extern __shared__ double2 sm[];
  const double* src = arr.src[blockIdx.y];
  double* dst = arr.dst[blockIdx.y];
  const int M = N >> 1, logn = logm + 1, lognl = 31 - __clz(nl);
  const int blk = xcd_logical_block<XMAJOR>();
  const int kp = blk / groups_per_plane, gp = blk - kp * groups_per_plane;
  const long long bs = off_src + kp * plane_src + gp * gstride_src;
  const long long bd = kp * plane_dst + gp * gstride_dst;
  double* smd = reinterpret_cast<double*>(sm);
  // the y transforms read their twiddles from an LDS copy after the lines (each radix-4
  // butterfly needs three per pass; from the caches they put a round trip in every pass);
  // the x transforms, whose forward pass was slower that way, read them from memory
  const double2* twl = tw;
  if (!XMAJOR) {
    double2* stw = sm + nl * (M + 1);
    for (int q = threadIdx.x; q < M; q += blockDim.x) stw[q] = tw[q];
    twl = stw;
  }
  // every load of a batch in flight before the LDS stores
  for (int q0 = threadIdx.x; q0 < nl * N; q0 += blockDim.x * FFT_LB_FWD) {
    double v[FFT_LB_FWD];
#pragma unroll
    for (int u = 0; u < FFT_LB_FWD; ++u) {
      const int q = q0 + u * blockDim.x;
      const int l = XMAJOR ? q >> logn : q & (nl - 1), e = XMAJOR ? q & (N - 1) : q >> lognl;
      v[u] = 0.0;
      if (q < nl * N) {
        if constexpr (FILL) {
          const int j = gp * nl + l;
          const long long c = (long long)(e + 1) + fs.sy * (j + 1) + fs.sz * (kp + 1);
          const double w0 = kp == fs.ktot - 1 ? 0.0 : fs.w[c], w1 = kp ? fs.w[c - fs.sz] : 0.0;
          v[u] = ((w0 - w1) * fs.cz + (fs.v[c] - fs.v[c + fs.below(j)]) * fs.cy +
                  (fs.u[c] - fs.u[e ? c - 1 : c + fs.itot - 1]) * fs.cx);
        } else {
          v[u] = src[bs + l * ls_src + e * es_src];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < FFT_LB_FWD; ++u) {
      const int q = q0 + u * blockDim.x;
      const int l = XMAJOR ? q >> logn : q & (nl - 1), e = XMAJOR ? q & (N - 1) : q >> lognl;
      if (q < nl * N) smd[2 * (l * (M + 1) + brev(e >> 1, logm)) + (e & 1)] = v[u];
    }
  }
  fft_stages<false>(sm, nl, M, logm, logn, twl);
  // X_k = E_k + W^k O_k, E_k = (Z_k + conj Z_M-k) / 2, O_k = (Z_k - conj Z_M-k) / 2i
  for (int q = threadIdx.x; q < nl * M; q += blockDim.x) {
    const int l = XMAJOR ? q >> logm : q & (nl - 1), k = XMAJOR ? q & (M - 1) : q >> lognl;
    const double2* z = sm + l * (M + 1);
    double* out = dst + bd + l * ls_dst;
    if (k == 0) {
      const double2 z0 = z[0];
      out[0] = z0.x + z0.y;
      out[es_dst] = z0.x - z0.y;
    } else {
      const double2 a = z[k], b = z[M - k];
      const double2 E = make_double2(0.5 * (a.x + b.x), 0.5 * (a.y - b.y));
      const double2 O = make_double2(0.5 * (a.y + b.y), -0.5 * (a.x - b.x));
      const double2 X = cmul(twl[k], O);
      out[(2 * k) * es_dst] = E.x + X.x;
      out[(2 * k + 1) * es_dst] = E.y + X.y;
    }
  }
}

// Inverse: packed half spectra -> real lines (scaled by 1/M here, 1/2 in the split).
template <bool XMAJOR>
__global__ void __launch_bounds__(FFT_THREADS)
    k_rfft_inv(Arrays arr, int N, int logm,
               int nl, int groups_per_plane, long long plane_src, long long plane_dst,
               long long gstride_src, long long gstride_dst, long long es_src, long long ls_src,
               long long es_dst, long long ls_dst, long long off_dst,
               const double2* __restrict__ tw) {
  extern __shared__ double2 sm[];
  const double* src = arr.src[blockIdx.y];
  double* dst = arr.dst[blockIdx.y];
  const int M = N >> 1, logn = logm + 1, lognl = 31 - __clz(nl);
  const int blk = xcd_logical_block<XMAJOR>();
  const int kp = blk / groups_per_plane, gp = blk - kp * groups_per_plane;
  const long long bs = kp * plane_src + gp * gstride_src;
  const long long bd = off_dst + kp * plane_dst + gp * gstride_dst;
  // twiddles from an LDS copy after the lines (as in k_rfft_fwd)
  double2* stw = sm + nl * (M + 1);
  for (int q = threadIdx.x; q < M; q += blockDim.x) stw[q] = tw[q];
  __syncthreads();
  // Z_k = E_k + i O_k, E_k = (X_k + conj X_M-k) / 2, O_k = (X_k - conj X_M-k) conj(W^k) / 2
  for (int q0 = threadIdx.x; q0 < nl * M; q0 += blockDim.x * FFT_LB_INV) {
    double2 va[FFT_LB_INV], vb[FFT_LB_INV];
#pragma unroll
    for (int u = 0; u < FFT_LB_INV; ++u) {
      const int q = q0 + u * blockDim.x;
      const int l = XMAJOR ? q >> logm : q & (nl - 1), k = XMAJOR ? q & (M - 1) : q >> lognl;
      const double* in = src + bs + l * ls_src;
      va[u] = make_double2(0.0, 0.0), vb[u] = va[u];
      if (q < nl * M) {
        if (k == 0) {
          va[u] = make_double2(in[0], in[es_src]);
        } else {
          va[u] = make_double2(in[(2 * k) * es_src], in[(2 * k + 1) * es_src]);
          vb[u] = make_double2(in[(2 * (M - k)) * es_src], in[(2 * (M - k) + 1) * es_src]);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < FFT_LB_INV; ++u) {
      const int q = q0 + u * blockDim.x;
      if (q >= nl * M) continue;
      const int l = XMAJOR ? q >> logm : q & (nl - 1), k = XMAJOR ? q & (M - 1) : q >> lognl;
      double2 Z;
      if (k == 0) {
        const double x0 = va[u].x, xm = va[u].y;
        Z = make_double2(0.5 * (x0 + xm), 0.5 * (x0 - xm));
      } else {
        const double2 a = va[u], b = vb[u];
        const double2 E = make_double2(0.5 * (a.x + b.x), 0.5 * (a.y - b.y));
        const double2 D = make_double2(0.5 * (a.x - b.x), 0.5 * (a.y + b.y));
        const double2 wc = make_double2(stw[k].x, -stw[k].y);
        const double2 O = cmul(D, wc);
        Z = make_double2(E.x - O.y, E.y + O.x);
      }
      sm[l * (M + 1) + brev(k, logm)] = Z;
    }
  }
  fft_stages<true>(sm, nl, M, logm, logn, stw);
  const double sc = 1.0 / (double)M;
  const double* smd = reinterpret_cast<const double*>(sm);
  for (int q = threadIdx.x; q < nl * N; q += blockDim.x) {
    const int l = XMAJOR ? q >> logn : q & (nl - 1), e = XMAJOR ? q & (N - 1) : q >> lognl;
    dst[bd + l * ls_dst + e * es_dst] = smd[2 * (l * (M + 1) + (e >> 1)) + (e & 1)] * sc;
  }
}

// ---- register transforms --------------------------------------------------------------------
// The transforms of lines that 8 values a thread cover (x lines of 16 .. 2048, y lines of
// 8 .. 1024 values): radix-8 passes in registers with two or three exchanges through LDS, where the
// kernels above go through LDS once per radix-4 pass and once more for the bit reversal, with a
// workgroup barrier each.  Bound by memory: at 1024 x 512 x 256 an array takes 422 us forward and
// 426 us inverse in x, 436 and 414 us in y (a copy of its 2.1 GB takes 438 us), 865 us with the
// divergence as the source; the kernels above took 569, 579, 553, 610 and 1029 us.
constexpr int REG_T = 256;  // threads of an x workgroup, and of a y workgroup up to 512 rows

// two neighbouring values of a row (the rows of the caller's fields start at odd elements)
struct __attribute__((packed, aligned(8))) Pair {
  double x, y;
};
__device__ __forceinline__ double2 load2(const double* p) {
  const Pair v = *reinterpret_cast<const Pair*>(p);
  return make_double2(v.x, v.y);
}
__device__ __forceinline__ void store2(double* p, double2 v) {
  *reinterpret_cast<Pair*>(p) = Pair{v.x, v.y};
}

// rows of the lines of one launch: line (j, k) at off + j row + k plane
struct Rows {
  long long off, row, plane;
  __device__ __forceinline__ long long at(int j, int k) const { return off + j * row + k * plane; }
};

// x lines: one line of M = itot / 2 complex values per M/8 lanes, 2048 / M lines a workgroup.  With
// M <= 512 a line stays within one wavefront and needs no workgroup barrier.
template <int LOGM>
struct XLine {
  using Line = fft::Line<LOGM, (LOGM > 9)>;
  static constexpr int M = Line::N, TPL = Line::TPL, PER = REG_T / TPL, PITCH = fft::pad(M) + 1;
};

// values 2q, 2q + 1 (q = t + TPL u) of x line (j, k): from `src`, the line's first value, or with
// FILL the divergence
template <int LOGM, bool FILL>
__device__ __forceinline__ void x_load(double2 (&a)[8], int t, const double* src,
                                       const FillSrc& fs, int j, int k) {
  constexpr int TPL = XLine<LOGM>::TPL;
  if constexpr (FILL) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const long long c = 2 * (t + TPL * u) + 1 + fs.sy * (j + 1) + fs.sz * (k + 1);
      // (w on the wall faces: loaded like the others, then 0)
      double2 w0 = load2(fs.w + c), w1 = load2(fs.w + c - fs.sz);
      if (k == fs.ktot - 1) w0 = make_double2(0.0, 0.0);
      if (k == 0) w1 = make_double2(0.0, 0.0);
      const double2 v0 = load2(fs.v + c), v1 = load2(fs.v + c + fs.below(j));
      const double2 u0 = load2(fs.u + c);
      const double2 u1 = make_double2(fs.u[u == 0 && t == 0 ? c + fs.itot - 1 : c - 1], u0.x);
      a[u] = make_double2(((w0.x - w1.x) * fs.cz + (v0.x - v1.x) * fs.cy + (u0.x - u1.x) * fs.cx),
                          ((w0.y - w1.y) * fs.cz + (v0.y - v1.y) * fs.cy + (u0.y - u1.y) * fs.cx));
    }
  } else {
#pragma unroll
    for (int u = 0; u < 8; ++u) a[u] = load2(src + 2 * (t + TPL * u));
  }
}

// the line's values into its packed half spectrum, a[u] = values 2q, 2q + 1 of it
template <int LOGM>
__device__ __forceinline__ void x_spectrum(double2 (&a)[8], double2* buf, int t,
                                           const double2* __restrict__ tw,
                                           const double2* __restrict__ twm) {
  using X = XLine<LOGM>;
  constexpr int M = X::M, TPL = X::TPL;
  constexpr bool WG = LOGM > 9;
  typename X::Line lw;
  lw.load(twm, t);
  lw.template run<false>(a, buf, t);
  // X_k = E_k + W^k O_k, E_k = (Z_k + conj Z_M-k) / 2, O_k = (Z_k - conj Z_M-k) / 2i
  fft::line_sync<WG>();
#pragma unroll
  for (int u = 0; u < 8; ++u) buf[fft::pad(t + TPL * u)] = a[u];
  fft::line_sync<WG>();
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const int q = t + TPL * u;
    const double2 b = buf[fft::pad((M - q) & (M - 1))], w = tw[q];
    const double2 E = make_double2(0.5 * (a[u].x + b.x), 0.5 * (a[u].y - b.y));
    const double2 O = make_double2(0.5 * (a[u].y + b.y), -0.5 * (a[u].x - b.x));
    double2 v = fft::add(E, fft::mul(w, O));
    if (u == 0 && t == 0) v = make_double2(a[0].x + a[0].y, a[0].x - a[0].y);
    a[u] = v;
  }
}

// and back
template <int LOGM>
__device__ __forceinline__ void x_values(double2 (&a)[8], double2* buf, int t,
                                         const double2* __restrict__ tw,
                                         const double2* __restrict__ twm) {
  using X = XLine<LOGM>;
  constexpr int M = X::M, TPL = X::TPL;
  constexpr bool WG = LOGM > 9;
  fft::line_sync<WG>();
#pragma unroll
  for (int u = 0; u < 8; ++u) buf[fft::pad(t + TPL * u)] = a[u];
  fft::line_sync<WG>();
  // Z_k = E_k + i O_k, E_k = (X_k + conj X_M-k) / 2, O_k = (X_k - conj X_M-k) conj(W^k) / 2
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const int q = t + TPL * u;
    const double2 b = buf[fft::pad((M - q) & (M - 1))], w = tw[q];
    const double2 E = make_double2(0.5 * (a[u].x + b.x), 0.5 * (a[u].y - b.y));
    const double2 D = make_double2(0.5 * (a[u].x - b.x), 0.5 * (a[u].y + b.y));
    const double2 O = fft::mul(D, make_double2(w.x, -w.y));
    double2 v = make_double2(E.x - O.y, E.y + O.x);
    if (u == 0 && t == 0)
      v = make_double2(0.5 * (a[0].x + a[0].y), 0.5 * (a[0].x - a[0].y));
    a[u] = v;
  }
  typename X::Line lw;
  lw.load(twm, t);
  lw.template run<true>(a, buf, t);
  const double sc = 1.0 / (double)M;
#pragma unroll
  for (int u = 0; u < 8; ++u) a[u] = make_double2(a[u].x * sc, a[u].y * sc);
}

template <int LOGM, bool FILL>
__global__ void __launch_bounds__(REG_T)
    k_x_fwd(Arrays arr, Rows rs, Rows rd, int logj, int lines, const double2* __restrict__ tw,
            const double2* __restrict__ twm, FillSrc fs) {
  using X = XLine<LOGM>;
  __shared__ double2 sm[X::PER * X::PITCH];
  const int t = threadIdx.x & (X::TPL - 1), own = threadIdx.x / X::TPL;
  const int line = blockIdx.x * X::PER + own;
  const bool live = line < lines;
  const int ln = live ? line : lines - 1, k = ln >> logj, j = ln & ((1 << logj) - 1);
  double2 a[8];
  x_load<LOGM, FILL>(a, t, FILL ? nullptr : arr.src[blockIdx.y] + rs.at(j, k), fs, j, k);
  x_spectrum<LOGM>(a, sm + own * X::PITCH, t, tw, twm);
  double* dst = arr.dst[blockIdx.y] + rd.at(j, k);
  if (live) {
#pragma unroll
    for (int u = 0; u < 8; ++u) store2(dst + 2 * (t + X::TPL * u), a[u]);
  }
}

template <int LOGM>
__global__ void __launch_bounds__(REG_T)
    k_x_inv(Arrays arr, Rows rs, Rows rd, int logj, int lines, const double2* __restrict__ tw,
            const double2* __restrict__ twm) {
  using X = XLine<LOGM>;
  __shared__ double2 sm[X::PER * X::PITCH];
  const int t = threadIdx.x & (X::TPL - 1), own = threadIdx.x / X::TPL;
  const int line = blockIdx.x * X::PER + own;
  const bool live = line < lines;
  const int ln = live ? line : lines - 1, k = ln >> logj, j = ln & ((1 << logj) - 1);
  double2 a[8];
  x_load<LOGM, false>(a, t, arr.src[blockIdx.y] + rs.at(j, k), FillSrc{}, j, k);
  x_values<LOGM>(a, sm + own * X::PITCH, t, tw, twm);
  double* dst = arr.dst[blockIdx.y] + rd.at(j, k);
  if (live) {
#pragma unroll
    for (int u = 0; u < 8; ++u) store2(dst + 2 * (t + X::TPL * u), a[u]);
  }
}

// y lines: two neighbouring real columns are the real and imaginary part of one complex line of
// N = jtot values (no twiddles in the split, 16-byte loads), neighbouring pairs on neighbouring
// lanes.  A workgroup holds COLS pairs: 64-byte row segments at 512 rows, 128 at 256.
template <int LOGN>
struct YLine {
  using Line = fft::Line<LOGN, true>;
  static constexpr int N = Line::N, TPL = Line::TPL;
  static constexpr int COLS = LOGN > 9 ? 4 : REG_T / TPL, T = COLS * TPL;
  // the pairs of a row lie in different banks: pitch = 16 / COLS mod 16 sixteen-byte slots
  static constexpr int SKEW = COLS >= 16 ? 1 : 16 / COLS;
  static constexpr int PITCH = fft::pad(N) + (SKEW - fft::pad(N) % 16 + 16) % 16;
  static constexpr int WAVES = T / 64;
};

// The two columns of a pair share their rounding: each gets about 1e-16 of the other's largest
// value, no more than the x transform left in either from the same row, except where a column is
// zero: in a flow uniform in x every column but the first is, and has to stay so for the flow to stay
// uniform to the last bit.  So a column of zeros gives zeros.
// y_mark: from the eight values a thread holds of each column, a bit per lane (nz: the first
// column's of each wavefront, then the second's); y_clear, a barrier later: the zero columns'
// values of v.
template <int LOGN>
__device__ __forceinline__ void y_mark(const double2 (&v)[8], unsigned long long* nz) {
  using Y = YLine<LOGN>;
  bool x = false, y = false;
#pragma unroll
  for (int u = 0; u < 8; ++u) x |= v[u].x != 0.0, y |= v[u].y != 0.0;
  const unsigned long long bx = __ballot(x), by = __ballot(y);
  if ((threadIdx.x & 63) == 0) nz[threadIdx.x >> 6] = bx, nz[Y::WAVES + (threadIdx.x >> 6)] = by;
}
template <int LOGN>
__device__ __forceinline__ void y_clear(double2 (&v)[8], const unsigned long long* nz, int col) {
  using Y = YLine<LOGN>;
  // wavefronts and, in each, lanes with values of column col
  constexpr int STEP = Y::COLS > 64 ? Y::COLS / 64 : 1;
  unsigned long long bx = 0, by = 0, lanes = 1;
#pragma unroll
  for (int l = Y::COLS; l < 64; l += Y::COLS) lanes |= 1ull << l;
  const int w0 = Y::COLS > 64 ? col >> 6 : 0;
#pragma unroll
  for (int w = 0; w < Y::WAVES; w += STEP) bx |= nz[w0 + w], by |= nz[Y::WAVES + w0 + w];
  const bool x = (bx >> (col & 63)) & lanes, y = (by >> (col & 63)) & lanes;
#pragma unroll
  for (int u = 0; u < 8; ++u) v[u] = make_double2(x ? v[u].x : 0.0, y ? v[u].y : 0.0);
}

// the packed half spectra of a pair of columns from its complex spectrum: rows 2k and 2k + 1
// (k = t + TPL u, u < 4) get Re and Im of X_k, rows 0 and 1 X_0 and X_N/2
template <int LOGN>
__device__ __forceinline__ void y_split(const double2 (&a)[8], double2* buf, int t,
                                        double2 (&row)[8]) {
  using Y = YLine<LOGN>;
  __syncthreads();
#pragma unroll
  for (int u = 4; u < 8; ++u) buf[fft::pad(t + Y::TPL * u)] = a[u];
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const bool first = u == 0 && t == 0;
    const int q = t + Y::TPL * u;
    const double2 b = buf[fft::pad(first ? Y::N / 2 : Y::N - q)];
    // A = (Z_k + conj Z_N-k) / 2, B = (Z_k - conj Z_N-k) / 2i
    row[2 * u] = make_double2(0.5 * (a[u].x + b.x), 0.5 * (a[u].y + b.y));
    row[2 * u + 1] = make_double2(0.5 * (a[u].y - b.y), -0.5 * (a[u].x - b.x));
    if (first) row[0] = a[0], row[1] = b;
  }
}

// the reverse: a[u] = Z_t+TPL u from the packed rows
template <int LOGN>
__device__ __forceinline__ void y_join(const double2 (&row)[8], double2* buf, int t,
                                       double2 (&a)[8]) {
  using Y = YLine<LOGN>;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const bool first = u == 0 && t == 0;
    const int q = t + Y::TPL * u;
    const double2 r = row[2 * u], i = row[2 * u + 1];  // (Re A, Re B), (Im A, Im B)
    a[u] = first ? r : make_double2(r.x - i.y, i.x + r.y);
    buf[fft::pad(first ? Y::N / 2 : Y::N - q)] = first ? i : make_double2(r.x + i.y, r.y - i.x);
  }
  __syncthreads();
#pragma unroll
  for (int u = 4; u < 8; ++u) a[u] = buf[fft::pad(t + Y::TPL * u)];
}

template <int LOGN, bool INV>
__global__ void __launch_bounds__(YLine<LOGN>::T)
    k_y(Arrays arr, int logc, long long pairs, const double2* __restrict__ twn) {
  using Y = YLine<LOGN>;
  __shared__ double2 sm[Y::COLS * Y::PITCH];
  __shared__ unsigned long long nz[2 * Y::WAVES];
  const int col = threadIdx.x & (Y::COLS - 1), t = threadIdx.x / Y::COLS;
  const long long g = (long long)xcd_logical_block<false>() * Y::COLS + col;
  const bool live = g < pairs;
  const long long gg = live ? g : pairs - 1, k = gg >> logc, c = gg - (k << logc);
  const long long pitch = 1LL << logc;  // pairs of a row
  double2* p = reinterpret_cast<double2*>(arr.dst[blockIdx.y]) + k * (pitch << LOGN) + c;
  double2* buf = sm + col * Y::PITCH;
  double2 a[8], row[8];
  typename Y::Line lw;
  if constexpr (!INV) {
#pragma unroll
    for (int u = 0; u < 8; ++u) a[u] = p[(t + Y::TPL * u) * pitch];
    lw.load(twn, t);
    y_mark<LOGN>(a, nz);
    lw.template run<false>(a, buf, t);
    y_split<LOGN>(a, buf, t, row);
    y_clear<LOGN>(row, nz, col);
    if (live) {
#pragma unroll
      for (int u = 0; u < 8; ++u) p[(2 * (t + Y::TPL * (u >> 1)) + (u & 1)) * pitch] = row[u];
    }
  } else {
#pragma unroll
    for (int u = 0; u < 8; ++u) row[u] = p[(2 * (t + Y::TPL * (u >> 1)) + (u & 1)) * pitch];
    lw.load(twn, t);
    y_mark<LOGN>(row, nz);
    y_join<LOGN>(row, buf, t, a);
    lw.template run<true>(a, buf, t);
    y_clear<LOGN>(a, nz, col);
    const double sc = 1.0 / (double)Y::N;
    if (live) {
#pragma unroll
      for (int u = 0; u < 8; ++u)
        p[(t + Y::TPL * u) * pitch] = make_double2(a[u].x * sc, a[u].y * sc);
    }
  }
}

// Planes of up to 8192 cells (itot, jtot >= 32): x and y transforms of a plane in one workgroup, the
// plane between them in LDS.  Bound by latency: on such grids a launch and its drain cost more than
// the pass over memory.  A step at 64^3 takes 68 us like this (82 with a launch per direction: 4.6
// and 5.2 us, against 6.6 for both), 64 x 64 x 256 126 (152), 128 x 64 x 250 218 (250), 32 x 32 x 16
// 47 (59).  A plane of 16384 values and the exchange buffer do not fit in LDS.
template <int LOGI, int LOGJ>
struct Plane {
  using X = XLine<LOGI - 1>;
  using Y = YLine<LOGJ>;
  static constexpr int PAIRS = 1 << (LOGI - 1), J = 1 << LOGJ;
  // rows of the columns that a wavefront's lanes hold together lie in different banks
  static constexpr int PITCH = PAIRS + (Y::COLS < 16 ? Y::COLS : 0);
  static constexpr int EX = X::PER * X::PITCH > Y::COLS * Y::PITCH ? X::PER * X::PITCH
                                                                   : Y::COLS * Y::PITCH;
};

template <int LOGI, int LOGJ, bool FILL>
__global__ void __launch_bounds__(REG_T)
    k_plane_fwd(Arrays arr, Rows rs, const double2* __restrict__ tw,
                const double2* __restrict__ twm, const double2* __restrict__ twn, FillSrc fs) {
  using P = Plane<LOGI, LOGJ>;
  using X = typename P::X;
  using Y = typename P::Y;
  static_assert(Y::T == REG_T, "one workgroup shape for both directions");
  __shared__ double2 pl[P::J * P::PITCH], ex[P::EX];
  __shared__ unsigned long long nz[2][2 * Y::WAVES];  // in turn: read until the next columns' barriers
  const int k = blockIdx.x;
  double2 a[8], row[8];
  for (int j0 = 0; j0 < P::J; j0 += X::PER) {
    const int t = threadIdx.x & (X::TPL - 1), own = threadIdx.x / X::TPL;
    const bool live = j0 + own < P::J;
    const int j = live ? j0 + own : P::J - 1;
    x_load<LOGI - 1, FILL>(a, t, FILL ? nullptr : arr.src[blockIdx.y] + rs.at(j, k), fs, j, k);
    x_spectrum<LOGI - 1>(a, ex + own * X::PITCH, t, tw, twm);
    if (live) {
#pragma unroll
      for (int u = 0; u < 8; ++u) pl[j * P::PITCH + t + X::TPL * u] = a[u];
    }
  }
  __syncthreads();
  double2* out = reinterpret_cast<double2*>(arr.dst[blockIdx.y]) + (long long)k * P::PAIRS * P::J;
  typename Y::Line lw;
  const int col = threadIdx.x & (Y::COLS - 1), t = threadIdx.x / Y::COLS;
  lw.load(twn, t);
  for (int c0 = 0; c0 < P::PAIRS; c0 += Y::COLS) {
    const bool live = c0 + col < P::PAIRS;
    const int c = live ? c0 + col : P::PAIRS - 1;
    double2* buf = ex + col * Y::PITCH;
#pragma unroll
    for (int u = 0; u < 8; ++u) a[u] = pl[(t + Y::TPL * u) * P::PITCH + c];
    unsigned long long* z = nz[(c0 / Y::COLS) & 1];
    y_mark<LOGJ>(a, z);
    lw.template run<false>(a, buf, t);
    y_split<LOGJ>(a, buf, t, row);
    y_clear<LOGJ>(row, z, col);
    if (live) {
#pragma unroll
      for (int u = 0; u < 8; ++u) out[(2 * (t + Y::TPL * (u >> 1)) + (u & 1)) * P::PAIRS + c] = row[u];
    }
  }
}

template <int LOGI, int LOGJ>
__global__ void __launch_bounds__(REG_T)
    k_plane_inv(Arrays arr, Rows rd, const double2* __restrict__ tw,
                const double2* __restrict__ twm, const double2* __restrict__ twn) {
  using P = Plane<LOGI, LOGJ>;
  using X = typename P::X;
  using Y = typename P::Y;
  __shared__ double2 pl[P::J * P::PITCH], ex[P::EX];
  __shared__ unsigned long long nz[2 * Y::WAVES];
  const int k = blockIdx.x;
  const double2* in =
      reinterpret_cast<const double2*>(arr.src[blockIdx.y]) + (long long)k * P::PAIRS * P::J;
  double2 a[8], row[8];
  {
    typename Y::Line lw;
    const int col = threadIdx.x & (Y::COLS - 1), t = threadIdx.x / Y::COLS;
    lw.load(twn, t);
    const double sc = 1.0 / (double)Y::N;
    for (int c0 = 0; c0 < P::PAIRS; c0 += Y::COLS) {
      const bool live = c0 + col < P::PAIRS;
      const int c = live ? c0 + col : P::PAIRS - 1;
      double2* buf = ex + col * Y::PITCH;
#pragma unroll
      for (int u = 0; u < 8; ++u) row[u] = in[(2 * (t + Y::TPL * (u >> 1)) + (u & 1)) * P::PAIRS + c];
      __syncthreads();  // the columns before these are done with buf and nz
      y_mark<LOGJ>(row, nz);
      y_join<LOGJ>(row, buf, t, a);
      lw.template run<true>(a, buf, t);
      y_clear<LOGJ>(a, nz, col);
      if (live) {
#pragma unroll
        for (int u = 0; u < 8; ++u)
          pl[(t + Y::TPL * u) * P::PITCH + c] = make_double2(a[u].x * sc, a[u].y * sc);
      }
    }
  }
  __syncthreads();
  for (int j0 = 0; j0 < P::J; j0 += X::PER) {
    const int t = threadIdx.x & (X::TPL - 1), own = threadIdx.x / X::TPL;
    const bool live = j0 + own < P::J;
    const int j = live ? j0 + own : P::J - 1;
#pragma unroll
    for (int u = 0; u < 8; ++u) a[u] = pl[j * P::PITCH + t + X::TPL * u];
    x_values<LOGI - 1>(a, ex + own * X::PITCH, t, tw, twm);
    double* dst = arr.dst[blockIdx.y] + rd.at(j, k);
    if (live) {
#pragma unroll
      for (int u = 0; u < 8; ++u) store2(dst + 2 * (t + X::TPL * u), a[u]);
    }
  }
}

// ---- Gaussian elimination in k (solver.f90:74-129) ------------------------------------------
// Wavenumber of packed position p of a length-n line: 0, n/2, or p/2.
__host__ __device__ __forceinline__ int wavenumber(int p, int n) {
  return p == 0 ? 0 : (p == 1 ? n / 2 : p >> 1);
}

// Reciprocal pivots per (wavenumber pair, k), built once: ztab[k][ky][kx] = z of
// solver.f90:80,89 (k < kmax), and at k = kmax the raw pivot bb - a d (:103-107).
__global__ void __launch_bounds__(256) k_ztab(int nkx, int nky, int ktot, int ne,
                                              const double* __restrict__ xrt,
                                              const double* __restrict__ yrt,
                                              const double* __restrict__ a,
                                              const double* __restrict__ b,
                                              const double* __restrict__ c,
                                              double* __restrict__ ztab) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long long)nkx * nky) return;
  const int kx = (int)(t % nkx), ky = (int)(t / nkx);
  const double xy = xrt[kx] + yrt[ky];
  const long long st = (long long)nkx * nky;
  double d = 0.0;
  for (int k = 0; k < ktot - 1; ++k) {
    const double bb = b[k] + xy;
    const double z = 1.0 / (bb - a[k] * d);
    ztab[k * st + t] = z;
    d = c[k] * z;
  }
  const double bb = (ne == 3) ? b[ktot - 1] : b[ktot - 1] + xy;
  ztab[(long long)(ktot - 1) * st + t] = bb - a[ktot - 1] * d;
}

// The systems of one launch: workgroup row blockIdx.y solves array p[y] with its coefficients.
struct Systems {
  double* p[3];
  const double* a[3];
  const double* c[3];
  const double* ztab[3];
};

// One lane per (i, j) mode of the compact spectral array, the forward sweep's values stored
// back into the array and read again by the back substitution (the path above 257 planes;
// k_tri_seg below takes every smaller grid in one pass).
__global__ void __launch_bounds__(TRI_MODES)
    k_tri(Systems sys, int itot, int jtot, int ktot) {
  double* __restrict__ p = sys.p[blockIdx.y];
  const double* __restrict__ a = sys.a[blockIdx.y];
  const double* __restrict__ c = sys.c[blockIdx.y];
  const double* __restrict__ ztab = sys.ztab[blockIdx.y];
  const long long plane = (long long)itot * jtot;
  const long long m = (long long)blockIdx.x * TRI_MODES + threadIdx.x;
  if (m >= plane) return;
  const int i = (int)(m % itot), j = (int)(m / itot);
  const int nkx = itot / 2 + 1, nky = jtot / 2 + 1;
  const long long zb = (long long)wavenumber(j, jtot) * nkx + wavenumber(i, itot);
  const long long zs = (long long)nkx * nky;
  double prev = 0.0;
  for (int k = 0; k < ktot - 1; ++k) {
    const double z = ztab[k * zs + zb];
    prev = (p[k * plane + m] - a[k] * prev) * z;
    p[k * plane + m] = prev;
  }
  const double zl = ztab[(long long)(ktot - 1) * zs + zb];
  double nxt = zl != 0.0 ? (p[(long long)(ktot - 1) * plane + m] - a[ktot - 1] * prev) / zl : 0.0;
  p[(long long)(ktot - 1) * plane + m] = nxt;
  for (int k = ktot - 2; k >= 0; --k) {
    const double d = c[k] * ztab[k * zs + zb];
    nxt = p[k * plane + m] - d * nxt;
    p[k * plane + m] = nxt;
  }
}

// One pass over the array for the same elimination.  A workgroup takes TRS_MODES modes (the
// lanes) and splits rows 0..ktot-2 into segments of TRS_LSEG rows, half a wavefront each, held in
// registers with their reciprocal pivots.  Each recurrence of the sweep is affine in the value
// it carries in from the previous segment, so
//   forward  y_k = (r_k - a_k y_k-1) z_k      over a segment: y_end = y0_end + G y_in,
//   backward x_k = y_k - d_k x_k+1             over a segment: x_start = x0_start + H x_in,
// where (y0, G) and (x0, H) come from a first pass started at 0 (G, H the products of the
// coefficients -a z and -d).  The carried values are composed through LDS, then every segment
// runs the sweep again from its true incoming value (the same expressions as k_tri inside a
// segment; only the carried values are re-associated).  The last segment also solves the
// last row (solver.f90:103-107, with its zero-pivot guard).  Reads the array and the pivots
// once and writes the solution once, against twice each for k_tri.
// Bound by memory, and by how much of it a compute unit keeps in flight: a workgroup loads, sweeps
// and stores in turn.  With 64 modes only one of 1024 threads fits (its registers hold the rows and
// pivots); 32 modes, whose rows are still two whole cache lines, let two take turns.  The systems of
// one launch and the rows 2j, 2j + 1, which read the same pivots, run close together on one XCD.
// 512 x 512 x 250, four systems: 1287 us with 64 modes, 1168 now (4.0 TB/s), 1460 with 16.
constexpr int TRS_LSEG = 16;                   // rows per segment (registers per lane: 2 x 16)
constexpr int TRS_MAXSEG = 16;                 // segments per workgroup
constexpr int TRS_MODES = 32;                  // modes per workgroup
__global__ void __launch_bounds__(TRS_MODES * TRS_MAXSEG, 4)
    k_tri_seg(Systems sys, int nsys, int itot, int jtot, int ktot) {
  const unsigned blk = xcd_contiguous(blockIdx.x, gridDim.x), sy = blk % nsys;
  double* __restrict__ p = sys.p[sy];
  const double* __restrict__ a = sys.a[sy];
  const double* __restrict__ c = sys.c[sy];
  const double* __restrict__ ztab = sys.ztab[sy];
  __shared__ double fy0[TRS_MAXSEG][TRS_MODES], fg[TRS_MAXSEG][TRS_MODES];
  __shared__ double bx0[TRS_MAXSEG][TRS_MODES], bh[TRS_MAXSEG][TRS_MODES];
  __shared__ double xlast[TRS_MODES];
  __shared__ double sa[TRS_MAXSEG * TRS_LSEG], sc[TRS_MAXSEG * TRS_LSEG];
  const int lane = threadIdx.x & (TRS_MODES - 1);
  const int s = threadIdx.x / TRS_MODES;
  const int nseg = blockDim.x / TRS_MODES;
  const long long plane = (long long)itot * jtot;
  const long long m = (long long)(blk / nsys) * TRS_MODES + lane;
  const bool live = m < plane;
  const int nk = ktot - 1;  // rows of the two recurrences
  const int k0 = min(s * TRS_LSEG, nk), n = min(TRS_LSEG, nk - k0);
  long long zb = 0;
  if (live) {
    const int i = (int)(m % itot), j = (int)(m / itot);
    zb = (long long)wavenumber(j, jtot) * (itot / 2 + 1) + wavenumber(i, itot);
  }
  const long long zs = (long long)(itot / 2 + 1) * (jtot / 2 + 1);
  // rows t >= n of a short segment are padding: they leave every carried value unchanged
  // (selects, so that the arrays stay in registers)
  // (every load is in bounds: lanes past the last mode read mode 0, then discard it)
  const long long mm = live ? m : 0;
  // a and c of the rows from LDS (as registers they would leave one workgroup a compute unit)
  for (int q = threadIdx.x; q < nseg * TRS_LSEG; q += blockDim.x)
    sa[q] = a[min(q, nk - 1)], sc[q] = c[min(q, nk - 1)];
  const double *ak = sa + s * TRS_LSEG, *ck = sc + s * TRS_LSEG;
  double r[TRS_LSEG], z[TRS_LSEG];
  const double alast = a[ktot - 1];
#pragma unroll
  for (int t = 0; t < TRS_LSEG; ++t) {
    const int k = k0 + min(t, max(n - 1, 0));
    const double rv = p[k * plane + mm], zv = ztab[k * zs + zb];
    r[t] = live && n > 0 ? rv : 0.0;
    z[t] = live && n > 0 ? zv : 1.0;
  }
  __syncthreads();
  // forward, first pass: the segment's map y_in -> y_end = y0 + G y_in
  {
    double y = 0.0, gm = 1.0;
#pragma unroll
    for (int t = 0; t < TRS_LSEG; ++t) {
      const double yn = (r[t] - ak[t] * y) * z[t];
      const double gn = gm * (-(ak[t] * z[t]));
      y = t < n ? yn : y;
      gm = t < n ? gn : gm;
    }
    fy0[s][lane] = y, fg[s][lane] = gm;
  }
  __syncthreads();
  double yin = 0.0;
  for (int q = 0; q < s; ++q) yin = fy0[q][lane] + fg[q][lane] * yin;
  // forward, second pass from the true incoming value (r becomes y)
  double prev = yin;
#pragma unroll
  for (int t = 0; t < TRS_LSEG; ++t) {
    const double yn = (r[t] - ak[t] * prev) * z[t];
    prev = t < n ? yn : prev;
    r[t] = prev;
  }
  // the last row, by the last wavefront: y_{ktot-2} is its carried-out value
  if (s == nseg - 1) {
    double nxt = 0.0;
    if (live) {
      const double zl = ztab[(long long)(ktot - 1) * zs + zb];
      nxt = zl != 0.0 ? (p[(long long)(ktot - 1) * plane + m] - alast * prev) / zl : 0.0;
      p[(long long)(ktot - 1) * plane + m] = nxt;
    }
    xlast[lane] = nxt;
  }
  // backward, first pass: the segment's map x_in -> x_start = x0 + H x_in, d_k = c_k z_k
  {
    double x = 0.0, hm = 1.0;
#pragma unroll
    for (int t = TRS_LSEG - 1; t >= 0; --t) {
      const double d = ck[t] * z[t];
      const double xn = r[t] - d * x;
      const double hn = hm * (-d);
      x = t < n ? xn : x;
      hm = t < n ? hn : hm;
    }
    bx0[s][lane] = x, bh[s][lane] = hm;
  }
  __syncthreads();
  double xin = xlast[lane];
  for (int q = nseg - 1; q > s; --q) xin = bx0[q][lane] + bh[q][lane] * xin;
  // backward, second pass: the solution
  double nxt = xin;
#pragma unroll
  for (int t = TRS_LSEG - 1; t >= 0; --t) {
    const double d = ck[t] * z[t];
    const double xn = r[t] - d * nxt;
    nxt = t < n ? xn : nxt;
    r[t] = nxt;
  }
  if (live) {
#pragma unroll
    for (int t = 0; t < TRS_LSEG; ++t)
      if (t < n) p[(k0 + t) * plane + m] = r[t];
  }
}

// ---- stencils --------------------------------------------------------------------------------
// The advection terms read each velocity field at offsets of at most one cell from (i, j, k),
// through an accessor A(di, dj, dk) = field(i + di, j + dj, k + dk) (planes staged in LDS by
// the k-marching kernel), in the reference's expressions and order.

// mom.f90:9-50 (momxad)
template <class A>
__device__ __forceinline__ double momxad(const FGrid& g, const A& Uo, const A& Vo, const A& Wo,
                                         const A& Uoo, const A& Voo, const A& Woo, double uwkm,
                                         double uwkp, double uwkmo, double uwkpo) {
  const double uuip = 0.25 * (Uo(1, 0, 0) + Uo(0, 0, 0)) * (Uo(1, 0, 0) + Uo(0, 0, 0));
  const double uuim = 0.25 * (Uo(-1, 0, 0) + Uo(0, 0, 0)) * (Uo(-1, 0, 0) + Uo(0, 0, 0));
  const double uvjp = 0.25 * (Uo(0, 1, 0) + Uo(0, 0, 0)) * (Vo(1, 0, 0) + Vo(0, 0, 0));
  const double uvjm = 0.25 * (Uo(0, -1, 0) + Uo(0, 0, 0)) * (Vo(1, -1, 0) + Vo(0, -1, 0));
  const double uuipo = 0.25 * (Uoo(1, 0, 0) + Uoo(0, 0, 0)) * (Uoo(1, 0, 0) + Uoo(0, 0, 0));
  const double uuimo = 0.25 * (Uoo(-1, 0, 0) + Uoo(0, 0, 0)) * (Uoo(-1, 0, 0) + Uoo(0, 0, 0));
  const double uvjpo = 0.25 * (Uoo(0, 1, 0) + Uoo(0, 0, 0)) * (Voo(1, 0, 0) + Voo(0, 0, 0));
  const double uvjmo = 0.25 * (Uoo(0, -1, 0) + Uoo(0, 0, 0)) * (Voo(1, -1, 0) + Voo(0, -1, 0));
  return g.dxi * ((1.5 * (-uuip + uuim)) - (.5 * (-uuipo + uuimo))) +
         g.dyi * ((1.5 * (-uvjp + uvjm)) - (.5 * (-uvjpo + uvjmo))) +
         g.dzi * ((1.5 * (-uwkp + uwkm)) - (.5 * (-uwkpo + uwkmo)));
}

// mom.f90:158-199 (momyad)
template <class A>
__device__ __forceinline__ double momyad(const FGrid& g, const A& Uo, const A& Vo, const A& Wo,
                                         const A& Uoo, const A& Voo, const A& Woo, double wvkm,
                                         double wvkp, double wvkmo, double wvkpo) {
  const double uvip = 0.25 * (Uo(0, 0, 0) + Uo(0, 1, 0)) * (Vo(0, 0, 0) + Vo(1, 0, 0));
  const double uvim = 0.25 * (Uo(-1, 0, 0) + Uo(-1, 1, 0)) * (Vo(0, 0, 0) + Vo(-1, 0, 0));
  const double vvjp = 0.25 * (Vo(0, 0, 0) + Vo(0, 1, 0)) * (Vo(0, 0, 0) + Vo(0, 1, 0));
  const double vvjm = 0.25 * (Vo(0, 0, 0) + Vo(0, -1, 0)) * (Vo(0, 0, 0) + Vo(0, -1, 0));
  const double uvipo = 0.25 * (Uoo(0, 0, 0) + Uoo(0, 1, 0)) * (Voo(0, 0, 0) + Voo(1, 0, 0));
  const double uvimo = 0.25 * (Uoo(-1, 0, 0) + Uoo(-1, 1, 0)) * (Voo(0, 0, 0) + Voo(-1, 0, 0));
  const double vvjpo = 0.25 * (Voo(0, 0, 0) + Voo(0, 1, 0)) * (Voo(0, 0, 0) + Voo(0, 1, 0));
  const double vvjmo = 0.25 * (Voo(0, 0, 0) + Voo(0, -1, 0)) * (Voo(0, 0, 0) + Voo(0, -1, 0));
  return g.dxi * ((1.5 * (-uvip + uvim)) - (.5 * (-uvipo + uvimo))) +
         g.dyi * ((1.5 * (-vvjp + vvjm)) - (.5 * (-vvjpo + vvjmo))) +
         g.dzi * ((1.5 * (-wvkp + wvkm)) - (.5 * (-wvkpo + wvkmo)));
}

// mom.f90:286-327 (momzad)
template <class A>
__device__ __forceinline__ double momzad(const FGrid& g, const A& Uo, const A& Vo, const A& Wo,
                                         const A& Uoo, const A& Voo, const A& Woo, double wwkm,
                                         double wwkp, double wwkmo, double wwkpo) {
  const double uwip = 0.25 * (Wo(0, 0, 0) + Wo(1, 0, 0)) * (Uo(0, 0, 0) + Uo(0, 0, 1));
  const double uwim = 0.25 * (Wo(0, 0, 0) + Wo(-1, 0, 0)) * (Uo(-1, 0, 0) + Uo(-1, 0, 1));
  const double vwjp = 0.25 * (Wo(0, 0, 0) + Wo(0, 1, 0)) * (Vo(0, 0, 0) + Vo(0, 0, 1));
  const double vwjm = 0.25 * (Wo(0, 0, 0) + Wo(0, -1, 0)) * (Vo(0, -1, 0) + Vo(0, -1, 1));
  const double uwipo = 0.25 * (Woo(0, 0, 0) + Woo(1, 0, 0)) * (Uoo(0, 0, 0) + Uoo(0, 0, 1));
  const double uwimo = 0.25 * (Woo(0, 0, 0) + Woo(-1, 0, 0)) * (Uoo(-1, 0, 0) + Uoo(-1, 0, 1));
  const double vwjpo = 0.25 * (Woo(0, 0, 0) + Woo(0, 1, 0)) * (Voo(0, 0, 0) + Voo(0, 0, 1));
  const double vwjmo = 0.25 * (Woo(0, 0, 0) + Woo(0, -1, 0)) * (Voo(0, -1, 0) + Voo(0, -1, 1));
  return g.dxi * ((1.5 * (-uwip + uwim)) - (.5 * (-uwipo + uwimo))) +
         g.dyi * ((1.5 * (-vwjp + vwjm)) - (.5 * (-vwjpo + vwjmo))) +
         g.dzi * ((1.5 * (-wwkp + wwkm)) - (.5 * (-wwkpo + wwkmo)));
}

// field(i + di, j + dj, k + dk), dk = 0 or 1, from the planes k and k+1 staged in LDS (row pitch w)
struct LAcc {
  const double* pl[2];  // &plane(i, j) of planes k, k+1
  int w;
  __device__ __forceinline__ double operator()(int di, int dj, int dk) const {
    return pl[dk][di + w * dj];
  }
};

// The fluxes through the face between planes k and k+1 (uwkp, wvkp, wwkp of mom.f90): the face
// below plane k+1 is the same, with its sums the other way round (uwkm, wvkm, wwkm), so the march
// carries them to the next plane.
struct FaceK {
  double u, v, w;
};
template <class A>
__device__ __forceinline__ FaceK face_k(const A& U, const A& V, const A& W) {
  return {0.25 * (U(0, 0, 1) + U(0, 0, 0)) * (W(1, 0, 0) + W(0, 0, 0)),
          0.25 * (W(0, 0, 0) + W(0, 1, 0)) * (V(0, 0, 1) + V(0, 0, 0)),
          0.25 * (W(0, 0, 0) + W(0, 0, 1)) * (W(0, 0, 0) + W(0, 0, 1))};
}

// p at a cell and its three next neighbours, and the forces there
struct CellIn {
  double p, pi, pj, pk, fx, fy, fz;
};

// The three right-hand sides of fftuvw.f90:30-105 at one interior cell, scaled by Rep
// (dwdt(:,:,kmax) = 0): -(dp/dx) + f, minus the advection terms, minus uo/dt.
template <class A>
__device__ __forceinline__ void mom_cell(const FGrid& g, double rep, double dt, const A& U,
                                         const A& V, const A& W, const A& UU, const A& VV,
                                         const A& WW, const CellIn& in, int k,
                                         FaceK& f, FaceK& fo, double& du, double& dv,
                                         double& dw) {
  const FaceK fp = face_k(U, V, W), fpo = face_k(UU, VV, WW);
  const double durk = (-g.dxi * ((in.pi - in.p))) + in.fx;
  const double dvrk = (-g.dyi * (in.pj - in.p)) + in.fy;
  const double dwrk = (-g.dzi * (in.pk - in.p)) + in.fz;
  du = -durk, dv = -dvrk, dw = -dwrk;
  du = du - momxad(g, U, V, W, UU, VV, WW, f.u, fp.u, fo.u, fpo.u);
  dv = dv - momyad(g, U, V, W, UU, VV, WW, f.v, fp.v, fo.v, fpo.v);
  dw = dw - momzad(g, U, V, W, UU, VV, WW, f.w, fp.w, fo.w, fpo.w);
  du = du - (U(0, 0, 0) / dt);
  dv = dv - (V(0, 0, 0) / dt);
  dw = dw - (W(0, 0, 0) / dt);
  du = du * rep;
  dv = dv * rep;
  dw = (k == g.ktot) ? 0.0 : dw * rep;
  f = fp, fo = fpo;
}

// fftuvw.f90:30-105 per interior cell, k-marching, into the compact arrays: a workgroup owns
// an MR_TI x MR_TJ tile of (i, j) columns and KB consecutive planes.  The six velocity fields'
// planes k and k+1 of the tile plus a one-cell apron sit in LDS; the fluxes through the face below
// plane k are carried in registers, so plane k-1 is not needed.  Each step starts the loads of
// plane k+2 and of the next cell's p and forces, computes plane k from what is there, and stores
// plane k+2 over plane k: no load is waited for before the arithmetic.  Every velocity value is
// read from HBM once per tile (plus the apron and the two extra planes).
// Bound by memory latency: 512 x 512 x 250 cells (6.9 GB) 1610 us with three planes in LDS and p
// and the forces loaded at their use, 1650 with the carried fluxes alone, 1484 with both (4.6 TB/s).
// At most three workgroups a compute unit: held to 128 registers for four, it spills (3330 us).
// 64 x 4 tiles: 1580; the tiles of an XCD made contiguous: slower (1650 -> 1700 before the
// earlier loads).
constexpr int MR_TI = 32, MR_TJ = 8;
constexpr int MR_W = MR_TI + 2, MR_H = MR_TJ + 2, MR_PL = MR_W * MR_H;
constexpr int MR_T = MR_TI * MR_TJ;
constexpr int MR_LD = (MR_PL + MR_T - 1) / MR_T;  // apron-plane cells per thread

__global__ void __launch_bounds__(MR_T, 3)
    k_mom_rhs_march(FGrid g, int KB, double rep, double dt, const double* __restrict__ uo,
                    const double* __restrict__ vo, const double* __restrict__ wo,
                    const double* __restrict__ uoo, const double* __restrict__ voo,
                    const double* __restrict__ woo, const double* __restrict__ p,
                    const double* __restrict__ fx, const double* __restrict__ fy,
                    const double* __restrict__ fz, double* __restrict__ cu,
                    double* __restrict__ cv, double* __restrict__ cw) {
  __shared__ double sp[6][2][MR_PL];
  const double* src[6] = {uo, vo, wo, uoo, voo, woo};
  const int tx = threadIdx.x % MR_TI, ty = threadIdx.x / MR_TI;
  const int i0 = blockIdx.x * MR_TI, j0 = blockIdx.y * MR_TJ;  // apron origin (halo index)
  const int kb0 = blockIdx.z * KB + 1;
  const int kb1 = min(kb0 + KB - 1, g.ktot);
  // the apron-plane cells this thread loads: c = tid + r MR_T
  long long off[MR_LD];
  bool ok[MR_LD];
#pragma unroll
  for (int r = 0; r < MR_LD; ++r) {
    const int c = threadIdx.x + r * MR_T;
    const int ii = c % MR_W, jj = c / MR_W;
    ok[r] = c < MR_PL && i0 + ii <= g.itot + 1 && j0 + jj <= g.jtot + 1;
    off[r] = ok[r] ? (long long)(i0 + ii) + g.sy * (j0 + jj) : 0;
  }
  // planes kb0-1 and kb0 into slots 0 and 1 (plane kk lives in slot (kk-kb0+1) & 1)
  for (int s0 = 0; s0 < 2; ++s0) {
    const long long kz = g.sz * (kb0 - 1 + s0);
#pragma unroll
    for (int f = 0; f < 6; ++f)
#pragma unroll
      for (int r = 0; r < MR_LD; ++r)
        if (threadIdx.x + r * MR_T < MR_PL) sp[f][s0][threadIdx.x + r * MR_T] = ok[r] ? src[f][off[r] + kz] : 0.0;
  }
  __syncthreads();
  const int i = i0 + tx + 1, j = j0 + ty + 1;
  const bool live = i <= g.itot && j <= g.jtot;
  const int me = (tx + 1) + MR_W * (ty + 1);
  FaceK face{}, faceo{};
  const long long q0 = live ? fidx(g, i, j, 0) : 0;
  CellIn in{}, nx{};
  nx.pk = live ? p[q0 + g.sz * kb0] : 0.0;
  // plane kb0-1 gives the faces below plane kb0 alone
  for (int k = kb0 - 1; k <= kb1; ++k) {
    const int s0 = (k - kb0 + 1) & 1, sp1 = s0 ^ 1;
    // prefetch plane k + 2 (the next step's k + 1)
    const bool more = k + 2 <= kb1 + 1;
    in = nx;
    if (live && more) {
      const long long q = q0 + g.sz * (k + 1);
      nx = CellIn{in.pk, p[q + 1], p[q + g.sy], p[q + g.sz], fx[q], fy[q], fz[q]};
    }
    double pre[6][MR_LD];
    if (more) {
      const long long kz = g.sz * (k + 2);
#pragma unroll
      for (int f = 0; f < 6; ++f)
#pragma unroll
        for (int r = 0; r < MR_LD; ++r) pre[f][r] = ok[r] ? src[f][off[r] + kz] : 0.0;
    }
    if (live) {
      LAcc A[6];
#pragma unroll
      for (int f = 0; f < 6; ++f) A[f] = LAcc{{&sp[f][s0][me], &sp[f][sp1][me]}, MR_W};
      if (k < kb0) {
        face = face_k(A[0], A[1], A[2]), faceo = face_k(A[3], A[4], A[5]);
      } else {
        double du, dv, dw;
        mom_cell(g, rep, dt, A[0], A[1], A[2], A[3], A[4], A[5], in, k, face, faceo, du, dv, dw);
        const long long t = (long long)(i - 1) + (long long)g.itot * ((j - 1) + (long long)g.jtot * (k - 1));
        cu[t] = du;
        cv[t] = dv;
        cw[t] = dw;
      }
    }
    __syncthreads();  // plane k is no longer read
    if (more) {
#pragma unroll
      for (int f = 0; f < 6; ++f)
#pragma unroll
        for (int r = 0; r < MR_LD; ++r)
          if (threadIdx.x + r * MR_T < MR_PL) sp[f][s0][threadIdx.x + r * MR_T] = pre[f][r];
    }
    __syncthreads();
  }
}

// fillps.f90:8-47 into the compact array
__global__ void __launch_bounds__(256) k_fillps(FGrid g, double dt, const double* __restrict__ u,
                                                const double* __restrict__ v,
                                                const double* __restrict__ w,
                                                double* __restrict__ cp) {
  const long long n = (long long)g.itot * g.jtot * g.ktot;
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int i = (int)(t % g.itot) + 1;
  const long long r = t / g.itot;
  const int j = (int)(r % g.jtot) + 1, k = (int)(r / g.jtot) + 1;
  const double dti = 1.0 / dt;
  const double dtidxi = dti * g.dxi, dtidyi = dti * g.dyi, dtidzi = dti * g.dzi;
  const long long q = fidx(g, i, j, k);
  cp[t] = ((w[q] - w[q - g.sz]) * dtidzi + (v[q] - v[q - g.sy]) * dtidyi +
           (u[q] - u[q - 1]) * dtidxi);
}

// a compact array into the interior of a field
__global__ void __launch_bounds__(256) k_to_field(FGrid g, const double* __restrict__ c,
                                                  double* __restrict__ f) {
  const long long n = (long long)g.itot * g.jtot * g.ktot;
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int i = (int)(t % g.itot) + 1;
  const long long r = t / g.itot;
  f[fidx(g, i, (int)(r % g.jtot) + 1, (int)(r / g.jtot) + 1)] = c[t];
}

// correc.f90:11-38
__global__ void __launch_bounds__(256) k_correc(FGrid g, double dt, double* __restrict__ u,
                                                double* __restrict__ v, double* __restrict__ w,
                                                const double* __restrict__ p) {
  const long long n = (long long)g.itot * g.jtot * g.ktot;
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int i = (int)(t % g.itot) + 1;
  const long long r = t / g.itot;
  const int j = (int)(r % g.jtot) + 1, k = (int)(r / g.jtot) + 1;
  const double factori = dt * g.dxi, factorj = dt * g.dyi, factork = dt * g.dzi;
  const long long q = fidx(g, i, j, k);
  u[q] = u[q] - factori * (p[q + 1] - p[q]);
  v[q] = v[q] - factorj * (p[q + g.sy] - p[q]);
  w[q] = w[q] - factork * (p[q + g.sz] - p[q]);
}

// correc (correc.f90:11-38) and pnew += p (main.f90:406-408) in one pass over the cells: the
// two touch disjoint outputs and both read p, which is then read once.  The p beyond the last cell
// of a line or row is the first one, above the last plane the cell's own (bound.f90:93-98): read
// there, so that p's halos are set with all others after this pass.  Two neighbouring cells a
// thread (itot is even).  Bound by memory: 1024 x 512 x 256 (9.7 GB) 1905 us a cell a thread from
// halos, 2010 from the interior, 1966 two cells a thread (4.9 TB/s); a step at 256 x 128 x 128
// 437 -> 432 us with the two cells.
__global__ void __launch_bounds__(256) k_correc_addp(FGrid g, int logh, int logj, double dt,
                                                     double* __restrict__ u,
                                                     double* __restrict__ v,
                                                     double* __restrict__ w,
                                                     const double* __restrict__ p,
                                                     double* __restrict__ pn) {
  const long long n = (long long)(g.itot / 2) * g.jtot * g.ktot;
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int h = (int)(t & ((1 << logh) - 1)), r = (int)(t >> logh);
  const int j = (r & ((1 << logj) - 1)) + 1, k = (r >> logj) + 1;
  const double factori = dt * g.dxi, factorj = dt * g.dyi, factork = dt * g.dzi;
  const long long q = fidx(g, 2 * h + 1, j, k);
  const double2 pq = load2(p + q);
  const double2 pi = make_double2(pq.y, p[h < (1 << logh) - 1 ? q + 2 : q + 2 - g.itot]);
  const double2 pj = load2(p + (j < g.jtot ? q + g.sy : q - (g.jtot - 1) * g.sy));
  const double2 pk = load2(p + (k < g.ktot ? q + g.sz : q));
  const double2 uq = load2(u + q), vq = load2(v + q), wq = load2(w + q), nq = load2(pn + q);
  store2(u + q, make_double2(uq.x - factori * (pi.x - pq.x), uq.y - factori * (pi.y - pq.y)));
  store2(v + q, make_double2(vq.x - factorj * (pj.x - pq.x), vq.y - factorj * (pj.y - pq.y)));
  store2(w + q, make_double2(wq.x - factork * (pk.x - pq.x), wq.y - factork * (pk.y - pq.y)));
  store2(pn + q, make_double2(nq.x + pq.x, nq.y + pq.y));
}

// Final value of a wall ghost / top face after the k step of bounduvw (bound.f90:38-56) or
// boundp (:93-98), at interior column (i, j).  kind 0: u or v (ghost = -interior), 1: w
// (0 on both wall faces, k1 copies kmax-1), 2: p (ghost = interior).
__device__ __forceinline__ double kstep(const FGrid& g, const double* f, int kind, int i, int j,
                                        int k) {
  const int kmax = g.ktot, k1 = g.ktot + 1;
  if (kind == 0) {
    if (k == 0) return -f[fidx(g, i, j, 1)];
    if (k == k1) return -f[fidx(g, i, j, kmax)];
  } else if (kind == 1) {
    if (k == 0 || k == kmax) return 0.0;
    if (k == k1) return f[fidx(g, i, j, kmax - 1)];
  } else {
    if (k == 0) return f[fidx(g, i, j, 1)];
    if (k == k1) return f[fidx(g, i, j, kmax)];
  }
  return f[fidx(g, i, j, k)];
}

// bounduvw / boundp in one launch: the k step, then updthalos in x, then in y
// (bound.f90:61-76, 100-104; bound.f90:141-190).  Every halo or ghost cell takes its final
// value straight from the interior column the sequence copies it from, and those interior
// values are not written here, so every cell is independent.  Threads [0, nfields * itot *
// jtot) take an interior column (its ghost planes k = 0 and ktot+1, and k = ktot for w); the
// rest one cell of a halo column: x halos i = 0, itot+1 for j = 0..jtot+1, then y halos
// j = 0, jtot+1 for i = 1..itot, every k (halo index fastest).
// kinds: the field kinds of kstep, four bits each.
struct Fields {
  double* f[5];
};
__global__ void __launch_bounds__(256) k_bound(FGrid g, Fields fs, int nfields, unsigned kinds) {
  const long long nin = (long long)g.itot * g.jtot;
  const long long nxh = 2LL * (g.jtot + 2), nh = nxh + 2LL * g.itot, K = g.ktot + 2;
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < nin * nfields) {
    const int fi = (int)(t / nin);
    const long long r = t - fi * nin;
    const int i = 1 + (int)(r % g.itot), j = 1 + (int)(r / g.itot);
    double* f = fs.f[fi];
    const int kind = (kinds >> (4 * fi)) & 15;
    f[fidx(g, i, j, 0)] = kstep(g, f, kind, i, j, 0);
    f[fidx(g, i, j, g.ktot + 1)] = kstep(g, f, kind, i, j, g.ktot + 1);
    if (kind == 1) f[fidx(g, i, j, g.ktot)] = 0.0;
    return;
  }
  const long long e = t - nin * nfields;
  if (e >= nh * K * nfields) return;
  const int fi = (int)(e / (nh * K));
  const long long r = e - fi * nh * K;
  const int k = (int)(r / nh);
  const long long h = r - k * nh;
  int i, j;
  if (h < nxh) {
    i = h < g.jtot + 2 ? 0 : g.itot + 1;
    j = (int)(h % (g.jtot + 2));
  } else {
    const long long hy = h - nxh;
    j = hy < g.itot ? 0 : g.jtot + 1;
    i = 1 + (int)(hy % g.itot);
  }
  double* f = fs.f[fi];
  const int kind = (kinds >> (4 * fi)) & 15;
  const int si = i == 0 ? g.itot : (i == g.itot + 1 ? 1 : i);
  const int sj = j == 0 ? g.jtot : (j == g.jtot + 1 ? 1 : j);
  f[fidx(g, i, j, k)] = kstep(g, f, kind, si, sj, k);
}

// indicator.f90:51-67: the central divergence of G = (gx, gy, gz), ((g(+1) - g(-1)) .5) d?i
// summed x + y + z, for every interior cell, into the compact array cp (the right-hand side
// of the indicator's Poisson solve) or, with f != nullptr, into the interior of the field f.
__global__ void __launch_bounds__(256) k_ind_div(FGrid g, const double* __restrict__ gx,
                                                 const double* __restrict__ gy,
                                                 const double* __restrict__ gz,
                                                 double* __restrict__ cp,
                                                 double* __restrict__ f) {
  const long long n = (long long)g.itot * g.jtot * g.ktot;
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int i = (int)(t % g.itot) + 1;
  const long long r = t / g.itot;
  const int j = (int)(r % g.jtot) + 1, k = (int)(r / g.jtot) + 1;
  const long long q = fidx(g, i, j, k);
  const double dgx = (gx[q + 1] - gx[q - 1]) * .5 * g.dxi;
  const double dgy = (gy[q + g.sy] - gy[q - g.sy]) * .5 * g.dyi;
  const double dgz = (gz[q + g.sz] - gz[q - g.sz]) * .5 * g.dzi;
  const double dg = dgx + dgy + dgz;
  if (f)
    f[q] = dg;
  else
    cp[t] = dg;
}

// indicator.f90:93-103: indic(i,j,k) = indi(i,j,k + ktot/4) for k <= kmax - ktot/4, else 0
// (the solution moved back down by the planes the capsules were shifted up)
__global__ void __launch_bounds__(256) k_ind_shift(FGrid g, const double* __restrict__ indi,
                                                   double* __restrict__ indic) {
  const long long n = (long long)g.itot * g.jtot * g.ktot;
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int i = (int)(t % g.itot) + 1;
  const long long r = t / g.itot;
  const int j = (int)(r % g.jtot) + 1, k = (int)(r / g.jtot) + 1;
  const int kq = g.ktot / 4;
  indic[fidx(g, i, j, k)] = k <= g.ktot - kq ? indi[fidx(g, i, j, k + kq)] : 0.0;
}

// indicator.f90:105-112: < .01 -> 0, >= .9 -> 1 (idempotent)
__device__ __forceinline__ double ind_threshold(double v) {
  if (v < .01) v = 0.;
  if (v >= .9) v = 1.;
  return v;
}

// indicator.f90:105-168 after boundind(indic), fused per interior cell: the thresholds, the
// viscosity visc0 (1 + (lambda - 1) indic) (:137-143) and the centrifugal buoyancy
//   forcey += .5 (indic(j) + indic(j+1)) sin(thetainc) tcoef          (:164)
//   forcez += .5 (indic(k) + indic(k+1)) (-cos(thetainc)) tcoef       (:165)
// The reference thresholds the whole interior before the force loop, so an interior
// neighbour is read thresholded and a halo neighbour (j+1 = j1, k+1 = k1) as boundind left
// it.  A neighbour is read here and thresholded on the spot: the threshold is idempotent, so
// reading it before or after its own thread rewrote it gives the same value.
__global__ void __launch_bounds__(256) k_ind_finish(FGrid g, double* __restrict__ indic,
                                                    double* __restrict__ visc,
                                                    double* __restrict__ forcey,
                                                    double* __restrict__ forcez, double lambda,
                                                    double visc0, double sin_t, double mcos_t,
                                                    double tcoef) {
  const long long n = (long long)g.itot * g.jtot * g.ktot;
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int i = (int)(t % g.itot) + 1;
  const long long r = t / g.itot;
  const int j = (int)(r % g.jtot) + 1, k = (int)(r / g.jtot) + 1;
  const long long q = fidx(g, i, j, k);
  const double v = ind_threshold(indic[q]);
  double vy = indic[q + g.sy], vz = indic[q + g.sz];
  if (j < g.jtot) vy = ind_threshold(vy);
  if (k < g.ktot) vz = ind_threshold(vz);
  indic[q] = v;
  visc[q] = visc0 * (1. + ((lambda - 1.) * v));
  forcey[q] = forcey[q] + (.5 * (v + vy) * sin_t * tcoef);
  forcez[q] = forcez[q] + (.5 * (v + vz) * mcos_t * tcoef);
}

// chkdiv.f90:7-61: per-block sums and maxima of the discrete divergence
__global__ void __launch_bounds__(256) k_div(FGrid g, const double* __restrict__ u,
                                             const double* __restrict__ v,
                                             const double* __restrict__ w,
                                             double* __restrict__ part) {
  __shared__ double ss[256], sm[256];
  const long long n = (long long)g.itot * g.jtot * g.ktot;
  double s = 0.0, m = 0.0;
  for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < n;
       t += (long long)gridDim.x * blockDim.x) {
    const int i = (int)(t % g.itot) + 1;
    const long long r = t / g.itot;
    const int j = (int)(r % g.jtot) + 1, k = (int)(r / g.jtot) + 1;
    const long long q = fidx(g, i, j, k);
    const double div = (w[q] - w[q - g.sz]) * g.dzi + (v[q] - v[q - g.sy]) * g.dyi +
                       (u[q] - u[q - 1]) * g.dxi;
    s = s + div;
    m = fmax(m, fabs(div));
  }
  ss[threadIdx.x] = s, sm[threadIdx.x] = m;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (threadIdx.x < h) {
      ss[threadIdx.x] = ss[threadIdx.x] + ss[threadIdx.x + h];
      sm[threadIdx.x] = fmax(sm[threadIdx.x], sm[threadIdx.x + h]);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) part[2 * blockIdx.x] = ss[0], part[2 * blockIdx.x + 1] = sm[0];
}

}  // namespace

struct fld_ctx {
  ibx_grid grid{};
  FGrid g{};
  double rep = 0, dt = 0;
  int device = 0;
  int cus = 256;
  hipStream_t own = nullptr, stream = nullptr;
  std::string err;
  long long ncomp = 0;                  // itot * jtot * ktot
  double* work[3] = {nullptr, nullptr, nullptr};  // compact spectral arrays
  double* ztab[4] = {nullptr, nullptr, nullptr, nullptr};  // index ne = 1..3
  double* coef[4] = {nullptr, nullptr, nullptr, nullptr};  // a, c per ne (2 * ktot each)
  double2* tw_x = nullptr;
  double2* tw_y = nullptr;
  double2* tw_xm = nullptr;  // exp(-2 pi i k / M), k < M = itot / 2
  double2* tw_yn = nullptr;  // exp(-2 pi i k / jtot), k < jtot
  double* part = nullptr;  // chkdiv partials
  int logmx = 0, logmy = 0;
  size_t lds_yf = 0, lds_yi = 0;
  int ylines_f = Y_LINES_FWD, ylines_i = Y_LINES_INV, xlines = 1;
};

namespace {

int fail(fld_ctx* c, int code, const std::string& msg) {
  if (c) c->err = msg;
  return code;
}

#define HIPF(ctx, call)                                                                      \
  do {                                                                                       \
    hipError_t e_ = (call);                                                                  \
    if (e_ != hipSuccess)                                                                    \
      return fail((ctx), FLD_E_HIP, std::string(#call) + ": " + hipGetErrorString(e_) +     \
                                        " (" + __FILE__ + ":" + std::to_string(__LINE__) + ")"); \
  } while (0)

inline unsigned nblocks(long long n, int b) { return (unsigned)((n + b - 1) / b); }

int ilog2(int n) {
  int l = 0;
  while ((1 << l) < n) ++l;
  return l;
}

bool pow2(int n) { return n >= 2 && (n & (n - 1)) == 0; }

// exp(-2 pi i k / n), k < count, from long-double sine and cosine
std::vector<double2> twiddles(int n, int count) {
  std::vector<double2> t((size_t)std::max(1, count));
  const long double pi = 3.141592653589793238462643383279502884L;
  for (int k = 0; k < count; ++k) {
    const long double a = 2.0L * pi * (long double)k / (long double)n;
    t[(size_t)k] = make_double2((double)cosl(a), (double)(-sinl(a)));
  }
  return t;
}

// initsolver.f90:108-132 by wavenumber: 0, 1 .. n/2 - 1, and n/2
std::vector<double> eigen(int n, double di) {
  std::vector<double> e((size_t)(n / 2 + 1));
  const double pi = std::acos(-1.0);
  e[0] = 0.0;
  for (int m = 1; m < n / 2; ++m) {
    const double s = std::sin((double)(2 * m) * pi / (2.0 * n));
    e[(size_t)m] = -(4.0 * di * di * (s * s));
  }
  e[(size_t)(n / 2)] = -(4.0 * di * di);
  return e;
}

// initsolver.f90:23-99 for e = 1, 2, 3 (main mesh)
void tridiag(const fld_ctx* c, int e, std::vector<double>& a, std::vector<double>& b,
             std::vector<double>& cc) {
  const int kmax = c->grid.ktot;
  const double dzi = c->grid.dzi;
  a.assign((size_t)kmax, 0.0), b.assign((size_t)kmax, 0.0), cc.assign((size_t)kmax, 0.0);
  for (int k = 0; k < kmax; ++k) {
    a[(size_t)k] = dzi * dzi;
    cc[(size_t)k] = dzi * dzi;
    b[(size_t)k] = -(a[(size_t)k] + cc[(size_t)k]);
  }
  if (e == 1) {
    b[0] = b[0] + a[0];
    b[(size_t)kmax - 1] = b[(size_t)kmax - 1] + cc[(size_t)kmax - 1];
    a[0] = 0.0;
    cc[(size_t)kmax - 1] = 0.0;
  } else {
    if (e == 2) {
      b[0] = b[0] - a[0];
      b[(size_t)kmax - 1] = b[(size_t)kmax - 1] - cc[(size_t)kmax - 1];
      a[0] = 0.0;
      cc[(size_t)kmax - 1] = 0.0;
    } else {
      b[(size_t)kmax - 1] = 1.0;
      a[0] = 0.0;
      a[(size_t)kmax - 1] = 0.0;
      cc[(size_t)kmax - 1] = 0.0;
    }
    for (int k = 0; k < kmax; ++k) b[(size_t)k] = b[(size_t)k] - (c->rep / c->dt);
    if (e == 3) b[(size_t)kmax - 1] = 1.0;
  }
}

// f(integral_constant<int, L>) for the run-time L in [LO, HI]
template <int LO, int HI, class F>
void with_log(int L, F&& f) {
  if constexpr (LO <= HI) {
    if (L == LO)
      f(std::integral_constant<int, LO>{});
    else
      with_log<LO + 1, HI>(L, f);
  }
}

bool reg_x(const fld_ctx* c) { return c->logmx >= 3 && c->logmx <= 10; }
bool reg_y(const fld_ctx* c) { return c->logmy >= 2 && c->logmy <= 9; }

// x transforms of n systems by the register kernels; fs: the pressure's divergence as the source
int reg_fft_x(fld_ctx* c, bool inv, int n, const Arrays& arr, bool src_field, bool dst_field,
              const FillSrc* fs) {
  const FGrid& g = c->g;
  const Rows field{1 + g.sy + g.sz, g.sy, g.sz}, compact{0, g.itot, (long long)g.itot * g.jtot};
  const Rows rs = src_field ? field : compact, rd = dst_field ? field : compact;
  const int lines = g.jtot * g.ktot, logj = c->logmy + 1;
  with_log<3, 10>(c->logmx, [&](auto l) {
    constexpr int L = decltype(l)::value;
    const dim3 nb(nblocks(lines, XLine<L>::PER), (unsigned)n);
    if (inv)
      k_x_inv<L><<<nb, REG_T, 0, c->stream>>>(arr, rs, rd, logj, lines, c->tw_x, c->tw_xm);
    else if (fs)
      k_x_fwd<L, true><<<nb, REG_T, 0, c->stream>>>(arr, rs, rd, logj, lines, c->tw_x, c->tw_xm, *fs);
    else
      k_x_fwd<L, false><<<nb, REG_T, 0, c->stream>>>(arr, rs, rd, logj, lines, c->tw_x, c->tw_xm,
                                                     FillSrc{});
  });
  HIPF(c, hipGetLastError());
  return FLD_OK;
}

int reg_fft_y(fld_ctx* c, bool inv, int n, const Arrays& arr) {
  const FGrid& g = c->g;
  const long long pairs = (long long)(g.itot / 2) * g.ktot;
  with_log<3, 10>(c->logmy + 1, [&](auto l) {
    constexpr int L = decltype(l)::value;
    const dim3 nb(nblocks(pairs, YLine<L>::COLS), (unsigned)n);
    if (inv)
      k_y<L, true><<<nb, YLine<L>::T, 0, c->stream>>>(arr, c->logmx, pairs, c->tw_yn);
    else
      k_y<L, false><<<nb, YLine<L>::T, 0, c->stream>>>(arr, c->logmx, pairs, c->tw_yn);
  });
  HIPF(c, hipGetLastError());
  return FLD_OK;
}

// x transforms of the interior lines of n fields (or compact arrays), forward or inverse
int fft_x(fld_ctx* c, bool inv, int n, const Arrays& arr, bool src_field, bool dst_field) {
  if (reg_x(c)) return reg_fft_x(c, inv, n, arr, src_field, dst_field, nullptr);
  const FGrid& g = c->g;
  const int N = g.itot, nl = c->xlines;
  const int gpp = g.jtot / nl;  // workgroups per k plane
  const long long cp = (long long)g.itot * g.jtot;
  const long long row_s = src_field ? g.sy : g.itot, plane_s = src_field ? g.sz : cp;
  const long long row_d = dst_field ? g.sy : g.itot, plane_d = dst_field ? g.sz : cp;
  const long long off = 1 + g.sy + g.sz;  // (1, 1, 1)
  // lines, plus the inverse's LDS copy of the twiddles
  const size_t lds = (size_t)nl * (N / 2 + 1) * sizeof(double2) + (inv ? (size_t)(N / 2) * sizeof(double2) : 0);
  const dim3 nb((unsigned)(gpp * g.ktot), (unsigned)n);
  if (!inv)
    k_rfft_fwd<true><<<nb, FFT_THREADS, lds, c->stream>>>(
        arr, N, c->logmx, nl, gpp, plane_s, plane_d, nl * row_s, nl * row_d, 1, row_s, 1, row_d,
        src_field ? off : 0, c->tw_x, FillSrc{});
  else
    k_rfft_inv<true><<<nb, FFT_THREADS, lds, c->stream>>>(
        arr, N, c->logmx, nl, gpp, plane_s, plane_d, nl * row_s, nl * row_d, 1, row_s, 1, row_d,
        dst_field ? off : 0, c->tw_x);
  HIPF(c, hipGetLastError());
  return FLD_OK;
}

// y transforms in place on n compact arrays
int fft_y(fld_ctx* c, bool inv, int n, double* const* a) {
  const FGrid& g = c->g;
  const int N = g.jtot, nl = inv ? c->ylines_i : c->ylines_f;
  const int gpp = g.itot / nl;
  const long long cp = (long long)g.itot * g.jtot;
  const dim3 nb((unsigned)(gpp * g.ktot), (unsigned)n);
  Arrays arr{};
  for (int i = 0; i < n; ++i) arr.src[i] = arr.dst[i] = a[i];
  if (reg_y(c)) return reg_fft_y(c, inv, n, arr);
  if (!inv)
    k_rfft_fwd<false><<<nb, FFT_THREADS, c->lds_yf, c->stream>>>(
        arr, N, c->logmy, nl, gpp, cp, cp, nl, nl, g.itot, 1, g.itot, 1, 0, c->tw_y, FillSrc{});
  else
    k_rfft_inv<false><<<nb, FFT_THREADS, c->lds_yi, c->stream>>>(
        arr, N, c->logmy, nl, gpp, cp, cp, nl, nl, g.itot, 1, g.itot, 1, 0, c->tw_y);
  HIPF(c, hipGetLastError());
  return FLD_OK;
}

int tri(fld_ctx* c, int n, double* const* a, const int* ne) {
  const FGrid& g = c->g;
  const long long modes = (long long)g.itot * g.jtot;
  Systems sys{};
  for (int i = 0; i < n; ++i)
    sys.p[i] = a[i], sys.a[i] = c->coef[ne[i]], sys.c[i] = c->coef[ne[i]] + g.ktot,
    sys.ztab[i] = c->ztab[ne[i]];
  const int nseg = std::max(1, (g.ktot - 1 + TRS_LSEG - 1) / TRS_LSEG);
  if (nseg <= TRS_MAXSEG)
    k_tri_seg<<<nblocks(modes, TRS_MODES) * (unsigned)n, TRS_MODES * nseg, 0, c->stream>>>(
        sys, n, g.itot, g.jtot, g.ktot);
  else
    k_tri<<<dim3(nblocks(modes, TRI_MODES), (unsigned)n), TRI_MODES, 0, c->stream>>>(
        sys, g.itot, g.jtot, g.ktot);
  HIPF(c, hipGetLastError());
  return FLD_OK;
}

// fillps (the divergence fs) already transformed in x, into the compact
// array dst: k_fillps and the pressure solve's forward x transform in one pass
int fft_x_fill(fld_ctx* c, const FillSrc& fs, double* dst) {
  const FGrid& g = c->g;
  const int N = g.itot, nl = c->xlines;
  const int gpp = g.jtot / nl;
  const long long cp = (long long)g.itot * g.jtot, row = g.itot;
  const size_t lds = (size_t)nl * (N / 2 + 1) * sizeof(double2);
  const unsigned nb = (unsigned)(gpp * g.ktot);
  const Arrays arr{{nullptr, nullptr, nullptr}, {dst, nullptr, nullptr}};
  if (reg_x(c)) return reg_fft_x(c, false, 1, arr, false, false, &fs);
  k_rfft_fwd<true, true><<<nb, FFT_THREADS, lds, c->stream>>>(
      arr, N, c->logmx, nl, gpp, cp, cp,
      nl * row, nl * row, 1, row, 1, row, 0, c->tw_x, fs);
  HIPF(c, hipGetLastError());
  return FLD_OK;
}

// f(LOGI, LOGJ as integral constants) where the plane kernels hold such a plane; the largest from
// 32 planes on (128 x 64 x 16: 68.4 us a step with them, 68.0 without)
template <class F>
bool with_plane(const fld_ctx* c, F&& f) {
  const int li = c->logmx + 1, lj = c->logmy + 1;
  if (li < 5 || lj < 5 || li + lj > (c->g.ktot >= 32 ? 13 : 12)) return false;
  with_log<5, 8>(li, [&](auto i) {
    constexpr int LI = decltype(i)::value;
    with_log<5, 13 - LI>(lj, [&](auto j) { f(i, j); });
  });
  return true;
}

// Forward x and y transforms of n systems io (fields or compact arrays, or the divergence fs) into
// the compact arrays a
int fft_xy(fld_ctx* c, int n, double* const* io, bool field, const FillSrc* fs, double* const* a) {
  const FGrid& g = c->g;
  const Rows rf{1 + g.sy + g.sz, g.sy, g.sz}, rc{0, g.itot, (long long)g.itot * g.jtot};
  Arrays arr{};
  for (int i = 0; i < n; ++i) arr.src[i] = io[i], arr.dst[i] = a[i];
  if (with_plane(c, [&](auto i, auto j) {
        constexpr int LI = decltype(i)::value, LJ = decltype(j)::value;
        const dim3 nb((unsigned)g.ktot, (unsigned)n);
        if (fs)
          k_plane_fwd<LI, LJ, true>
              <<<nb, REG_T, 0, c->stream>>>(arr, rc, c->tw_x, c->tw_xm, c->tw_yn, *fs);
        else
          k_plane_fwd<LI, LJ, false><<<nb, REG_T, 0, c->stream>>>(
              arr, field ? rf : rc, c->tw_x, c->tw_xm, c->tw_yn, FillSrc{});
      })) {
    HIPF(c, hipGetLastError());
    return FLD_OK;
  }
  const int rv = fs ? fft_x_fill(c, *fs, a[0]) : fft_x(c, false, n, arr, field, false);
  return rv ? rv : fft_y(c, false, n, a);
}

// and back, into the interiors of the fields out
int ifft_xy(fld_ctx* c, int n, double* const* a, double* const* out) {
  const FGrid& g = c->g;
  const Rows rf{1 + g.sy + g.sz, g.sy, g.sz};
  Arrays arr{};
  for (int i = 0; i < n; ++i) arr.src[i] = a[i], arr.dst[i] = out[i];
  if (with_plane(c, [&](auto i, auto j) {
        constexpr int LI = decltype(i)::value, LJ = decltype(j)::value;
        k_plane_inv<LI, LJ><<<dim3((unsigned)g.ktot, (unsigned)n), REG_T, 0, c->stream>>>(
            arr, rf, c->tw_x, c->tw_xm, c->tw_yn);
      })) {
    HIPF(c, hipGetLastError());
    return FLD_OK;
  }
  const int rv = fft_y(c, true, n, a);
  return rv ? rv : fft_x(c, true, n, arr, false, true);
}

// n solver1d of the sources io (as fft_xy's), through the compact arrays a, into the interiors of
// the fields out
int solve(fld_ctx* c, int n, double* const* io, bool field, const FillSrc* fs, double* const* a,
          const int* ne, double* const* out) {
  int rc;
  if ((rc = fft_xy(c, n, io, field, fs, a)) || (rc = tri(c, n, a, ne))) return rc;
  return ifft_xy(c, n, a, out);
}

// halos and wall ghosts of nfields fields; kinds: kstep's kind of each, four bits
constexpr unsigned KIND_UVW = 0x100, KIND_P = 0x2, KIND_STEP = 0x22100;
int bound(fld_ctx* c, const Fields& fs, int nfields, unsigned kinds) {
  const FGrid& g = c->g;
  const long long n = ((long long)g.itot * g.jtot +
                       (2LL * (g.jtot + 2) + 2LL * g.itot) * (g.ktot + 2)) * nfields;
  k_bound<<<nblocks(n, 256), 256, 0, c->stream>>>(g, fs, nfields, kinds);
  HIPF(c, hipGetLastError());
  return FLD_OK;
}

}  // namespace

extern "C" {

int fld_create(fld_ctx** out, const ibx_grid* gr, double rep, double dt, int device) {
  if (!out || !gr) return FLD_E_ARG;
  *out = nullptr;
  if (!pow2(gr->itot) || !pow2(gr->jtot) || gr->itot < 4 || gr->jtot < 4 || gr->ktot < 2)
    return FLD_E_ARG;
  // one line of each transform must fit in LDS
  if ((size_t)(gr->itot / 2 + 1) * sizeof(double2) > LDS_MAX ||
      (size_t)(gr->jtot / 2 + 1) * sizeof(double2) > LDS_MAX)
    return FLD_E_ARG;
  if (!(rep > 0 && dt > 0 && gr->dxi > 0 && gr->dyi > 0 && gr->dzi > 0)) return FLD_E_ARG;
  fld_ctx* c = new fld_ctx();
  c->grid = *gr;
  c->rep = rep, c->dt = dt, c->device = device;
  FGrid& g = c->g;
  g.itot = gr->itot, g.jtot = gr->jtot, g.ktot = gr->ktot;
  g.sy = gr->itot + 2;
  g.sz = (long long)(gr->itot + 2) * (gr->jtot + 2);
  g.dxi = gr->dxi, g.dyi = gr->dyi, g.dzi = gr->dzi;
  c->ncomp = (long long)g.itot * g.jtot * g.ktot;
  c->logmx = ilog2(g.itot / 2), c->logmy = ilog2(g.jtot / 2);
  c->xlines = std::min(g.jtot, std::max(1, 2048 / g.itot));
  // columns per workgroup of the LDS y transforms (jtot of 4, or above 1024); 8 both ways was best
  // when they took every length (512 rows: forward 543 us against 604 with 4 and 744 with 2;
  // inverse 602 us against 674 with 16)
  auto lines = [&](int want) {
    int nl = std::min(g.itot, want);
    while (nl > 1 && (size_t)nl * (g.jtot / 2 + 1) * sizeof(double2) > LDS_MAX / 2) nl >>= 1;
    return nl;
  };
  c->ylines_f = lines(Y_LINES_FWD), c->ylines_i = lines(Y_LINES_INV);
  // lines plus the LDS copy of the twiddles
  c->lds_yf = ((size_t)c->ylines_f * (g.jtot / 2 + 1) + g.jtot / 2) * sizeof(double2);
  c->lds_yi = ((size_t)c->ylines_i * (g.jtot / 2 + 1) + g.jtot / 2) * sizeof(double2);
  auto bail = [&](int code, const char* what) {
    fld_destroy(c);
    (void)what;
    return code;
  };
  if (hipSetDevice(device) != hipSuccess) return bail(FLD_E_HIP, "device");
  (void)hipDeviceGetAttribute(&c->cus, hipDeviceAttributeMultiprocessorCount, device);
  if (hipStreamCreateWithFlags(&c->own, hipStreamNonBlocking) != hipSuccess)
    return bail(FLD_E_HIP, "stream");
  c->stream = c->own;
  for (auto& w : c->work)
    if (hipMalloc(&w, (size_t)c->ncomp * sizeof(double)) != hipSuccess) return bail(FLD_E_HIP, "work");
  // dynamic LDS above the default limit for the y transform and the elimination
  if (hipFuncSetAttribute((const void*)k_rfft_fwd<false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)LDS_MAX) != hipSuccess ||
      hipFuncSetAttribute((const void*)k_rfft_inv<false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)LDS_MAX) != hipSuccess ||
      hipFuncSetAttribute((const void*)k_rfft_fwd<true>, hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)LDS_MAX) != hipSuccess ||
      hipFuncSetAttribute((const void*)k_rfft_fwd<true, true>,
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_MAX) != hipSuccess ||
      hipFuncSetAttribute((const void*)k_rfft_inv<true>, hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)LDS_MAX) != hipSuccess)
    return bail(FLD_E_HIP, "lds");
  // twiddles, eigenvalues, coefficients and the pivot tables of e = 1, 2, 3
  const std::vector<double2> twx = twiddles(g.itot, g.itot / 2), twy = twiddles(g.jtot, g.jtot / 2);
  const std::vector<double2> twxm = twiddles(g.itot / 2, g.itot / 2), twyn = twiddles(g.jtot, g.jtot);
  const std::vector<double> xrt = eigen(g.itot, g.dxi), yrt = eigen(g.jtot, g.dyi);
  double *dx = nullptr, *dy = nullptr, *dabc = nullptr;
  bool ok = hipMalloc(&c->tw_x, twx.size() * sizeof(double2)) == hipSuccess &&
            hipMalloc(&c->tw_y, twy.size() * sizeof(double2)) == hipSuccess &&
            hipMalloc(&c->tw_xm, twxm.size() * sizeof(double2)) == hipSuccess &&
            hipMalloc(&c->tw_yn, twyn.size() * sizeof(double2)) == hipSuccess &&
            hipMalloc(&dx, xrt.size() * sizeof(double)) == hipSuccess &&
            hipMalloc(&dy, yrt.size() * sizeof(double)) == hipSuccess &&
            hipMalloc(&dabc, 3 * (size_t)g.ktot * sizeof(double)) == hipSuccess &&
            hipMalloc(&c->part, 2 * 1024 * sizeof(double)) == hipSuccess;
  ok = ok && hipMemcpy(c->tw_x, twx.data(), twx.size() * sizeof(double2), hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(c->tw_y, twy.data(), twy.size() * sizeof(double2), hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(c->tw_xm, twxm.data(), twxm.size() * sizeof(double2), hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(c->tw_yn, twyn.data(), twyn.size() * sizeof(double2), hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(dx, xrt.data(), xrt.size() * sizeof(double), hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(dy, yrt.data(), yrt.size() * sizeof(double), hipMemcpyHostToDevice) == hipSuccess;
  const int nkx = g.itot / 2 + 1, nky = g.jtot / 2 + 1;
  for (int ne = 1; ok && ne <= 3; ++ne) {
    std::vector<double> a, b, cc;
    tridiag(c, ne, a, b, cc);
    std::vector<double> abc(a);
    abc.insert(abc.end(), b.begin(), b.end());
    abc.insert(abc.end(), cc.begin(), cc.end());
    std::vector<double> ac(a);
    ac.insert(ac.end(), cc.begin(), cc.end());
    ok = hipMalloc(&c->coef[ne], 2 * (size_t)g.ktot * sizeof(double)) == hipSuccess &&
         hipMemcpy(c->coef[ne], ac.data(), ac.size() * sizeof(double), hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(dabc, abc.data(), abc.size() * sizeof(double), hipMemcpyHostToDevice) == hipSuccess &&
         hipMalloc(&c->ztab[ne], (size_t)nkx * nky * g.ktot * sizeof(double)) == hipSuccess;
    if (ok) {
      k_ztab<<<nblocks((long long)nkx * nky, 256), 256, 0, c->own>>>(
          nkx, nky, g.ktot, ne, dx, dy, dabc, dabc + g.ktot, dabc + 2 * g.ktot, c->ztab[ne]);
      ok = hipGetLastError() == hipSuccess && hipStreamSynchronize(c->own) == hipSuccess;
    }
  }
  if (dx) (void)hipFree(dx);
  if (dy) (void)hipFree(dy);
  if (dabc) (void)hipFree(dabc);
  if (!ok) return bail(FLD_E_HIP, "tables");
  *out = c;
  return FLD_OK;
}

void fld_destroy(fld_ctx* c) {
  if (!c) return;
  (void)hipSetDevice(c->device);
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  for (auto& w : c->work)
    if (w) (void)hipFree(w);
  for (int ne = 1; ne <= 3; ++ne) {
    if (c->ztab[ne]) (void)hipFree(c->ztab[ne]);
    if (c->coef[ne]) (void)hipFree(c->coef[ne]);
  }
  if (c->tw_x) (void)hipFree(c->tw_x);
  if (c->tw_y) (void)hipFree(c->tw_y);
  if (c->tw_xm) (void)hipFree(c->tw_xm);
  if (c->tw_yn) (void)hipFree(c->tw_yn);
  if (c->part) (void)hipFree(c->part);
  if (c->own) (void)hipStreamDestroy(c->own);
  delete c;
}

const char* fld_last_error(const fld_ctx* c) { return c ? c->err.c_str() : "null context"; }

int fld_set_stream(fld_ctx* c, void* s) {
  if (!c) return FLD_E_ARG;
  c->stream = s ? (hipStream_t)s : c->own;
  return FLD_OK;
}

int fld_sync(fld_ctx* c) {
  if (!c) return FLD_E_ARG;
  HIPF(c, hipSetDevice(c->device));
  HIPF(c, hipStreamSynchronize(c->stream));
  return FLD_OK;
}

int fld_solver1d_dev(fld_ctx* c, double* p, int ne) {
  if (!c) return FLD_E_ARG;
  if (!p) return fail(c, FLD_E_ARG, "null field");
  if (ne < 1 || ne > 3) return fail(c, FLD_E_ARG, "ne must be 1, 2 or 3");
  HIPF(c, hipSetDevice(c->device));
  return solve(c, 1, &p, true, nullptr, c->work, &ne, &p);
}

int fld_fftuvw_dev(fld_ctx* c, double* unew, double* vnew, double* wnew, const double* uo,
                   const double* vo, const double* wo, const double* uoo, const double* voo,
                   const double* woo, const double* pnew, const double* fx, const double* fy,
                   const double* fz) {
  if (!c) return FLD_E_ARG;
  if (!(unew && vnew && wnew && uo && vo && wo && uoo && voo && woo && pnew && fx && fy && fz))
    return fail(c, FLD_E_ARG, "null field");
  HIPF(c, hipSetDevice(c->device));
  // planes per workgroup: 32 (two extra planes read per 32) while that gives two workgroups a
  // compute unit (asking for four changes nothing: 441 against 439 us for a step at
  // 256 x 128 x 128), fewer on smaller grids, where the march along k
  // is a serial chain of plane loads (64^3 cells: 66 us with 32 planes, 32 workgroups)
  const unsigned ti = (unsigned)((c->grid.itot + MR_TI - 1) / MR_TI);
  const unsigned tj = (unsigned)((c->grid.jtot + MR_TJ - 1) / MR_TJ);
  int kb = 32;
  while (kb > 2 && (long long)ti * tj * ((c->grid.ktot + kb - 1) / kb) < 2LL * c->cus) kb >>= 1;
  const dim3 mgrid(ti, tj, (unsigned)((c->grid.ktot + kb - 1) / kb));
  k_mom_rhs_march<<<mgrid, MR_T, 0, c->stream>>>(c->g, kb, c->rep, c->dt, uo, vo, wo, uoo, voo,
                                                 woo, pnew, fx, fy, fz, c->work[0], c->work[1],
                                                 c->work[2]);
  HIPF(c, hipGetLastError());
  const int ne[3] = {2, 2, 3};
  double* const out[3] = {unew, vnew, wnew};
  return solve(c, 3, c->work, false, nullptr, c->work, ne, out);
}

int fld_bounduvw_dev(fld_ctx* c, double* u, double* v, double* w) {
  if (!c) return FLD_E_ARG;
  if (!(u && v && w)) return fail(c, FLD_E_ARG, "null field");
  HIPF(c, hipSetDevice(c->device));
  return bound(c, Fields{{u, v, w, nullptr}}, 3, KIND_UVW);
}

int fld_boundp_dev(fld_ctx* c, double* p) {
  if (!c) return FLD_E_ARG;
  if (!p) return fail(c, FLD_E_ARG, "null field");
  HIPF(c, hipSetDevice(c->device));
  return bound(c, Fields{{p, nullptr, nullptr, nullptr}}, 1, KIND_P);
}

int fld_fillps_dev(fld_ctx* c, const double* u, const double* v, const double* w, double* p) {
  if (!c) return FLD_E_ARG;
  if (!(u && v && w && p)) return fail(c, FLD_E_ARG, "null field");
  HIPF(c, hipSetDevice(c->device));
  k_fillps<<<nblocks(c->ncomp, 256), 256, 0, c->stream>>>(c->g, c->dt, u, v, w, c->work[0]);
  k_to_field<<<nblocks(c->ncomp, 256), 256, 0, c->stream>>>(c->g, c->work[0], p);
  HIPF(c, hipGetLastError());
  return FLD_OK;
}

int fld_correc_dev(fld_ctx* c, double* u, double* v, double* w, const double* p) {
  if (!c) return FLD_E_ARG;
  if (!(u && v && w && p)) return fail(c, FLD_E_ARG, "null field");
  HIPF(c, hipSetDevice(c->device));
  k_correc<<<nblocks(c->ncomp, 256), 256, 0, c->stream>>>(c->g, c->dt, u, v, w, p);
  HIPF(c, hipGetLastError());
  return FLD_OK;
}

int fld_step_dev(fld_ctx* c, double* unew, double* vnew, double* wnew, double* pnew, double* p,
                 const double* uo, const double* vo, const double* wo, const double* uoo,
                 const double* voo, const double* woo, const double* fx, const double* fy,
                 const double* fz) {
  if (!c) return FLD_E_ARG;
  if (!(pnew && p)) return fail(c, FLD_E_ARG, "null field");
  int rc = fld_fftuvw_dev(c, unew, vnew, wnew, uo, vo, wo, uoo, voo, woo, pnew, fx, fy, fz);
  if (rc) return rc;
  const int ne = 1;
  // the reference sets the halos of the velocities before fillps and those of p before correc:
  // the two passes read the interior values behind them instead, and one launch sets all at the
  // end (64^3 cells: 87.4 -> 82.3 us a step)
  const FGrid& g = c->g;
  const double dti = 1.0 / c->dt;
  const FillSrc fs{unew, vnew, wnew,   dti * g.dxi, dti * g.dyi, dti * g.dzi,
                   g.sy, g.sz, g.itot, g.jtot,      g.ktot};
  if ((rc = solve(c, 1, c->work, false, &fs, c->work, &ne, &p))) return rc;
  // correc and pnew += p fused (the reference's bounduvw between them reads neither p nor
  // pnew), then bounduvw, boundp(pnew) and boundp(p)
  k_correc_addp<<<nblocks(c->ncomp / 2, 256), 256, 0, c->stream>>>(
      c->g, c->logmx, c->logmy + 1, c->dt, unew, vnew, wnew, p, pnew);
  HIPF(c, hipGetLastError());
  return bound(c, Fields{{unew, vnew, wnew, pnew, p}}, 5, KIND_STEP);
}

int fld_indicator_div_dev(fld_ctx* c, const double* gx, const double* gy, const double* gz,
                          double* indi) {
  if (!c) return FLD_E_ARG;
  if (!(gx && gy && gz && indi)) return fail(c, FLD_E_ARG, "null field");
  HIPF(c, hipSetDevice(c->device));
  k_ind_div<<<nblocks(c->ncomp, 256), 256, 0, c->stream>>>(c->g, gx, gy, gz, nullptr, indi);
  HIPF(c, hipGetLastError());
  return FLD_OK;
}

static int ind_finish(fld_ctx* c, double* indi, double* indic, double* visc, double* forcey,
                      double* forcez, double lambda, double visc0, double sin_t, double cos_t,
                      double tcoef) {
  int rc;
  if ((rc = bound(c, Fields{{indi, nullptr, nullptr, nullptr}}, 1, KIND_P))) return rc;  // boundind(indi)
  k_ind_shift<<<nblocks(c->ncomp, 256), 256, 0, c->stream>>>(c->g, indi, indic);
  HIPF(c, hipGetLastError());
  if ((rc = bound(c, Fields{{indic, nullptr, nullptr, nullptr}}, 1, KIND_P))) return rc;  // boundind(indic)
  k_ind_finish<<<nblocks(c->ncomp, 256), 256, 0, c->stream>>>(c->g, indic, visc, forcey, forcez,
                                                              lambda, visc0, sin_t, -cos_t,
                                                              tcoef);
  HIPF(c, hipGetLastError());
  return bound(c, Fields{{visc, nullptr, nullptr, nullptr}}, 1, KIND_P);  // boundp(visc)
}

static bool ind_args_ok(double lambda, double visc0, double sin_t, double cos_t, double tcoef) {
  return std::isfinite(lambda) && std::isfinite(visc0) && std::isfinite(sin_t) &&
         std::isfinite(cos_t) && std::isfinite(tcoef);
}

int fld_indicator_finish_dev(fld_ctx* c, double* indi, double* indic, double* visc,
                             double* forcey, double* forcez, double lambda, double visc0,
                             double sin_t, double cos_t, double tcoef) {
  if (!c) return FLD_E_ARG;
  if (!(indi && indic && visc && forcey && forcez)) return fail(c, FLD_E_ARG, "null field");
  if (!ind_args_ok(lambda, visc0, sin_t, cos_t, tcoef))
    return fail(c, FLD_E_ARG, "non-finite indicator constant");
  HIPF(c, hipSetDevice(c->device));
  return ind_finish(c, indi, indic, visc, forcey, forcez, lambda, visc0, sin_t, cos_t, tcoef);
}

int fld_indicator_dev(fld_ctx* c, const double* gx, const double* gy, const double* gz,
                      double* indi, double* indic, double* visc, double* forcey, double* forcez,
                      double lambda, double visc0, double sin_t, double cos_t, double tcoef) {
  if (!c) return FLD_E_ARG;
  if (!(gx && gy && gz && indi && indic && visc && forcey && forcez))
    return fail(c, FLD_E_ARG, "null field");
  if (!ind_args_ok(lambda, visc0, sin_t, cos_t, tcoef))
    return fail(c, FLD_E_ARG, "non-finite indicator constant");
  HIPF(c, hipSetDevice(c->device));
  // divergence straight into the solver's compact array, solve (initsolver(0) and
  // solver1d(indi, 0) are the pressure solve, ne = 1), solution into the interior of indi
  k_ind_div<<<nblocks(c->ncomp, 256), 256, 0, c->stream>>>(c->g, gx, gy, gz, c->work[0], nullptr);
  HIPF(c, hipGetLastError());
  const int ne = 1;
  int rc = solve(c, 1, c->work, false, nullptr, c->work, &ne, &indi);
  if (rc) return rc;
  return ind_finish(c, indi, indic, visc, forcey, forcez, lambda, visc0, sin_t, cos_t, tcoef);
}

int fld_chkdiv_dev(fld_ctx* c, const double* u, const double* v, const double* w,
                   double* divtot, double* divmax) {
  if (!c) return FLD_E_ARG;
  if (!(u && v && w && divtot && divmax)) return fail(c, FLD_E_ARG, "null pointer");
  HIPF(c, hipSetDevice(c->device));
  const unsigned nb = std::min<unsigned>(1024, nblocks(c->ncomp, 256));
  k_div<<<nb, 256, 0, c->stream>>>(c->g, u, v, w, c->part);
  HIPF(c, hipGetLastError());
  std::vector<double> h(2 * (size_t)nb);
  HIPF(c, hipMemcpyAsync(h.data(), c->part, h.size() * sizeof(double), hipMemcpyDeviceToHost,
                         c->stream));
  HIPF(c, hipStreamSynchronize(c->stream));
  double s = 0.0, m = 0.0;
  for (unsigned b = 0; b < nb; ++b) s += h[2 * b], m = std::max(m, h[2 * b + 1]);
  *divtot = s, *divmax = m;
  return FLD_OK;
}

}  // extern "C"
