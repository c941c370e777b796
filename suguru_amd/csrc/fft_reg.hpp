// fft_reg.hpp -- register transforms of libfluid: a complex line of N = 8 .. 1024 values held by
// N/8 threads, eight values each, exchanged through LDS between passes of radix 8.
#pragma once
#include <hip/hip_runtime.h>

#pragma clang fp contract(off)

namespace fft {

__device__ __forceinline__ double2 mul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 add(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 sub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }

// a times -i (forward) or +i (inverse)
template <bool INV>
__device__ __forceinline__ double2 turn(double2 a) {
  return INV ? make_double2(-a.y, a.x) : make_double2(a.y, -a.x);
}

template <bool INV>
__device__ __forceinline__ void dft4(double2& a0, double2& a1, double2& a2, double2& a3) {
  const double2 s = add(a0, a2), d = sub(a0, a2), t = add(a1, a3), u = turn<INV>(sub(a1, a3));
  a0 = add(s, t), a1 = add(d, u), a2 = sub(s, t), a3 = sub(d, u);
}

template <bool INV>
__device__ __forceinline__ void dft8(double2 (&a)[8]) {
  constexpr double h = 0.70710678118654752440;  // sqrt(1/2)
  double2 e0 = a[0], e1 = a[2], e2 = a[4], e3 = a[6], o0 = a[1], o1 = a[3], o2 = a[5], o3 = a[7];
  dft4<INV>(e0, e1, e2, e3);
  dft4<INV>(o0, o1, o2, o3);
  // o1 exp(-+ i pi/4), o2 (-+ i), o3 exp(-+ 3 i pi/4)
  const double2 t1 = turn<INV>(o1), t3 = turn<INV>(o3);
  o1 = make_double2(h * (o1.x + t1.x), h * (o1.y + t1.y));
  o2 = turn<INV>(o2);
  o3 = make_double2(h * (t3.x - o3.x), h * (t3.y - o3.y));
  a[0] = add(e0, o0), a[1] = add(e1, o1), a[2] = add(e2, o2), a[3] = add(e3, o3);
  a[4] = sub(e0, o0), a[5] = sub(e1, o1), a[6] = sub(e2, o2), a[7] = sub(e3, o3);
}

// LDS index of element i of a line: one pad per eight, so that the stride-8 stores of the first
// exchange spread over the banks.
__host__ __device__ constexpr int pad(int i) { return i + (i >> 3); }

// Between the threads of a line.  Within one wavefront (WG false) LDS operations complete in
// order and only the compiler has to keep them so; otherwise a workgroup barrier.
template <bool WG>
__device__ __forceinline__ void line_sync() {
  if constexpr (WG) {
    __syncthreads();
  } else {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

// Line of N = 2^LOGN values: thread t < TPL holds x[t + TPL u] in a[u] before and X[t + TPL u]
// after the transform (Stockham passes of radix 8 and a last one of 2, 4 or 8: self-sorting).
// WG: the threads of a line lie in several wavefronts; every thread of the workgroup calls run.
template <int LOGN, bool WG>
struct Line {
  static constexpr int N = 1 << LOGN, TPL = N / 8;
  static_assert(LOGN >= 3 && LOGN <= 10 && (WG || TPL <= 64), "length");
  static constexpr int radix(int L) { return N / L >= 8 ? 8 : N / L; }
  static constexpr int count(int L) {  // twiddles of the passes from product L on
    return L >= N ? 0 : (L > 1 ? 8 - 8 / radix(L) : 0) + count(L * radix(L));
  }
  static constexpr int NW = count(1) > 0 ? count(1) : 1;

  double2 w[NW];  // this thread's twiddles, pass by pass

  // table: exp(-2 pi i q / N), q < N
  template <int L = 1, int AT = 0>
  __device__ __forceinline__ void load(const double2* __restrict__ table, int t) {
    if constexpr (L < N) {
      constexpr int R = radix(L);
      if constexpr (L > 1) {
#pragma unroll
        for (int s = 0; s < 8 / R; ++s) {
          const int k = (t + TPL * s) & (L - 1);
#pragma unroll
          for (int r = 1; r < R; ++r) w[AT + s * (R - 1) + r - 1] = table[k * r * (N / (L * R))];
        }
      }
      load<L * R, AT + (L > 1 ? 8 - 8 / R : 0)>(table, t);
    }
  }

  // buf: the line's pad(N) values of LDS, free after the line's threads have synchronized once more
  template <bool INV, int L = 1, int AT = 0>
  __device__ __forceinline__ void run(double2 (&a)[8], double2* buf, int t) const {
    constexpr int R = radix(L);
    if constexpr (L > 1) {
#pragma unroll
      for (int s = 0; s < 8 / R; ++s)
#pragma unroll
        for (int r = 1; r < R; ++r) {
          double2 v = w[AT + s * (R - 1) + r - 1];
          if (INV) v.y = -v.y;
          a[s + r * (8 / R)] = mul(v, a[s + r * (8 / R)]);
        }
    }
    if constexpr (R == 8) {
      dft8<INV>(a);
    } else if constexpr (R == 4) {
      dft4<INV>(a[0], a[2], a[4], a[6]);
      dft4<INV>(a[1], a[3], a[5], a[7]);
    } else {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const double2 x = a[s], y = a[s + 4];
        a[s] = add(x, y), a[s + 4] = sub(x, y);
      }
    }
    if constexpr (L * R < N) {
      line_sync<WG>();
#pragma unroll
      for (int s = 0; s < 8 / R; ++s) {
        const int q = t + TPL * s, k = q & (L - 1);
#pragma unroll
        for (int r = 0; r < R; ++r) buf[pad((q - k) * R + k + r * L)] = a[s + r * (8 / R)];
      }
      line_sync<WG>();
#pragma unroll
      for (int u = 0; u < 8; ++u) a[u] = buf[pad(t + TPL * u)];
      run<INV, L * R, AT + (L > 1 ? 8 - 8 / R : 0)>(a, buf, t);
    }
  }
};

}  // namespace fft
