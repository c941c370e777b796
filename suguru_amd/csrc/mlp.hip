// mlp.hip -- the learned membrane-traction surrogate: an MLP trained and run with hand-written
// BF16 MFMA kernels (v_mfma_f32_16x16x32_bf16) accumulating in FP32, on gfx950.
//
// Layers: din -> width (SiLU) -> ... (nhidden hidden layers) -> dout (linear).  Every GEMM
// dimension is padded to a multiple of 64 with zeros, so the tiles need no bounds checks;
// padded rows/columns of the weights stay zero (their gradients are zero and Adam keeps them
// at zero), so the padded network equals the unpadded one.
//
// GEMM: C[M x N] = A[M x K] B[K x N], BM x BN tile per 256-thread workgroup, each wavefront a
// quarter of it as 16 x 16 MFMA 16x16x32 blocks; A and B are staged through LDS with k
// contiguous, so that each lane's MFMA operand (8 consecutive k) is one 16-byte read.
// A is either row-major [M x K] or its transpose ([K x M], for dW = dZ^T H); B is either
// [K x N] row-major (dX = dZ W) or [N x K] row-major (forward: B = W^T).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "../../include/memb.h"

namespace mlp {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int TK = 64, THREADS = 256;
constexpr int LDK = TK + 8;  // LDS row stride in bf16 (pads rows apart by 16 bytes)
constexpr int GROUP = 8;     // layers per grouped launch

__device__ inline __bf16 to_bf16(float f) { return (__bf16)f; }  // round to nearest even
__device__ inline float silu(float z) { return z / (1.0f + __expf(-z)); }
__device__ inline float dsilu(float z) {
  const float s = 1.0f / (1.0f + __expf(-z));
  return s * (1.0f + z * (1.0f - s));
}

enum Epi {
  EPI_BIAS_SILU = 0,  // Z = acc + b (fp32 out0, unless null), H = bf16(silu(Z)) (out1)
  EPI_OUT = 1,        // y = omean + oscale (acc + b), the real rows and columns only (out0)
  EPI_DSILU = 2,      // dZ = bf16(acc * silu'(Z)), Z read from aux (fp32) (out1)
  EPI_F32 = 3,        // plain fp32 store (weight gradients) (out0)
  EPI_LOSS = 4,       // Y = acc + b, dY = bf16(2 (Y - t') w / (batch dout)) (out1), loss partials
};

// One product and what its epilogue reads and writes (ldc: row pitch of out0 / out1 / aux).
struct GemmArgs {
  int K, lda, ldb, ldc;
  const __bf16* A;
  const __bf16* B;
  const float* bias;
  const float* aux;      // EPI_DSILU: Z; EPI_LOSS: the targets t [batch][dout]
  float* out0;
  __bf16* out1;
  const float* omean;    // EPI_OUT, EPI_LOSS
  const float* oscale;
  const float* wt;       // EPI_LOSS: per-output weights or null
  float* part;           // EPI_LOSS: one partial sum per workgroup, or null
  int batch, dout;       // EPI_OUT, EPI_LOSS: the unpadded extents
};

// One TK-deep slice of an operand tile of R rows (rows = m of A, n of B) from memory into
// registers, then into LDS as [row][k].  T = false: memory is [row][k], 16 bytes (8 k) per load.
// T = true: memory is [k][row]; a thread loads a pair of rows for 8 consecutive k (8 loads of
// 4 bytes) and transposes the 8 x 2 block in registers, so that LDS gets 16-byte stores
// either way.
template <int R, bool T>
struct Slice {
  static constexpr int NV = T ? (R * TK / 16 + THREADS - 1) / THREADS
                              : (R * TK / 8 + THREADS - 1) / THREADS;
  static constexpr int ITEMS = T ? R * TK / 16 : R * TK / 8;
  bf16x8 v[NV][T ? 2 : 1];
  __device__ __forceinline__ void load(const __bf16* __restrict__ g, int ld, int r0, int k0) {
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      const int t = threadIdx.x + u * THREADS;
      if (ITEMS % THREADS && t >= ITEMS) continue;
      if (!T) {
        const int r = t / (TK / 8), kc = (t % (TK / 8)) * 8;
        v[u][0] = *reinterpret_cast<const bf16x8*>(&g[(size_t)(r0 + r) * ld + k0 + kc]);
      } else {
        const int kc = (t / (R / 2)) * 8, r = (t % (R / 2)) * 2;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const bf16x2 w = *reinterpret_cast<const bf16x2*>(&g[(size_t)(k0 + kc + e) * ld + r0 + r]);
          v[u][0][e] = w[0];
          v[u][T ? 1 : 0][e] = w[1];
        }
      }
    }
  }
  __device__ __forceinline__ void store(__bf16* s) const {
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      const int t = threadIdx.x + u * THREADS;
      if (ITEMS % THREADS && t >= ITEMS) continue;
      if (!T) {
        const int r = t / (TK / 8), kc = (t % (TK / 8)) * 8;
        *reinterpret_cast<bf16x8*>(&s[r * LDK + kc]) = v[u][0];
      } else {
        const int kc = (t / (R / 2)) * 8, r = (t % (R / 2)) * 2;
        *reinterpret_cast<bf16x8*>(&s[r * LDK + kc]) = v[u][0];
        *reinterpret_cast<bf16x8*>(&s[(r + 1) * LDK + kc]) = v[u][T ? 1 : 0];
      }
    }
  }
};

// A: if !TA, A[m][k] = Ag[m * lda + k]; if TA, A[m][k] = Ag[k * lda + m]
// B: if TB,  B[k][n] = Bg[n * ldb + k]; if !TB, B[k][n] = Bg[k * ldb + n]
// Tile (m0, n0) of BM x BN: four wavefronts in a 2 x 2 arrangement, each owning (BM/2) x (BN/2)
// as 16 x 16 MFMA blocks.  The matrices are small enough to sit in the caches, so a tile is bound
// by the round trips of its K-slices, not by the matrix cores: TK = 64, two LDS buffers with one
// barrier per slice, and PF slices of loads in flight in registers ahead of the one in LDS.  A
// 512-deep layer of 64 rows takes 4.6 us like this (6.1 us with one slice ahead, 8.4-11 us with
// 32-deep slices and none ahead, as k_gemm had before).  The transposed operands hold 4-byte
// pairs, so one slice ahead is all that pays (weight gradients 12.9 us, 18.5 with three).  Each
// output element sums its 32-deep K-steps in the same order whatever the tile, so every tile
// gives the same bits.
template <int BM, int BN, bool TA, bool TB, int EPI>
__device__ __forceinline__ void gemm_tile(const GemmArgs& q, int m0, int n0) {
  constexpr int FM = BM / 32, FN = BN / 32;  // MFMA blocks per wavefront
  __shared__ __attribute__((aligned(16))) __bf16 smem[2 * (BM + BN) * LDK];
  // buffer c: A rows, then B rows
  auto As = [&](int c) { return smem + c * (BM + BN) * LDK; };
  auto Bs = [&](int c) { return smem + c * (BM + BN) * LDK + BM * LDK; };
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int wm = (wv >> 1) * (BM / 2), wn = (wv & 1) * (BN / 2);
  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // PF slices in flight in registers ahead of the one in LDS
  constexpr int PF = TA || !TB ? (BM >= 64 ? 1 : 2) : (BM >= 64 ? 3 : 4);
  Slice<BM, TA> sa[PF];
  Slice<BN, !TB> sb[PF];
#pragma unroll
  for (int p = 0; p < PF; ++p)
    if (p * TK < q.K) {
      sa[p].load(q.A, q.lda, m0, p * TK);
      sb[p].load(q.B, q.ldb, n0, p * TK);
    }
  int cur = 0;
  for (int kb = 0; kb < q.K; kb += PF * TK) {
#pragma unroll
    for (int p = 0; p < PF; ++p) {
      const int k0 = kb + p * TK;
      if (k0 >= q.K) break;
      // buffer `cur` was last read two slices ago, before the previous slice's barrier
      sa[p].store(As(cur));
      sb[p].store(Bs(cur));
      __syncthreads();
      if (k0 + PF * TK < q.K) {
        sa[p].load(q.A, q.lda, m0, k0 + PF * TK);
        sb[p].load(q.B, q.ldb, n0, k0 + PF * TK);
      }
#pragma unroll
      for (int kk = 0; kk < TK; kk += 32) {
        // operands: lane holds row (lane % 16), k = 8 (lane / 16) .. +7
        bf16x8 a[FM], b[FN];
#pragma unroll
        for (int i = 0; i < FM; ++i)
          a[i] = *reinterpret_cast<const bf16x8*>(
              &As(cur)[(wm + i * 16 + (lane & 15)) * LDK + kk + 8 * (lane >> 4)]);
#pragma unroll
        for (int j = 0; j < FN; ++j)
          b[j] = *reinterpret_cast<const bf16x8*>(
              &Bs(cur)[(wn + j * 16 + (lane & 15)) * LDK + kk + 8 * (lane >> 4)]);
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
      }
      cur ^= 1;
    }
  }
  // result: lane holds rows 4 (lane / 16) + r, column lane % 16 of each 16 x 16 block
  float loss = 0.0f;
  // the output goes through LDS: the rows of y have no alignment, so whole row segments of the
  // tile are written by consecutive lanes instead of 16 columns of four rows per store
  float* tile = reinterpret_cast<float*>(smem);
  static_assert(BM * (BN + 1) * sizeof(float) <= sizeof(smem), "output tile in the operand buffers");
  if (EPI == EPI_OUT) __syncthreads();
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int col = n0 + wn + j * 16 + (lane & 15);
      const float bias = EPI == EPI_BIAS_SILU || EPI == EPI_OUT || EPI == EPI_LOSS ? q.bias[col] : 0.0f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + wm + i * 16 + 4 * (lane >> 4) + r;
        const size_t o = (size_t)row * q.ldc + col;
        const float v = acc[i][j][r];
        if (EPI == EPI_BIAS_SILU) {
          const float zz = v + bias;
          if (q.out0) q.out0[o] = zz;
          q.out1[o] = to_bf16(silu(zz));
        } else if (EPI == EPI_OUT) {
          tile[(row - m0) * (BN + 1) + col - n0] = v + bias;
        } else if (EPI == EPI_DSILU) {
          q.out1[o] = to_bf16(v * dsilu(q.aux[o]));
        } else if (EPI == EPI_LOSS) {
          // loss = mean((Y - t')^2 w) over batch x dout with t' = (t - omean) / oscale
          float g = 0.0f;
          if (row < q.batch && col < q.dout) {
            const float w = q.wt ? q.wt[col] : 1.0f;
            const float d =
                (v + bias) - (q.aux[(size_t)row * q.dout + col] - q.omean[col]) / q.oscale[col];
            const float inv = 1.0f / ((float)q.batch * (float)q.dout);
            loss += d * d * w * inv;
            g = 2.0f * d * w * inv;
          }
          q.out1[o] = to_bf16(g);
        } else {
          q.out0[o] = v;
        }
      }
    }
  if (EPI == EPI_OUT) {
    __syncthreads();
    const int c = tid % BN, col = n0 + c;
    if (col < q.dout) {
      const float om = q.omean[col], os = q.oscale[col];
#pragma unroll 4
      for (int r = tid / BN; r < BM && m0 + r < q.batch; r += THREADS / BN)
        q.out0[(size_t)(m0 + r) * q.dout + col] = om + os * tile[r * (BN + 1) + c];
    }
  }
  if (EPI == EPI_LOSS) {
    __shared__ float red[THREADS / 64];
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) loss += __shfl_down(loss, s);
    if (lane == 0) red[wv] = loss;
    __syncthreads();
    if (tid == 0 && q.part) q.part[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
  }
}

template <int BM, int BN, bool TA, bool TB, int EPI>
__global__ void __launch_bounds__(THREADS) k_gemm(GemmArgs q, int tiles_n) {
  // workgroup b runs on XCD b % 8 (round-robin dispatch): with a multiple of 8 tiles, each XCD
  // takes a contiguous eighth of them, tiles_n tiles per row block, so that its L2 reads an
  // eighth of A instead of all of it
  const unsigned nb = gridDim.x, b = blockIdx.x;
  const int t = (nb & 7u) ? (int)b : (int)((b & 7u) * (nb >> 3) + (b >> 3));
  gemm_tile<BM, BN, TA, TB, EPI>(q, t / tiles_n * BM, t % tiles_n * BN);
}

// x[batch][din] fp32 -> X[Mp][Dp] bf16 with (x - mean) * scale, zero padding.  One column of
// IN_ROWS rows per thread, neighbouring threads on neighbouring columns (the rows of x have no
// 16-byte alignment), every load of a thread in flight together.
constexpr int IN_ROWS = 8;
__global__ void __launch_bounds__(THREADS)
    k_input(int batch, int din, int Mp, int Dp, const float* __restrict__ x,
            const float* __restrict__ mean, const float* __restrict__ scale,
            __bf16* __restrict__ X) {
  const int c = blockIdx.x * THREADS + threadIdx.x, r0 = blockIdx.y * IN_ROWS;
  if (c >= Dp) return;
  float v[IN_ROWS];
#pragma unroll
  for (int e = 0; e < IN_ROWS; ++e)
    v[e] = r0 + e < batch && c < din ? x[(size_t)(r0 + e) * din + c] : 0.0f;
  const float mu = c < din ? mean[c] : 0.0f, sc = c < din ? scale[c] : 0.0f;
#pragma unroll
  for (int e = 0; e < IN_ROWS; ++e)
    X[(size_t)(r0 + e) * Dp + c] = to_bf16(r0 + e < batch && c < din ? (v[e] - mu) * sc : 0.0f);
}

// The weight and bias gradients of up to GROUP layers in one launch: they are independent of
// each other once the backward chain has left every dZ_i.
//   db_i[c] = sum over rows of dZ_i[r][c]: a workgroup takes CS_COLS columns; its threads bring
// CS_ROWS rows at a time into LDS with every load in flight, and CS_COLS of them add a column
// each in row order.  (One thread per column reading its rows from memory one after the other
// took 53 us per layer at 512 rows.)
//   dW_i = dZ_i^T H_{i-1} ([out x in], K = batch rows): one BM x BN tile per workgroup.
// cfirst[i] / first[i]: layer i's first column / tile workgroup; the column sums come first.
constexpr int CS_COLS = 32, CS_ROWS = 256;
struct GroupArgs {
  int n, first[GROUP + 1], tiles_n[GROUP], cfirst[GROUP + 1];
  GemmArgs g[GROUP];
  float* db[GROUP];
};

__device__ __forceinline__ void colsum(const __bf16* __restrict__ dZ, int rows, int ld, int c0,
                                       float* __restrict__ db) {
  __shared__ __attribute__((aligned(16))) __bf16 s[CS_ROWS][CS_COLS];
  const int tid = threadIdx.x;
  float sum = 0.0f;
  for (int r0 = 0; r0 < rows; r0 += CS_ROWS) {
    const int nr = min(CS_ROWS, rows - r0);  // rows are padded to a multiple of 128
#pragma unroll
    for (int u = 0; u < CS_ROWS * CS_COLS / 8 / THREADS; ++u) {
      const int t = tid + u * THREADS, r = t / (CS_COLS / 8), c = (t % (CS_COLS / 8)) * 8;
      if (r < nr)
        *reinterpret_cast<bf16x8*>(&s[r][c]) =
            *reinterpret_cast<const bf16x8*>(&dZ[(size_t)(r0 + r) * ld + c0 + c]);
    }
    __syncthreads();
    if (tid < CS_COLS) {
#pragma unroll 32
      for (int r = 0; r < nr; ++r) sum += (float)s[r][tid];
    }
    __syncthreads();
  }
  if (tid < CS_COLS) db[c0 + tid] = sum;
}

template <int BM, int BN>
__global__ void __launch_bounds__(THREADS) k_grads(GroupArgs a) {
  const int ncol = a.cfirst[a.n];
  int i = 0;
  if ((int)blockIdx.x < ncol) {
    while ((int)blockIdx.x >= a.cfirst[i + 1]) ++i;
    colsum(a.g[i].A, a.g[i].K, a.g[i].lda, (blockIdx.x - a.cfirst[i]) * CS_COLS, a.db[i]);
    return;
  }
  const int b = blockIdx.x - ncol;
  while (b >= a.first[i + 1]) ++i;
  const int t = b - a.first[i];
  const GemmArgs q = a.g[i];
  gemm_tile<BM, BN, true, false, EPI_F32>(q, t / a.tiles_n[i] * BM, t % a.tiles_n[i] * BN);
}

// Adam on fp32 masters; refreshes the bf16 copy.  Padded entries have zero gradient and stay 0.
// Up to 2 GROUP arrays (weights and biases) in one launch, four values per thread; first[i]:
// array i's first workgroup.
struct AdamArgs {
  int n, first[2 * GROUP + 1];
  long long len[2 * GROUP];
  float lr, b1, b2, eps, c1, c2;
  float* w[2 * GROUP];
  const float* g[2 * GROUP];
  float* m[2 * GROUP];
  float* v[2 * GROUP];
  __bf16* wb[2 * GROUP];
};

__global__ void __launch_bounds__(THREADS) k_adam(AdamArgs a) {
  int i = 0;
  while (i + 1 < a.n && (int)blockIdx.x >= a.first[i + 1]) ++i;
  const long long q = 4 * ((long long)(blockIdx.x - a.first[i]) * THREADS + threadIdx.x);
  if (q >= a.len[i]) return;  // lengths are multiples of 64
  f32x4 w = *reinterpret_cast<f32x4*>(a.w[i] + q), m = *reinterpret_cast<f32x4*>(a.m[i] + q),
        v = *reinterpret_cast<f32x4*>(a.v[i] + q);
  const f32x4 g = *reinterpret_cast<const f32x4*>(a.g[i] + q);
  bf16x4 wb;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float gg = g[e];
    // the fused products are written out: which of the two the compiler fuses is left to it
    // otherwise, and Adam's division by |g| carries that rounding on through the steps
    const float mm = __builtin_fmaf(1.0f - a.b1, gg, a.b1 * m[e]);
    const float vv = __builtin_fmaf(gg, (1.0f - a.b2) * gg, a.b2 * v[e]);
    m[e] = mm, v[e] = vv;
    const float ww = w[e] - a.lr * (mm / a.c1) / (sqrtf(vv / a.c2) + a.eps);
    w[e] = ww;
    wb[e] = to_bf16(ww);
  }
  *reinterpret_cast<f32x4*>(a.m[i] + q) = m;
  *reinterpret_cast<f32x4*>(a.v[i] + q) = v;
  *reinterpret_cast<f32x4*>(a.w[i] + q) = w;
  if (a.wb[i]) *reinterpret_cast<bf16x4*>(a.wb[i] + q) = wb;
}

__global__ void k_to_bf16(long long n, const float* __restrict__ a, __bf16* __restrict__ b) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < n) b[q] = to_bf16(a[q]);
}

inline int pad64(int v) { return (v + 63) / 64 * 64; }
inline int pad128(int v) { return (v + 127) / 128 * 128; }  // batch rows
inline unsigned nblk(long long n, int t = 256) { return (unsigned)((n + t - 1) / t); }

}  // namespace mlp

using namespace mlp;

struct memb_mlp {
  int device = 0;
  int cus = 256;  // compute units of the device (GEMM tile choice)
  hipStream_t own = nullptr, stream = nullptr;
  std::string err;
  int din = 0, width = 0, nh = 0, dout = 0, maxb = 0;
  int Dp = 0, Wp = 0, Op = 0, Mp = 0, nl = 0;
  std::vector<int> in_p, out_p, in_r, out_r;  // padded and real layer shapes
  // per layer: fp32 master W [out_p][in_p], b [out_p]; bf16 W copy; Adam moments; grads
  std::vector<float*> W, b, mW, vW, mb, vb, gW, gb;
  std::vector<__bf16*> Wb;
  // activations
  __bf16* X = nullptr;             // [Mp][Dp]
  std::vector<float*> Z;           // hidden pre-activations [Mp][Wp]
  std::vector<__bf16*> H;          // hidden activations [Mp][Wp]
  std::vector<__bf16*> dZ;         // per layer, gradient of the pre-activation [Mp][out_p]
  // loss partials, one per workgroup of the last layer, in pinned host memory, and its device
  // address: allocated by the first call that asks for the loss (an allocation and its release take
  // 0.5 ms, which a network that only infers need not pay; such a call waits, so it is not captured)
  float* hpart = nullptr;
  float* part = nullptr;
  size_t npart = 0;
  float *mean = nullptr, *scale = nullptr;    // input normalisation [Dp]
  float *omean = nullptr, *oscale = nullptr;  // output de-normalisation [Op]
  long long step = 0;
  std::vector<void*> allocs;
};

namespace {
int mfail(memb_mlp* m, int code, const std::string& s) {
  if (m) m->err = s;
  return code;
}
#define XCHK(m, call)                                                                    \
  do {                                                                                   \
    hipError_t e_ = (call);                                                              \
    if (e_ != hipSuccess)                                                                \
      return mfail((m), MEMB_E_HIP, std::string(#call) + ": " + hipGetErrorString(e_));  \
  } while (0)

template <typename T>
int dalloc(memb_mlp* m, T** p, size_t n) {
  void* d = nullptr;
  XCHK(m, hipMalloc(&d, n * sizeof(T)));
  XCHK(m, hipMemset(d, 0, n * sizeof(T)));
  m->allocs.push_back(d);
  *p = (T*)d;
  return MEMB_OK;
}

// 64 x 64 tiles where there is at least one per compute unit, 32 x 32 below (training batches,
// small inference batches): a forward pass of 2048 rows takes 48 us with 64 x 64 hidden layers (256
// tiles) and 54 us with 32 x 32; 4096 rows 67 and 78 us; a training step of 512 rows, whose
// hidden layers have 64 tiles of 64 x 64, 142 us with 32 x 32.  128 x 128 tiles were slower
// everywhere (8192 rows: 150 against 121 us).
template <bool TA, bool TB, int EPI>
int gemm(memb_mlp* m, int M, int N, const GemmArgs& q) {
  if (M % 64 || N % 64 || q.K % TK) return mfail(m, MEMB_E_ARG, "gemm shape not padded");
  const int b = (long long)(M / 64) * (N / 64) >= m->cus ? 64 : 32;
  const unsigned grid = (unsigned)(M / b) * (N / b);
  if (b == 64)
    k_gemm<64, 64, TA, TB, EPI><<<grid, THREADS, 0, m->stream>>>(q, N / b);
  else
    k_gemm<32, 32, TA, TB, EPI><<<grid, THREADS, 0, m->stream>>>(q, N / b);
  m->npart = grid;
  XCHK(m, hipGetLastError());
  return MEMB_OK;
}

// The hidden layers; keep: store the pre-activations Z for a backward pass.
int forward_hidden(memb_mlp* m, int batch, const float* x, bool keep) {
  const int Mp = pad128(batch);
  k_input<<<dim3(nblk(m->Dp, THREADS), Mp / IN_ROWS), THREADS, 0, m->stream>>>(
      batch, m->din, Mp, m->Dp, x, m->mean, m->scale, m->X);
  for (int i = 0; i < m->nl - 1; ++i) {
    GemmArgs q{};
    q.K = q.lda = q.ldb = m->in_p[i], q.ldc = m->out_p[i];
    q.A = i == 0 ? m->X : m->H[i - 1], q.B = m->Wb[i], q.bias = m->b[i];
    q.out0 = keep ? m->Z[i] : nullptr, q.out1 = m->H[i];
    int rc = gemm<false, true, EPI_BIAS_SILU>(m, Mp, m->out_p[i], q);
    if (rc) return rc;
  }
  return MEMB_OK;
}

// The arguments of the last layer's product, whose epilogue forms the output or the loss
GemmArgs last_layer(const memb_mlp* m, int batch) {
  const int i = m->nl - 1;
  GemmArgs q{};
  q.K = q.lda = q.ldb = m->in_p[i], q.ldc = m->out_p[i];
  q.A = i == 0 ? m->X : m->H[i - 1], q.B = m->Wb[i], q.bias = m->b[i];
  q.omean = m->omean, q.oscale = m->oscale, q.batch = batch, q.dout = m->dout;
  return q;
}

// Forward, loss and every gradient, enqueued; with want_loss the nloss loss partials are in hpart
// once the stream has come this far.
int backward(memb_mlp* m, int batch, const float* x, const float* t, const float* wt,
             bool want_loss, size_t& nloss) {
  if (want_loss && !m->hpart) {
    const size_t parts = (size_t)(m->Mp / 32) * (m->Op / 32);  // the smallest tile's workgroups
    XCHK(m, hipHostMalloc((void**)&m->hpart, parts * sizeof(float), hipHostMallocMapped));
    XCHK(m, hipHostGetDevicePointer((void**)&m->part, m->hpart, 0));
  }
  int rc = forward_hidden(m, batch, x, true);
  if (rc) return rc;
  const int Mp = pad128(batch), last = m->nl - 1;
  {
    GemmArgs q = last_layer(m, batch);
    q.aux = t, q.wt = wt, q.out1 = m->dZ[last], q.part = want_loss ? m->part : nullptr;
    if ((rc = gemm<false, true, EPI_LOSS>(m, Mp, m->out_p[last], q))) return rc;
    nloss = m->npart;
  }
  for (int i = last; i > 0; --i) {
    // dZ_{i-1} = (dZ_i W_i) * silu'(Z_{i-1}): [Mp x in], K = out
    GemmArgs q{};
    q.K = q.lda = m->out_p[i], q.ldb = q.ldc = m->in_p[i];
    q.A = m->dZ[i], q.B = m->Wb[i], q.aux = m->Z[i - 1], q.out1 = m->dZ[i - 1];
    if ((rc = gemm<false, false, EPI_DSILU>(m, Mp, m->in_p[i], q))) return rc;
  }
  for (int i0 = 0; i0 < m->nl; i0 += GROUP) {
    const int n = std::min(GROUP, m->nl - i0);
    GroupArgs g{};
    g.n = n;
    for (int k = 0; k < n; ++k) {
      const int i = i0 + k;
      g.tiles_n[k] = m->in_p[i] / 64;
      g.first[k + 1] = g.first[k] + m->out_p[i] / 64 * g.tiles_n[k];
      GemmArgs& q = g.g[k];
      q.K = Mp, q.lda = m->out_p[i], q.ldb = q.ldc = m->in_p[i];
      q.A = m->dZ[i], q.B = i == 0 ? m->X : m->H[i - 1], q.out0 = m->gW[i];
      g.cfirst[k + 1] = g.cfirst[k] + m->out_p[i] / CS_COLS;
      g.db[k] = m->gb[i];
    }
    k_grads<64, 64><<<g.cfirst[n] + g.first[n], THREADS, 0, m->stream>>>(g);
  }
  XCHK(m, hipGetLastError());
  return MEMB_OK;
}

// Waits for the step and adds its loss partials in workgroup order.
int read_loss(memb_mlp* m, size_t nloss, float* loss) {
  XCHK(m, hipStreamSynchronize(m->stream));
  float s = 0.0f;
  for (size_t i = 0; i < nloss; ++i) s += m->hpart[i];
  *loss = s;
  return MEMB_OK;
}
}  // namespace

extern "C" {

int memb_mlp_create(memb_mlp** out, int din, int width, int nhidden, int dout, int max_batch,
                    int device) {
  if (!out || din <= 0 || width <= 0 || nhidden <= 0 || dout <= 0 || max_batch <= 0)
    return MEMB_E_ARG;
  memb_mlp* m = new memb_mlp();
  *out = m;
  m->device = device;
  XCHK(m, hipSetDevice(device));
  XCHK(m, hipStreamCreate(&m->own));
  m->stream = m->own;
  (void)hipDeviceGetAttribute(&m->cus, hipDeviceAttributeMultiprocessorCount, device);
  m->din = din, m->width = width, m->nh = nhidden, m->dout = dout, m->maxb = max_batch;
  m->Dp = pad64(din), m->Wp = pad64(width), m->Op = pad64(dout), m->Mp = pad128(max_batch);
  m->nl = nhidden + 1;
  for (int i = 0; i < m->nl; ++i) {
    m->in_p.push_back(i == 0 ? m->Dp : m->Wp);
    m->in_r.push_back(i == 0 ? din : width);
    m->out_p.push_back(i == m->nl - 1 ? m->Op : m->Wp);
    m->out_r.push_back(i == m->nl - 1 ? dout : width);
  }
  int rc;
  for (int i = 0; i < m->nl; ++i) {
    const size_t nw = (size_t)m->out_p[i] * m->in_p[i], nb = m->out_p[i];
    float *w, *bb, *a1, *a2, *a3, *a4, *g1, *g2;
    __bf16* wb;
    if ((rc = dalloc(m, &w, nw)) || (rc = dalloc(m, &bb, nb)) || (rc = dalloc(m, &a1, nw)) ||
        (rc = dalloc(m, &a2, nw)) || (rc = dalloc(m, &a3, nb)) || (rc = dalloc(m, &a4, nb)) ||
        (rc = dalloc(m, &g1, nw)) || (rc = dalloc(m, &g2, nb)) || (rc = dalloc(m, &wb, nw)))
      return rc;
    m->W.push_back(w), m->b.push_back(bb), m->mW.push_back(a1), m->vW.push_back(a2);
    m->mb.push_back(a3), m->vb.push_back(a4), m->gW.push_back(g1), m->gb.push_back(g2);
    m->Wb.push_back(wb);
  }
  for (int i = 0; i < nhidden; ++i) {
    float* z;
    __bf16* h;
    if ((rc = dalloc(m, &z, (size_t)m->Mp * m->Wp)) || (rc = dalloc(m, &h, (size_t)m->Mp * m->Wp)))
      return rc;
    m->Z.push_back(z), m->H.push_back(h);
  }
  for (int i = 0; i < m->nl; ++i) {
    __bf16* d;
    if ((rc = dalloc(m, &d, (size_t)m->Mp * m->out_p[i]))) return rc;
    m->dZ.push_back(d);
  }
  if ((rc = dalloc(m, &m->X, (size_t)m->Mp * m->Dp)) ||
      (rc = dalloc(m, &m->mean, (size_t)m->Dp)) || (rc = dalloc(m, &m->scale, (size_t)m->Dp)) ||
      (rc = dalloc(m, &m->omean, (size_t)m->Op)) || (rc = dalloc(m, &m->oscale, (size_t)m->Op)))
    return rc;
  std::vector<float> one(std::max(m->Dp, m->Op), 1.0f);
  XCHK(m, hipMemcpy(m->scale, one.data(), m->Dp * sizeof(float), hipMemcpyHostToDevice));
  XCHK(m, hipMemcpy(m->oscale, one.data(), m->Op * sizeof(float), hipMemcpyHostToDevice));
  return MEMB_OK;
}

void memb_mlp_destroy(memb_mlp* m) {
  if (!m) return;
  (void)hipSetDevice(m->device);
  if (m->stream) (void)hipStreamSynchronize(m->stream);
  for (void* p : m->allocs) (void)hipFree(p);
  if (m->hpart) (void)hipHostFree(m->hpart);
  if (m->own) (void)hipStreamDestroy(m->own);
  delete m;
}

const char* memb_mlp_last_error(const memb_mlp* m) { return m ? m->err.c_str() : "null mlp"; }

int memb_mlp_set_stream(memb_mlp* m, void* s) {
  if (!m) return MEMB_E_ARG;
  m->stream = s ? (hipStream_t)s : m->own;
  return MEMB_OK;
}

int memb_mlp_num_layers(const memb_mlp* m) { return m ? m->nl : 0; }

int memb_mlp_layer_shape(const memb_mlp* m, int i, int* out_dim, int* in_dim) {
  if (!m || i < 0 || i >= m->nl) return MEMB_E_ARG;
  if (out_dim) *out_dim = m->out_r[i];
  if (in_dim) *in_dim = m->in_r[i];
  return MEMB_OK;
}

int memb_mlp_set_norm(memb_mlp* m, const float* mean, const float* scale, const float* out_mean,
                      const float* out_scale) {
  if (!m || !mean || !scale || !out_mean || !out_scale) return MEMB_E_ARG;
  for (int c = 0; c < m->dout; ++c)
    if (!(out_scale[c] > 0.0f)) return mfail(m, MEMB_E_ARG, "out_scale must be positive");
  XCHK(m, hipSetDevice(m->device));
  XCHK(m, hipMemcpy(m->mean, mean, m->din * sizeof(float), hipMemcpyHostToDevice));
  XCHK(m, hipMemcpy(m->scale, scale, m->din * sizeof(float), hipMemcpyHostToDevice));
  XCHK(m, hipMemcpy(m->omean, out_mean, m->dout * sizeof(float), hipMemcpyHostToDevice));
  XCHK(m, hipMemcpy(m->oscale, out_scale, m->dout * sizeof(float), hipMemcpyHostToDevice));
  return MEMB_OK;
}

int memb_mlp_set_layer(memb_mlp* m, int i, const float* W, const float* b) {
  if (!m || i < 0 || i >= m->nl || !W || !b) return MEMB_E_ARG;
  XCHK(m, hipSetDevice(m->device));
  const int op = m->out_p[i], ip = m->in_p[i], orr = m->out_r[i], ir = m->in_r[i];
  std::vector<float> w((size_t)op * ip, 0.0f), bb(op, 0.0f);
  for (int r = 0; r < orr; ++r) {
    for (int c = 0; c < ir; ++c) w[(size_t)r * ip + c] = W[(size_t)r * ir + c];
    bb[r] = b[r];
  }
  XCHK(m, hipMemcpy(m->W[i], w.data(), w.size() * sizeof(float), hipMemcpyHostToDevice));
  XCHK(m, hipMemcpy(m->b[i], bb.data(), bb.size() * sizeof(float), hipMemcpyHostToDevice));
  k_to_bf16<<<nblk((long long)w.size()), 256, 0, m->stream>>>((long long)w.size(), m->W[i], m->Wb[i]);
  XCHK(m, hipGetLastError());
  XCHK(m, hipStreamSynchronize(m->stream));
  return MEMB_OK;
}

static int get_padded(memb_mlp* m, int i, const float* dW, const float* db, float* W, float* b) {
  const int op = m->out_p[i], ip = m->in_p[i], orr = m->out_r[i], ir = m->in_r[i];
  std::vector<float> w((size_t)op * ip), bb(op);
  XCHK(m, hipSetDevice(m->device));
  XCHK(m, hipStreamSynchronize(m->stream));
  XCHK(m, hipMemcpy(w.data(), dW, w.size() * sizeof(float), hipMemcpyDeviceToHost));
  XCHK(m, hipMemcpy(bb.data(), db, bb.size() * sizeof(float), hipMemcpyDeviceToHost));
  for (int r = 0; r < orr; ++r) {
    for (int c = 0; c < ir; ++c) W[(size_t)r * ir + c] = w[(size_t)r * ip + c];
    b[r] = bb[r];
  }
  return MEMB_OK;
}

int memb_mlp_get_layer(memb_mlp* m, int i, float* W, float* b) {
  if (!m || i < 0 || i >= m->nl || !W || !b) return MEMB_E_ARG;
  return get_padded(m, i, m->W[i], m->b[i], W, b);
}

int memb_mlp_get_grad(memb_mlp* m, int i, float* dW, float* db) {
  if (!m || i < 0 || i >= m->nl || !dW || !db) return MEMB_E_ARG;
  return get_padded(m, i, m->gW[i], m->gb[i], dW, db);
}

int memb_mlp_init(memb_mlp* m, uint64_t seed) {
  if (!m) return MEMB_E_ARG;
  std::mt19937_64 rng(seed);
  for (int i = 0; i < m->nl; ++i) {
    const int orr = m->out_r[i], ir = m->in_r[i];
    const float a = std::sqrt(6.0f / (float)(ir + orr));
    std::uniform_real_distribution<float> U(-a, a);
    std::vector<float> w((size_t)orr * ir), bb(orr, 0.0f);
    for (auto& v : w) v = U(rng);
    int rc = memb_mlp_set_layer(m, i, w.data(), bb.data());
    if (rc) return rc;
  }
  m->step = 0;
  return MEMB_OK;
}

int memb_mlp_forward(memb_mlp* m, int batch, const float* x, float* y) {
  if (!m || batch <= 0 || batch > m->maxb || !x || !y) return MEMB_E_ARG;
  XCHK(m, hipSetDevice(m->device));
  int rc = forward_hidden(m, batch, x, false);
  if (rc) return rc;
  GemmArgs q = last_layer(m, batch);
  q.out0 = y;
  return gemm<false, true, EPI_OUT>(m, pad128(batch), m->out_p[m->nl - 1], q);
}

int memb_mlp_grad_only(memb_mlp* m, int batch, const float* x, const float* t, const float* wt,
                       float* loss) {
  if (!m || batch <= 0 || batch > m->maxb || !x || !t) return MEMB_E_ARG;
  XCHK(m, hipSetDevice(m->device));
  size_t nloss = 0;
  int rc = backward(m, batch, x, t, wt, loss != nullptr, nloss);
  if (rc || !loss) return rc;
  return read_loss(m, nloss, loss);
}

int memb_mlp_train_step(memb_mlp* m, int batch, const float* x, const float* t, const float* wt,
                        float lr, float* loss) {
  if (!m || batch <= 0 || batch > m->maxb || !x || !t) return MEMB_E_ARG;
  XCHK(m, hipSetDevice(m->device));
  size_t nloss = 0;
  int rc = backward(m, batch, x, t, wt, loss != nullptr, nloss);
  if (rc) return rc;
  ++m->step;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float c1 = 1.0f - std::pow(b1, (float)m->step), c2 = 1.0f - std::pow(b2, (float)m->step);
  for (int i0 = 0; i0 < m->nl; i0 += GROUP) {
    AdamArgs a{};
    a.lr = lr, a.b1 = b1, a.b2 = b2, a.eps = eps, a.c1 = c1, a.c2 = c2;
    auto add = [&](long long n, float* w, float* g, float* mo, float* vo, __bf16* wb) {
      const int k = a.n++;
      a.len[k] = n, a.w[k] = w, a.g[k] = g, a.m[k] = mo, a.v[k] = vo, a.wb[k] = wb;
      a.first[k + 1] = a.first[k] + (int)nblk(n / 4, THREADS);
    };
    for (int i = i0; i < std::min(i0 + GROUP, m->nl); ++i) {
      add((long long)m->out_p[i] * m->in_p[i], m->W[i], m->gW[i], m->mW[i], m->vW[i], m->Wb[i]);
      add(m->out_p[i], m->b[i], m->gb[i], m->mb[i], m->vb[i], nullptr);
    }
    k_adam<<<a.first[a.n], THREADS, 0, m->stream>>>(a);
  }
  XCHK(m, hipGetLastError());
  return loss ? read_loss(m, nloss, loss) : MEMB_OK;
}

}  // extern "C"
