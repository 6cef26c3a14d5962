// Point-set MLP of the learned block proposal on gfx950 matrix cores.
//
//   k_gemm       C = act(alpha * A B^T + bias) (+ C), A and B bf16 with any
//                strides, FP32 accumulation on v_mfma_f32_16x16x16_bf16,
//                32 x 32 per wave (2 x 2 MFMA tiles), K in steps of 16:
//                64 x 64 output tile per 256-lane workgroup, or, for long
//                sums on few tiles, 32 x 32 with the sum cut over 16 waves.
//   k_point_pool the shared per-point MLP 3 -> 64 -> 128 -> 256 (ReLU) fused
//                with the max-pool over each scene's points: 64 points at a
//                time, layer 1 on the VALU in FP32, layers 2 and 3 on
//                MFMA with bf16 activations staged in LDS, then a per-channel
//                (max, first argmax) reduction merged across workgroups with
//                one 64-bit atomic max per channel.
//   k_adam       Adam step on FP32 master weights plus their bf16 copy.
//
// MFMA 16x16x16 bf16 lane layout (wave64): A holds row (lane % 16), k =
// 4 (lane / 16) + i; B holds column (lane % 16), same k; the four results
// are rows 4 (lane / 16) + j of column (lane % 16).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "../../include/set_proposal.h"

namespace sp {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint16_t f2bf(float f) {
  // round to nearest even; NaN stays NaN
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

__device__ __forceinline__ f32x4 mfma(bf16x4 a, bf16x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

struct GemmArgs {
  int M, N, K;
  const uint16_t* A;
  long lda_m, lda_k;
  const uint16_t* B;
  long ldb_n, ldb_k;
  const float* bias;
  float alpha;
  int relu, accumulate;
  float* C;
  long ldc;
  uint16_t* Cb;  // optional bf16 copy of the result (same ldc)
};

// How a wave reads an operand's fragment, 32 rows by 16 k as two 16 x 16 MFMA
// tiles, four k of a row a lane: element by element at any strides; in one
// 8-byte load where k is contiguous; or, where the rows are contiguous, as the
// pairs of rows 2 r, 2 r + 1 at four k, tile 0 taking the even rows and tile 1
// the odd ones.
enum class Read { kAny, kQuads, kPairs };
__device__ inline int row_of(Read how, int tile, int r) { return how == Read::kPairs ? 2 * r + tile : 16 * tile + r; }

template <Read how>
__device__ inline void read_fragment(bf16x4 (&f)[2], const uint16_t* X, long ld_row, long ld_k, int row0, int rows,
                                     int k0, int K) {
  const int lane = threadIdx.x & 63, r = lane & 15, k = k0 + (lane >> 4) * 4;
  if (how == Read::kPairs) {
    const int row = row0 + 2 * r;
    uint32_t p[4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
      p[t] = row < rows && k + t < K ? *reinterpret_cast<const uint32_t*>(X + row + (long)(k + t) * ld_k) : 0u;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      f[0][t] = (short)(p[t] & 0xFFFFu);
      f[1][t] = (short)(p[t] >> 16);
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = row0 + 16 * i + r;
    if (how == Read::kQuads) {
      f[i] = row < rows && k < K ? *reinterpret_cast<const bf16x4*>(X + row * ld_row + k) : bf16x4{0, 0, 0, 0};
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t)
        f[i][t] = row < rows && k + t < K ? (short)X[row * ld_row + (k + t) * ld_k] : (short)0;
    }
  }
}

// kSlices == 1: 64 x 64 of C a workgroup, 32 x 32 a wave, each element's
// products summed over k in steps of 16 in order.  kSlices > 1: 32 x 32 a
// workgroup, every wave a slice of k of its own, the slices' sums added in
// order in LDS.  The latter is for few tiles and long sums, where the chain of
// steps down one wave bounds the product: the weight gradients of 8,192 rows
// (128 x 64 and 256 x 128 by 8,192) were two and eight
// workgroups, 237 us each, and take 25 and 29; read element by element, where 4
// k are now one load, the 8,192 x 128 by 256 input gradient took 21 us, now 10.
constexpr int kDeepSlices = 16;
template <int kSlices, Read kA, Read kB>
__global__ __launch_bounds__(kSlices == 1 ? 256 : kSlices * 64) void k_gemm(GemmArgs g) {
  __shared__ float s_sum[kSlices == 1 ? 1 : kSlices][kSlices == 1 ? 1 : 16 * 64 + 16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m0 = kSlices == 1 ? blockIdx.y * 64 + (wave >> 1) * 32 : blockIdx.y * 32;
  const int n0 = kSlices == 1 ? blockIdx.x * 64 + (wave & 1) * 32 : blockIdx.x * 32;
  const int r = lane & 15, kq = (lane >> 4) * 4;
  const int steps = (g.K + 15) / 16, per = (steps + kSlices - 1) / kSlices;
  const int first = kSlices == 1 ? 0 : wave * per, last = min(steps, first + per);
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
  for (int s = first; s < last; ++s) {
    bf16x4 a[2], b[2];
    read_fragment<kA>(a, g.A, g.lda_m, g.lda_k, m0, g.M, 16 * s, g.K);
    read_fragment<kB>(b, g.B, g.ldb_n, g.ldb_k, n0, g.N, 16 * s, g.K);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = mfma(a[i], b[j], acc[i][j]);
  }
  auto store = [&](int i, int j, int t, float sum) {
    const int m = m0 + row_of(kA, i, kq + t);
    const int n = n0 + row_of(kB, j, r);
    if (m >= g.M || n >= g.N) return;
    float v = g.alpha * sum;
    if (g.bias) v += g.bias[n];
    if (g.relu) v = v > 0.0f ? v : 0.0f;
    float* c = g.C + (long)m * g.ldc + n;
    if (g.accumulate) v += *c;
    *c = v;
    if (g.Cb) g.Cb[(long)m * g.ldc + n] = f2bf(v);
  };
  if (kSlices == 1) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int t = 0; t < 4; ++t) store(i, j, t, acc[i][j][t]);
    return;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int t = 0; t < 4; ++t) s_sum[wave][(8 * i + 4 * j + t) * 64 + lane] = acc[i][j][t];
  __syncthreads();
  // wave w: result w of every lane, (i, j, t) = (w / 8, w / 4 % 2, w % 4)
  static_assert(kSlices == 1 || kSlices == 16, "a result a wave");
  float sum = 0.0f;
  for (int w = 0; w < kSlices; ++w) sum += s_sum[w][wave * 64 + lane];
  store(wave >> 3, wave >> 2 & 1, wave & 3, sum);
}

// ---------------------------------------------------------------------------
constexpr int kPts = 64;              // points per workgroup
constexpr int kH1 = 64, kH2 = 128, kH3 = 256;
constexpr int kPad = 4;               // bf16 padding per LDS row (bank spread)
constexpr int kPoolBlocks = 512;      // workgroups of the pool together

struct PoolArgs {
  int B, N;
  const float* pts;      // B x N x 3
  const float* W1;       // 64 x 3
  const float* b1;       // 64
  const uint16_t* W2;    // 128 x 64 bf16
  const float* b2;
  const uint16_t* W3;    // 256 x 128 bf16
  const float* b3;
  unsigned long long* pooled;  // B x 256: (value bits << 32) | (0xffffffff - point)
};

// A workgroup walks every gridDim.x-th group of 64 points of its scene with its
// waves' weights in registers (wave w: channels [32 w, 32 w + 32) of layer 2 and
// [64 w, 64 w + 64) of layer 3), and keeps its channels' maxima there too.
// Loading the 80 KB of weights for every 64 points bound it: 308 us for 32
// scenes of 20,000 points, now 131 (53 GFLOP, 400 TFLOP/s), two workgroups a CU
// and a share of the points each (one, three or four a CU: 214, 159, 138).
__global__ __launch_bounds__(256, 2) void k_point_pool(PoolArgs a) {
  __shared__ __align__(16) uint16_t s_h1[kPts][kH1 + kPad];
  __shared__ __align__(16) uint16_t s_h2[kPts][kH2 + kPad];
  __shared__ float4 s_x[kPts];
  const int b = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, kq = (lane >> 4) * 4;
  auto quad = [](const uint16_t* p) { return *reinterpret_cast<const bf16x4*>(p); };
  const bool aligned = ((reinterpret_cast<uintptr_t>(a.W2) | reinterpret_cast<uintptr_t>(a.W3)) & 7u) == 0u;
  auto weights = [&](const uint16_t* p) {
    if (aligned) return quad(p);
    return bf16x4{(short)p[0], (short)p[1], (short)p[2], (short)p[3]};
  };
  bf16x4 w2[2][kH1 / 16], w3[4][kH2 / 16];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int k = 0; k < kH1 / 16; ++k) w2[j][k] = weights(a.W2 + (long)(wave * 32 + j * 16 + r) * kH1 + 16 * k + kq);
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int k = 0; k < kH2 / 16; ++k) w3[j][k] = weights(a.W3 + (long)(wave * 64 + j * 16 + r) * kH2 + 16 * k + kq);
  float bias2[2], bias3[4];
#pragma unroll
  for (int j = 0; j < 2; ++j) bias2[j] = a.b2[wave * 32 + j * 16 + r];
#pragma unroll
  for (int j = 0; j < 4; ++j) bias3[j] = a.b3[wave * 64 + j * 16 + r];
  // layer 1 (FP32): lane = channel, 16 points a wave
  const float w1x = a.W1[3 * lane], w1y = a.W1[3 * lane + 1], w1z = a.W1[3 * lane + 2], bias1 = a.b1[lane];
  auto layer1 = [&](int p0) {  // by wave: its own points' coordinates through LDS
    if (lane < 16) {
      const int p = p0 + wave * 16 + lane;
      const float* x = a.pts + ((long)b * a.N + (p < a.N ? p : 0)) * 3;
      s_x[wave * 16 + lane] = make_float4(x[0], x[1], x[2], 0.0f);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float4 x = s_x[wave * 16 + i];
      const float h = ((w1x * x.x + w1y * x.y) + w1z * x.z) + bias1;
      s_h1[wave * 16 + i][lane] = f2bf(h > 0.0f ? h : 0.0f);  // points past the end: never looked at
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  // (max, first argmax) of each channel over the lane's points, which come in
  // rising order: a later one has to be larger.  ReLU: nothing is below the 0 of
  // the lane's first point.
  float best[4];
  int bp[4];
  const int first = blockIdx.x * kPts + kq, stride = gridDim.x * kPts;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    best[j] = first < a.N ? 0.0f : -1.0f;
    bp[j] = first;
  }
  if ((int)blockIdx.x * kPts < a.N) layer1(blockIdx.x * kPts);
  for (int p0 = blockIdx.x * kPts; p0 < a.N; p0 += stride) {  // uniform
    __syncthreads();
    {  // layer 2
      f32x4 acc[4][2];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int k = 0; k < kH1 / 16; ++k) {
        bf16x4 av[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) av[i] = quad(&s_h1[i * 16 + r][16 * k + kq]);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[i][j] = mfma(av[i], w2[j][k], acc[i][j]);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const float v = acc[i][j][t] + bias2[j];
            s_h2[i * 16 + kq + t][wave * 32 + j * 16 + r] = f2bf(v > 0.0f ? v : 0.0f);
          }
    }
    __syncthreads();
    if (p0 + stride < a.N) layer1(p0 + stride);  // layer 2 is done with s_h1
    // layer 3, two blocks of 16 points at a time
#pragma unroll
    for (int i0 = 0; i0 < 4; i0 += 2) {
      f32x4 acc[2][4];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int k = 0; k < kH2 / 16; ++k) {
        bf16x4 av[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) av[i] = quad(&s_h2[(i0 + i) * 16 + r][16 * k + kq]);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[i][j] = mfma(av[i], w3[j][k], acc[i][j]);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const int p = p0 + (i0 + i) * 16 + kq + t;
            const float v = acc[i][j][t] + bias3[j];
            const bool up = v > best[j] && p < a.N;
            best[j] = up ? v : best[j];
            bp[j] = up ? p : bp[j];
          }
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
#pragma unroll
    for (int off = 16; off < 64; off <<= 1) {
      const float ov = __shfl_xor(best[j], off, 64);
      const int op = __shfl_xor(bp[j], off, 64);
      if (ov > best[j] || (ov == best[j] && op < bp[j])) {
        best[j] = ov;
        bp[j] = op;
      }
    }
    if (lane < 16 && best[j] >= 0.0f) {
      const unsigned long long key = ((unsigned long long)__float_as_uint(best[j]) << 32) |
                                     (unsigned long long)(0xffffffffu - (uint32_t)bp[j]);
      atomicMax(a.pooled + (long)b * kH3 + wave * 64 + j * 16 + r, key);
    }
  }
}

__global__ void k_fill_u64(unsigned long long* p, unsigned long long v, long n) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

__global__ void k_unpack_pool(const unsigned long long* pooled, long n, float* value, int* index) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const unsigned long long k = pooled[i];
  value[i] = __uint_as_float((uint32_t)(k >> 32));
  index[i] = (int)(0xffffffffu - (uint32_t)(k & 0xffffffffull));
}

__global__ void k_to_bf16(const float* x, uint16_t* y, long n) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = f2bf(x[i]);
}

__global__ void k_adam(float* p, uint16_t* pb, const float* g, float* m, float* v, long n, float lr, float b1,
                       float b2, float eps, float c1, float c2) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * (gi * gi);
  m[i] = mi;
  v[i] = vi;
  const float mh = mi / c1, vh = vi / c2;
  const float pi = p[i] - lr * mh / (sqrtf(vh) + eps);
  p[i] = pi;
  if (pb) pb[i] = f2bf(pi);
}

unsigned blocks(long n, int t = 256) { return (unsigned)((n + t - 1) / t); }

}  // namespace sp

using namespace sp;

extern "C" {

int sp_gemm_bf16(int M, int N, int K, const uint16_t* A, long lda_m, long lda_k, const uint16_t* B, long ldb_n,
                 long ldb_k, const float* bias, float alpha, int relu, int accumulate, float* C, long ldc,
                 uint16_t* C_bf16, sp_stream_t stream) {
  if (M < 0 || N < 0 || K < 0 || (M > 0 && N > 0 && (!A || !B || !C))) return 1;
  if (M == 0 || N == 0) return 0;
  GemmArgs g{M, N, K, A, lda_m, lda_k, B, ldb_n, ldb_k, bias, alpha, relu, accumulate, C, ldc, C_bf16};
  // whole 8-byte quads of k, or whole 4-byte pairs of rows, at their alignment
  auto how = [K](const uint16_t* X, long ld_row, long ld_k, int rows) {
    const uintptr_t at = reinterpret_cast<uintptr_t>(X);
    if (ld_k == 1 && K % 4 == 0 && ld_row % 4 == 0 && at % 8 == 0) return Read::kQuads;
    if (ld_row == 1 && rows % 2 == 0 && ld_k % 2 == 0 && at % 4 == 0) return Read::kPairs;
    return Read::kAny;
  };
  const Read ra = how(A, lda_m, lda_k, M), rb = how(B, ldb_n, ldb_k, N);
  // Long sums on few enough tiles, us with the sum cut and whole: 128 x 64 by 512
  // 9 and 16, by 1,024 9 and 30; 512 x 512 by 4,096 17 and 156; 1,024 x 1,024 by
  // 4,096 51 and 159; but 2,048 x 2,048 by 2,048 98 and 85.
  const long tiles = (long)((M + 63) / 64) * ((N + 63) / 64);
  const bool deep = K >= 512 && tiles <= 256;
  const hipStream_t st = (hipStream_t)stream;
  auto launch = [&](auto a, auto b) {
    constexpr Read kA = decltype(a)::value, kB = decltype(b)::value;
    if (deep)
      hipLaunchKernelGGL((k_gemm<kDeepSlices, kA, kB>), dim3((N + 31) / 32, (M + 31) / 32), dim3(kDeepSlices * 64), 0,
                         st, g);
    else
      hipLaunchKernelGGL((k_gemm<1, kA, kB>), dim3((N + 63) / 64, (M + 63) / 64), dim3(256), 0, st, g);
  };
  using Any = std::integral_constant<Read, Read::kAny>;
  using Quads = std::integral_constant<Read, Read::kQuads>;
  using Pairs = std::integral_constant<Read, Read::kPairs>;
  auto with_b = [&](auto a) {
    if (rb == Read::kQuads) launch(a, Quads{});
    else if (rb == Read::kPairs) launch(a, Pairs{});
    else launch(a, Any{});
  };
  if (ra == Read::kQuads) with_b(Quads{});
  else if (ra == Read::kPairs) with_b(Pairs{});
  else with_b(Any{});
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int sp_point_pool(int B, int N, const float* pts, const float* W1, const float* b1, const uint16_t* W2,
                  const float* b2, const uint16_t* W3, const float* b3, float* value, int* index,
                  unsigned long long* scratch, sp_stream_t stream) {
  if (B < 0 || N < 0) return 1;
  if (B == 0) return 0;
  if (!pts || !W1 || !b1 || !W2 || !b2 || !W3 || !b3 || !value || !index || !scratch) return 1;
  hipStream_t st = (hipStream_t)stream;
  const long n = (long)B * kH3;
  hipLaunchKernelGGL(k_fill_u64, dim3(blocks(n)), dim3(256), 0, st, scratch, 0ull, n);
  if (N > 0) {
    PoolArgs a{B, N, pts, W1, b1, W2, b2, W3, b3, scratch};
    // two workgroups a CU between them, at least one a scene
    const int groups = (N + kPts - 1) / kPts, share = (kPoolBlocks + B - 1) / B;
    hipLaunchKernelGGL(k_point_pool, dim3(groups < share ? groups : share, B), dim3(256), 0, st, a);
  }
  hipLaunchKernelGGL(k_unpack_pool, dim3(blocks(n)), dim3(256), 0, st, scratch, n, value, index);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int sp_to_bf16(const float* x, uint16_t* y, long n, sp_stream_t stream) {
  if (n <= 0) return n < 0 ? 1 : 0;
  hipLaunchKernelGGL(k_to_bf16, dim3(blocks(n)), dim3(256), 0, (hipStream_t)stream, x, y, n);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int sp_adam(float* param, uint16_t* param_bf16, const float* grad, float* m, float* v, long n, float lr,
            float beta1, float beta2, float eps, int step, sp_stream_t stream) {
  if (n <= 0 || step < 1) return n < 0 || step < 1 ? 1 : 0;
  const float c1 = 1.0f - powf(beta1, (float)step), c2 = 1.0f - powf(beta2, (float)step);
  hipLaunchKernelGGL(k_adam, dim3(blocks(n)), dim3(256), 0, (hipStream_t)stream, param, param_bf16, grad, m, v, n,
                     lr, beta1, beta2, eps, c1, c2);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

}  // extern "C"
