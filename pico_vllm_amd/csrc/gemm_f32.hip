// True float32 matrix product C = A W^T (+ bias) on the float32 matrix instruction (v_mfma_f32_32x32x2_f32: products and
// sums in float32, no reduced precision).  Every output element is accumulated in an order that depends on K alone, so a
// row's result does not depend on how many other rows the call has, nor on how the work was dealt out.
//
// The sum is a tree over k: 16 products one after the other (eight instructions on one accumulator), 16 such sums (256),
// then the `ranges` of K, each of as many 256s as there are ranges (both about sqrt(K / 256)): four short chains in place
// of one long one.  Error against 64 bits, in units of 2^-24 of the result's rms, measured: 1.93 at K = 1,536, 2.12 at
// 8,960, 2.34 at 27,648 (plain FMA in a tree of radix 16 over four levels: 1.96, 2.28, 2.39; one running sum would give
// 0.2 sqrt(K)).
//
// Bound by the matrix instruction (157 TFLOP/s) from about 64 rows on, by the stream of W below.  A wave owns 32 x 32
// outputs, so that the tree's four levels are 64 registers and four workgroups share a compute unit; its operands come
// from LDS (64 of 128 B a cycle at most), a stage of 32 k behind.  Tiles that read the same rows of W are neighbours on
// one die.  Where the tiles alone leave the chip idle (less than two a compute unit) every range of K is a workgroup
// of its own, its sum goes to a slab, and a second launch adds the slabs in the order in which one workgroup would have.
// 320 rows, microseconds a call with plain FMA in 64 x 64 tiles and with this: 17,920 x 1,536 575 / 234 (75 TFLOP/s);
// 1,536 x 8,960 1,421 / 123; 1,536 x 1,536 183 / 34.  2,048 rows of 17,920 x 1,536: 3,299 / 1,171 (96 TFLOP/s).  One row of
// 151,936 x 1,536: 1,070 / 270 (3.5 TB/s).
#include "common.h"

typedef float f32x16 __attribute__((ext_vector_type(16)));

#define BK 32          // k of a stage
#define ST (BK + 4)    // row stride in LDS: 16-byte reads of neighbouring rows fall on different banks
#define GROUP 256      // k of the tree's second level

// How K is cut: the number of ranges, each of `len` k (the last takes what is left).  The host allocates a slab a range.
__host__ __device__ inline int f32_ranges(int K, int& len) {
  const int groups = (K + GROUP - 1) / GROUP;
  int r = 1;
  while (r * r < groups) r++;
  const int per = (groups + r - 1) / r;
  len = per * GROUP;
  return (groups + per - 1) / per;
}

__device__ __forceinline__ float4 zero_from(float4 v, int k, int K) {
  v.x = k < K ? v.x : 0.f; v.y = k + 1 < K ? v.y : 0.f; v.z = k + 2 < K ? v.z : 0.f; v.w = k + 3 < K ? v.w : 0.f;
  return v;
}

// Four k of a row from k on.  VEC: rows of whole aligned fours, so one load; what lies behind K reads as zero (from an
// address inside the row).  Otherwise four clamped loads.
template <bool VEC>
__device__ __forceinline__ float4 fetch4(const float* row, int k, int K) {
  if (VEC) return *reinterpret_cast<const float4*>(row + (k < K ? k : 0));
  return make_float4(row[min(k, K - 1)], row[min(k + 1, K - 1)], row[min(k + 2, K - 1)], row[min(k + 3, K - 1)]);
}
template <bool VEC>
__device__ __forceinline__ float4 fetch4(const bf16_t* row, int k, int K) {
  if (VEC) {
    const uint2 v = *reinterpret_cast<const uint2*>(row + (k < K ? k : 0));
    return make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16),
                       __uint_as_float(v.y & 0xffff0000u));
  }
  return make_float4(bf16_to_f32(row[min(k, K - 1)]), bf16_to_f32(row[min(k + 1, K - 1)]),
                     bf16_to_f32(row[min(k + 2, K - 1)]), bf16_to_f32(row[min(k + 3, K - 1)]));
}

// A [M, K] row stride lda; W [N, K] row stride ldw; C [M, N] row stride ldc.  TA is the storage type of A (float, or
// bfloat16 bits that are widened on load).  WM x 2 waves of 32 x 32 outputs.  grid (8 ceil(n_tiles / 8) m_tiles, 1) with
// `slabs` null, (.., ranges) with slabs [ranges, M, N].
template <typename TA, int WM, bool VEC>
__global__ __launch_bounds__(128 * WM, 4) void gemm_f32_kernel(const TA* __restrict__ A, const float* __restrict__ W,
                                                               const float* __restrict__ bias, float* __restrict__ C,
                                                               float* __restrict__ slabs, int M, int N, int K, int lda,
                                                               int ldw, int ldc, int m_tiles) {
  constexpr int TM = 32 * WM, TN = 64, THREADS = 128 * WM;
  constexpr int NA = TM * BK / 4 / THREADS, NW = TN * BK / 4 / THREADS;     // pieces of four a thread
  __shared__ __attribute__((aligned(16))) float As[2][TM * ST];
  __shared__ __attribute__((aligned(16))) float Ws[2][TN * ST];
  // dies take workgroups in turn: the tiles of one strip of W stay on one die
  const int die = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int n0 = ((local / m_tiles) * 8 + die) * TN, m0 = local % m_tiles * TM;
  if (n0 >= N) return;
  int len;
  f32_ranges(K, len);
  const int k_first = slabs ? blockIdx.y * len : 0, k_end = slabs ? min(K, k_first + len) : K;

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l = lane & 31, half = lane >> 5;
  const int wm = wave >> 1, wn = wave & 1;
  const TA* a_row[NA];
  const float* w_row[NW];
  int a_at[NA], w_at[NW];
  const int kc = threadIdx.x % (BK / 4) * 4;
#pragma unroll
  for (int i = 0; i < NA; i++) {
    const int r = (threadIdx.x + THREADS * i) / (BK / 4);
    a_row[i] = A + (size_t)min(m0 + r, M - 1) * lda;
    a_at[i] = r * ST + kc;
  }
#pragma unroll
  for (int i = 0; i < NW; i++) {
    const int r = (threadIdx.x + THREADS * i) / (BK / 4);
    w_row[i] = W + (size_t)min(n0 + r, N - 1) * ldw;
    w_at[i] = r * ST + kc;
  }
  float4 av[NA], wv[NW];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < NW; i++) wv[i] = fetch4<VEC>(w_row[i], k0 + kc, K);
#pragma unroll
    for (int i = 0; i < NA; i++) av[i] = fetch4<VEC>(a_row[i], k0 + kc, K);
  };
  auto put = [&](int b, int k0) {
    const bool edge = k0 + BK > K;
#pragma unroll
    for (int i = 0; i < NW; i++) *reinterpret_cast<float4*>(&Ws[b][w_at[i]]) = edge ? zero_from(wv[i], k0 + kc, K) : wv[i];
#pragma unroll
    for (int i = 0; i < NA; i++) *reinterpret_cast<float4*>(&As[b][a_at[i]]) = edge ? zero_from(av[i], k0 + kc, K) : av[i];
  };

  f32x16 l1 = {}, l2 = {}, l3 = {};
  const float* ap = &As[0][(32 * wm + l) * ST + 4 * half];
  const float* wp = &Ws[0][(32 * wn + l) * ST + 4 * half];
  fetch(k_first);
  put(0, k_first);
  int buf = 0;
  for (int k0 = k_first; k0 < k_end; k0 += BK, buf ^= 1) {
    __syncthreads();
    const bool more = k0 + BK < k_end;
    if (more) fetch(k0 + BK);
    const float* a = ap + buf * (TM * ST);
    const float* w = wp + buf * (TN * ST);
#pragma unroll
    for (int g = 0; g < BK; g += 16) {
      // 16 k: this half of the lanes holds 0..3 and 8..11 (or 4..7 and 12..15) of them
      const float4 a0 = *reinterpret_cast<const float4*>(a + g), a1 = *reinterpret_cast<const float4*>(a + g + 8);
      const float4 w0 = *reinterpret_cast<const float4*>(w + g), w1 = *reinterpret_cast<const float4*>(w + g + 8);
      f32x16 l0 = {};
      l0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.x, w0.x, l0, 0, 0, 0);
      l0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.y, w0.y, l0, 0, 0, 0);
      l0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.z, w0.z, l0, 0, 0, 0);
      l0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.w, w0.w, l0, 0, 0, 0);
      l0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.x, w1.x, l0, 0, 0, 0);
      l0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.y, w1.y, l0, 0, 0, 0);
      l0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.z, w1.z, l0, 0, 0, 0);
      l0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.w, w1.w, l0, 0, 0, 0);
      l1 += l0;
    }
    if (more) put(buf ^ 1, k0 + BK);
    const int done = k0 + BK - k_first;
    if (done % GROUP == 0) {
      l2 += l1;
      l1 = {};
    }
    if (!slabs && (done % len == 0 || !more)) {      // the same for all threads
      l3 += l1 + l2;
      l1 = {};
      l2 = {};
    }
  }
  const int n = n0 + 32 * wn + l;
  if (n >= N) return;
  const float b = !slabs && bias ? bias[n] : 0.f;
  if (slabs) l3 = l1 + l2;
  float* out = slabs ? slabs + (size_t)blockIdx.y * M * N : C;
  const int ldo = slabs ? N : ldc;
#pragma unroll
  for (int r = 0; r < 16; r++) {
    const int m = m0 + 32 * wm + 8 * (r >> 2) + 4 * half + (r & 3);
    if (m < M) out[(size_t)m * ldo + n] = slabs ? l3[r] : l3[r] + b;
  }
}

// C = the slabs one after the other, + bias.  A thread a column of a row; grid (ceil(N / 256), M).
__global__ __launch_bounds__(256) void gemm_f32_join_kernel(const float* __restrict__ slabs, int ranges,
                                                            const float* __restrict__ bias, float* __restrict__ C, int M,
                                                            int N, int ldc) {
  const int n = blockIdx.x * 256 + threadIdx.x, m = blockIdx.y;
  if (n >= N) return;
  const float* p = slabs + (size_t)m * N + n;
  const size_t step = (size_t)M * N;
  float sum = 0.f;
  int s = 0;
  for (; s + 4 <= ranges; s += 4) {                  // four loads in flight
    const float v0 = p[s * step], v1 = p[(s + 1) * step], v2 = p[(s + 2) * step], v3 = p[(s + 3) * step];
    sum += v0; sum += v1; sum += v2; sum += v3;
  }
  for (; s < ranges; s++) sum += p[s * step];
  C[(size_t)m * ldc + n] = sum + (bias ? bias[n] : 0.f);
}

// The number of slabs [M, N] that a call of these sizes wants as its workspace; 0: none.  Tiles of 64 x 64 (32 x 64 up to
// 32 rows) and the ranges are the units of work; below two tiles a compute unit (four fit) the ranges are dealt out too.
extern "C" int pico_gemm_f32_slabs(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const long long tiles = (long long)((N + 63) / 64) * (M <= 32 ? 1 : (M + 63) / 64);
  int len;
  const int ranges = f32_ranges(K, len);
  return tiles < 512 && ranges > 1 ? ranges : 0;
}

template <typename TA, int WM>
static void launch_gemm_f32(const TA* A, const float* W, const float* bias, float* C, float* slabs, int M, int N, int K,
                            int lda, int ldw, int ldc, hipStream_t stream) {
  const int m_tiles = (M + 32 * WM - 1) / (32 * WM), n_tiles = (N + 63) / 64;
  int len;
  const int ranges = f32_ranges(K, len);
  const dim3 grid((n_tiles + 7) / 8 * 8 * m_tiles, slabs ? ranges : 1);
  const bool vec = K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && (uintptr_t)A % (4 * sizeof(TA)) == 0 && (uintptr_t)W % 16 == 0;
  if (vec)
    gemm_f32_kernel<TA, WM, true><<<grid, 128 * WM, 0, stream>>>(A, W, bias, C, slabs, M, N, K, lda, ldw, ldc, m_tiles);
  else
    gemm_f32_kernel<TA, WM, false><<<grid, 128 * WM, 0, stream>>>(A, W, bias, C, slabs, M, N, K, lda, ldw, ldc, m_tiles);
  if (slabs) gemm_f32_join_kernel<<<dim3((N + 255) / 256, M), 256, 0, stream>>>(slabs, ranges, bias, C, M, N, ldc);
}

// `slabs`: float [pico_gemm_f32_slabs(M, N, K), M, N], or null where that is 0 (null is taken everywhere: the bits are the
// same).
extern "C" int pico_gemm_f32(const void* A, int a_dtype, const float* W, const float* bias, float* C, float* slabs, int M,
                             int N, int K, int lda, int ldw, int ldc, hipStream_t stream) {
  PICO_REQUIRE(M >= 0 && N > 0 && K > 0, "pico_gemm_f32: bad sizes M=%d N=%d K=%d", M, N, K);
  PICO_REQUIRE(lda >= K && ldw >= K && ldc >= N, "pico_gemm_f32: a row stride is smaller than its row");
  if (M == 0) return 0;
  PICO_REQUIRE((long long)((N + 511) / 512) * 8 * ((M + 31) / 32) < (1LL << 31), "pico_gemm_f32: M=%d, N=%d are too large for one launch", M, N);
  PICO_REQUIRE(!slabs || M <= 65535, "pico_gemm_f32: M=%d is too large for a call with slabs", M);
  if (a_dtype == PICO_DTYPE_F32) {
    if (M <= 32) launch_gemm_f32<float, 1>((const float*)A, W, bias, C, slabs, M, N, K, lda, ldw, ldc, stream);
    else launch_gemm_f32<float, 2>((const float*)A, W, bias, C, slabs, M, N, K, lda, ldw, ldc, stream);
  } else if (a_dtype == PICO_DTYPE_BF16) {
    if (M <= 32) launch_gemm_f32<bf16_t, 1>((const bf16_t*)A, W, bias, C, slabs, M, N, K, lda, ldw, ldc, stream);
    else launch_gemm_f32<bf16_t, 2>((const bf16_t*)A, W, bias, C, slabs, M, N, K, lda, ldw, ldc, stream);
  } else {
    PICO_REQUIRE(false, "pico_gemm_f32: unknown dtype %d", a_dtype);
  }
  PICO_LAUNCH_CHECK();
  return 0;
}
