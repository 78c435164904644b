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
// outputs, so that the tree's four levels are 64 registers and three or four workgroups share a compute unit; its operands come
// from LDS (64 of 128 B a cycle at most), stages of 32 k.  Tiles that read the same rows of W are neighbours on
// one die.  Where the tiles alone leave the chip idle (less than two a compute unit) every range of K is a workgroup
// of its own, its sum goes to a slab, and a second launch adds the slabs in the order in which one workgroup would have.
// 320 rows, microseconds a call with plain FMA in 64 x 64 tiles and with this: 17,920 x 1,536 575 / 206 (86 TFLOP/s);
// 1,536 x 8,960 1,421 / 104; 1,536 x 1,536 183 / 32.  2,048 rows of 17,920 x 1,536: 3,299 / 1,120 (101 TFLOP/s; the library's
// product, which sums in one chain, 1,030).  One row of 151,936 x 1,536: 1,070 / 230 (4.1 TB/s).
#include "common.h"

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

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

// The same sums where both operands are float32 rows of whole aligned fours: a stage goes from memory straight to one of NBUF LDS
// buffers (buffer_load .. lds, eight rows of 128 bytes an instruction, their sixteen-byte chunks xor-swizzled by the row so that the
// operand reads of 16 rows meet every bank once).  The operands of 16 k are read under the products of the 16 before, and their sums
// join the others under the products behind them; the one barrier of a stage stands where its last operands are in registers.
// (Through registers, with every wave waiting for its operands and its sums in turn, the matrix instruction was busy 56 % of
// the time at 320 rows and 67 % at 2,048.)  What lies outside a matrix (rows behind the last, k behind K) arrives as zeros.
// Up to 32 rows the stream of W bounds a call and workgroups side by side count: two buffers (two 220, three 240, four 255 us, 1 row of
// 151,936 x 1,536).  Microseconds through registers and so: 1 row of 151,936 x 1,536 268 and 230, 32 rows 283 and 266; 17,920 x 1,536
// 100 rows 114 and 104, 320 211 and 206, 2,048 1,135 and 1,120; 1,536 x 8,960 33 rows 50 and 45, 320 108 and 104.
// (The operands are read as native vectors: in front of a read of float4, a class, the compiler waits for all copies.)
constexpr int fs_bytes(int WM) { return (32 * WM + 64) * BK * 4; }
constexpr int fs_buffers(int WM) { return WM == 1 ? 2 : 3; }
template <int WM>
__global__ __launch_bounds__(128 * WM, 3) void gemm_f32_stream_kernel(const float* A, const float* W,
                                                                      const float* bias, float* C,
                                                                      float* slabs, int M, int N, int K, int lda,
                                                                      int ldw, int ldc, int m_tiles) {
#ifdef __HIP_DEVICE_COMPILE__      // (buffer resources exist on the device only)
  constexpr int TM = 32 * WM, TN = 64, WAVES = 2 * WM, COPIES = (TM + TN) / 8 / WAVES, NBUF = fs_buffers(WM), STAGE = fs_bytes(WM);
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  // dies take workgroups in turn: the tiles of one strip of W stay on one die
  const int die = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int n0 = ((local / m_tiles) * 8 + die) * TN, m0 = local % m_tiles * TM;
  if (n0 >= N) return;
  int len;
  f32_ranges(K, len);
  const int k_first = slabs ? blockIdx.y * len : 0, k_end = slabs ? min(K, k_first + len) : K;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = lane & 31, half = lane >> 5;
  const int wm = wave >> 1, wn = wave & 1;

  auto source = [](const float* base, long long rows, int ld, int K) {
    const long long bytes = ((rows - 1) * ld + K) * 4;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, (int)min(bytes, (long long)0x7fffffff), 0x00020000);
  };
  const __amdgpu_buffer_rsrc_t as = source(A + (size_t)m0 * lda, M - m0, lda, K), ws = source(W + (size_t)n0 * ldw, N - n0, ldw, K);
  // copy j of this wave brings rows 8 (j WAVES + wave) .. + 7 of [A's tile | W's tile]; lane: row lane / 8, chunk lane % 8 there
  uint32_t off[COPIES];
  const uint32_t kbyte = (uint32_t)(((lane & 7) ^ (4 * (wave & 1) + (lane >> 4))) << 4);
#pragma unroll
  for (int j = 0; j < COPIES; j++) {
    const int r = (j * WAVES + wave) * 8 + (lane >> 3);
    off[j] = (uint32_t)(r < TM ? r * lda : (r - TM) * ldw) * 4;
  }
  auto ask = [&](int b, int k0) {
    const uint32_t k = (uint32_t)k0 * 4 + kbyte, at = k < (uint32_t)K * 4 ? k : 0x80000000u;
#pragma unroll
    for (int j = 0; j < COPIES; j++)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(j * WAVES * 8 < TM ? as : ws, (__attribute__((address_space(3))) void*)(smem + b * STAGE + (j * WAVES + wave) * 1024),
                                               16, off[j] + at, 0, 0, 0);
  };
  static_assert(TM % (8 * WAVES) == 0, "a copy of all waves is of one operand");
  const int sw = (l >> 1) & 7;                              // of row l and of row 32 + l
  const char* ap = smem + (32 * wm + l) * 128;
  const char* wp = smem + (TM + 32 * wn + l) * 128;
  // operands of 16 k: this half of the lanes holds 0..3 and 8..11 (or 4..7 and 12..15) of them
  f32x4 a0[2], a1[2], w0[2], w1[2];
  f32x16 l0[2], l1 = {}, l2 = {}, l3 = {};
  auto read = [&](int b, int g) {
    const int c0 = ((4 * g + half) ^ sw) << 4, c1 = ((4 * g + 2 + half) ^ sw) << 4;
    a0[g] = *reinterpret_cast<const f32x4*>(ap + b * STAGE + c0);
    w0[g] = *reinterpret_cast<const f32x4*>(wp + b * STAGE + c0);
    a1[g] = *reinterpret_cast<const f32x4*>(ap + b * STAGE + c1);
    w1[g] = *reinterpret_cast<const f32x4*>(wp + b * STAGE + c1);
  };
  // the products of group g, the sums of the group before joining theirs under them
  auto multiply = [&](int g) {
    l0[g] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0[g].x, w0[g].x, f32x16{}, 0, 0, 0);
    l0[g] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0[g].y, w0[g].y, l0[g], 0, 0, 0);
    l0[g] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0[g].z, w0[g].z, l0[g], 0, 0, 0);
    l0[g] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0[g].w, w0[g].w, l0[g], 0, 0, 0);
    l0[g] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[g].x, w1[g].x, l0[g], 0, 0, 0);
    l0[g] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[g].y, w1[g].y, l0[g], 0, 0, 0);
    l0[g] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[g].z, w1[g].z, l0[g], 0, 0, 0);
    l0[g] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[g].w, w1[g].w, l0[g], 0, 0, 0);
    l1 += l0[g ^ 1];
    __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
#pragma unroll
    for (int i = 0; i < 6; i++) {
      __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // what is summed up to k = done (all sums of the groups are in l1)
  auto close = [&](int done) {
    if (done % GROUP == 0) {
      l2 += l1;
      l1 = {};
    }
    if (!slabs && (done % len == 0 || k_first + done >= k_end)) {      // the same for all threads
      l3 += l1 + l2;
      l1 = {};
      l2 = {};
    }
  };
#pragma unroll
  for (int b = 0; b < NBUF - 1; b++) ask(b, k_first + b * BK);
  l0[1] = {};
  constexpr int LEFT = (NBUF - 2) * COPIES;                  // copies that may be on their way when a stage is begun
  __builtin_amdgcn_s_waitcnt((LEFT & 15) | (LEFT >> 4 << 14) | (7 << 4) | (15 << 8));
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  ask(NBUF - 1, k_first + (NBUF - 1) * BK);
  read(0, 0);
  int buf = 0;
  for (int k0 = k_first; k0 < k_end; k0 += BK) {
    const int next = buf + 1 == NBUF ? 0 : buf + 1;
    __builtin_amdgcn_sched_barrier(0);
    read(buf, 1);
    multiply(0);
    if (k0 > k_first) close(k0 - k_first);
    // this wave's copies of the next stage have landed and its reads of this one are done; behind the barrier all waves'
    __builtin_amdgcn_s_waitcnt((LEFT & 15) | (LEFT >> 4 << 14) | (7 << 4));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    ask(buf, k0 + NBUF * BK);
    read(next, 0);
    multiply(1);
    buf = next;
  }
  l1 += l0[1];
  close((k_end - k_first + BK - 1) / BK * BK);
  __builtin_amdgcn_s_waitcnt(0x0070);                        // the last copies (zeros) are in before LDS is given back
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
#endif
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
  if constexpr (sizeof(TA) == 4) {
    // (a tile's rows within 2^31 bytes of its first)
    static const hipError_t room = hipFuncSetAttribute((const void*)&gemm_f32_stream_kernel<WM>, hipFuncAttributeMaxDynamicSharedMemorySize, fs_buffers(WM) * fs_bytes(WM));
    if (vec && lda < (1 << 23) && ldw < (1 << 23) && room == hipSuccess)
      gemm_f32_stream_kernel<WM><<<grid, 128 * WM, fs_buffers(WM) * fs_bytes(WM), stream>>>(A, W, bias, C, slabs, M, N, K, lda, ldw, ldc, m_tiles);
    else
      gemm_f32_kernel<TA, WM, false><<<grid, 128 * WM, 0, stream>>>(A, W, bias, C, slabs, M, N, K, lda, ldw, ldc, m_tiles);
  } else if (vec) {
    gemm_f32_kernel<TA, WM, true><<<grid, 128 * WM, 0, stream>>>(A, W, bias, C, slabs, M, N, K, lda, ldw, ldc, m_tiles);
  } else {
    gemm_f32_kernel<TA, WM, false><<<grid, 128 * WM, 0, stream>>>(A, W, bias, C, slabs, M, N, K, lda, ldw, ldc, m_tiles);
  }
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
