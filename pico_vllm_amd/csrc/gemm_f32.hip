// True float32 matrix product C = A W^T (+ bias): every number is three bfloat16 pieces that hold all of its 24 bits, and the products
// of the pieces run on the bfloat16 matrix instruction (split3.h; six instructions of 16 k are 6/16 of the float32 instruction's time).
// Every output element is accumulated in an order that depends on K alone, so a row's result does not depend on how many
// other rows the call has, nor on how the work was dealt out.
//
// The sum is a tree over k: 16 products an instruction, 16 instructions (256 k) on one accumulator, then the `ranges` of K, each of
// as many 256s as there are ranges (both about sqrt(K / 256)); the small terms of a range are one sum beside that, 2^-8 of it.
// A result that is not finite (split3.h) is made again on the float32 instruction, element by element, so that it
// too depends on its own row and column alone: one infinite number in 320 rows of 17,920 x 1,536 141 and 182 us, in 1 of 1,536 x 1,536 18
// and 34.  Error against 64 bits, in units of 2^-24 of the result's rms, on the float32
// instruction (16 products a sum, 16 sums) and so: 1.93 and 1.68 at K = 1,536, 2.13 and 1.90 at 8,960, 2.28 and 2.06 at 18,944 (one
// running sum would give 0.2 sqrt(K)).
//
// Over 32 rows bound by the vector instructions that take operands apart and by the matrix instruction, about as much by either, up
// to there by the stream of W; with few tiles by the chain of a range's stages (0.8 us each).  Tiles that read the same rows
// of W are neighbours on one die.  Where the tiles alone leave the chip idle (less than two a compute unit) every range of K is a
// workgroup of its own, its sum goes to a slab, and a second launch adds the slabs in the order in which one workgroup would have.
// Microseconds on the float32 instruction and so, in one process: 320 rows of 17,920 x 1,536 184 / 140, 1,536 x 8,960 98 / 85, 1,536
// x 1,536 31 / 28; 2,048 rows of 17,920 x 1,536 1,060 / 761; one row of 151,936 x 1,536 212 / 187 (5.0 TB/s), 32 rows 230 / 208.
#include "split3.h"

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

#define F32_OUT 0x80000000u          // added to an offset: behind the end of any buffer (at most 2^31 - 1 bytes)
#ifdef __HIP_DEVICE_COMPILE__
__device__ __forceinline__ __amdgpu_buffer_rsrc_t f32_rows(const float* base, long long rows, int ld, int K) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, (int)min(((rows - 1) * ld + K) * 4, (long long)0x7fffffff), 0x00020000);
}
#endif

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

// Eight k of a row, in loads of four where they all lie in it
typedef float f32_four __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ void fetch8(const float* row, int k, int K, float (&v)[8]) {
  if (k + 8 <= K) {
    const f32_four a = *reinterpret_cast<const f32_four*>(row + k), b = *reinterpret_cast<const f32_four*>(row + k + 4);
#pragma unroll
    for (int i = 0; i < 4; i++) { v[i] = a[i]; v[4 + i] = b[i]; }
    return;
  }
#pragma unroll
  for (int i = 0; i < 8; i++) v[i] = k + i < K ? row[k + i] : 0.f;
}
__device__ __forceinline__ void fetch8(const bf16_t* row, int k, int K, float (&v)[8]) {
#pragma unroll
  for (int i = 0; i < 8; i++) v[i] = k + i < K ? bf16_to_f32(row[k + i]) : 0.f;
}

// A wave's 32 x 32 block over k_first .. k_end on the float32 instruction, straight from memory: lane (l, half) has row l of A and of
// W (`a_row`, `w_row`) and of 16 k the half'th eight.
template <typename TA>
__device__ __forceinline__ s3_f32x16 plain_block(const TA* a_row, const float* w_row, int k_first, int k_end, int K, int half) {
  s3_f32x16 sum = {}, group = {};
#pragma unroll 1
  for (int k0 = k_first; k0 < k_end; k0 += 16) {
    s3_f32x16 few = {};
    float a[8], w[8];
    fetch8(a_row, k0 + 8 * half, K, a);
    fetch8(w_row, k0 + 8 * half, K, w);
#pragma unroll
    for (int i = 0; i < 8; i++) few = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], w[i], few, 0, 0, 0);
    group += few;
    if ((k0 - k_first) % GROUP == GROUP - 16) {
      sum += group;
      group = {};
    }
  }
  return sum + group;
}

// What a range of K comes to: the sums of its large and of its small terms; results that split3.h says are made again.
template <typename TA>
__device__ __forceinline__ s3_f32x16 range_sum(const s3_f32x16& big, const s3_f32x16& small, const TA* a_row, const float* w_row, int k_first,
                                               int k_end, int K, int half) {
  s3_f32x16 sum = (big + small) * S3_BACK;
  bool odd = false;
#pragma unroll
  for (int r = 0; r < 16; r++) odd = odd || s3_redo(sum[r]);
  if (__any(odd)) {
    const s3_f32x16 plain = plain_block(a_row, w_row, k_first, k_end, K, half);
#pragma unroll
    for (int r = 0; r < 16; r++) sum[r] = s3_redo(sum[r]) ? plain[r] : sum[r];
  }
  return sum;
}

// A [M, K] row stride lda; W [N, K] row stride ldw; C [M, N] row stride ldc.  TA is the storage type of A (float, or
// bfloat16 bits that are widened on load).  WM x 2 waves of 32 x 32 outputs.  grid (8 ceil(n_tiles / 8) m_tiles, 1) with
// `slabs` null, (.., ranges) with slabs [ranges, M, N].
template <typename TA, int WM, bool VEC>
__global__ __launch_bounds__(128 * WM, 2) void gemm_f32_kernel(const TA* __restrict__ A, const float* __restrict__ W,
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

  s3_f32x16 big = {}, small = {}, l2 = {}, l3 = {};
  const float* ap = &As[0][(32 * wm + l) * ST + 8 * half];
  const float* wp = &Ws[0][(32 * wn + l) * ST + 8 * half];
  const int n = n0 + 32 * wn + l;
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
    for (int g = 0; g < BK; g += 16)                    // 16 k: this half of the lanes holds 0..7 (or 8..15) of them
      split_multiply<sizeof(TA) == 2>(split8(*reinterpret_cast<const float4*>(a + g), *reinterpret_cast<const float4*>(a + g + 4)),
                                      split8(*reinterpret_cast<const float4*>(w + g), *reinterpret_cast<const float4*>(w + g + 4)), big, small);
    if (more) put(buf ^ 1, k0 + BK);
    const int done = k0 + BK - k_first;
    if (done % GROUP == 0) {
      l2 += big;
      big = {};
    }
    if (done % len == 0 || !more) {                      // the same for all threads
      l3 += range_sum(l2 + big, small, A + (size_t)min(m0 + 32 * wm + l, M - 1) * lda, W + (size_t)min(n, N - 1) * ldw, k0 / len * len, min(K, k0 + BK), K, half);
      big = {};
      l2 = {};
      small = {};
    }
  }
  if (n >= N) return;
  const float b = !slabs && bias ? bias[n] : 0.f;
  float* out = slabs ? slabs + (size_t)blockIdx.y * M * N : C;
  const int ldo = slabs ? N : ldc;
#pragma unroll
  for (int r = 0; r < 16; r++) {
    const int m = m0 + 32 * wm + 8 * (r >> 2) + 4 * half + (r & 3);
    if (m < M) out[(size_t)m * ldo + n] = slabs ? l3[r] : l3[r] + b;
  }
}

// The same sums where both operands are float32 rows of whole aligned fours, up to 32 rows: the stream of W bounds a call.  A
// stage of 32 k goes from memory straight to one of two LDS buffers (buffer_load .. lds, eight rows of 128 bytes an instruction,
// their sixteen-byte chunks xor-swizzled by the row so that the operand reads of 16 rows meet every bank once); a wave has 32 x 32
// outputs, and the one barrier of a stage stands where its operands are in registers.  What lies outside a matrix (rows
// behind the last, k behind K) arrives as zeros.  (Three buffers instead of two 240 us, four 255, two 220: 1 row of 151,936 x 1,536 on
// the float32 instruction.  Four where there are few tiles: 1,536 x 8,960 46 us, two 43: a stage's own chain, not memory.)
// (The operands are read as native vectors: in front of a read of float4, a class, the compiler waits for all copies.)
#define FS_STAGE ((32 + 64) * BK * 4)
__global__ __launch_bounds__(128, 3) void gemm_f32_stream_kernel(const float* A, const float* W, const float* bias, float* C, float* slabs, int M,
                                                                 int N, int K, int lda, int ldw, int ldc) {
#ifdef __HIP_DEVICE_COMPILE__      // (buffer resources exist on the device only)
  __shared__ __attribute__((aligned(1024))) char smem[2 * FS_STAGE];
  const int n0 = blockIdx.x * 64;
  int len;
  f32_ranges(K, len);
  const int k_first = slabs ? blockIdx.y * len : 0, k_end = slabs ? min(K, k_first + len) : K;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = lane & 31, half = lane >> 5;
  const __amdgpu_buffer_rsrc_t as = f32_rows(A, M, lda, K), ws = f32_rows(W + (size_t)n0 * ldw, N - n0, ldw, K);
  // copy j of this wave brings rows 8 (2 j + wave) .. + 7 of [A's tile | W's tile]; lane: row lane / 8, chunk lane % 8 there
  uint32_t off[6];
  const uint32_t kbyte = (uint32_t)(((lane & 7) ^ (4 * wave + (lane >> 4))) << 4);
#pragma unroll
  for (int j = 0; j < 6; j++) {
    const int r = (j * 2 + wave) * 8 + (lane >> 3);
    off[j] = (uint32_t)(r < 32 ? r * lda : (r - 32) * ldw) * 4;
  }
  auto ask = [&](int b, int k0) {
    const uint32_t k = (uint32_t)k0 * 4 + kbyte, at = k < (uint32_t)K * 4 ? k : F32_OUT;
#pragma unroll
    for (int j = 0; j < 6; j++)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(j < 2 ? as : ws, (__attribute__((address_space(3))) void*)(smem + b * FS_STAGE + (j * 2 + wave) * 1024), 16,
                                               off[j] + at, 0, 0, 0);
  };
  const int sw = (l >> 1) & 7;                              // of row l and of row 32 + l
  const char* ap = smem + l * 128;
  const char* wp = smem + (32 + 32 * wave + l) * 128;
  s3_f32x16 big = {}, small = {}, l2 = {}, l3 = {};
  const int n = n0 + 32 * wave + l;
  ask(0, k_first);
  ask(1, k_first + BK);
  int buf = 0;
  for (int k0 = k_first; k0 < k_end; k0 += BK, buf ^= 1) {
    // this wave's copies of this stage have landed; behind the barrier all waves'
    __builtin_amdgcn_s_waitcnt(6 | (7 << 4) | (15 << 8));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    f32x4 a[2][2], w[2][2];                                 // of 16 k this half of the lanes holds 0..7 (or 8..15)
#pragma unroll
    for (int g = 0; g < 2; g++)
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const int c = ((4 * g + 2 * half + i) ^ sw) << 4;
        a[g][i] = *reinterpret_cast<const f32x4*>(ap + buf * FS_STAGE + c);
        w[g][i] = *reinterpret_cast<const f32x4*>(wp + buf * FS_STAGE + c);
      }
    // they are in registers, so the buffer may be filled again
    __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    ask(buf, k0 + 2 * BK);
#pragma unroll
    for (int g = 0; g < 2; g++) split_multiply(split8(a[g][0], a[g][1]), split8(w[g][0], w[g][1]), big, small);
    const int done = k0 + BK - k_first;
    if (done % GROUP == 0) {
      l2 += big;
      big = {};
    }
    if (done % len == 0 || k0 + BK >= k_end) {              // the same for all threads
      l3 += range_sum(l2 + big, small, A + (size_t)min(l, M - 1) * lda, W + (size_t)min(n, N - 1) * ldw, k0 / len * len, min(K, k0 + BK), K, half);
      big = {};
      l2 = {};
      small = {};
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0070);                        // the last copies (zeros) are in before LDS is given back
  if (n >= N) return;
  const float b = !slabs && bias ? bias[n] : 0.f;
  float* out = slabs ? slabs + (size_t)blockIdx.y * M * N : C;
  const int ldo = slabs ? N : ldc;
#pragma unroll
  for (int r = 0; r < 16; r++) {
    const int m = 8 * (r >> 2) + 4 * half + (r & 3);
    if (m < M) out[(size_t)m * ldo + n] = slabs ? l3[r] : l3[r] + b;
  }
#endif
}

// The same sums over 32 rows: the operands are taken apart once a workgroup, on their way from memory through registers to LDS,
// where a stage of 32 k lies as three planes of bfloat16 rows of 64 bytes, their sixteen-byte chunks xor-swizzled by a quarter of the
// row: LDS serves sixteen lanes of a read or write at a time, and sixteen rows of one chunk, or four rows whole, so meet every bank
// once (swizzled by half of the row, which is right for eight lanes, two lanes met in each bank: 300 rows of 17,920 x 1,536 148 us and
// so 143, 100 rows 84 and 78).  Four waves (2 x 2) of 32 x 32 NW outputs.  A stage's numbers are asked for AHEAD stages ahead, lie in
// registers, and are taken apart under the products of the stage in front.
constexpr int fp_plane(int NW) { return (64 + 64 * NW) * BK * 2; }
// Rows may start anywhere: a load of four to registers needs no more alignment than one.  (Through gemm_f32_kernel, where every wave takes its
// operands apart by itself, 64 such rows of 32,000 x 1,024 95 us and so 64, 320 of 17,920 x 1,536 262 and 145.)  EVEN: whole fours; else
// the four numbers that K ends in are asked for one by one.
template <int NW, int AHEAD, bool EVEN>
__global__ __launch_bounds__(256, NW == 1 && AHEAD == 2 ? 3 : 2) void gemm_f32_planes_kernel(const float* A, const float* W, const float* bias, float* C, float* slabs,
                                                                               int M, int N, int K, int lda, int ldw, int ldc, int m_tiles) {
#ifdef __HIP_DEVICE_COMPILE__      // (buffer resources exist on the device only)
  constexpr int TM = 64, TN = 64 * NW, PLANE = fp_plane(NW), STAGE = 3 * PLANE, PIECES = (TM + TN) / 64;
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
  const __amdgpu_buffer_rsrc_t as = f32_rows(A + (size_t)m0 * lda, M - m0, lda, K), ws = f32_rows(W + (size_t)n0 * ldw, N - n0, ldw, K);
  // a thread's pieces: eight k (chunk threadIdx.x % 4 of a stage) of row threadIdx.x / 4 of A's tile, and of every 64 rows of W's
  const int prow = threadIdx.x >> 2, chunk = threadIdx.x & 3;
  uint32_t off[PIECES];
  off[0] = (uint32_t)(prow * lda) * 4;
#pragma unroll
  for (int j = 1; j < PIECES; j++) off[j] = (uint32_t)((prow + 64 * (j - 1)) * ldw) * 4;
  char* put_at = smem + prow * 64 + ((chunk ^ ((prow >> 2) & 3)) << 4);
  f32x4 raw[AHEAD][PIECES][2];
  auto ask = [&](int set, int k0) {
    const uint32_t k = (uint32_t)(k0 + 8 * chunk) * 4, end = (uint32_t)K * 4;
    if (!EVEN && k0 + BK > K) {
#pragma unroll
      for (int j = 0; j < PIECES; j++)
#pragma unroll
        for (int i = 0; i < 8; i++)
          raw[set][j][i / 4][i % 4] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(j == 0 ? as : ws, off[j] + (k + 4 * i < end ? k + 4 * i : F32_OUT), 0, 0));
      return;
    }
#pragma unroll
    for (int j = 0; j < PIECES; j++)
#pragma unroll
      for (int i = 0; i < 2; i++)
        raw[set][j][i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(j == 0 ? as : ws, off[j] + (k + 16 * i < end ? k + 16 * i : F32_OUT), 0, 0));
  };
  auto put = [&](int set, int b) {
#pragma unroll
    for (int j = 0; j < PIECES; j++) {
      const Split8 s = split8(raw[set][j][0], raw[set][j][1]);
      char* dst = put_at + b * STAGE + j * (64 * 64);
      *reinterpret_cast<s3_u32x4*>(dst) = s.h;
      *reinterpret_cast<s3_u32x4*>(dst + PLANE) = s.m;
      *reinterpret_cast<s3_u32x4*>(dst + 2 * PLANE) = s.l;
    }
  };
  const int sw = (l >> 2) & 3;
  const char* ap = smem + (32 * wm + l) * 64;
  const char* wp = smem + (TM + 32 * NW * wn + l) * 64;
  auto read = [&](const char* p, int b, int g) {
    const char* at = p + b * STAGE + (((2 * g + half) ^ sw) << 4);
    Split8 s;
    s.h = *reinterpret_cast<const s3_u32x4*>(at);
    s.m = *reinterpret_cast<const s3_u32x4*>(at + PLANE);
    s.l = *reinterpret_cast<const s3_u32x4*>(at + 2 * PLANE);
    return s;
  };
  s3_f32x16 big[NW], small[NW], l2[NW], l3[NW];
#pragma unroll
  for (int j = 0; j < NW; j++) big[j] = small[j] = l2[j] = l3[j] = s3_f32x16{};
  auto stage = [&](int k0, int i) {                          // the i'th stage of AHEAD
    const int b = i & 1, next = (i + 1) % AHEAD;
    __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4));   // this wave's part of the stage is written; behind the barrier all waves'
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < 2; g++) {
      const Split8 a = read(ap, b, g);
      Split8 w[NW];
#pragma unroll
      for (int j = 0; j < NW; j++) w[j] = read(wp + j * (32 * 64), b, g);
#pragma unroll
      for (int j = 0; j < NW; j++) split_multiply(a, w[j], big[j], small[j]);
      if (g == 0) {
        put(next, b ^ 1);
        ask(next, k0 + (AHEAD + 1) * BK);
      }
    }
    const int done = k0 + BK - k_first;
    if (done % GROUP == 0) {
#pragma unroll
      for (int j = 0; j < NW; j++) {
        l2[j] += big[j];
        big[j] = s3_f32x16{};
      }
    }
    if (done % len == 0 || k0 + BK >= k_end) {              // the same for all threads
#pragma unroll
      for (int j = 0; j < NW; j++) {
        const int n = n0 + 32 * (NW * wn + j) + l;
        l3[j] += range_sum(l2[j] + big[j], small[j], A + (size_t)min(m0 + 32 * wm + l, M - 1) * lda, W + (size_t)min(n, N - 1) * ldw, k0 / len * len,
                           min(K, k0 + BK), K, half);
        big[j] = l2[j] = small[j] = s3_f32x16{};
      }
    }
  };
#pragma unroll
  for (int i = 0; i < AHEAD; i++) ask(i, k_first + i * BK);
  put(0, 0);
  ask(0, k_first + AHEAD * BK);
  for (int k0 = k_first; k0 < k_end; k0 += AHEAD * BK)
#pragma unroll
    for (int i = 0; i < AHEAD; i++)
      if (k0 + i * BK < k_end) stage(k0 + i * BK, i);
  float* out = slabs ? slabs + (size_t)blockIdx.y * M * N : C;
  const int ldo = slabs ? N : ldc;
#pragma unroll
  for (int j = 0; j < NW; j++) {
    const int n = n0 + 32 * (NW * wn + j) + l;
    if (n >= N) continue;
    const float b = !slabs && bias ? bias[n] : 0.f;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int m = m0 + 32 * wm + 8 * (r >> 2) + 4 * half + (r & 3);
      if (m < M) out[(size_t)m * ldo + n] = slabs ? l3[j][r] : l3[j][r] + b;
    }
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

// Tiles of 64 x 128 instead of 64 x 64: an operand is read from LDS for half as many products, so where they are more than the
// chip holds at once (17,920 x 1,536: 700 tiles, 320 rows, 138 us, in tiles of 64 x 64 153; 560 tiles, 256 rows, 135 and 128).
static bool f32_wide(int M, int N) { return (long long)((N + 127) / 128) * ((M + 63) / 64) >= 600; }

// The number of slabs [M, N] that a call of these sizes wants as its workspace; 0: none.  Tiles of 64 x 64 (32 x 64 up to
// 32 rows) and the ranges are the units of work; below two tiles a compute unit (four fit) the ranges are dealt out too.
extern "C" int pico_gemm_f32_slabs(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const long long tiles = (long long)((N + 63) / 64) * (M <= 32 ? 1 : (M + 63) / 64);
  int len;
  const int ranges = f32_ranges(K, len);
  return tiles < 512 && ranges > 1 ? ranges : 0;
}

template <int NW, int AHEAD, bool EVEN>
static bool launch_planes_of(const float* A, const float* W, const float* bias, float* C, float* slabs, int M, int N, int K, int lda, int ldw, int ldc,
                          int ranges, hipStream_t stream) {
  constexpr int bytes = 6 * fp_plane(NW);
  static const hipError_t room = hipFuncSetAttribute((const void*)&gemm_f32_planes_kernel<NW, AHEAD, EVEN>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (room != hipSuccess) return false;
  const int m_tiles = (M + 63) / 64, n_tiles = (N + 64 * NW - 1) / (64 * NW);
  gemm_f32_planes_kernel<NW, AHEAD, EVEN>
      <<<dim3((n_tiles + 7) / 8 * 8 * m_tiles, ranges), 256, bytes, stream>>>(A, W, bias, C, slabs, M, N, K, lda, ldw, ldc, m_tiles);
  return true;
}
template <int NW, int AHEAD>
static bool launch_planes(const float* A, const float* W, const float* bias, float* C, float* slabs, int M, int N, int K, int lda, int ldw, int ldc,
                          int ranges, hipStream_t stream) {
  return K % 4 == 0 ? launch_planes_of<NW, AHEAD, true>(A, W, bias, C, slabs, M, N, K, lda, ldw, ldc, ranges, stream)
                    : launch_planes_of<NW, AHEAD, false>(A, W, bias, C, slabs, M, N, K, lda, ldw, ldc, ranges, stream);
}

template <typename TA, int WM>
static void launch_gemm_f32(const TA* A, const float* W, const float* bias, float* C, float* slabs, int M, int N, int K,
                            int lda, int ldw, int ldc, hipStream_t stream) {
  const int m_tiles = (M + 32 * WM - 1) / (32 * WM), n_tiles = (N + 63) / 64;
  int len;
  const int all = f32_ranges(K, len), ranges = slabs ? all : 1;
  const dim3 grid((n_tiles + 7) / 8 * 8 * m_tiles, ranges);
  const bool vec = K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && (uintptr_t)A % (4 * sizeof(TA)) == 0 && (uintptr_t)W % 16 == 0;
  bool done = false;
  if constexpr (sizeof(TA) == 4) {
    // (a tile's rows within 2^31 bytes of its first; copies to LDS want whole aligned fours)
    if ((vec || WM == 2) && lda < (1 << 23) && ldw < (1 << 23)) {
      if (WM == 1) {
        gemm_f32_stream_kernel<<<dim3(n_tiles, ranges), 128, 0, stream>>>(A, W, bias, C, slabs, M, N, K, lda, ldw, ldc);
        done = true;
      } else if (f32_wide(M, N) && ldw < (1 << 22)) {
        done = launch_planes<2, 2>(A, W, bias, C, slabs, M, N, K, lda, ldw, ldc, ranges, stream);
      } else {                                               // few workgroups: reads ahead take the registers of a third one a unit
        done = (long long)n_tiles * m_tiles * ranges <= 512 ? launch_planes<1, 4>(A, W, bias, C, slabs, M, N, K, lda, ldw, ldc, ranges, stream)
                                                            : launch_planes<1, 2>(A, W, bias, C, slabs, M, N, K, lda, ldw, ldc, ranges, stream);
      }
    }
  }
  if (!done && vec)
    gemm_f32_kernel<TA, WM, true><<<grid, 128 * WM, 0, stream>>>(A, W, bias, C, slabs, M, N, K, lda, ldw, ldc, m_tiles);
  else if (!done)
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
