// Plain paged attention in float32 arithmetic, for every batch shape (prompt portions beside decode tokens), any head size up to
// 256, any page size, an optional window.  Two kernels: the attention of the 32-bit engine on the float32 matrix
// instruction, and one wave per (query token, query head) for what that does not take (bfloat16 of sizes that the bfloat16
// matrix-core kernels refuse, head and page sizes that are no multiples of 4).
//
//   query head h reads kv head h / (nq / nkv)              (pico_vllm/kernels/attention.py:31,139)
//   s_k = (q . K_k) * scale, keys k <= position visible     (attention.py:190-197)
//   window > 0: only keys k > position - window
//   online softmax over blocks of keys, o = sum p_k V_k / sum p_k   (attention.py:199-211)
//
// Keys are visited in blocks of 64 aligned to absolute positions, so the result at a
// position does not depend on how the sequence was cut into steps.
#include "common.h"

template <typename T>
__global__ __launch_bounds__(64) void paged_attention_ref_kernel(
    const T* __restrict__ q, int q_stride, const T* __restrict__ k_cache, const T* __restrict__ v_cache,
    const int* __restrict__ block_table, int max_pages, const int* __restrict__ positions,
    const int* __restrict__ token_seq, T* __restrict__ out, int nq, int nkv, int d, int P, int window, float scale,
    int num_pages) {
  extern __shared__ float lds[];
  float* qs = lds;       // [d]
  float* ps = lds + d;   // [64]
  const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const int g = h / (nq / nkv);
  const int pos = positions[t];
  const int* bt = block_table + (size_t)token_seq[t] * max_pages;
  const int lo = window > 0 ? max(0, pos - window + 1) : 0;
  const T* qrow = q + (size_t)t * q_stride + (size_t)h * d;
  for (int j = lane; j < d; j += 64) qs[j] = load_f32(qrow + j);
  __syncthreads();

  float m = -INFINITY, l = 0.f;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int c0 = (lo / 64) * 64; c0 <= pos; c0 += 64) {
    const int key = c0 + lane;
    const bool valid = key >= lo && key <= pos;
    float s = -INFINITY;
    if (valid) {
      int page = bt[key / P];
      page = min(max(page, 0), num_pages - 1);
      const T* kp = k_cache + (((size_t)page * nkv + g) * P + key % P) * d;
      float dot = 0.f;
      for (int j = 0; j < d; j++) dot = fmaf(qs[j], load_f32(kp + j), dot);
      s = dot * scale;
    }
    const float m_new = fmaxf(m, wave_max(s));
    const float alpha = expf(m - m_new);
    const float p = valid ? expf(s - m_new) : 0.f;
    l = l * alpha + wave_sum(p);
    __syncthreads();
    ps[lane] = p;
    __syncthreads();
    // the block's part of P V is summed on its own and then joins the running sum: two short sums instead of one
    // over the whole context
    float blk[4] = {0.f, 0.f, 0.f, 0.f};
    const int kend = min(64, pos - c0 + 1);
    for (int kk = max(0, lo - c0); kk < kend; kk++) {
      const int kpos = c0 + kk;
      int page = bt[kpos / P];
      page = min(max(page, 0), num_pages - 1);
      const T* vp = v_cache + ((size_t)page * nkv + g) * d * P + kpos % P;
      const float pk = ps[kk];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int dim = lane + 64 * i;
        if (dim < d) blk[i] = fmaf(pk, load_f32(vp + (size_t)dim * P), blk[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i] = fmaf(acc[i], alpha, blk[i]);
    m = m_new;
  }
  T* o = out + ((size_t)t * nq + h) * d;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int dim = lane + 64 * i;
    if (dim < d) store_f32(o + dim, acc[i] / l);
  }
}

// ---------------------------------------------------------------------------
// 32-bit.  A workgroup takes 16 columns, neighbouring (token, head) pairs of one kv head, so a key and a value are read once for
// them and both products are contractions for v_mfma_f32_16x16x4f32 (exact 32-bit products and sums).  Its four waves take a
// quarter of every 64 keys each, 16 by absolute position, with a softmax of their own, and are joined at the end in a fixed
// order: nothing is exchanged on the way, and no barrier stands between the loads.  S = K Q^T: lane (i, h) holds key i of the
// quarter, dims 16 b + 4 h .. + 3; it comes out with column i and keys 4 h .. + 3 in a lane, which is how the second product,
// O^T = V P, wants its probabilities; lane (i, h) holds dim 16 b + i of V, keys 4 h .. + 3.  Keys and page numbers of the next
// 64 are asked for while this one's values are multiplied.
// Tokens of several sequences in one tile are served sequence by sequence.  A column that sees none of the 16 keys keeps what it
// has, and where only some are seen and a value is not finite the keys are taken one at a time: what a column does not see
// does not reach it, be it infinite.
// Bound by the chain of one column's blocks (loads, products, softmax), not by the matrix cores: 300 tokens of 12 heads of 128
// over two 20 us (a wave a token and head: 188), 2,048 tokens 250 (7,720), eight single tokens behind 4,000 513 (1,610), 40
// behind 900 of 28 heads over four 134 (470).  Error against 64 bits 1.9e-7 to 3.1e-7 (3.0e-7 to 4.8e-7: one chain over a head).
// ---------------------------------------------------------------------------
struct Attn32Args {
  const float* q;
  const float* k;
  const float* v;
  const int* table;
  const int* positions;
  const int* token_seq;
  float* out;
  int q_stride, max_pages, T, nq, nkv, d, P, window, num_pages;
  float scale;
};
typedef float a32_f32x4 __attribute__((ext_vector_type(4)));

template <int DB>      // blocks of 16 dims
__global__ __launch_bounds__(256) void attention_f32_kernel(const Attn32Args a) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  constexpr int ROW = 16 * DB + 4;
  float* obuf = lds;                        // [4][16][ROW]
  float* ml = lds + 4 * 16 * ROW;           // [4][16][2]
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, i = lane & 15, h = lane >> 4;
  const int R = a.nq / a.nkv, g = blockIdx.y, cols = a.T * R, tile = gridDim.x - 1 - blockIdx.x;    // the longest rows first
  const int c = tile * 16 + i, cc = min(c, cols - 1), t = cc / R;
  const int pos = a.positions[t], seq = a.token_seq[t], lo = a.window > 0 ? max(0, pos - a.window + 1) : 0;
  const float* qrow = a.q + (size_t)t * a.q_stride + (size_t)(g * R + cc % R) * a.d;
  a32_f32x4 qv[DB], kv[DB], o[DB];
#pragma unroll
  for (int b = 0; b < DB; b++) {
    const int at = 16 * b + 4 * h;
#pragma unroll
    for (int r = 0; r < 4; r++) qv[b][r] = at + r < a.d ? qrow[at + r] : 0.f;
    o[b] = a32_f32x4{0.f, 0.f, 0.f, 0.f};
  }
  float m = -INFINITY, l = 0.f;
  bool todo = c < cols;
  for (unsigned long long left = __ballot(todo); left; left = __ballot(todo)) {
    const int cur = __builtin_amdgcn_readfirstlane(__shfl(seq, __ffsll(left) - 1));
    const bool in = todo && seq == cur;
    todo = todo && !in;
    int hi = in ? pos : -1, low = in ? lo : 0x7fffffff;
#pragma unroll
    for (int x = 1; x < 16; x *= 2) { hi = max(hi, __shfl_xor(hi, x)); low = min(low, __shfl_xor(low, x)); }
    hi = __builtin_amdgcn_readfirstlane(hi);
    low = __builtin_amdgcn_readfirstlane(low);
    const int* bt = a.table + (size_t)cur * a.max_pages;
    auto page = [&](int key) { return min(max(bt[min(key / a.P, a.max_pages - 1)], 0), a.num_pages - 1); };
    auto load_k = [&](int k0, int pg) {
      const int key = k0 + i;
      const float* kp = a.k + (((size_t)pg * a.nkv + g) * a.P + key % a.P) * a.d;
#pragma unroll
      for (int b = 0; b < DB; b++) kv[b] = *reinterpret_cast<const a32_f32x4*>(kp + (16 * b + 4 * h < a.d ? 16 * b + 4 * h : 0));
    };
    int k0 = low / 64 * 64 + 16 * wave;
    int kpage = page(k0 + i), vpage = page(k0 + 4 * h);
    load_k(k0, kpage);
    for (; k0 <= hi; k0 += 64) {
      const int kpage_n = page(k0 + 64 + i), vpage_n = page(k0 + 64 + 4 * h);
      a32_f32x4 vv[DB];
      const float* vp = a.v + ((size_t)vpage * a.nkv + g) * a.d * a.P + (k0 + 4 * h) % a.P;
#pragma unroll
      for (int b = 0; b < DB; b++) vv[b] = *reinterpret_cast<const a32_f32x4*>(vp + (size_t)min(16 * b + i, a.d - 1) * a.P);
      a32_f32x4 s0{0.f, 0.f, 0.f, 0.f}, s1 = s0;
#pragma unroll
      for (int b = 0; b < DB; b++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const float kj = 16 * b + 4 * h < a.d ? kv[b][j] : 0.f;
          if (b & 1) s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kj, qv[b][j], s1, 0, 0, 0);
          else s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kj, qv[b][j], s0, 0, 0, 0);
        }
      if (k0 + 64 <= hi) load_k(k0 + 64, kpage_n);
      vpage = vpage_n;
      bool valid[4], some = false, all = true;
      float s[4], top = -INFINITY;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int key = k0 + 4 * h + r;
        valid[r] = in && key >= lo && key <= pos;
        s[r] = valid[r] ? (s0[r] + s1[r]) * a.scale : -INFINITY;
        top = fmaxf(top, s[r]);
        some = some || valid[r];
        all = all && valid[r];
      }
      top = fmaxf(top, __shfl_xor(top, 16));
      top = fmaxf(top, __shfl_xor(top, 32));
      const unsigned long long seen = __ballot(some);
      const bool sees = ((seen >> i) | (seen >> (16 + i)) | (seen >> (32 + i)) | (seen >> (48 + i))) & 1;     // this column any of the 16
      const float m_new = fmaxf(m, top), base = m_new == -INFINITY ? 0.f : m_new;
      const float alpha = expf(m - base);
      float p[4], part = 0.f;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        p[r] = valid[r] ? expf(s[r] - base) : 0.f;
        part += p[r];
      }
      bool finite = true;
      if (__ballot(in && !all)) {
#pragma unroll
        for (int b = 0; b < DB; b++)
#pragma unroll
          for (int j = 0; j < 4; j++) finite = finite && fabsf(vv[b][j]) < INFINITY;
        finite = !__ballot(!finite);
      }
      if (finite) {
#pragma unroll
        for (int b = 0; b < DB; b++) {
          a32_f32x4 blk{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int j = 0; j < 4; j++) blk = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[b][j], p[j], blk, 0, 0, 0);
#pragma unroll
          for (int r = 0; r < 4; r++) o[b][r] = sees ? fmaf(o[b][r], alpha, blk[r]) : o[b][r];
        }
      } else {
#pragma unroll
        for (int b = 0; b < DB; b++) {
          a32_f32x4 blk{0.f, 0.f, 0.f, 0.f};
          for (int hh = 0; hh < 4; hh++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
              const int key = k0 + 4 * hh + j;
              const bool see = in && key >= lo && key <= pos;
              const a32_f32x4 one = __builtin_amdgcn_mfma_f32_16x16x4f32(h == hh ? vv[b][j] : 0.f, h == hh ? p[j] : 0.f,
                                                                         a32_f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
              for (int r = 0; r < 4; r++) blk[r] = see ? blk[r] + one[r] : blk[r];
            }
#pragma unroll
          for (int r = 0; r < 4; r++) o[b][r] = sees ? fmaf(o[b][r], alpha, blk[r]) : o[b][r];
        }
      }
      if (sees) {
        l = l * alpha + part;
        m = m_new;
      }
    }
  }
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);
#pragma unroll
  for (int b = 0; b < DB; b++) *reinterpret_cast<a32_f32x4*>(obuf + (wave * 16 + i) * ROW + 16 * b + 4 * h) = o[b];
  if (h == 0) { ml[(wave * 16 + i) * 2] = m; ml[(wave * 16 + i) * 2 + 1] = l; }
  __syncthreads();
  // sixteen threads a column
  const int col = threadIdx.x >> 4, cw = tile * 16 + col;
  if (cw >= cols) return;
  float f[4], top = -INFINITY, sum = 0.f;
#pragma unroll
  for (int w = 0; w < 4; w++) top = fmaxf(top, ml[(w * 16 + col) * 2]);
#pragma unroll
  for (int w = 0; w < 4; w++) {
    const float mw = ml[(w * 16 + col) * 2];
    f[w] = mw == -INFINITY ? 0.f : expf(mw - top);
    sum = fmaf(ml[(w * 16 + col) * 2 + 1], f[w], sum);
  }
  float* dst = a.out + ((size_t)(cw / R) * a.nq + g * R + cw % R) * a.d;
  for (int j = (threadIdx.x & 15) * 4; j < a.d; j += 64) {
    a32_f32x4 x{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 4; w++) {
      const a32_f32x4 ow = *reinterpret_cast<const a32_f32x4*>(obuf + (w * 16 + col) * ROW + j);
#pragma unroll
      for (int r = 0; r < 4; r++) x[r] = ml[(w * 16 + col) * 2] == -INFINITY ? x[r] : fmaf(ow[r], f[w], x[r]);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) dst[j + r] = x[r] / sum;
  }
}

template <int DB>
static int attention_f32(const Attn32Args& a, hipStream_t stream) {
  constexpr int bytes = (4 * 16 * (16 * DB + 4) + 4 * 16 * 2) * (int)sizeof(float);
  static const hipError_t room = hipFuncSetAttribute((const void*)&attention_f32_kernel<DB>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  PICO_REQUIRE(room == hipSuccess, "pico_paged_attention_ref: %s", hipGetErrorString(room));
  const long long tiles = ((long long)a.T * (a.nq / a.nkv) + 15) / 16;
  attention_f32_kernel<DB><<<dim3((unsigned)tiles, a.nkv), 256, bytes, stream>>>(a);
  PICO_LAUNCH_CHECK();
  return 0;
}

extern "C" int pico_paged_attention_ref(const void* q, int q_stride, int dtype, const void* k_cache,
                                        const void* v_cache, const int* block_table, int max_pages,
                                        const int* positions, const int* token_seq, void* out, int T, int nq,
                                        int nkv, int d, int P, int window, float scale, int num_pages,
                                        hipStream_t stream) {
  PICO_REQUIRE(T >= 0 && nq > 0 && nkv > 0 && d > 0 && P > 0 && max_pages > 0 && num_pages > 0,
               "pico_paged_attention_ref: bad sizes");
  PICO_REQUIRE(nq % nkv == 0, "pico_paged_attention_ref: %d query heads are not a multiple of %d kv heads", nq, nkv);
  PICO_REQUIRE(d <= 256, "pico_paged_attention_ref: head size %d is larger than 256", d);
  PICO_REQUIRE(nq <= 65535, "pico_paged_attention_ref: too many heads");
  PICO_REQUIRE(q_stride >= nq * d, "pico_paged_attention_ref: query row stride too small");
  if (T == 0) return 0;
  if (dtype == PICO_DTYPE_F32 && d % 4 == 0 && P % 4 == 0 && ((uintptr_t)k_cache | (uintptr_t)v_cache) % 16 == 0 &&
      (long long)T * (nq / nkv) < (1LL << 30)) {
    const Attn32Args a{(const float*)q, (const float*)k_cache, (const float*)v_cache, block_table, positions, token_seq, (float*)out,
                       q_stride, max_pages, T, nq, nkv, d, P, window, num_pages, scale};
    return d <= 64 ? attention_f32<4>(a, stream) : d <= 128 ? attention_f32<8>(a, stream) : attention_f32<16>(a, stream);
  }
  dim3 grid(T, nq);
  const size_t lds = (size_t)(d + 64) * sizeof(float);
  if (dtype == PICO_DTYPE_F32)
    paged_attention_ref_kernel<float><<<grid, 64, lds, stream>>>(
        (const float*)q, q_stride, (const float*)k_cache, (const float*)v_cache, block_table, max_pages, positions,
        token_seq, (float*)out, nq, nkv, d, P, window, scale, num_pages);
  else if (dtype == PICO_DTYPE_BF16)
    paged_attention_ref_kernel<bf16_t><<<grid, 64, lds, stream>>>(
        (const bf16_t*)q, q_stride, (const bf16_t*)k_cache, (const bf16_t*)v_cache, block_table, max_pages,
        positions, token_seq, (bf16_t*)out, nq, nkv, d, P, window, scale, num_pages);
  else
    PICO_REQUIRE(false, "pico_paged_attention_ref: unknown dtype %d", dtype);
  PICO_LAUNCH_CHECK();
  return 0;
}
