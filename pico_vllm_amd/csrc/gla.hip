// Gated linear attention: a recurrent mixer whose state is a matrix per head.
//
//   per head, with key channels c and value channels v:
//     S_t[c][v] = alpha_t[c] * S_(t-1)[c][v] + k_t[c] * v_t[v]          (a decay per key channel)
//     o_t[v]    = sum_c S_t[c][v] * q_t[c] * qscale
//   alpha_t = sigmoid(z_t)^(1 / tau),  z_t = A2 (A1 h_t) + b           (a low-rank projection; A1 h_t comes with q, k, v)
//   out_t = rmsnorm_v(o_t) * w * silu(g_t)                             (every head by itself, one weight for all heads)
//   or out_t = rmsnorm(o_t) * w * sigmoid(g_t) with all heads of a token as one row (pico_gated_row_norm)
// Optionally q, k and v go through z sigmoid(z) as they are read, and a head's decay is a constant.
//
// The state lives in float32, one [heads, dk, dv] block per state slot; decays, their logarithms, the recurrence and
// the head norm are float32 whatever the storage type T of the projections.  Every sum runs in an order that depends
// on the sizes alone, so a token's output does not depend on how its sequence was cut into steps.
#include "common.h"

// log(sigmoid(z)) = -log(1 + e^-z), without overflow on either side; one logarithm and exponential serve both, as lanes of a
// wave that differ in sign would go through the two in turn.
__device__ __forceinline__ float log_sigmoid(float z) {
  const float l = log1pf(expf(-fabsf(z)));
  return z >= 0.f ? -l : z - l;
}

// ---------------------------------------------------------------------------
// Logarithm of the decay: out[t][c] = log(sigmoid(z)) / tau, z = sum_r a2[c][r] * x[t][r] + b[c].
// x: the low-rank activations (columns of a wider row, stride ldx); a2 [C, R]; b float32 [C].  grid (ceil(T / TOK), ceil(C / 256)),
// any C and R.  A thread makes one channel of TOK tokens, so that a2 is read once for them: 2,048 tokens, 768 channels of
// rank 32 13.7 us, 16.5 with a token a workgroup and a logarithm for either sign; few tokens keep one, to fill the chip.
// ---------------------------------------------------------------------------
#define GLA_DECAY_TOKENS 8
template <typename T, int TOK>
__global__ __launch_bounds__(256) void gla_decay_kernel(const T* __restrict__ x, int ldx, const T* __restrict__ a2,
                                                        const float* __restrict__ b, float inv_tau, float* __restrict__ out,
                                                        int tokens, int C, int R) {
  extern __shared__ float xs[];                         // [R][TOK]
  const int t0 = blockIdx.x * TOK, c = blockIdx.y * 256 + threadIdx.x;
  for (int i = threadIdx.x; i < R * TOK; i += blockDim.x) xs[i] = load_f32(x + (size_t)min(t0 + i % TOK, tokens - 1) * ldx + i / TOK);
  __syncthreads();
  if (c >= C) return;
  const T* w = a2 + (size_t)c * R;
  float z[TOK];
#pragma unroll
  for (int k = 0; k < TOK; k++) z[k] = b ? b[c] : 0.f;
  constexpr int V = 16 / sizeof(T);
  int r = 0;
  if (R % V == 0 && (uintptr_t)a2 % 16 == 0)            // a lane's row of a2 in whole aligned sixteens: its lines are asked for once
#pragma unroll 2
    for (; r < R; r += V) {
      alignas(16) T wv[V];
      *reinterpret_cast<uint4*>(wv) = *reinterpret_cast<const uint4*>(w + r);
#pragma unroll
      for (int i = 0; i < V; i++)
#pragma unroll
        for (int k = 0; k < TOK; k++) z[k] = fmaf(load_f32(wv + i), xs[(r + i) * TOK + k], z[k]);
    }
  for (; r < R; r++) {
    const float wr = load_f32(w + r);
#pragma unroll
    for (int k = 0; k < TOK; k++) z[k] = fmaf(wr, xs[r * TOK + k], z[k]);
  }
#pragma unroll
  for (int k = 0; k < TOK; k++) {
    if (t0 + k >= tokens) break;
    out[(size_t)(t0 + k) * C + c] = log_sigmoid(z[k]) * inv_tau;
  }
}

extern "C" int pico_gla_decay(const void* x, int ldx, int dtype, const void* a2, const float* b, float tau, float* out,
                              int T, int C, int R, hipStream_t stream) {
  PICO_REQUIRE(T >= 0 && C > 0 && R > 0 && ldx >= R && R <= 8192, "pico_gla_decay: bad sizes");
  PICO_REQUIRE((C + 255) / 256 <= 65535, "pico_gla_decay: sizes beyond the grid");
  PICO_REQUIRE(tau > 0.f, "pico_gla_decay: tau must be positive");
  if (T == 0) return 0;
  // blocks of tokens where they still fill the chip and their activations fit LDS
  const bool many = T >= 64 && R <= 1024;
  const int tok = many ? GLA_DECAY_TOKENS : 1;
  const size_t lds = (size_t)R * tok * sizeof(float);
  const dim3 grid((T + tok - 1) / tok, (C + 255) / 256);
#define DECAY(TT)                                                                                                            \
  do {                                                                                                                       \
    if (many) gla_decay_kernel<TT, GLA_DECAY_TOKENS><<<grid, 256, lds, stream>>>((const TT*)x, ldx, (const TT*)a2, b, 1.0f / tau, out, T, C, R); \
    else gla_decay_kernel<TT, 1><<<grid, 256, lds, stream>>>((const TT*)x, ldx, (const TT*)a2, b, 1.0f / tau, out, T, C, R);  \
  } while (0)
  if (dtype == PICO_DTYPE_F32) DECAY(float);
  else if (dtype == PICO_DTYPE_BF16) DECAY(bf16_t);
  else PICO_REQUIRE(false, "pico_gla_decay: unknown dtype %d", dtype);
#undef DECAY
  PICO_LAUNCH_CHECK();
  return 0;
}

// ---------------------------------------------------------------------------
// The recurrence, token by token.  grid (sequences, heads, ceil(dv / 64)); a workgroup owns 64 value channels of one head of
// one sequence; wave w of its NW owns key channels 32 w ..  A thread keeps a patch of 8 key by 4 value channels of the state in
// registers over all tokens of the step (lane l: values 4 (l mod 16) .., keys 8 (l / 16) ..), so that the 24 numbers of q, k
// and decays and the 4 of v that it reads of a token out of LDS serve 96 operations; the wave's four partial outputs of a
// value are added by lane swaps that leave each lane one value.  Tokens are taken TB (8 or 16) at a time: they are staged in
// LDS while the next block's travel from memory in registers; the waves' partial outputs meet in LDS and are summed in
// wave order.
// What bounds it is the vector pipe, 3 operations a state element and token (2 where no outputs are made); with one value
// and 32 key channels a lane it was LDS, which hands every lane its own copy of 96 numbers a token.  A prompt of 2,048 tokens,
// 12 heads of 64 x 128: chunks of 64 take 43 us with outputs and 26 without, before 81 and 48.
//
// Long portions are cut into chunks of `chunk` tokens that run side by side (the recurrence is linear in the state):
//   GLA_LOCAL:  every chunk from a state of zero, no outputs; leaves its state in ws[chunk] and the sum of its decays'
//               logarithms in ws_decay[chunk]
//   (gla_combine_kernel walks a sequence's chunks: ws[j] <- the state in front of chunk j, and the slot's final state)
//   GLA_FROM:   every chunk again from ws[chunk], writing the outputs
// GLA_WHOLE is the plain walk from the slot's state (a sequence is one chunk).  blockIdx.x = sequence * max_chunks + chunk.
// ---------------------------------------------------------------------------
typedef float f32x4 __attribute__((ext_vector_type(4)));

#define GLA_CPT 32
#define GLA_KEYS 8          // of a lane
#define GLA_WHOLE 0
#define GLA_LOCAL 1
#define GLA_FROM 2

// FUSED: the decays are made inside the walk (log_decay is null) instead of read.  FEW: blocks of two tokens.  wide: the states' rows are whole aligned fours.
template <typename T, int MODE, int NW, bool FUSED, bool FEW = false>
__global__ __launch_bounds__(64 * NW) void gla_scan_kernel(const T* __restrict__ x, int ldx, int q_col, int k_col, int v_col,
                                                       const float* __restrict__ log_decay,
                                                       const int* __restrict__ cu_seqlens,
                                                       const int* __restrict__ state_slots, float* __restrict__ state,
                                                       float* __restrict__ out, int H, int dk, int dv, float qscale,
                                                       int num_slots, int chunk, int max_chunks, float* __restrict__ ws,
                                                       float* __restrict__ ws_decay, const T* __restrict__ a2,
                                                       const float* __restrict__ a2_bias, int a_col, int R, float inv_tau,
                                                       const float* __restrict__ head_decay, int silu, int wide) {
  constexpr int TB = FEW ? 2 : NW <= 4 ? 16 : 8, CP = NW * GLA_CPT, NL = TB / 2, NV = TB / NW;
  __shared__ float qs[TB * CP], ks[TB * CP], as[TB * CP], vs[TB * 64], po[TB * NW * 64];
  // head_decay given: every key channel of head h decays by the constant head_decay[h] at every token (log_decay, a2
  // are not read); the decay is multiplied in as it is, no logarithm and exponential between
  const float fixed = head_decay ? head_decay[blockIdx.y] : 0.f;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int b = MODE == GLA_WHOLE ? blockIdx.x : blockIdx.x / max_chunks, h = blockIdx.y, v0 = blockIdx.z * 64;
  int t_begin = cu_seqlens[b], t_end = cu_seqlens[b + 1];
  if (MODE != GLA_WHOLE) {
    t_begin += (blockIdx.x % max_chunks) * chunk;
    t_end = min(t_end, t_begin + chunk);
  }
  const int slot = state_slots[b];
  if (slot < 0 || slot >= num_slots || t_end <= t_begin) return;
  const int live = (dk + GLA_CPT - 1) / GLA_CPT;        // waves that own key channels at all
  const int ck = (lane >> 4) * GLA_KEYS, c0 = wave * GLA_CPT + ck, vl = 4 * (lane & 15), v = v0 + vl;
  float* sp = MODE == GLA_WHOLE ? state + ((size_t)slot * H + h) * dk * dv : ws + ((size_t)blockIdx.x * H + h) * dk * dv;
  // Every load below is unconditional, from an address clamped into the tensor, and what must not count is cleared
  // afterwards: a load inside a branch is waited for inside that branch, and a thread's loads of a block then queue
  // one behind the other's latency instead of travelling together.
  f32x4 S[GLA_KEYS];
  if (MODE != GLA_LOCAL) {
    if (wide) {
#pragma unroll
      for (int c = 0; c < GLA_KEYS; c++) S[c] = *reinterpret_cast<const f32x4*>(sp + (size_t)min(c0 + c, dk - 1) * dv + min(v, dv - 4));
    } else {
#pragma unroll
      for (int c = 0; c < GLA_KEYS; c++)
#pragma unroll
        for (int j = 0; j < 4; j++) S[c][j] = sp[(size_t)min(c0 + c, dk - 1) * dv + min(v + j, dv - 1)];
    }
  }
#pragma unroll
  for (int c = 0; c < GLA_KEYS; c++)
#pragma unroll
    for (int j = 0; j < 4; j++) S[c][j] = (MODE != GLA_LOCAL && v + j < dv && c0 + c < dk) ? S[c][j] : 0.f;
  // A thread stages TB / 2 elements (tokens tt0, tt0 + 2, .., channel cc) of a block's q, k and decays and TB / NW of its v
  // (tokens wave, wave + NW, .., channel lane).  The next block's values travel in registers while this block is walked.
  const int tt0 = (int)threadIdx.x >= CP ? 1 : 0, cc = (int)threadIdx.x - tt0 * CP;
  T rq[NL], rk[NL], rv[NV];
  float ra[NL], decayed = 0.f;                          // (decayed: the logarithms of this thread's tokens in the chunk, added up)
  const int c_in = min(cc, dk - 1), v_in = min(v0 + lane, dv - 1);
  auto fetch = [&](int t0) {
    const int nb = min(TB, t_end - t0);
#pragma unroll
    for (int j = 0; j < NL; j++) {
      const int tt = min(tt0 + 2 * j, nb - 1);
      const T* row = x + (size_t)(t0 + tt) * ldx + (size_t)h * dk + c_in;
      rq[j] = MODE != GLA_LOCAL ? row[q_col] : row[k_col];
      rk[j] = row[k_col];
      if (head_decay) {
        ra[j] = 0.f;
      } else if (!FUSED) {
        ra[j] = log_decay[(size_t)(t0 + tt) * H * dk + (size_t)h * dk + c_in];
      } else if (tt0 + 2 * j >= nb) {
        ra[j] = 0.f;                                    // no such token in this block: nothing to work out
      } else {
        // the decay's logarithm made here from the low-rank activations (as gla_decay_kernel does): one launch less
        const T* xa = x + (size_t)(t0 + tt) * ldx + a_col;
        const T* w = a2 + ((size_t)h * dk + c_in) * R;
        float z = a2_bias ? a2_bias[h * dk + c_in] : 0.f;
        for (int r = 0; r < R; r++) z = fmaf(load_f32(w + r), load_f32(xa + r), z);
        ra[j] = log_sigmoid(z) * inv_tau;
      }
    }
#pragma unroll
    for (int j = 0; j < NV; j++) rv[j] = x[(size_t)(t0 + min(wave + j * NW, nb - 1)) * ldx + v_col + (size_t)h * dv + v_in];
  };
  fetch(t_begin);
  for (int t0 = t_begin; t0 < t_end; t0 += TB) {
    const int nb = min(TB, t_end - t0);
    __syncthreads();                                    // the last block's staged values and partial outputs have been read
#pragma unroll
    for (int j = 0; j < NL; j++) {
      const int tt = tt0 + 2 * j, i = tt * CP + cc;     // a workgroup has 2 CP threads
      const bool in = tt < nb && cc < dk;
      const float qv = load_f32(&rq[j]), kv = load_f32(&rk[j]);
      if (MODE != GLA_LOCAL) qs[i] = in ? (silu ? silu_f(qv) : qv) * qscale : 0.f;
      ks[i] = in ? (silu ? silu_f(kv) : kv) : 0.f;
      as[i] = in ? (head_decay ? fixed : expf(ra[j])) : 1.f;
      if (MODE == GLA_LOCAL) decayed += in ? ra[j] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < NV; j++) {
      const float x0 = load_f32(&rv[j]);
      vs[(wave + j * NW) * 64 + lane] = (wave + j * NW < nb && v0 + lane < dv) ? (silu ? silu_f(x0) : x0) : 0.f;
    }
    __syncthreads();
    if (t0 + TB < t_end) fetch(t0 + TB);
    auto token = [&](int tt) {
      const f32x4* a4 = reinterpret_cast<const f32x4*>(as + tt * CP + c0);
      const f32x4* k4 = reinterpret_cast<const f32x4*>(ks + tt * CP + c0);
      const f32x4* q4 = reinterpret_cast<const f32x4*>(qs + tt * CP + c0);
      const f32x4 vt = *reinterpret_cast<const f32x4*>(vs + tt * 64 + vl);
      float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < GLA_KEYS / 4; c++) {
        const f32x4 av = a4[c], kv = k4[c];
        f32x4 qv = {0.f, 0.f, 0.f, 0.f};
        if (MODE != GLA_LOCAL) qv = q4[c];
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
          for (int j = 0; j < 4; j++) {
            S[4 * c + i][j] = fmaf(av[i], S[4 * c + i][j], kv[i] * vt[j]);
            if (MODE != GLA_LOCAL) acc[j] = fmaf(S[4 * c + i][j], qv[i], acc[j]);
          }
      }
      if (MODE != GLA_LOCAL) {
        // lane (group g, l) is left with value 4 l + g of the four groups' sums
        const auto e = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[0]), __float_as_uint(acc[2]), false, false);
        const auto f = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[1]), __float_as_uint(acc[3]), false, false);
        const float e2 = __uint_as_float(e[0]) + __uint_as_float(e[1]), f2 = __uint_as_float(f[0]) + __uint_as_float(f[1]);
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(e2), __float_as_uint(f2), false, false);
        po[(tt * NW + wave) * 64 + vl + (lane >> 4)] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
      }
    };
    if (wave < live) {
      if (nb == TB) {                                   // whole blocks in one piece: a token's reads travel under the one before
#pragma unroll
        for (int tt = 0; tt < TB; tt++) token(tt);
      } else {
#pragma unroll 1
        for (int tt = 0; tt < nb; tt++) token(tt);
      }
    }
    if (MODE == GLA_LOCAL) continue;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NV; j++) {
      const int tt = wave + j * NW;
      float sum = 0.f;
      for (int w = 0; w < live; w++) sum += po[(tt * NW + w) * 64 + lane];
      if (tt < nb && v0 + lane < dv) out[(size_t)(t0 + tt) * H * dv + (size_t)h * dv + v0 + lane] = sum;
    }
  }
  if (MODE != GLA_FROM) {
    if (wide) {
#pragma unroll
      for (int c = 0; c < GLA_KEYS; c++)
        if (v < dv && c0 + c < dk) *reinterpret_cast<f32x4*>(sp + (size_t)(c0 + c) * dv + v) = S[c];
    } else {
#pragma unroll
      for (int c = 0; c < GLA_KEYS; c++)
#pragma unroll
        for (int j = 0; j < 4; j++)
          if (v + j < dv && c0 + c < dk) sp[(size_t)(c0 + c) * dv + v + j] = S[c][j];
    }
  }
  if (MODE == GLA_LOCAL && blockIdx.z == 0) {
    // the chunk's decays multiplied up, as the sum of their logarithms, for the walk over the chunks
    __syncthreads();
    if (tt0) as[cc] = decayed;
    __syncthreads();
    if (!tt0 && cc < dk)
      ws_decay[((size_t)blockIdx.x * H + h) * dk + cc] = head_decay ? (float)(t_end - t_begin) * logf(fixed) : decayed + as[cc];
  }
}

// The walk over a sequence's chunks, one thread per state element: ws[j] becomes the state in front of chunk j, the
// slot gets the state behind the last chunk.  grid (sequences, heads, ceil(dk dv / 256)).  32 chunks of 12 states of 64 x 128
// 10.3 us, with every chunk's state asked for in its turn 15.6.
#define GLA_AHEAD 8
__global__ __launch_bounds__(256) void gla_combine_kernel(const int* __restrict__ cu_seqlens,
                                                          const int* __restrict__ state_slots, float* __restrict__ state,
                                                          float* __restrict__ ws, const float* __restrict__ ws_decay, int H,
                                                          int dk, int dv, int num_slots, int chunk, int max_chunks) {
  const int b = blockIdx.x, h = blockIdx.y, e = blockIdx.z * 256 + threadIdx.x;
  if (e >= dk * dv) return;
  const int slot = state_slots[b], n = cu_seqlens[b + 1] - cu_seqlens[b];
  if (slot < 0 || slot >= num_slots || n <= 0) return;
  const int c = e / dv;
  float* sp = state + ((size_t)slot * H + h) * dk * dv + e;
  float S = *sp;
  const int chunks = (n + chunk - 1) / chunk;
  const size_t step = (size_t)H * dk * dv, step_d = (size_t)H * dk;
  float* w = ws + ((size_t)b * max_chunks * H + h) * dk * dv + e;
  const float* wd = ws_decay + ((size_t)b * max_chunks * H + h) * dk + c;
  // the next chunks' states and decays are asked for before the ones in hand are walked
  float local[GLA_AHEAD], decay[GLA_AHEAD];
  auto fetch = [&](int j0) {
#pragma unroll
    for (int a = 0; a < GLA_AHEAD; a++) {
      const int j = min(j0 + a, chunks - 1);
      local[a] = w[j * step];
      decay[a] = wd[j * step_d];
    }
  };
  fetch(0);
  for (int j0 = 0; j0 < chunks; j0 += GLA_AHEAD) {
    float L[GLA_AHEAD], D[GLA_AHEAD];
#pragma unroll
    for (int a = 0; a < GLA_AHEAD; a++) { L[a] = local[a]; D[a] = expf(decay[a]); }
    if (j0 + GLA_AHEAD < chunks) fetch(j0 + GLA_AHEAD);
#pragma unroll
    for (int a = 0; a < GLA_AHEAD; a++) {
      if (j0 + a >= chunks) break;
      w[(j0 + a) * step] = S;
      S = fmaf(D[a], S, L[a]);
    }
  }
  *sp = S;
}

// log_decay null (chunk == 0 only): the decays are made inside the walk from x[:, a_col : a_col + R], a2 [H dk, R] and
// a2_bias, as pico_gla_decay makes them.
// chunk == 0: every sequence walked whole from its slot.  chunk > 0: sequences cut into chunks of that many tokens that
// run side by side (three launches); ws float32 [num_seqs * max_chunks, H, dk, dv], ws_decay [num_seqs * max_chunks, H, dk],
// max_chunks at least the chunks of the longest sequence.
extern "C" int pico_gla_scan(const void* x, int ldx, int dtype, int q_col, int k_col, int v_col, const float* log_decay,
                             const int* cu_seqlens, const int* state_slots, float* state, float* out, int num_seqs,
                             int T, int H, int dk, int dv, float qscale, int num_slots, int chunk, int max_chunks,
                             float* ws, float* ws_decay, const void* a2, const float* a2_bias, int a_col, int R, float tau,
                             const float* head_decay, int silu, hipStream_t stream) {
  PICO_REQUIRE(head_decay != nullptr || log_decay != nullptr || (chunk == 0 && a2 != nullptr && R > 0 && a_col >= 0 && ldx >= a_col + R && tau > 0.f),
               "pico_gla_scan: without the decays' logarithms the walk needs what makes them, and runs whole");
  PICO_REQUIRE(num_seqs >= 0 && T >= 0 && H > 0 && dk > 0 && dv > 0 && num_slots > 0, "pico_gla_scan: bad sizes");
  PICO_REQUIRE(dk <= 8 * GLA_CPT, "pico_gla_scan: at most %d key channels a head, got %d", 8 * GLA_CPT, dk);
  PICO_REQUIRE(q_col >= 0 && k_col >= 0 && v_col >= 0 && ldx >= q_col + H * dk && ldx >= k_col + H * dk && ldx >= v_col + H * dv,
               "pico_gla_scan: the row of %d columns does not hold q, k and v", ldx);
  PICO_REQUIRE(H <= 65535 && (dv + 63) / 64 <= 65535 && (dk * dv + 255) / 256 <= 65535, "pico_gla_scan: sizes beyond the grid");
  PICO_REQUIRE(chunk == 0 || (chunk > 0 && max_chunks > 0 && ws != nullptr && ws_decay != nullptr &&
                              (long long)max_chunks * chunk >= T && (long long)num_seqs * max_chunks < (1ll << 31)),
               "pico_gla_scan: chunks need room for their states and must cover the step's tokens");
  if (num_seqs == 0 || T == 0) return 0;
  // A step of few tokens with one wave a workgroup: blocks of two tokens, so that a thread fetches next to nothing for tokens that
  // are not there.  (12 heads of 32 x 64, 8 requests of one token: 3.7 us, in blocks of 16 6.2.  With more waves a thread's share of a block
  // is smaller: 64 x 128 5.9, with a value and 32 keys a lane 6.1.)
  const bool few = chunk == 0 && T <= 2 * num_seqs;
  const int wide = dv % 4 == 0 && ((uintptr_t)state | (uintptr_t)ws) % 16 == 0, vb = (dv + 63) / 64;
#define GLA_ARGS(TT)                                                                                                       \
  (const TT*)x, ldx, q_col, k_col, v_col, log_decay, cu_seqlens, state_slots, state, out, H, dk, dv, qscale, num_slots,   \
      chunk, max_chunks, ws, ws_decay, (const TT*)a2, a2_bias, a_col, R, 1.0f / (tau > 0.f ? tau : 1.f), head_decay, silu, wide
#define GLA_WAVES(TT, MODE, GX, FUSED)                                                                                     \
  do {                                                                                                                     \
    if (dk <= 32 && few) gla_scan_kernel<TT, MODE, 1, FUSED, MODE == GLA_WHOLE><<<dim3(GX, H, vb), 64, 0, stream>>>(GLA_ARGS(TT)); \
    else if (dk <= 32) gla_scan_kernel<TT, MODE, 1, FUSED><<<dim3(GX, H, vb), 64, 0, stream>>>(GLA_ARGS(TT));                   \
    else if (dk <= 64) gla_scan_kernel<TT, MODE, 2, FUSED><<<dim3(GX, H, vb), 128, 0, stream>>>(GLA_ARGS(TT));             \
    else if (dk <= 128) gla_scan_kernel<TT, MODE, 4, FUSED><<<dim3(GX, H, vb), 256, 0, stream>>>(GLA_ARGS(TT));            \
    else gla_scan_kernel<TT, MODE, 8, FUSED><<<dim3(GX, H, vb), 512, 0, stream>>>(GLA_ARGS(TT));                           \
  } while (0)
#define GLA_LAUNCH(TT, MODE, GX)                                                                                           \
  do {                                                                                                                     \
    constexpr bool whole = MODE == GLA_WHOLE;                                                                              \
    if (log_decay == nullptr && head_decay == nullptr && whole) GLA_WAVES(TT, MODE, GX, whole);                            \
    else GLA_WAVES(TT, MODE, GX, false);                                                                                   \
  } while (0)
#define GLA_RUN(TT)                                                                                                        \
  if (chunk == 0) {                                                                                                        \
    GLA_LAUNCH(TT, GLA_WHOLE, num_seqs);                                                                                   \
  } else {                                                                                                                 \
    GLA_LAUNCH(TT, GLA_LOCAL, num_seqs * max_chunks);                                                                      \
    gla_combine_kernel<<<dim3(num_seqs, H, (dk * dv + 255) / 256), 256, 0, stream>>>(cu_seqlens, state_slots, state, ws,   \
                                                                                     ws_decay, H, dk, dv, num_slots, chunk, \
                                                                                     max_chunks);                          \
    GLA_LAUNCH(TT, GLA_FROM, num_seqs * max_chunks);                                                                       \
  }
  if (dtype == PICO_DTYPE_F32) {
    GLA_RUN(float)
  } else if (dtype == PICO_DTYPE_BF16) {
    GLA_RUN(bf16_t)
  } else {
    PICO_REQUIRE(false, "pico_gla_scan: unknown dtype %d", dtype);
  }
#undef GLA_RUN
#undef GLA_LAUNCH
#undef GLA_WAVES
#undef GLA_ARGS
  PICO_LAUNCH_CHECK();
  return 0;
}

// ---------------------------------------------------------------------------
// Head norm and gate: out[t][h][v] = o[t][h][v] / sqrt(mean_v(o^2) + eps) * w[v] * silu(g[t][h][v]).
// o float32 [T, H dv]; g: columns of a wider row of type T (stride ldg); out type T [T, H dv].  grid (T, H), one wave.
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(64) void gla_out_kernel(const float* __restrict__ o, const T* __restrict__ g, int ldg,
                                                     const float* __restrict__ w, float eps, T* __restrict__ out, int H,
                                                     int dv, int sigmoid_gate) {
  const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const float* orow = o + ((size_t)t * H + h) * dv;
  float ss = 0.f;
  for (int v = lane; v < dv; v += 64) ss = fmaf(orow[v], orow[v], ss);
  ss = wave_sum(ss);
  const float r = 1.0f / sqrtf(ss / (float)dv + eps);
  const T* grow = g + (size_t)t * ldg + (size_t)h * dv;
  T* dst = out + ((size_t)t * H + h) * dv;
  for (int v = lane; v < dv; v += 64) {
    const float gv = load_f32(grow + v);
    // the gate: silu(g), or sigmoid(g)
    store_f32(dst + v, orow[v] * r * w[v] * ((sigmoid_gate ? 1.0f : gv) / (1.0f + expf(-gv))));
  }
}

extern "C" int pico_gla_out(const float* o, const void* g, int ldg, int dtype, const float* w, float eps, void* out, int T,
                            int H, int dv, int sigmoid_gate, hipStream_t stream) {
  PICO_REQUIRE(T >= 0 && H > 0 && dv > 0 && ldg >= H * dv && H <= 65535, "pico_gla_out: bad sizes");
  if (T == 0) return 0;
  const dim3 grid(T, H);
  if (dtype == PICO_DTYPE_F32)
    gla_out_kernel<float><<<grid, 64, 0, stream>>>(o, (const float*)g, ldg, w, eps, (float*)out, H, dv, sigmoid_gate);
  else if (dtype == PICO_DTYPE_BF16)
    gla_out_kernel<bf16_t><<<grid, 64, 0, stream>>>(o, (const bf16_t*)g, ldg, w, eps, (bf16_t*)out, H, dv, sigmoid_gate);
  else
    PICO_REQUIRE(false, "pico_gla_out: unknown dtype %d", dtype);
  PICO_LAUNCH_CHECK();
  return 0;
}

// ---------------------------------------------------------------------------
// Norm over all heads of a token at once, and gate: out[t][i] = o[t][i] / sqrt(mean_i(o^2) + eps) * w[i] * sigmoid(g[t][i]).
// o float32 [T, N]; g: columns of a wider row of type T (stride ldg); out rows of type T (stride ldo).  One workgroup a
// token, its row in registers: thread i owns entries i, i + blockDim, ..; the number of threads goes with N alone.
// ---------------------------------------------------------------------------
#define ROW_NORM_VPT 8
template <typename T>
__global__ __launch_bounds__(1024) void gated_row_norm_kernel(const float* __restrict__ o, const T* __restrict__ g, int ldg,
                                                              const float* __restrict__ w, float eps, T* __restrict__ out,
                                                              int ldo, int N) {
  __shared__ float scratch[16];
  const int t = blockIdx.x;
  float v[ROW_NORM_VPT], gv[ROW_NORM_VPT], wv[ROW_NORM_VPT];
#pragma unroll
  for (int j = 0; j < ROW_NORM_VPT; j++) {
    if (j * (int)blockDim.x >= N) break;
    const int i = min(j * (int)blockDim.x + (int)threadIdx.x, N - 1);
    v[j] = o[(size_t)t * N + i];
    gv[j] = load_f32(g + (size_t)t * ldg + i);
    wv[j] = w[i];
  }
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < ROW_NORM_VPT; j++)
    if (j * (int)blockDim.x + (int)threadIdx.x < N) ss = fmaf(v[j], v[j], ss);
  const float r = 1.0f / sqrtf(block_sum(ss, scratch) / (float)N + eps);
#pragma unroll
  for (int j = 0; j < ROW_NORM_VPT; j++) {
    const int i = j * (int)blockDim.x + (int)threadIdx.x;
    if (i < N) store_f32(out + (size_t)t * ldo + i, v[j] * r * wv[j] / (1.0f + expf(-gv[j])));
  }
}

extern "C" int pico_gated_row_norm(const float* o, const void* g, int ldg, int dtype, const float* w, float eps, void* out,
                                   int ldo, int T, int N, hipStream_t stream) {
  PICO_REQUIRE(T >= 0 && N > 0 && ldg >= N && ldo >= N && eps > 0.f, "pico_gated_row_norm: bad sizes");
  PICO_REQUIRE(N <= 1024 * ROW_NORM_VPT, "pico_gated_row_norm: rows of at most %d entries, got %d", 1024 * ROW_NORM_VPT, N);
  if (T == 0) return 0;
  const int threads = N <= 256 ? 64 : N <= 2048 ? 256 : 1024;
  if (dtype == PICO_DTYPE_F32)
    gated_row_norm_kernel<float><<<T, threads, 0, stream>>>(o, (const float*)g, ldg, w, eps, (float*)out, ldo, N);
  else if (dtype == PICO_DTYPE_BF16)
    gated_row_norm_kernel<bf16_t><<<T, threads, 0, stream>>>(o, (const bf16_t*)g, ldg, w, eps, (bf16_t*)out, ldo, N);
  else
    PICO_REQUIRE(false, "pico_gated_row_norm: unknown dtype %d", dtype);
  PICO_LAUNCH_CHECK();
  return 0;
}
