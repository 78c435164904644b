// A selective state-space mixer: a short causal convolution per channel and a recurrence whose decay, input and
// output weights depend on the token.
//
//   xc[t][c] = act(bias[c] + sum_j w[j][c] * x[t - (taps - 1) + j][c])          zeros before a sequence's start; act is
//                                                                           silu, or nothing; w is kept tap by tap,
//                                                                           [taps, C]: neighbours read neighbours
//   dt[t][c] = softplus(dtp[t][c] + dt_bias[c]),   A[c][n] = -exp(A_log[c][n])
//   S[c][n] <- exp(dt A) S + dt xc[t][c] B[t][n];   y[t][c] = sum_n S[c][n] C[t][n] + D[c] xc[t][c]
//   out[t][c] = y[t][c] * silu(z[t][c])
//
// A request's state slot holds, per channel, the N elements of S and behind them the last taps - 1 inputs of the
// convolution (float32 [slots, channels, N + taps - 1]).  Step sizes, decays, the recurrence and its state are
// float32 whatever the storage type of the projections; every sum runs in an order that depends on the sizes alone.
#include "common.h"

#define SSM_MAX_TAPS 16

// what follows the convolution: silu, or nothing
__device__ __forceinline__ float conv_act(float v, int silu) { return silu ? silu_f(v) : v; }
// the decay exp(dt A) of an element: the library's exponential in the 32-bit engine; with bfloat16 storage the
// hardware's (exp2 of the argument times log2 e; the argument is at most 0, the relative error a few 1e-7)
template <typename T> __device__ __forceinline__ float decay_exp(float v);
template <> __device__ __forceinline__ float decay_exp<float>(float v) { return expf(v); }
template <> __device__ __forceinline__ float decay_exp<bf16_t>(float v) { return __expf(v); }

// grid (T, ceil(C / 256)): one thread per (token, channel).  Inputs before the portion come from the slot's history.
template <typename T>
__global__ __launch_bounds__(256) void causal_conv_kernel(const T* __restrict__ x, int ldx, const float* __restrict__ w,
                                                          const float* __restrict__ bias, const int* __restrict__ token_seq,
                                                          const int* __restrict__ cu_seqlens,
                                                          const int* __restrict__ state_slots, const float* __restrict__ state,
                                                          int num_slots, int C, int N, int taps, int silu, T* __restrict__ out) {
  const int t = blockIdx.x, c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= C) return;
  const int b = token_seq[t], first = cu_seqlens[b];
  const int slot = min(max(state_slots[b], 0), num_slots - 1);
  const float* hist = state + ((size_t)slot * C + c) * (N + taps - 1) + N;
  float acc = bias ? bias[c] : 0.f;
  for (int j = 0; j < taps; j++) {
    const int src = t - (taps - 1) + j;                 // token index of this tap's input
    const float v = src >= first ? load_f32(x + (size_t)src * ldx + c) : hist[(taps - 1) + (src - first)];
    acc = fmaf(w[(size_t)j * C + c], v, acc);
  }
  store_f32(out + (size_t)t * C + c, conv_act(acc, silu));
}

// The same for bfloat16 and up to four taps with four neighbouring channels (8-byte accesses; C and the row stride multiples of 4) and
// CONV_TOKENS neighbouring tokens a thread: the taps' weights, twice the bytes of the inputs they meet, are read once a thread, and a
// row once for all its taps, all of a thread's rows asked for at once.  grid (ceil(T / CONV_TOKENS), ceil(C / 4 / 64)).
// Bound by that one latency and the silu; eight channels or eight tokens a thread leave half the waves to hide it.  Microseconds with the
// history's launch, a token and eight channels a thread / 8 channels, 8 tokens / 4, 8 / 4, 4: 2,052 tokens of 3,328 channels 29 / 19 / 16 /
// 15; 1,377 of 3,072 21 / 16 / 12 / 11.
#define CONV_TOKENS 4
template <int TAPS>
__global__ __launch_bounds__(64) void causal_conv_rows_kernel(const bf16_t* __restrict__ x, int ldx, const float* __restrict__ w,
                                                              const float* __restrict__ bias, const int* __restrict__ token_seq,
                                                              const int* __restrict__ cu_seqlens,
                                                              const int* __restrict__ state_slots, const float* __restrict__ state,
                                                              int num_slots, int T, int C, int N, int silu, bf16_t* __restrict__ out) {
  constexpr int W = 4;
  const int t0 = blockIdx.x * CONV_TOKENS, c0 = (blockIdx.y * 64 + threadIdx.x) * W;
  if (c0 >= C) return;
  constexpr int ROWS = CONV_TOKENS + TAPS - 1;
  uint32_t raw[ROWS][W / 2];
#pragma unroll
  for (int r = 0; r < ROWS; r++) {
    const uint2 v = *reinterpret_cast<const uint2*>(x + (size_t)min(max(t0 - (TAPS - 1) + r, 0), T - 1) * ldx + c0);
    raw[r][0] = v.x; raw[r][1] = v.y;
  }
  float wt[TAPS][W], b[W];
#pragma unroll
  for (int i = 0; i < W; i++) b[i] = bias ? bias[c0 + i] : 0.f;
#pragma unroll
  for (int j = 0; j < TAPS; j++) {
    const float4 v = *reinterpret_cast<const float4*>(w + (size_t)j * C + c0);
    wt[j][0] = v.x; wt[j][1] = v.y; wt[j][2] = v.z; wt[j][3] = v.w;
  }
#pragma unroll
  for (int k = 0; k < CONV_TOKENS; k++) {
    const int t = t0 + k;
    if (t >= T) return;
    const int s = token_seq[t], first = cu_seqlens[s];
    float acc[W];
#pragma unroll
    for (int i = 0; i < W; i++) acc[i] = b[i];
#pragma unroll
    for (int j = 0; j < TAPS; j++) {
      const int src = t - (TAPS - 1) + j;
      float v[W];
#pragma unroll
      for (int i = 0; i < W; i += 2) {
        v[i] = __uint_as_float(raw[k + j][i / 2] << 16);
        v[i + 1] = __uint_as_float(raw[k + j][i / 2] & 0xffff0000u);
      }
      if (src < first) {                                   // (the same for the whole wave: a sequence's first tokens)
        const int slot = min(max(state_slots[s], 0), num_slots - 1);
#pragma unroll
        for (int i = 0; i < W; i++) v[i] = state[((size_t)slot * C + c0 + i) * (N + TAPS - 1) + N + (TAPS - 1) + (src - first)];
      }
#pragma unroll
      for (int i = 0; i < W; i++) acc[i] = fmaf(wt[j][i], v[i], acc[i]);
    }
    *reinterpret_cast<uint2*>(out + (size_t)t * C + c0) = make_uint2(pack2_bf16(conv_act(acc[0], silu), conv_act(acc[1], silu)),
                                                                    pack2_bf16(conv_act(acc[2], silu), conv_act(acc[3], silu)));
  }
}

// The same for bfloat16 with eight neighbouring channels a thread (16-byte accesses; C and the row stride multiples of 8).
// grid (T, ceil(C / 8 / 256)).
__global__ __launch_bounds__(256) void causal_conv8_kernel(const bf16_t* __restrict__ x, int ldx, const float* __restrict__ w,
                                                           const float* __restrict__ bias, const int* __restrict__ token_seq,
                                                           const int* __restrict__ cu_seqlens,
                                                           const int* __restrict__ state_slots, const float* __restrict__ state,
                                                           int num_slots, int C, int N, int taps, int silu, bf16_t* __restrict__ out) {
  const int t = blockIdx.x, c0 = (blockIdx.y * blockDim.x + threadIdx.x) * 8;
  if (c0 >= C) return;
  const int b = token_seq[t], first = cu_seqlens[b];
  const int slot = min(max(state_slots[b], 0), num_slots - 1);
  float acc[8];
#pragma unroll
  for (int i = 0; i < 8; i++) acc[i] = bias ? bias[c0 + i] : 0.f;
  for (int j = 0; j < taps; j++) {
    const int src = t - (taps - 1) + j;
    float v[8];
    if (src >= first) {
      const uint4 r = *reinterpret_cast<const uint4*>(x + (size_t)src * ldx + c0);
      v[0] = __uint_as_float(r.x << 16); v[1] = __uint_as_float(r.x & 0xffff0000u);
      v[2] = __uint_as_float(r.y << 16); v[3] = __uint_as_float(r.y & 0xffff0000u);
      v[4] = __uint_as_float(r.z << 16); v[5] = __uint_as_float(r.z & 0xffff0000u);
      v[6] = __uint_as_float(r.w << 16); v[7] = __uint_as_float(r.w & 0xffff0000u);
    } else {
#pragma unroll
      for (int i = 0; i < 8; i++) v[i] = state[((size_t)slot * C + c0 + i) * (N + taps - 1) + N + (taps - 1) + (src - first)];
    }
    const float4 w0 = *reinterpret_cast<const float4*>(w + (size_t)j * C + c0), w1 = *reinterpret_cast<const float4*>(w + (size_t)j * C + c0 + 4);
    acc[0] = fmaf(w0.x, v[0], acc[0]); acc[1] = fmaf(w0.y, v[1], acc[1]); acc[2] = fmaf(w0.z, v[2], acc[2]); acc[3] = fmaf(w0.w, v[3], acc[3]);
    acc[4] = fmaf(w1.x, v[4], acc[4]); acc[5] = fmaf(w1.y, v[5], acc[5]); acc[6] = fmaf(w1.z, v[6], acc[6]); acc[7] = fmaf(w1.w, v[7], acc[7]);
  }
  uint4 o;
  o.x = pack2_bf16(conv_act(acc[0], silu), conv_act(acc[1], silu));
  o.y = pack2_bf16(conv_act(acc[2], silu), conv_act(acc[3], silu));
  o.z = pack2_bf16(conv_act(acc[4], silu), conv_act(acc[5], silu));
  o.w = pack2_bf16(conv_act(acc[6], silu), conv_act(acc[7], silu));
  *reinterpret_cast<uint4*>(out + (size_t)t * C + c0) = o;
}

// grid (sequences, ceil(C / 256)): the slot's history becomes the last taps - 1 inputs behind this step's tokens.
template <typename T>
__global__ __launch_bounds__(256) void conv_history_kernel(const T* __restrict__ x, int ldx, const int* __restrict__ cu_seqlens,
                                                           const int* __restrict__ state_slots, float* __restrict__ state,
                                                           int num_slots, int C, int N, int taps) {
  const int b = blockIdx.x, c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= C) return;
  const int first = cu_seqlens[b], n = cu_seqlens[b + 1] - first, slot = state_slots[b];
  if (n <= 0 || slot < 0 || slot >= num_slots) return;
  float* hist = state + ((size_t)slot * C + c) * (N + taps - 1) + N;
  float keep[SSM_MAX_TAPS];
  for (int k = 0; k < taps - 1; k++) {
    const int at = n + k;                               // index in [old history | this step's inputs]
    keep[k] = at < taps - 1 ? hist[at] : load_f32(x + (size_t)(first + at - (taps - 1)) * ldx + c);
  }
  for (int k = 0; k < taps - 1; k++) hist[k] = keep[k];
}

// Every sequence brings ONE token (a decode step): convolution and history in one launch, a thread per (sequence,
// channel), which reads its history before it writes it.  grid (sequences, ceil(C / 256)).
template <typename T>
__global__ __launch_bounds__(256) void causal_conv_step_kernel(const T* __restrict__ x, int ldx, const float* __restrict__ w,
                                                               const float* __restrict__ bias, const int* __restrict__ cu_seqlens,
                                                               const int* __restrict__ state_slots, float* __restrict__ state,
                                                               int num_slots, int C, int N, int taps, int silu, T* __restrict__ out) {
  const int b = blockIdx.x, c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= C) return;
  const int t = cu_seqlens[b], slot = state_slots[b];
  if (cu_seqlens[b + 1] != t + 1 || slot < 0 || slot >= num_slots) return;
  float* hist = state + ((size_t)slot * C + c) * (N + taps - 1) + N;
  const float xv = load_f32(x + (size_t)t * ldx + c);
  float acc = bias ? bias[c] : 0.f;
  float keep[SSM_MAX_TAPS];
  for (int j = 0; j < taps - 1; j++) {
    keep[j] = hist[j];
    acc = fmaf(w[(size_t)j * C + c], keep[j], acc);
  }
  acc = fmaf(w[(size_t)(taps - 1) * C + c], xv, acc);
  for (int j = 0; j + 1 < taps - 1; j++) hist[j] = keep[j + 1];
  if (taps > 1) hist[taps - 2] = xv;
  store_f32(out + (size_t)t * C + c, conv_act(acc, silu));
}

extern "C" int pico_causal_conv(const void* x, int ldx, int dtype, const float* w, const float* bias, const int* token_seq,
                                const int* cu_seqlens, const int* state_slots, float* state, int num_slots, int T, int B,
                                int C, int N, int taps, void* out, int single, int silu, hipStream_t stream) {
  PICO_REQUIRE(T >= 0 && B >= 0 && C > 0 && N >= 0 && taps >= 1 && taps <= SSM_MAX_TAPS && ldx >= C && num_slots > 0,
               "pico_causal_conv: bad sizes (1 to %d taps)", SSM_MAX_TAPS);
  if (T == 0 || B == 0) return 0;
  const int cb = (C + 255) / 256;
  PICO_REQUIRE(cb <= 65535, "pico_causal_conv: too many channels");
  if (single) {               // one token a sequence (the caller says so; a sequence of another length is left alone)
    PICO_REQUIRE(T == B, "pico_causal_conv: a step of single tokens has as many tokens as sequences");
    if (dtype == PICO_DTYPE_F32)
      causal_conv_step_kernel<float><<<dim3(B, cb), 256, 0, stream>>>((const float*)x, ldx, w, bias, cu_seqlens, state_slots, state,
                                                                      num_slots, C, N, taps, silu, (float*)out);
    else if (dtype == PICO_DTYPE_BF16)
      causal_conv_step_kernel<bf16_t><<<dim3(B, cb), 256, 0, stream>>>((const bf16_t*)x, ldx, w, bias, cu_seqlens, state_slots, state,
                                                                       num_slots, C, N, taps, silu, (bf16_t*)out);
    else
      PICO_REQUIRE(false, "pico_causal_conv: unknown dtype %d", dtype);
    PICO_LAUNCH_CHECK();
    return 0;
  }
  if (dtype == PICO_DTYPE_F32) {
    causal_conv_kernel<float><<<dim3(T, cb), 256, 0, stream>>>((const float*)x, ldx, w, bias, token_seq, cu_seqlens, state_slots,
                                                               state, num_slots, C, N, taps, silu, (float*)out);
    if (taps > 1)
      conv_history_kernel<float><<<dim3(B, cb), 256, 0, stream>>>((const float*)x, ldx, cu_seqlens, state_slots, state, num_slots, C, N, taps);
  } else if (dtype == PICO_DTYPE_BF16) {
    // Few entries are a thread's latency, which a token and a channel a thread keeps shortest: one chain of loads, and not four tokens
    // one behind the other where sequences begin.  Microseconds, that / four tokens and channels, four taps: 8 requests of a token
    // 5.4 / 8.6 (3,072 channels); 200 tokens of 3,072 7.3 / 7.3, 300 7.9 / 7.4, 700 14.9 / 8.5; 300 of 1,664 6.7 / 6.9, 500 7.6 / 7.0; 64 of
    // 7,168 8.2 / 8.0, 96 8.5 / 7.6; 1,000 of 512 6.2 / 6.7, 1,377 7.2 / 6.6: they meet at 0.6 million entries.  More taps than four, that /
    // eight channels a thread: 5 taps, 500 tokens of 3,072 12.1 / 14.6, 700 18.5 / 17.6, 1,377 34 / 23; 8 taps, 1,000 of 1,664 23 / 21, 700
    // 14 / 17, 300 of 7,168 30 / 27; 12 taps, 1,377 of 3,072 61 / 40.
    const long long entries = (long long)T * C;
    if (entries >= 600000 && C % 4 == 0 && ldx % 4 == 0 && taps >= 2 && taps <= 4 && ((uintptr_t)x | (uintptr_t)out) % 8 == 0 && (uintptr_t)w % 16 == 0) {
      const dim3 grid((T + CONV_TOKENS - 1) / CONV_TOKENS, (C / 4 + 63) / 64);
      PICO_REQUIRE(grid.y <= 65535, "pico_causal_conv: too many channels");
#define CONV_ROWS(TAPS) causal_conv_rows_kernel<TAPS><<<grid, 64, 0, stream>>>((const bf16_t*)x, ldx, w, bias, token_seq, cu_seqlens, state_slots, \
                                                                             state, num_slots, T, C, N, silu, (bf16_t*)out)
      if (taps == 4) CONV_ROWS(4);
      else if (taps == 3) CONV_ROWS(3);
      else CONV_ROWS(2);
#undef CONV_ROWS
    } else if (taps > 4 && entries >= (taps < 8 ? 2000000 : 1600000) && C % 8 == 0 && ldx % 8 == 0 && ((uintptr_t)x | (uintptr_t)out | (uintptr_t)w) % 16 == 0) {
      causal_conv8_kernel<<<dim3(T, (C / 8 + 255) / 256), 256, 0, stream>>>((const bf16_t*)x, ldx, w, bias, token_seq, cu_seqlens,
                                                                            state_slots, state, num_slots, C, N, taps, silu, (bf16_t*)out);
    } else {
      causal_conv_kernel<bf16_t><<<dim3(T, cb), 256, 0, stream>>>((const bf16_t*)x, ldx, w, bias, token_seq, cu_seqlens, state_slots,
                                                                  state, num_slots, C, N, taps, silu, (bf16_t*)out);
    }
    if (taps > 1)
      conv_history_kernel<bf16_t><<<dim3(B, cb), 256, 0, stream>>>((const bf16_t*)x, ldx, cu_seqlens, state_slots, state, num_slots, C, N, taps);
  } else {
    PICO_REQUIRE(false, "pico_causal_conv: unknown dtype %d", dtype);
  }
  PICO_LAUNCH_CHECK();
  return 0;
}

// ---------------------------------------------------------------------------
// The recurrence.  grid (sequences, ceil(C / channels a workgroup)); LPC lanes (a power of two: 1 up to 16 state
// elements, so that a lane owns at most 16) share a channel, lane l of them owns state elements l, l + LPC, .. (NPL of
// them); the sum over n is a lane's chain and then a butterfly over the LPC lanes.  Tokens are taken SSM_TB at a time:
// a thread's own values (its channel's input, step size and gate: neighbouring threads read neighbouring channels)
// travel together in registers, and the tokens' B and C rows, which all channels share, are staged in LDS.
// ---------------------------------------------------------------------------
#define SSM_TB 16
#define SSM_WHOLE 0
#define SSM_LOCAL 1
#define SSM_FROM 2

// Long portions are cut into chunks of `chunk` tokens that run side by side (the recurrence is linear in the state):
//   SSM_LOCAL: every chunk from a state of zero, no outputs; leaves its state in ws[chunk] and the sum of its step
//              sizes in ws_dt[chunk] (the chunk's decay of element n is exp(A[c][n] * that sum))
//   (ssm_combine_kernel walks a sequence's chunks: ws[j] <- the state in front of chunk j, and the slot's final state)
//   SSM_FROM:  every chunk again from ws[chunk], writing the outputs
// SSM_WHOLE is the plain walk from the slot's state.  blockIdx.x = sequence * max_chunks + chunk.
template <typename T, int NPL, int MODE>
__global__ __launch_bounds__(256) void selective_scan_kernel(const T* __restrict__ xc, const float* __restrict__ dtp,
                                                             const float* __restrict__ dt_bias, const T* __restrict__ bc,
                                                             int ldbc, int b_col, int c_col, const float* __restrict__ A_log,
                                                             const float* __restrict__ D, const T* __restrict__ z, int ldz,
                                                             const int* __restrict__ cu_seqlens,
                                                             const int* __restrict__ state_slots, float* __restrict__ state,
                                                             int num_slots, int C, int N, int hist, int LPC,
                                                             T* __restrict__ out, int chunk, int max_chunks,
                                                             float* __restrict__ ws, float* __restrict__ ws_dt) {
  extern __shared__ float bcs[];                         // [SSM_TB][2 N]: the block's B and C rows, shared by all channels
  const int b = MODE == SSM_WHOLE ? blockIdx.x : blockIdx.x / max_chunks;
  const int per = blockDim.x / LPC;                      // channels a workgroup
  const int c = blockIdx.y * per + threadIdx.x / LPC, l = threadIdx.x % LPC;
  int t_begin = cu_seqlens[b], t_end = cu_seqlens[b + 1];
  const int slot = state_slots[b];
  if (MODE != SSM_WHOLE) {
    t_begin += (blockIdx.x % max_chunks) * chunk;
    t_end = min(t_end, t_begin + chunk);
  }
  if (slot < 0 || slot >= num_slots || t_end <= t_begin) return;      // the whole workgroup alike
  const bool c_ok = c < C;
  const int ci = min(c, C - 1);
  float* sp = MODE == SSM_WHOLE ? state + ((size_t)slot * C + ci) * (N + hist) : ws + ((size_t)blockIdx.x * C + ci) * N;
  float S[NPL], A[NPL];
  int ni[NPL];
  bool n_ok[NPL];
#pragma unroll
  for (int j = 0; j < NPL; j++) {
    const int n = l + j * LPC;
    n_ok[j] = n < N;
    ni[j] = min(n, N - 1);
    S[j] = (MODE != SSM_LOCAL && n_ok[j]) ? sp[ni[j]] : 0.f;
    A[j] = -expf(A_log[(size_t)ci * N + ni[j]]);
  }
  const float bias = dt_bias[ci], Dc = D[ci];
  float dt_sum = 0.f;
  for (int t0 = t_begin; t0 < t_end; t0 += SSM_TB) {
    const int nb = min(SSM_TB, t_end - t0);
    // a thread's own values of the block's tokens travel while the B and C rows are staged
    float xv[SSM_TB], dv[SSM_TB], zv[SSM_TB];
#pragma unroll
    for (int k = 0; k < SSM_TB; k++) {
      const size_t t = (size_t)(t0 + min(k, nb - 1));
      xv[k] = load_f32(xc + t * C + ci);
      dv[k] = dtp[t * C + ci];
      zv[k] = MODE != SSM_LOCAL ? load_f32(z + t * ldz + ci) : 0.f;
    }
    __syncthreads();                                     // the last block's rows have been read
    for (int i = threadIdx.x; i < nb * 2 * N; i += blockDim.x) {
      const int k = i / (2 * N), e = i % (2 * N);
      bcs[i] = load_f32(bc + (size_t)(t0 + k) * ldbc + (e < N ? b_col + e : c_col + e - N));
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < SSM_TB; k++) {
      if (k >= nb) break;
      const float pre = dv[k] + bias;
      const float dt = pre > 20.f ? pre : log1pf(expf(pre));
      const float dx = dt * xv[k];
      dt_sum += dt;
      const float* Bk = bcs + k * 2 * N;
      float y = 0.f;
#pragma unroll
      for (int j = 0; j < NPL; j++) {
        S[j] = n_ok[j] ? fmaf(decay_exp<T>(dt * A[j]), S[j], dx * Bk[ni[j]]) : 0.f;
        if (MODE != SSM_LOCAL) y = fmaf(S[j], Bk[N + ni[j]], y);
      }
      if (MODE != SSM_LOCAL) {
        for (int off = LPC >> 1; off > 0; off >>= 1) y += __shfl_xor(y, off, 64);
        if (l == 0 && c_ok) store_f32(out + (size_t)(t0 + k) * C + c, fmaf(Dc, xv[k], y) * silu_f(zv[k]));
      }
    }
  }
  if (c_ok && MODE != SSM_FROM) {
#pragma unroll
    for (int j = 0; j < NPL; j++)
      if (n_ok[j]) sp[ni[j]] = S[j];
    if (MODE == SSM_LOCAL && l == 0) ws_dt[(size_t)blockIdx.x * C + c] = dt_sum;
  }
}

// The two passes over chunks for 16 state elements a channel and bfloat16, a channel a lane.  A chunk's B and C rows are staged in
// LDS once, as floats, and read back four at a time; a lane's own values travel eight tokens ahead of their use; the first pass
// leaves the step sizes (softplus: a quarter of its instructions) for the second.  LOCAL: dt_ws is written, FROM: read.
// Chunks are numbered through: a sequence's first is scan16_first of its number and its first token, which leaves room for the
// last chunk of each sequence to be partly empty and makes T / chunk + sequences of them at most.
// 1,377 tokens of 3,072 channels: 36 and 27 us in chunks of 33 tokens, where the general kernel (rows and values fetched 16 tokens at
// a time, one wave a SIMD in chunks of 64) took 87 and 106; bound by the vector units (an exponential and three multiplications
// an element, the softplus) at two waves a SIMD.  The step sizes stay the library's log1p(e^x): a form from the
// hardware's exponential and logarithm took 11 us less and was off by 6e-8 instead of 3.3e-8 in the mean.
#define SSM_AHEAD 8
__device__ __forceinline__ int scan16_first(int b, int first_token, int chunk) { return first_token / chunk + b; }
template <int MODE>
__global__ __launch_bounds__(256) void scan16_kernel(const bf16_t* __restrict__ xc, const float* __restrict__ dtp,
                                                     const float* __restrict__ dt_bias, const bf16_t* __restrict__ bc, int ldbc,
                                                     int b_col, int c_col, const float* __restrict__ A_log,
                                                     const float* __restrict__ D, const bf16_t* __restrict__ z, int ldz,
                                                     const int* __restrict__ cu_seqlens, const int* __restrict__ state_slots,
                                                     int num_slots, int C, bf16_t* __restrict__ out, int chunk, int num_seqs,
                                                     float* __restrict__ ws, float* __restrict__ ws_dt, float* __restrict__ dt_ws) {
  constexpr int N = 16;
  extern __shared__ __attribute__((aligned(16))) float rows[];            // [chunk][B, and C for the second pass]
  constexpr int ROW = MODE == SSM_LOCAL ? N : 2 * N;
  const int c = blockIdx.y * 256 + threadIdx.x, ci = min(c, C - 1);
  // the last sequence whose first chunk is not behind this one, 64 sequences at a time, one a lane
  int b = 0;
  for (int b0 = 0; b0 < num_seqs; b0 += 64) {
    const int bl = b0 + (int)(threadIdx.x & 63);
    const unsigned long long here = __builtin_amdgcn_ballot_w64(bl < num_seqs && scan16_first(bl, cu_seqlens[min(bl, num_seqs - 1)], chunk) <= (int)blockIdx.x);
    if (here) b = b0 + 63 - __builtin_clzll(here);
  }
  b = __builtin_amdgcn_readfirstlane(b);
  const int slot = state_slots[b], t_first = cu_seqlens[b];
  const int t_begin = t_first + ((int)blockIdx.x - scan16_first(b, t_first, chunk)) * chunk, t_end = min(cu_seqlens[b + 1], t_begin + chunk);
  if (slot < 0 || slot >= num_slots || t_end <= t_begin) return;         // the whole workgroup alike
  const int n = t_end - t_begin;
  const bool c_ok = c < C;
  float* sp = ws + ((size_t)blockIdx.x * C + ci) * N;
  float xv[2][SSM_AHEAD], dv[2][SSM_AHEAD], zv[2][SSM_AHEAD];
  auto fetch = [&](int set, int k0) {
#pragma unroll
    for (int k = 0; k < SSM_AHEAD; k++) {
      const size_t t = (size_t)(t_begin + min(k0 + k, n - 1));
      xv[set][k] = load_f32(xc + t * C + ci);
      dv[set][k] = (MODE == SSM_LOCAL ? dtp : dt_ws)[t * C + ci];
      zv[set][k] = MODE == SSM_FROM ? load_f32(z + t * ldz + ci) : 0.f;
    }
  };
  fetch(0, 0);
  float S[N], A[N];
#pragma unroll
  for (int j = 0; j < N; j += 4) {
    const float4 a = *reinterpret_cast<const float4*>(A_log + (size_t)ci * N + j);
    A[j] = a.x; A[j + 1] = a.y; A[j + 2] = a.z; A[j + 3] = a.w;
    const float4 v = MODE == SSM_FROM ? *reinterpret_cast<const float4*>(sp + j) : make_float4(0.f, 0.f, 0.f, 0.f);
    S[j] = v.x; S[j + 1] = v.y; S[j + 2] = v.z; S[j + 3] = v.w;
  }
  for (int i = threadIdx.x; i < n * ROW; i += 256) {
    const int k = i / ROW, e = i % ROW;
    rows[i] = load_f32(bc + (size_t)(t_begin + k) * ldbc + (e < N ? b_col + e : c_col + e - N));
  }
#pragma unroll
  for (int j = 0; j < N; j++) A[j] = -expf(A[j]) * 1.4426950408889634f;    // decays through 2^x
  const float bias = dt_bias[ci], Dc = D[ci];
  float dt_sum = 0.f;
  __syncthreads();
  auto token = [&](int k, float x, float d, float g) {
    const size_t t = (size_t)(t_begin + k);
    float dt = d;
    if (MODE == SSM_LOCAL) {
      const float pre = d + bias;
      dt = pre > 20.f ? pre : log1pf(expf(pre));
      dt_sum += dt;
      if (c_ok) dt_ws[t * C + c] = dt;
    }
    const float dx = dt * x;
    const float4* r = reinterpret_cast<const float4*>(rows + k * ROW);
    float y = 0.f;
#pragma unroll
    for (int j = 0; j < N; j += 4) {
      const float4 B = r[j / 4];
      S[j] = fmaf(__builtin_amdgcn_exp2f(dt * A[j]), S[j], dx * B.x);
      S[j + 1] = fmaf(__builtin_amdgcn_exp2f(dt * A[j + 1]), S[j + 1], dx * B.y);
      S[j + 2] = fmaf(__builtin_amdgcn_exp2f(dt * A[j + 2]), S[j + 2], dx * B.z);
      S[j + 3] = fmaf(__builtin_amdgcn_exp2f(dt * A[j + 3]), S[j + 3], dx * B.w);
      if (MODE == SSM_FROM) {
        const float4 Cr = r[N / 4 + j / 4];
        y = fmaf(S[j + 3], Cr.w, fmaf(S[j + 2], Cr.z, fmaf(S[j + 1], Cr.y, fmaf(S[j], Cr.x, y))));
      }
    }
    if (MODE == SSM_FROM && c_ok) out[t * C + c] = f32_to_bf16(fmaf(Dc, x, y) * silu_f(g));
  };
  for (int k0 = 0; k0 < n; k0 += 2 * SSM_AHEAD) {
    fetch(1, k0 + SSM_AHEAD);
#pragma unroll
    for (int k = 0; k < SSM_AHEAD; k++)
      if (k0 + k < n) token(k0 + k, xv[0][k], dv[0][k], zv[0][k]);
    fetch(0, k0 + 2 * SSM_AHEAD);
#pragma unroll
    for (int k = 0; k < SSM_AHEAD; k++)
      if (k0 + SSM_AHEAD + k < n) token(k0 + SSM_AHEAD + k, xv[1][k], dv[1][k], zv[1][k]);
  }
  if (MODE == SSM_LOCAL && c_ok) {
#pragma unroll
    for (int j = 0; j < N; j += 4) *reinterpret_cast<float4*>(sp + j) = make_float4(S[j], S[j + 1], S[j + 2], S[j + 3]);
    ws_dt[(size_t)blockIdx.x * C + c] = dt_sum;
  }
}

// The walk over a sequence's chunks, one thread per state element: ws[j] becomes the state in front of chunk j, the
// slot gets the state behind the last chunk.  grid (sequences, ceil(C N / 256)).  through: chunks are numbered as scan16_first says.
__global__ __launch_bounds__(256) void ssm_combine_kernel(const int* __restrict__ cu_seqlens, const int* __restrict__ state_slots,
                                                          float* __restrict__ state, float* __restrict__ ws,
                                                          const float* __restrict__ ws_dt, const float* __restrict__ A_log,
                                                          int num_slots, int C, int N, int hist, int chunk, int max_chunks, int through) {
  const int b = blockIdx.x, e = blockIdx.y * 256 + threadIdx.x;
  if (e >= C * N) return;
  const int slot = state_slots[b], n_tok = cu_seqlens[b + 1] - cu_seqlens[b];
  if (slot < 0 || slot >= num_slots || n_tok <= 0) return;
  const int c = e / N, n = e % N;
  const float A = -expf(A_log[e]);
  float* sp = state + ((size_t)slot * C + c) * (N + hist) + n;
  float S = *sp;
  const int chunks = (n_tok + chunk - 1) / chunk;
  const size_t first = through ? (size_t)scan16_first(b, cu_seqlens[b], chunk) : (size_t)b * max_chunks;
  if (chunks <= 2) {                                     // (single tokens: nothing that is not used is asked for)
    for (int j = 0; j < chunks; j++) {
      const size_t at = first + j;
      const float local = ws[(at * C + c) * N + n], sum = ws_dt[at * C + c];
      ws[(at * C + c) * N + n] = S;
      S = fmaf(expf(A * sum), S, local);
    }
    *sp = S;
    return;
  }
  // the values of sixteen chunks at a time, those of the next sixteen on their way: one after the other, a chunk would cost a
  // memory latency (a store stands between the loads)
  constexpr int AHEAD = 16;
  float local[2][AHEAD], sum[2][AHEAD];
  auto fetch = [&](int set, int j0) {
#pragma unroll
    for (int k = 0; k < AHEAD; k++) {
      const size_t at = first + min(j0 + k, chunks - 1);
      local[set][k] = ws[(at * C + c) * N + n];
      sum[set][k] = ws_dt[at * C + c];
    }
  };
  auto walk = [&](int set, int j0) {
#pragma unroll
    for (int k = 0; k < AHEAD; k++) {
      if (j0 + k >= chunks) break;
      ws[((first + j0 + k) * C + c) * N + n] = S;
      S = fmaf(expf(A * sum[set][k]), S, local[set][k]);
    }
  };
  fetch(0, 0);
  for (int j0 = 0; j0 < chunks; j0 += 2 * AHEAD) {
    if (j0 + AHEAD < chunks) fetch(1, j0 + AHEAD);
    walk(0, j0);
    if (j0 + 2 * AHEAD < chunks) fetch(0, j0 + 2 * AHEAD);
    if (j0 + AHEAD < chunks) walk(1, j0 + AHEAD);
  }
  *sp = S;
}

// chunk == 0: every sequence walked whole from its slot.  chunk > 0: sequences cut into chunks of that many tokens that
// run side by side (three launches); ws float32 [num_seqs * max_chunks, C, N], ws_dt [num_seqs * max_chunks, C],
// max_chunks at least the chunks of the longest sequence.  dt_ws [T, C] chooses the passes for 16 state elements and bfloat16, for
// which ws and ws_dt hold T / chunk + num_seqs chunks, numbered through; null: the general kernels.
extern "C" int pico_selective_scan(const void* xc, const float* dtp, const float* dt_bias, const void* bc, int ldbc, int b_col,
                                   int c_col, const float* A_log, const float* D, const void* z, int ldz, int dtype,
                                   const int* cu_seqlens, const int* state_slots, float* state, int num_slots, int B, int T,
                                   int C, int N, int hist, void* out, int chunk, int max_chunks, float* ws, float* ws_dt,
                                   float* dt_ws, hipStream_t stream) {
  PICO_REQUIRE(B >= 0 && T >= 0 && C > 0 && N > 0 && N <= 256 && hist >= 0 && num_slots > 0 && ldz >= C &&
                   b_col >= 0 && c_col >= 0 && ldbc >= b_col + N && ldbc >= c_col + N,
               "pico_selective_scan: bad sizes (at most 256 state elements a channel)");
  PICO_REQUIRE(chunk == 0 || (chunk > 0 && max_chunks > 0 && ws != nullptr && ws_dt != nullptr &&
                              (long long)max_chunks * chunk >= T && (long long)B * max_chunks < (1ll << 31)),
               "pico_selective_scan: chunks need room for their states and must cover the step's tokens");
  if (B == 0 || T == 0) return 0;
  int lpc = 1;
  while (lpc * 16 < N) lpc *= 2;                         // up to 16 state elements a lane
  const int need = (N + lpc - 1) / lpc;
  const int npl = need <= 1 ? 1 : need <= 2 ? 2 : need <= 4 ? 4 : need <= 8 ? 8 : 16;
  const size_t lds = (size_t)SSM_TB * 2 * N * sizeof(float);
  const int per = 256 / lpc;
  const int gy = (C + per - 1) / per;
  PICO_REQUIRE(gy <= 65535 && ((long long)C * N + 255) / 256 <= 65535, "pico_selective_scan: too many channels");
  if (dt_ws != nullptr) {
    // (no way back to the general kernels: they number the chunks otherwise, and need room for more of them)
    PICO_REQUIRE(dtype == PICO_DTYPE_BF16 && N == 16 && chunk > 0 && chunk <= 256 && ((uintptr_t)A_log | (uintptr_t)ws) % 16 == 0,
                 "pico_selective_scan: chunks numbered through want 16 state elements, bfloat16, chunks of up to 256 tokens and aligned A_log and ws");
    const dim3 grid(T / chunk + B, (C + 255) / 256);
#define SSM_16 (const bf16_t*)xc, dtp, dt_bias, (const bf16_t*)bc, ldbc, b_col, c_col, A_log, D, (const bf16_t*)z, ldz, cu_seqlens, \
               state_slots, num_slots, C, (bf16_t*)out, chunk, B, ws, ws_dt, dt_ws
    scan16_kernel<SSM_LOCAL><<<grid, 256, chunk * 16 * sizeof(float), stream>>>(SSM_16);
    ssm_combine_kernel<<<dim3(B, (C * N + 255) / 256), 256, 0, stream>>>(cu_seqlens, state_slots, state, ws, ws_dt, A_log, num_slots, C, N,
                                                                         hist, chunk, max_chunks, 1);
    scan16_kernel<SSM_FROM><<<grid, 256, chunk * 32 * sizeof(float), stream>>>(SSM_16);
#undef SSM_16
    PICO_LAUNCH_CHECK();
    return 0;
  }
#define SSM_ARGS(TT)                                                                                                    \
  (const TT*)xc, dtp, dt_bias, (const TT*)bc, ldbc, b_col, c_col, A_log, D, (const TT*)z, ldz, cu_seqlens, state_slots, \
      state, num_slots, C, N, hist, lpc, (TT*)out, chunk, max_chunks, ws, ws_dt
#define SSM_LAUNCH(TT, MODE, GX)                                                                              \
  do {                                                                                                        \
    if (npl == 1) selective_scan_kernel<TT, 1, MODE><<<dim3(GX, gy), 256, lds, stream>>>(SSM_ARGS(TT));       \
    else if (npl == 2) selective_scan_kernel<TT, 2, MODE><<<dim3(GX, gy), 256, lds, stream>>>(SSM_ARGS(TT));  \
    else if (npl == 4) selective_scan_kernel<TT, 4, MODE><<<dim3(GX, gy), 256, lds, stream>>>(SSM_ARGS(TT));  \
    else if (npl == 8) selective_scan_kernel<TT, 8, MODE><<<dim3(GX, gy), 256, lds, stream>>>(SSM_ARGS(TT));  \
    else selective_scan_kernel<TT, 16, MODE><<<dim3(GX, gy), 256, lds, stream>>>(SSM_ARGS(TT));               \
  } while (0)
#define SSM_RUN(TT)                                                                                                        \
  if (chunk == 0) {                                                                                                        \
    SSM_LAUNCH(TT, SSM_WHOLE, B);                                                                                          \
  } else {                                                                                                                 \
    SSM_LAUNCH(TT, SSM_LOCAL, B * max_chunks);                                                                             \
    ssm_combine_kernel<<<dim3(B, (C * N + 255) / 256), 256, 0, stream>>>(cu_seqlens, state_slots, state, ws, ws_dt, A_log, \
                                                                         num_slots, C, N, hist, chunk, max_chunks, 0);     \
    SSM_LAUNCH(TT, SSM_FROM, B * max_chunks);                                                                              \
  }
  if (dtype == PICO_DTYPE_F32) {
    SSM_RUN(float)
  } else if (dtype == PICO_DTYPE_BF16) {
    SSM_RUN(bf16_t)
  } else {
    PICO_REQUIRE(false, "pico_selective_scan: unknown dtype %d", dtype);
  }
#undef SSM_RUN
#undef SSM_LAUNCH
#undef SSM_ARGS
  PICO_LAUNCH_CHECK();
  return 0;
}
