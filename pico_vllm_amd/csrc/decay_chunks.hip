// Linear attention with a constant decay a head (the recurrence of gla.hip with one number in place of a token's decays), in
// chunks that run side by side on the matrix cores:
//
//   S_t = g S_(t-1) + k_t v_t^T,   o_t = S_t^T q_t          (per head; g the head's decay, S [dk, dv])
//
// With i, j counted inside a chunk of n <= 64 tokens and S0 the state in front of it
//
//   o_i = sum_(j <= i) g^(i - j) (q_i . k_j) v_j + g^(i + 1) S0^T q_i
//   S_n = g^n S0 + L,   L = sum_j g^(n - 1 - j) k_j v_j^T
//
// Three launches: every chunk's L from zero; a walk over a sequence's chunks that turns the L's into the states in front
// of the chunks and leaves the slot's new state; every chunk's outputs.  The operands are bfloat16 rows; state, decays and sums are
// float32 as the walk's are, in another order, and keep their 24 bits on the way (decay_pieces_*: what is multiplied with
// the rows is taken apart; of numbers below 2^-110 what is above 2^-134 is left).  Rows that go through z sigmoid(z) as they are read are float32 numbers on both sides of a product: those run
// on v_mfma_f32_32x32x2_f32 (decay_chunk_*).
//
// VAR: the decay changes from token to token (one number a head), g^(i - j) becomes the product of the decays behind j up to
// i, a written key has a factor, and heads share queries and keys (a state-space duality layer).
//
// 2,048 tokens of 48 heads of 128 x 64 over two heads of queries and keys: 71 us; 125 with all products on the float32 instruction, 366
// for the walk in chunks on the vector units; 300 tokens 26, 31 and 151; error against 64 bits 0.86e-7, 1.05e-7 and 1.3e-7.  12 heads of
// 64 x 128 with a constant decay: 1,377 tokens 31 us and 40, error 2.2e-7 and 2.7e-7.  Bound by the states' traffic (52 MB written,
// walked and read), the float32 instruction by itself and by LDS, which lets one of its workgroups onto a compute unit at 128 key channels.
//
// decay_chunk_*: a workgroup (four waves) owns one chunk, one head and 32 NBLK value columns; its rows lie in LDS as float32.  An operand
// tile of the products is 32 rows (lane % 32) by 2 k (lane / 32); which k a step takes is free as long as both operands
// agree, so lane half h takes k = 8 b + 4 h + 0..3 over four steps: four contiguous floats where k runs along a row.
#include "split3.h"

typedef s3_f32x16 f32x16;

#define DC_CHUNK 64

struct ChunkArgs {
  const bf16_t* x;             // [T, ld]; q, k, v of head h from columns q_col + h dk, k_col + h dk, v_col + h dv
  int ld, q_col, k_col, v_col;
  const int* cu_seqlens;
  const int* state_slots;
  const float* decay;          // [H]
  float* state;                // [slots, H, dk, dv]
  float* ws;                   // [chunks, H, dk, dv]
  float* out;                  // [T, H dv]
  int H, dk, dv, num_slots, num_seqs, chunks, silu;      // chunks: room for so many, at least those of the step
  float qscale;
  // VAR: a decay and a factor on the written key of every token and head; `share` heads read one head of queries and keys;
  // ws_decay [chunks, H]: a chunk's decays multiplied up
  const float* g;              // [T, H]
  const float* beta;           // [T, H]
  float* ws_decay;
  int share;
};

// lc[i] = log2 of the product of the decays of tokens 0 .. i of a chunk (tokens from n on: no decay), in 64 bits, so that the
// decay between two tokens, 2^(lc[i] - lc[j]), is as exact as a float holds it however far down the chunk they stand; be[i]:
// the factors.  A decay of zero counts as 2^-4096; one that is not a number makes all tokens from its own on so.  Wave 0 fills
// them; the caller's barrier follows.
__device__ __forceinline__ void chunk_decays(const ChunkArgs& a, int t0, int n, int h, double* lc, float* be) {
  if (threadIdx.x >= 64) return;
  const int i = threadIdx.x;
  const size_t at = (size_t)(t0 + min(i, n - 1)) * a.H + h;
  const float g = a.g[at], b = a.beta[at];
  const double lg = log2((double)g);
  double x = i < n ? (lg < -4096.0 ? -4096.0 : lg) : 0.0;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const double y = __shfl_up(x, o);
    x += i >= o ? y : 0.0;
  }
  lc[i] = x;
  be[i] = i < n ? b : 0.f;
}
__device__ __forceinline__ float between(double from, double to) { return exp2f((float)(to - from)); }

// g^n for n >= 0 (lg = log2 g); g = 1 exactly stays 1
__device__ __forceinline__ float decay_power(float lg, int n) { return exp2f(lg * (float)n); }

__device__ __forceinline__ float act8(uint32_t w, bool high, int silu) {
  const float z = high ? __uint_as_float(w & 0xffff0000u) : __uint_as_float(w << 16);
  return silu ? z / (1.0f + __expf(-z)) : z;
}

// A thread's pieces (8 columns of a row each) of 64 rows x COLS columns: asked for by `fetch`, written to LDS by `put`.
// Rows from n on and columns from `cols` on (a multiple of 8) read as zero; every load is from an address inside.
template <int COLS>
struct Rows {
  static constexpr int N = DC_CHUNK * COLS / 8 / 256;
  static_assert(N >= 1, "at least one piece a thread");
  uint4 v[N];
  __device__ __forceinline__ void fetch(const bf16_t* src, int ld, int n, int cols) {
#pragma unroll
    for (int i = 0; i < N; i++) {
      const int u = threadIdx.x + 256 * i, r = u / (COLS / 8), c = u % (COLS / 8) * 8;
      v[i] = *reinterpret_cast<const uint4*>(src + (size_t)min(r, n - 1) * ld + (c < cols ? c : 0));
    }
  }
  // FINITE: an Inf or NaN is written as zero; returns whether this thread had one.
  template <bool FINITE = false, typename F>
  __device__ __forceinline__ bool put(float* dst, int stride, int n, int cols, int silu, F factor) {
    bool odd = false;
#pragma unroll
    for (int i = 0; i < N; i++) {
      const int u = threadIdx.x + 256 * i, r = u / (COLS / 8), c = u % (COLS / 8) * 8;
      const float f = (r < n && c < cols) ? factor(r) : 0.f;
      float4 a, b;
      a.x = act8(v[i].x, false, silu) * f; a.y = act8(v[i].x, true, silu) * f;
      a.z = act8(v[i].y, false, silu) * f; a.w = act8(v[i].y, true, silu) * f;
      b.x = act8(v[i].z, false, silu) * f; b.y = act8(v[i].z, true, silu) * f;
      b.z = act8(v[i].w, false, silu) * f; b.w = act8(v[i].w, true, silu) * f;
      if (!(r < n && c < cols)) a = b = make_float4(0.f, 0.f, 0.f, 0.f);
      if (FINITE) {
        float e[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int j = 0; j < 8; j++) {
          const bool ok = fabsf(e[j]) < INFINITY;
          odd = odd || !ok;
          e[j] = ok ? e[j] : 0.f;
        }
        a = make_float4(e[0], e[1], e[2], e[3]);
        b = make_float4(e[4], e[5], e[6], e[7]);
      }
      *reinterpret_cast<float4*>(dst + r * stride + c) = a;
      *reinterpret_cast<float4*>(dst + r * stride + c + 4) = b;
    }
    return odd;
  }
};

__device__ __forceinline__ f32x16 mfma32(float a, float b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }

__device__ __forceinline__ f32x16 zero16() {
  f32x16 z;
#pragma unroll
  for (int r = 0; r < 16; r++) z[r] = 0.f;
  return z;
}

// The chunks of a step are counted sequence by sequence (workgroup and place in ws alike).  Which tokens a workgroup has;
// false: none.
__device__ __forceinline__ bool chunk_tokens(const ChunkArgs& a, int& t0, int& n) {
  int j = blockIdx.x, b = 0, end = 0;
  for (; b < a.num_seqs; b++) {
    t0 = a.cu_seqlens[b];
    end = a.cu_seqlens[b + 1];
    const int chunks = (end - t0 + DC_CHUNK - 1) / DC_CHUNK;
    if (j < chunks) break;
    j -= chunks;
  }
  if (b == a.num_seqs) return false;
  t0 += j * DC_CHUNK;
  n = min(DC_CHUNK, end - t0);
  const int slot = a.state_slots[b];
  return slot >= 0 && slot < a.num_slots;
}

// L of every chunk into ws.  Wave w: value columns 32 (w % NBLK) .. of the workgroup's; with fewer than four column blocks
// the waves of one share the key channels.
template <int DKP, int NBLK>
__global__ __launch_bounds__(256) void decay_chunk_state_kernel(const ChunkArgs a) {
  constexpr int KS = DKP + 4, NB = 32 * NBLK, VS = NB + 8, CB = DKP / 32, SHARE = 4 / NBLK;
  __shared__ __attribute__((aligned(16))) float ks[DC_CHUNK * KS];
  __shared__ __attribute__((aligned(16))) float vs[DC_CHUNK * VS];
  int t0, n;
  if (!chunk_tokens(a, t0, n)) return;
  const int h = blockIdx.y, n0 = blockIdx.z * NB, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l = lane & 31, half = lane >> 5;
  const float lg = log2f(a.decay[h]);
  const bf16_t* row = a.x + (size_t)t0 * a.ld;
  Rows<DKP> k;
  Rows<NB> v;
  k.fetch(row + a.k_col + h * a.dk, a.ld, n, a.dk);
  v.fetch(row + a.v_col + h * a.dv + n0, a.ld, n, a.dv - n0);
  k.put(ks, KS, n, a.dk, a.silu, [&](int r) { return decay_power(lg, n - 1 - r); });
  v.put(vs, VS, n, a.dv - n0, a.silu, [&](int) { return 1.0f; });
  __syncthreads();
  const int nb = wave % NBLK, c_first = wave / NBLK;
  const float* vp = vs + 4 * half * VS + 32 * nb + l;
  f32x16 acc[(CB + SHARE - 1) / SHARE];
#pragma unroll
  for (int i = 0; i < (CB + SHARE - 1) / SHARE; i++) acc[i] = zero16();
  auto eight = [&](int j) {                              // tokens j .. j + 7
    float b[4];
#pragma unroll
    for (int s = 0; s < 4; s++) b[s] = vp[(j + s) * VS];
#pragma unroll
    for (int i = 0; i < (CB + SHARE - 1) / SHARE; i++) {
      const int cb = min(c_first + i * SHARE, CB - 1);
      const float* kp = ks + (j + 4 * half) * KS + 32 * cb + l;
#pragma unroll
      for (int s = 0; s < 4; s++) acc[i] = mfma32(kp[s * KS], b[s], acc[i]);
    }
  };
  if (n > DC_CHUNK / 2) {
#pragma unroll 2
    for (int j = 0; j < DC_CHUNK; j += 8) eight(j);
  } else {                                               // (rows from n on are zero: 42 us of a launch of short ones become 31)
    for (int j = 0; j < n; j += 8) eight(j);
  }
  float* ws = a.ws + ((size_t)blockIdx.x * a.H + h) * a.dk * a.dv;
  const int col = n0 + 32 * nb + l;
  if (col >= a.dv) return;
#pragma unroll
  for (int i = 0; i < (CB + SHARE - 1) / SHARE; i++) {
    const int cb = c_first + i * SHARE;
    if (cb >= CB) break;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int c = 32 * cb + 8 * (r >> 2) + 4 * half + (r & 3);
      if (c < a.dk) ws[(size_t)c * a.dv + col] = acc[i][r];
    }
  }
}

// The walk over a sequence's chunks, a thread V neighbouring state elements: ws becomes the state in front of every chunk, the
// slot gets the state behind the last.  The loads of 8 / V chunks travel together.  grid (sequences, heads,
// ceil(dk dv / (256 V))).  One element a thread fills the chip for one sequence; with many sequences of few chunks each it is the
// number of workgroups that costs: 40 single tokens beside a portion of 300, 48 heads of 128 x 64, 83 us with one, 41 with four.
template <bool VAR, int V>
__global__ __launch_bounds__(256) void decay_chunk_walk_kernel(const ChunkArgs a) {
  constexpr int DC_AHEAD = 8 / V;
  typedef float vec __attribute__((ext_vector_type(V)));
  const int b = blockIdx.x, h = blockIdx.y, size = a.dk * a.dv, e = (blockIdx.z * 256 + threadIdx.x) * V;
  const int slot = a.state_slots[b], n = a.cu_seqlens[b + 1] - a.cu_seqlens[b];
  if (slot < 0 || slot >= a.num_slots || n <= 0) return;
  // the sequence's first chunk: a lane counts a sequence in front of it (with 41 sequences 225 us for the launch where a
  // workgroup counts them one after the other, 83 so)
  int first = 0;
  if (b > 0) {
    for (int i = threadIdx.x & 63; i < b; i += 64) first += (a.cu_seqlens[i + 1] - a.cu_seqlens[i] + DC_CHUNK - 1) / DC_CHUNK;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) first += __shfl_xor(first, o);
  }
  if (e >= size) return;
  const float lg = VAR ? 0.f : log2f(a.decay[h]), whole = decay_power(lg, DC_CHUNK);
  const float* wd = VAR ? a.ws_decay + (size_t)first * a.H + h : nullptr;
  vec* sp = reinterpret_cast<vec*>(a.state + ((size_t)slot * a.H + h) * size + e);
  float* w = a.ws + ((size_t)first * a.H + h) * size + e;
  const size_t step = (size_t)a.H * size;
  const int chunks = (n + DC_CHUNK - 1) / DC_CHUNK;
  vec S = *sp;
  for (int j0 = 0; j0 < chunks; j0 += DC_AHEAD) {
    vec local[DC_AHEAD];
    float decay[VAR ? DC_AHEAD : 1];
#pragma unroll
    for (int i = 0; i < DC_AHEAD; i++) {
      local[i] = *reinterpret_cast<const vec*>(w + min(j0 + i, chunks - 1) * step);
      if (VAR) decay[VAR ? i : 0] = wd[(size_t)min(j0 + i, chunks - 1) * a.H];
    }
#pragma unroll
    for (int i = 0; i < DC_AHEAD; i++) {
      if (j0 + i >= chunks) break;
      *reinterpret_cast<vec*>(w + (j0 + i) * step) = S;
      const int left = n - (j0 + i) * DC_CHUNK;
      const float g = VAR ? decay[VAR ? i : 0] : left < DC_CHUNK ? decay_power(lg, left) : whole;
#pragma unroll
      for (int v = 0; v < V; v++) S[v] = fmaf(g, S[v], local[i][v]);
    }
  }
  *sp = S;
}

// The outputs of every chunk.  Wave w: value columns 32 (w % NBLK) ..; with four column blocks it makes both blocks of 32
// tokens, with two one of them.  Products of queries and keys are made by three waves (the block of later keys and earlier
// queries is empty) and meet the values through LDS, where they take the keys' place.
//
// A token's weight on a later one is 0, and 0 * Inf is NaN: the products see an Inf or NaN among the values as zero, and
// where there is one it is added afterwards to the tokens from its own on.
template <int DKP, int NBLK>
__global__ __launch_bounds__(256) void decay_chunk_out_kernel(const ChunkArgs a) {
  __shared__ bool odd_values[4];
  constexpr int KS = DKP + 4, PS = DC_CHUNK + 4, NB = 32 * NBLK, VS = NB + 8, IB = NBLK == 4 ? 2 : 1;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float* qs = lds;
  float* ks = qs + DC_CHUNK * KS;                        // the keys, then the weighted products [64][PS]
  float* vs = ks + DC_CHUNK * (KS > PS ? KS : PS);
  int t0, n;
  if (!chunk_tokens(a, t0, n)) return;
  const int h = blockIdx.y, n0 = blockIdx.z * NB, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l = lane & 31, half = lane >> 5;
  const int nb = wave % NBLK, ib0 = NBLK == 4 ? 0 : wave / NBLK, col = n0 + 32 * nb + l;
  const float lg = log2f(a.decay[h]);
  const bf16_t* row = a.x + (size_t)t0 * a.ld;
  Rows<DKP> q, k;
  Rows<NB> v;
  q.fetch(row + a.q_col + h * a.dk, a.ld, n, a.dk);
  k.fetch(row + a.k_col + h * a.dk, a.ld, n, a.dk);
  v.fetch(row + a.v_col + h * a.dv + n0, a.ld, n, a.dv - n0);
  // the state in front of the chunk as an operand: rows 8 b + 4 half + 0..3, this lane's column
  float s0[DKP / 2];
  {
    const float* sp = a.ws + ((size_t)blockIdx.x * a.H + h) * a.dk * a.dv + min(col, a.dv - 1);
#pragma unroll
    for (int i = 0; i < DKP / 2; i++) s0[i] = sp[(size_t)min(i / 4 * 8 + 4 * half + i % 4, a.dk - 1) * a.dv];
  }
  q.put(qs, KS, n, a.dk, a.silu, [&](int) { return a.qscale; });
  k.put(ks, KS, n, a.dk, a.silu, [&](int) { return 1.0f; });
  const bool odd = __any(v.template put<true>(vs, VS, n, a.dv - n0, a.silu, [&](int) { return 1.0f; }));
  if (lane == 0) odd_values[wave] = odd;
  __syncthreads();
  // queries and keys: wave 0 block (0, 0), wave 1 (1, 0), wave 2 (1, 1)
  const int pi = wave == 0 ? 0 : 1, pj = wave == 2 ? 1 : 0;
  f32x16 p = zero16();
  if (wave < 3) {
    const float* qp = qs + (32 * pi + l) * KS + 4 * half;
    const float* kp = ks + (32 * pj + l) * KS + 4 * half;
#pragma unroll 4
    for (int c = 0; c < DKP; c += 8) {
      const float4 qv = *reinterpret_cast<const float4*>(qp + c), kv = *reinterpret_cast<const float4*>(kp + c);
      p = mfma32(qv.x, kv.x, p);
      p = mfma32(qv.y, kv.y, p);
      p = mfma32(qv.z, kv.z, p);
      p = mfma32(qv.w, kv.w, p);
    }
  }
  // what the state contributes: the two halves of the key channels are summed apart (half as long a chain)
  f32x16 acc[IB], half_sum[IB];
#pragma unroll
  for (int i = 0; i < IB; i++) acc[i] = half_sum[i] = zero16();
#pragma unroll
  for (int c = 0; c < DKP; c += 8) {
    if (c == DKP / 2) {
#pragma unroll
      for (int i = 0; i < IB; i++) {
        half_sum[i] = acc[i];
        acc[i] = zero16();
      }
    }
#pragma unroll
    for (int i = 0; i < IB; i++) {
      const float4 qv = *reinterpret_cast<const float4*>(qs + (32 * (ib0 + i) + l) * KS + 4 * half + c);
      // (rows of the state from dk on stand beside zeros of q; they are another row's numbers, finite as the state is)
      acc[i] = mfma32(qv.x, s0[c / 2], acc[i]);
      acc[i] = mfma32(qv.y, s0[c / 2 + 1], acc[i]);
      acc[i] = mfma32(qv.z, s0[c / 2 + 2], acc[i]);
      acc[i] = mfma32(qv.w, s0[c / 2 + 3], acc[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < IB; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int t = 32 * (ib0 + i) + 8 * (r >> 2) + 4 * half + (r & 3);
      acc[i][r] = (acc[i][r] + half_sum[i][r]) * decay_power(lg, t + 1);
    }
  __syncthreads();                                       // every wave is done with the keys
  if (wave < 3) {
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int i = 32 * pi + 8 * (r >> 2) + 4 * half + (r & 3), j = 32 * pj + l;
      ks[i * PS + j] = j <= i ? p[r] * decay_power(lg, i - j) : 0.f;
    }
  }
  __syncthreads();
  const float* vp = vs + 4 * half * VS + 32 * nb + l;
#pragma unroll
  for (int i = 0; i < IB; i++) {
    const int ib = ib0 + i;
    const float* pp = ks + (32 * ib + l) * PS + 4 * half;
#pragma unroll 4
    for (int j = 0; j < 32 * (ib + 1); j += 8) {
      const float4 pv = *reinterpret_cast<const float4*>(pp + j);
      acc[i] = mfma32(pv.x, vp[j * VS], acc[i]);
      acc[i] = mfma32(pv.y, vp[(j + 1) * VS], acc[i]);
      acc[i] = mfma32(pv.z, vp[(j + 2) * VS], acc[i]);
      acc[i] = mfma32(pv.w, vp[(j + 3) * VS], acc[i]);
    }
  }
  if (col >= a.dv) return;
  if (odd_values[0] || odd_values[1] || odd_values[2] || odd_values[3]) {
    const bf16_t* vcol = row + a.v_col + h * a.dv + col;
#pragma unroll 1
    for (int j = 0; j < n; j++) {
      const float x = act8(vcol[(size_t)j * a.ld], false, a.silu);
      if (fabsf(x) < INFINITY) continue;
#pragma unroll
      for (int i = 0; i < IB; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
          const int t = 32 * (ib0 + i) + 8 * (r >> 2) + 4 * half + (r & 3);
          if (t >= j) acc[i][r] = fmaf(ks[t * PS + j], x, acc[i][r]);
        }
    }
  }
#pragma unroll
  for (int i = 0; i < IB; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int t = 32 * (ib0 + i) + 8 * (r >> 2) + 4 * half + (r & 3);
      if (t < n) a.out[(size_t)(t0 + t) * a.H * a.dv + (size_t)h * a.dv + col] = acc[i][r];
    }
}

// ---------------------------------------------------------------------------
// Rows that are read as they stand (no z sigmoid(z)): q, k and v are bfloat16 numbers, and what they are multiplied with, state, weighted
// values and weighted products, is taken apart into three of them (split3.h; three instructions of 16 k, 3/16 of the float32
// instruction's time).  Products of queries and keys are the bfloat16 instruction's own.  All of a tile in LDS is bfloat16: a
// third of the bytes, so that three workgroups share a compute unit.  Pieces of numbers below 2^-110 end at 2^-133 (scaled, as in
// split3.h, states of 2^80 and more would not be numbers).
// ---------------------------------------------------------------------------
#define DC_TS (DC_CHUNK + 8)             // row stride of [channel][token] and [token][token] planes: 16-byte reads of rows meet every bank once

// Two numbers' pieces; what is not finite (or rounds to it) is its own upper piece.
__device__ __forceinline__ void split2_any(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
  h = pack2_bf16(a, b);
  const float ha = s3_low(h), hb = s3_high(h);
  a = fabsf(ha) < INFINITY ? a - ha : 0.f;
  b = fabsf(hb) < INFINITY ? b - hb : 0.f;
  m = pack2_bf16(a, b);
  l = pack2_bf16(a - s3_low(m), b - s3_high(m));
}

// 64 rows x COLS columns on their way to LDS turned around: a thread has two neighbouring rows of eight columns.
template <int COLS>
struct Turned {
  static constexpr int UNITS = 32 * COLS / 8, N = (UNITS + 255) / 256;
  uint4 v[N][2];
  __device__ __forceinline__ int pair(int i) const { return (threadIdx.x + 256 * i) % 32; }
  __device__ __forceinline__ int col(int i) const { return (threadIdx.x + 256 * i) / 32 * 8; }
  __device__ __forceinline__ void fetch(const bf16_t* src, int ld, int n, int cols) {
#pragma unroll
    for (int i = 0; i < N; i++) {
      const int c = col(i) < cols ? col(i) : 0;
#pragma unroll
      for (int k = 0; k < 2; k++) v[i][k] = *reinterpret_cast<const uint4*>(src + (size_t)min(2 * pair(i) + k, n - 1) * ld + c);
    }
  }
  // use(column, row pair, word of the two rows' numbers in it): rows from n on and columns from `cols` on are zero
  template <typename F>
  __device__ __forceinline__ void each(int n, int cols, F use) const {
#pragma unroll
    for (int i = 0; i < N; i++) {
      if (COLS % 64 != 0 && (int)threadIdx.x + 256 * i >= UNITS) break;
      const int r = 2 * pair(i);
      const uint32_t a[4] = {v[i][0].x, v[i][0].y, v[i][0].z, v[i][0].w}, b[4] = {v[i][1].x, v[i][1].y, v[i][1].z, v[i][1].w};
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const int c = col(i) + j;
        const uint32_t lo = (j & 1) ? a[j / 2] >> 16 : a[j / 2] & 0xffffu, hi = (j & 1) ? b[j / 2] & 0xffff0000u : b[j / 2] << 16;
        use(c, r, c < cols ? (r < n ? lo : 0u) | (r + 1 < n ? hi : 0u) : 0u);
      }
    }
  }
};

__device__ __forceinline__ s3_u32x4 dc_read(const bf16_t* p) { return *reinterpret_cast<const s3_u32x4*>(p); }

template <int DKP, int NBLK>
constexpr int dc_state_bytes() { return (DKP + 3 * 32 * NBLK) * DC_TS * 2; }
template <int DKP, int NBLK>
constexpr int dc_out_bytes() {
  const int rows = 2 * DC_CHUNK * (DKP + 8), planes = 3 * DC_CHUNK * DC_TS;
  return ((rows > planes ? rows : planes) + 32 * NBLK * DC_TS) * 2;
}

// L of every chunk into ws, as decay_chunk_state_kernel; the weights on the values.
template <int DKP, int NBLK, bool VAR>
__global__ __launch_bounds__(256, 2) void decay_pieces_state_kernel(const ChunkArgs a) {
  constexpr int NB = 32 * NBLK, CB = DKP / 32, SHARE = 4 / NBLK, PLANE = NB * DC_TS;
  __shared__ double lc[VAR ? DC_CHUNK : 1];
  __shared__ float be[VAR ? DC_CHUNK : 1];
  extern __shared__ __attribute__((aligned(16))) float lds[];
  bf16_t* kt = reinterpret_cast<bf16_t*>(lds);                // [DKP][DC_TS]
  bf16_t* vt = kt + DKP * DC_TS;                              // three planes of [NB][DC_TS]
  int t0, n;
  if (!chunk_tokens(a, t0, n)) return;
  const int h = blockIdx.y, n0 = blockIdx.z * NB, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l = lane & 31, half = lane >> 5;
  const float lg = VAR ? 0.f : log2f(a.decay[h]);
  const bf16_t* row = a.x + (size_t)t0 * a.ld;
  Turned<DKP> k;
  Turned<NB> v;
  k.fetch(row + a.k_col + (VAR ? h / a.share : h) * a.dk, a.ld, n, a.dk);
  v.fetch(row + a.v_col + h * a.dv + n0, a.ld, n, a.dv - n0);
  if (VAR) {
    chunk_decays(a, t0, n, h, lc, be);
    __syncthreads();
    if (threadIdx.x == 0 && n0 == 0) a.ws_decay[(size_t)blockIdx.x * a.H + h] = exp2f((float)lc[n - 1]);
  }
  k.each(n, a.dk, [&](int c, int r, uint32_t w) { *reinterpret_cast<uint32_t*>(kt + c * DC_TS + r) = w; });
  const int pair = 2 * (threadIdx.x % 32);                    // this thread's rows (of every unit)
  float f[2];
#pragma unroll
  for (int i = 0; i < 2; i++) f[i] = pair + i < n ? (VAR ? be[pair + i] * between(lc[pair + i], lc[n - 1]) : decay_power(lg, n - 1 - pair - i)) : 0.f;
  v.each(n, a.dv - n0, [&](int c, int r, uint32_t w) {
    uint32_t p[3];
    split2_any(r < n ? s3_low(w) * f[0] : 0.f, r + 1 < n ? s3_high(w) * f[1] : 0.f, p[0], p[1], p[2]);
#pragma unroll
    for (int i = 0; i < 3; i++) *reinterpret_cast<uint32_t*>(vt + i * PLANE + c * DC_TS + r) = p[i];
  });
  __syncthreads();
  const int nb = wave % NBLK, c_first = wave / NBLK;
  f32x16 acc[(CB + SHARE - 1) / SHARE];
#pragma unroll
  for (int i = 0; i < (CB + SHARE - 1) / SHARE; i++) acc[i] = zero16();
#pragma unroll
  for (int j = 0; j < DC_CHUNK; j += 16) {
    if (j >= n) break;                                        // (rows from n on are zero)
    const bf16_t* vp = vt + (32 * nb + l) * DC_TS + j + 8 * half;
    const s3_u32x4 vl = dc_read(vp + 2 * PLANE), vm = dc_read(vp + PLANE), vh = dc_read(vp);
#pragma unroll
    for (int i = 0; i < (CB + SHARE - 1) / SHARE; i++) {
      const s3_u32x4 kk = dc_read(kt + (32 * min(c_first + i * SHARE, CB - 1) + l) * DC_TS + j + 8 * half);
      acc[i] = mfma16(kk, vl, acc[i]);
      acc[i] = mfma16(kk, vm, acc[i]);
      acc[i] = mfma16(kk, vh, acc[i]);
    }
  }
  float* ws = a.ws + ((size_t)blockIdx.x * a.H + h) * a.dk * a.dv;
  const int col = n0 + 32 * nb + l;
  if (col >= a.dv) return;
#pragma unroll
  for (int i = 0; i < (CB + SHARE - 1) / SHARE; i++) {
    const int cb = c_first + i * SHARE;
    if (cb >= CB) break;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int c = 32 * cb + 8 * (r >> 2) + 4 * half + (r & 3);
      if (c < a.dk) ws[(size_t)c * a.dv + col] = acc[i][r];
    }
  }
}

// The outputs of every chunk, as decay_chunk_out_kernel.  The products of queries and keys are made turned around (a lane has
// a query, a register a key), so that a lane writes four neighbouring keys' pieces at a time.
template <int DKP, int NBLK, bool VAR>
__global__ __launch_bounds__(256, 2) void decay_pieces_out_kernel(const ChunkArgs a) {
  constexpr int QS = DKP + 8, NB = 32 * NBLK, IB = NBLK == 4 ? 2 : 1, PLANE = DC_CHUNK * DC_TS, UNITS = DC_CHUNK * DKP / 8 / 256;
  static_assert(UNITS >= 1, "at least one piece a thread");
  __shared__ double lc[VAR ? DC_CHUNK : 1];
  __shared__ float be[VAR ? DC_CHUNK : 1];
  __shared__ bool odd_values[4];
  extern __shared__ __attribute__((aligned(16))) float lds[];
  bf16_t* qs = reinterpret_cast<bf16_t*>(lds);                // [64][QS], then the weighted products' planes [64][DC_TS]
  bf16_t* ks = qs + DC_CHUNK * QS;
  bf16_t* ps = qs;
  bf16_t* vt = qs + (2 * DC_CHUNK * QS > 3 * PLANE ? 2 * DC_CHUNK * QS : 3 * PLANE);      // [NB][DC_TS]
  int t0, n;
  if (!chunk_tokens(a, t0, n)) return;
  const int h = blockIdx.y, n0 = blockIdx.z * NB, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l = lane & 31, half = lane >> 5;
  const int nb = wave % NBLK, ib0 = NBLK == 4 ? 0 : wave / NBLK, col = n0 + 32 * nb + l;
  const float lg = VAR ? 0.f : log2f(a.decay[h]);
  const bf16_t* row = a.x + (size_t)t0 * a.ld;
  const bf16_t* qrow = row + a.q_col + (VAR ? h / a.share : h) * a.dk;
  const bf16_t* krow = row + a.k_col + (VAR ? h / a.share : h) * a.dk;
  uint4 qv[UNITS], kv[UNITS];
#pragma unroll
  for (int i = 0; i < UNITS; i++) {
    const int u = threadIdx.x + 256 * i, r = u / (DKP / 8), c = u % (DKP / 8) * 8;
    const size_t at = (size_t)min(r, n - 1) * a.ld + (c < a.dk ? c : 0);
    qv[i] = *reinterpret_cast<const uint4*>(qrow + at);
    kv[i] = *reinterpret_cast<const uint4*>(krow + at);
  }
  Turned<NB> v;
  v.fetch(row + a.v_col + h * a.dv + n0, a.ld, n, a.dv - n0);
  // the state in front of the chunk as an operand: of 16 channels the half'th eight, this lane's column
  float s0[DKP / 2];
  {
    const float* sp = a.ws + ((size_t)blockIdx.x * a.H + h) * a.dk * a.dv + min(col, a.dv - 1);
#pragma unroll
    for (int i = 0; i < DKP / 2; i++) s0[i] = sp[(size_t)min(i / 8 * 16 + 8 * half + i % 8, a.dk - 1) * a.dv];
  }
#pragma unroll
  for (int i = 0; i < UNITS; i++) {
    const int u = threadIdx.x + 256 * i, r = u / (DKP / 8), c = u % (DKP / 8) * 8;
    const bool in = r < n && c < a.dk;
    *reinterpret_cast<uint4*>(qs + r * QS + c) = in ? qv[i] : make_uint4(0, 0, 0, 0);
    *reinterpret_cast<uint4*>(ks + r * QS + c) = in ? kv[i] : make_uint4(0, 0, 0, 0);
  }
  bool odd = false;                                           // an Inf or NaN among the values is written as zero
  v.each(n, a.dv - n0, [&](int c, int r, uint32_t w) {
    const bool lo = (w & 0x7f80u) == 0x7f80u, hi = (w & 0x7f800000u) == 0x7f800000u;
    odd = odd || lo || hi;
    *reinterpret_cast<uint32_t*>(vt + c * DC_TS + r) = (lo ? 0u : w & 0xffffu) | (hi ? 0u : w & 0xffff0000u);
  });
  odd = __any(odd);
  if (lane == 0) odd_values[wave] = odd;
  if (VAR) chunk_decays(a, t0, n, h, lc, be);
  __syncthreads();
  // keys by queries: wave 0 queries 0 .. 31 and keys 0 .. 31, wave 1 the later queries, wave 2 the later of both
  const int pi = wave == 0 ? 0 : 1, pj = wave == 2 ? 1 : 0;
  f32x16 p = zero16();
  if (wave < 3) {
#pragma unroll
    for (int c = 0; c < DKP; c += 16)
      p = mfma16(dc_read(ks + (32 * pj + l) * QS + c + 8 * half), dc_read(qs + (32 * pi + l) * QS + c + 8 * half), p);
  }
  // what the state contributes
  f32x16 acc[IB];
#pragma unroll
  for (int i = 0; i < IB; i++) acc[i] = zero16();
#pragma unroll
  for (int c = 0; c < DKP; c += 16) {
    s3_u32x4 sh, sm, sl;
#pragma unroll
    for (int w = 0; w < 4; w++) {
      uint32_t x, y, z;
      split2_any(s0[c / 2 + 2 * w], s0[c / 2 + 2 * w + 1], x, y, z);
      sh[w] = x; sm[w] = y; sl[w] = z;
    }
#pragma unroll
    for (int i = 0; i < IB; i++) {
      // (rows of the state from dk on stand beside zeros of q; they are another row's numbers, finite as the state is)
      const s3_u32x4 qq = dc_read(qs + (32 * (ib0 + i) + l) * QS + c + 8 * half);
      acc[i] = mfma16(qq, sl, acc[i]);
      acc[i] = mfma16(qq, sm, acc[i]);
      acc[i] = mfma16(qq, sh, acc[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < IB; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int t = 32 * (ib0 + i) + 8 * (r >> 2) + 4 * half + (r & 3);
      acc[i][r] *= (VAR ? exp2f((float)lc[t]) : decay_power(lg, t + 1)) * a.qscale;
    }
  __syncthreads();                                            // every wave is done with the queries and keys
  if (wave < 3) {
    const int i = 32 * pi + l;
#pragma unroll
    for (int r = 0; r < 16; r += 4) {
      const int j0 = 32 * pj + 2 * r + 4 * half;
      float w[4];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int j = j0 + e;
        w[e] = j <= i ? p[r + e] * a.qscale * (VAR ? be[j] * between(lc[j], lc[i]) : decay_power(lg, i - j)) : 0.f;
      }
      uint32_t x[3], y[3];
      split2_any(w[0], w[1], x[0], x[1], x[2]);
      split2_any(w[2], w[3], y[0], y[1], y[2]);
#pragma unroll
      for (int e = 0; e < 3; e++) *reinterpret_cast<uint2*>(ps + e * PLANE + i * DC_TS + j0) = make_uint2(x[e], y[e]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < IB; i++) {
    const int ib = ib0 + i;
    const bf16_t* pp = ps + (32 * ib + l) * DC_TS + 8 * half;
#pragma unroll
    for (int j = 0; j < DC_CHUNK; j += 16) {
      if (j >= 32 * (ib + 1)) break;
      const s3_u32x4 vv = dc_read(vt + (32 * nb + l) * DC_TS + j + 8 * half);
      acc[i] = mfma16(dc_read(pp + 2 * PLANE + j), vv, acc[i]);
      acc[i] = mfma16(dc_read(pp + PLANE + j), vv, acc[i]);
      acc[i] = mfma16(dc_read(pp + j), vv, acc[i]);
    }
  }
  if (col >= a.dv) return;
  if (odd_values[0] || odd_values[1] || odd_values[2] || odd_values[3]) {
    const bf16_t* vcol = row + a.v_col + h * a.dv + col;
#pragma unroll 1
    for (int j = 0; j < n; j++) {
      const float x = bf16_to_f32(vcol[(size_t)j * a.ld]);
      if (fabsf(x) < INFINITY) continue;
#pragma unroll
      for (int i = 0; i < IB; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
          const int t = 32 * (ib0 + i) + 8 * (r >> 2) + 4 * half + (r & 3);
          const bf16_t* w = ps + t * DC_TS + j;
          // (the block of later keys and earlier queries is not written)
          if (t >= j) acc[i][r] = fmaf(bf16_to_f32(w[0]) + (bf16_to_f32(w[PLANE]) + bf16_to_f32(w[2 * PLANE])), x, acc[i][r]);
        }
    }
  }
#pragma unroll
  for (int i = 0; i < IB; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int t = 32 * (ib0 + i) + 8 * (r >> 2) + 4 * half + (r & 3);
      if (t < n) a.out[(size_t)(t0 + t) * a.H * a.dv + (size_t)h * a.dv + col] = acc[i][r];
    }
}

// The walk between the chunks' two launches
template <bool VAR>
static void launch_walk(const ChunkArgs& a, int num_seqs, hipStream_t stream) {
  if (num_seqs > 4 && (uintptr_t)a.state % 16 == 0 && (uintptr_t)a.ws % 16 == 0)       // (dv is a multiple of 8)
    decay_chunk_walk_kernel<VAR, 4><<<dim3(num_seqs, a.H, (a.dk * a.dv + 1023) / 1024), 256, 0, stream>>>(a);
  else
    decay_chunk_walk_kernel<VAR, 1><<<dim3(num_seqs, a.H, (a.dk * a.dv + 255) / 256), 256, 0, stream>>>(a);
}

template <int DKP, int NBLK>
static int launch_chunks(const ChunkArgs& a, int num_seqs, hipStream_t stream) {
  constexpr int KS = DKP + 4, PS = DC_CHUNK + 4, VS = 32 * NBLK + 8;
  constexpr int bytes = DC_CHUNK * (KS + (KS > PS ? KS : PS) + VS) * (int)sizeof(float);
  static const hipError_t room = hipFuncSetAttribute((const void*)decay_chunk_out_kernel<DKP, NBLK>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  PICO_REQUIRE(room == hipSuccess, "pico_decay_chunks: %d bytes of LDS refused", bytes);
  const dim3 grid(a.chunks, a.H, (a.dv + 32 * NBLK - 1) / (32 * NBLK));
  decay_chunk_state_kernel<DKP, NBLK><<<grid, 256, 0, stream>>>(a);
  launch_walk<false>(a, num_seqs, stream);
  decay_chunk_out_kernel<DKP, NBLK><<<grid, 256, bytes, stream>>>(a);
  PICO_LAUNCH_CHECK();
  return 0;
}

template <int DKP, int NBLK, bool VAR>
static int launch_pieces(const ChunkArgs& a, int num_seqs, hipStream_t stream) {
  constexpr int first = dc_state_bytes<DKP, NBLK>(), last = dc_out_bytes<DKP, NBLK>();
  static const hipError_t room1 = hipFuncSetAttribute((const void*)decay_pieces_state_kernel<DKP, NBLK, VAR>, hipFuncAttributeMaxDynamicSharedMemorySize, first);
  static const hipError_t room2 = hipFuncSetAttribute((const void*)decay_pieces_out_kernel<DKP, NBLK, VAR>, hipFuncAttributeMaxDynamicSharedMemorySize, last);
  PICO_REQUIRE(room1 == hipSuccess && room2 == hipSuccess, "pico_decay_chunks: %d and %d bytes of LDS refused", first, last);
  const dim3 grid(a.chunks, a.H, (a.dv + 32 * NBLK - 1) / (32 * NBLK));
  decay_pieces_state_kernel<DKP, NBLK, VAR><<<grid, 256, first, stream>>>(a);
  launch_walk<VAR>(a, num_seqs, stream);
  decay_pieces_out_kernel<DKP, NBLK, VAR><<<grid, 256, last, stream>>>(a);
  PICO_LAUNCH_CHECK();
  return 0;
}

template <bool VAR>
static int pick_chunks(const ChunkArgs& a, int num_seqs, hipStream_t stream) {
  const bool wide = a.dv > 64;
#define PICK(DKP)                                                                                                                \
  do {                                                                                                                           \
    if (!VAR && a.silu) return wide ? launch_chunks<DKP, 4>(a, num_seqs, stream) : launch_chunks<DKP, 2>(a, num_seqs, stream);    \
    return wide ? launch_pieces<DKP, 4, VAR>(a, num_seqs, stream) : launch_pieces<DKP, 2, VAR>(a, num_seqs, stream);              \
  } while (0)
  if (a.dk <= 32) PICK(32);
  if (a.dk <= 64) PICK(64);
  if (a.dk <= 96) PICK(96);
  PICK(128);
#undef PICK
}

extern "C" int pico_decay_chunk_tokens() { return DC_CHUNK; }

// x bfloat16 [T, ld]; ws float32 [chunks, H, dk, dv], chunks at least T / 64 + num_seqs.
extern "C" int pico_decay_chunks(const void* x, int ld, int q_col, int k_col, int v_col, const int* cu_seqlens, const int* state_slots,
                                 const float* decay, float* state, float* out, float* ws, int num_seqs, int T, int H, int dk, int dv,
                                 float qscale, int num_slots, int chunks, int silu, hipStream_t stream) {
  PICO_REQUIRE(num_seqs >= 0 && T >= 0 && H > 0 && H <= 65535 && dk > 0 && dv > 0 && num_slots > 0, "pico_decay_chunks: bad sizes");
  PICO_REQUIRE(dk <= 128 && dk % 8 == 0 && dv % 8 == 0, "pico_decay_chunks: keys of a multiple of 8 up to 128 and values of a multiple of 8, got %d and %d", dk, dv);
  PICO_REQUIRE(q_col >= 0 && k_col >= 0 && v_col >= 0 && ld >= q_col + H * dk && ld >= k_col + H * dk && ld >= v_col + H * dv,
               "pico_decay_chunks: the row of %d columns does not hold q, k and v", ld);
  PICO_REQUIRE((ld | q_col | k_col | v_col) % 8 == 0 && (uintptr_t)x % 16 == 0, "pico_decay_chunks: rows and columns must start on 16 bytes");
  PICO_REQUIRE(chunks >= T / DC_CHUNK + num_seqs && ws && state && out && decay,
               "pico_decay_chunks: chunks need room for their states and must cover the step's tokens");
  PICO_REQUIRE((dv + 63) / 64 <= 65535 && (dk * dv + 255) / 256 <= 65535, "pico_decay_chunks: sizes beyond the grid");
  if (num_seqs == 0 || T == 0) return 0;
  const ChunkArgs a{(const bf16_t*)x, ld, q_col, k_col, v_col, cu_seqlens, state_slots, decay, state, ws, out, H, dk, dv, num_slots, num_seqs, chunks, silu, qscale,
                    nullptr, nullptr, nullptr, 1};
  return pick_chunks<false>(a, num_seqs, stream);
}

// The same with a decay `g` and a factor `beta` on the written key of every token and head (float32 [T, H] each) and `share`
// heads to a head of q and k; x as it stands (no silu), q and k of head h from columns q_col + h / share * dk, ..  ws_decay
// float32 [chunks, H].
extern "C" int pico_ssd_chunks(const void* x, int ld, int q_col, int k_col, int v_col, const int* cu_seqlens, const int* state_slots,
                               const float* g, const float* beta, float* state, float* out, float* ws, float* ws_decay, int num_seqs,
                               int T, int H, int share, int dk, int dv, int num_slots, int chunks, hipStream_t stream) {
  PICO_REQUIRE(num_seqs >= 0 && T >= 0 && H > 0 && H <= 65535 && dk > 0 && dv > 0 && num_slots > 0 && share > 0 && H % share == 0,
               "pico_ssd_chunks: bad sizes");
  PICO_REQUIRE(dk <= 128 && dk % 8 == 0 && dv % 8 == 0, "pico_ssd_chunks: keys of a multiple of 8 up to 128 and values of a multiple of 8, got %d and %d", dk, dv);
  PICO_REQUIRE(q_col >= 0 && k_col >= 0 && v_col >= 0 && ld >= q_col + H / share * dk && ld >= k_col + H / share * dk && ld >= v_col + H * dv,
               "pico_ssd_chunks: the row of %d columns does not hold q, k and v", ld);
  PICO_REQUIRE((ld | q_col | k_col | v_col) % 8 == 0 && (uintptr_t)x % 16 == 0, "pico_ssd_chunks: rows and columns must start on 16 bytes");
  PICO_REQUIRE(chunks >= T / DC_CHUNK + num_seqs && ws && ws_decay && state && out && g && beta,
               "pico_ssd_chunks: chunks need room for their states and must cover the step's tokens");
  PICO_REQUIRE((dv + 63) / 64 <= 65535 && (dk * dv + 255) / 256 <= 65535, "pico_ssd_chunks: sizes beyond the grid");
  if (num_seqs == 0 || T == 0) return 0;
  const ChunkArgs a{(const bf16_t*)x, ld, q_col, k_col, v_col, cu_seqlens, state_slots, nullptr, state, ws, out, H, dk, dv, num_slots, num_seqs, chunks, 0, 1.0f,
                    g, beta, ws_decay, share};
  return pick_chunks<true>(a, num_seqs, stream);
}
