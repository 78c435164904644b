// Prompt portions of attention through a latent, with the heads' own keys and values: bfloat16, compiled for one set of sizes
// (unrotated and rotated key entries of a head, value entries, entries of the latent).
//
// The cache keeps a latent c and a rotated part kr a token.  Single tokens attend in the latent's space, where keys are
// rank + rot and values rank entries for every head; a portion of many tokens pays that for every (token, key) pair, and is
// better off with a head's own keys and values, which are products of the latents, once a key:
//   k_h = [Wuk_h c | kr],  v_h = Wuv_h c
// (12 heads, 128 + 64 and 128 entries, a latent of 256 + 64: 320 multiplications a pair instead of 576).
//   latent_expand_kernel   the keys and values of all heads for all tokens of the portions' sequences, 64 tokens a tile:
//                          kx [tile][head][64][D], vx [tile][head][V][64] (values transposed), kr [tile][64][R]
//   latent_prompt_kernel   attention over them
//   latent_join_kernel     puts together the tiles whose keys were shared by several workgroups
// Sequences are the step's from `lead` on (the ones in front of them are single tokens and not served here).
#include "common.h"

#if !defined(PICO_LAT_D) || !defined(PICO_LAT_R) || !defined(PICO_LAT_V) || !defined(PICO_LAT_RANK)
#error "compile with -DPICO_LAT_D=<key> -DPICO_LAT_R=<rotated> -DPICO_LAT_V=<value> -DPICO_LAT_RANK=<latent>"
#endif
constexpr int D = PICO_LAT_D, R = PICO_LAT_R, V = PICO_LAT_V, RANK = PICO_LAT_RANK;
static_assert((D == 32 || D == 64 || D == 128) && (R == 32 || R == 64 || R == 128) && (V == 32 || V == 64 || V == 128), "sizes of 32, 64 or 128");
static_assert(RANK % 32 == 0 && RANK >= 32 && RANK <= 256, "a latent of whole 32s up to 256");

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int TK = 64;                     // keys of a tile, the unit in which keys are dealt out
constexpr int TQ = 128;                    // queries of a workgroup: 32 a wave
constexpr int PART_ROW = V + 4;            // floats of a row of a part: sums, maximum, sum of the weights, padding

template <int N> struct Int { static constexpr int value = N; };

struct LatentArgs {
  const bf16_t* q;                         // [T, >= H (D + R)], rows and heads on 8 bytes
  const float* cos_sin;                    // [T, R / 2, 2]
  const bf16_t *k_cache, *uk, *uv;         // latents [page][P][RANK + R]; [H D, RANK], [H V, RANK]
  const int *block_table, *cu_seqlens, *context_lens;
  bf16_t *kx, *vx, *kr, *out;
  float* part;                             // [H][slots][2][TQ][PART_ROW]
  const bf16_t* gate;
  int q_stride, gate_stride, out_stride, H, num_seqs, max_pages, num_pages, pshift, cap_tiles, slots, least, num_tokens, first_token;
  float scale;
};

// Tiles of TQ queries and the tiles of keys that each reads, of a sequence of `ctx` tokens of which n are new: query tile i
// reads ceil(keys up to its last query / 64); whole tiles of queries end 128 keys apart.
__device__ __forceinline__ int units_before(int i, int first) { return i * first + i * (i + 1); }
__device__ __forceinline__ int seq_tiles(int n, int ctx) { return n > 0 ? (ctx + TK - 1) / TK : 0; }
__device__ __forceinline__ int seq_first(int n, int ctx) { return (ctx - n + TK - 1) / TK; }
__device__ __forceinline__ int seq_units(int n, int ctx) {
  const int whole = n / TQ;
  return units_before(whole, seq_first(n, ctx)) + (n % TQ ? (ctx + TK - 1) / TK : 0);
}
static_assert(TQ == 2 * TK, "units_before: a whole tile of queries adds two tiles of keys");

// tiles of keys of a piece
__device__ __forceinline__ int piece(const LatentArgs& a, int total) { return max(a.least, (total + a.slots - 1) / a.slots); }

struct Place { int b, tok0, n, ctx, units, tiles; };      // a sequence, and what lies in front of it

__device__ __forceinline__ int wave_scan(int v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int d = 1; d < 64; d *= 2) {
    const int o = __shfl_up(v, d);
    if (lane >= d) v += o;
  }
  return v;
}

// The first sequence for which pick(first token, new tokens, units in front, units up to its end, tiles in front, up to its
// end) holds; all lanes of the wave alike.  total: the units of all sequences, total_tiles: their tiles of keys.
template <typename Pick>
__device__ __forceinline__ bool find_place(const LatentArgs& a, Place& at, int& total, int& total_tiles, Pick pick) {
  const int lane = threadIdx.x & 63;
  int units0 = 0, tiles0 = 0;
  bool found = false;
  for (int base = 0; base < a.num_seqs; base += 64) {
    const int b = base + lane;
    const bool real = b < a.num_seqs;
    const int t0 = real ? a.cu_seqlens[b] : 0, n = real ? a.cu_seqlens[b + 1] - t0 : 0, c = real ? a.context_lens[b] : 0;
    const int u = seq_units(n, c), k = seq_tiles(n, c), ui = wave_scan(u), ki = wave_scan(k);
    const unsigned long long hit = __builtin_amdgcn_ballot_w64(real && n > 0 && pick(t0, n, units0 + ui - u, units0 + ui, tiles0 + ki - k, tiles0 + ki));
    if (!found && hit) {
      const int l = __builtin_ctzll(hit);
      at.b = base + l;
      at.tok0 = __builtin_amdgcn_readlane(t0, l);
      at.n = __builtin_amdgcn_readlane(n, l);
      at.ctx = __builtin_amdgcn_readlane(c, l);
      at.units = units0 + __builtin_amdgcn_readlane(ui - u, l);
      at.tiles = tiles0 + __builtin_amdgcn_readlane(ki - k, l);
      found = true;
    }
    units0 += __builtin_amdgcn_readlane(ui, 63);
    tiles0 += __builtin_amdgcn_readlane(ki, 63);
  }
  total = units0;
  total_tiles = tiles0;
  return found;
}

// ---- keys and values of the heads ---------------------------------------------------------------------------------------
// A wave has 32 outputs of a head (of its keys or of its values), whose matrix rows stay in its registers (RANK / 8 of them a
// lane); the four waves of a workgroup share the latents that stream by, 64 tokens at a time, through two LDS buffers.  (A wave
// reading its latents from the L2 by itself: 32 lines an instruction, 16 bytes of each, and as many instructions as products;
// 6,144 tokens of 12 heads about 50 us, so 27; what is left is the latency of a tile's copy, five tiles a workgroup.)  A row in LDS is an odd number of 16-byte chunks: 16 rows meet every bank once.
// v_mfma_f32_32x32x16_bf16 (A 32x16, B 16x32): lane l = (c, h) supplies A[c][8 h + 0..7] and B[8 h + 0..7][c] and receives
// D[8 (r / 4) + 4 h + r % 4][c] in register r: what lies along the rows is contiguous in a lane, so keys are [output x token] and
// values [token x output].
constexpr int EB = RANK / 16, EROW = RANK / 8 + 1, ECOPIES = (TK * EROW + 255) / 256, ESTAGE = ECOPIES * 4096;
__global__ __launch_bounds__(256, 2) void latent_expand_kernel(const LatentArgs a) {
#ifdef __HIP_DEVICE_COMPILE__
  extern __shared__ __attribute__((aligned(16))) char le_smem[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, l32 = lane & 31, h = lane >> 5;
  constexpr int KB = D / 32, NB = KB + V / 32, ROW = RANK + R;
  const int P = 1 << a.pshift;
  Place at{0, 0, 0, 0, 0, 0};
  int total, tiles;
  find_place(a, at, total, tiles, [](int, int, int, int, int, int) { return false; });
  tiles = min(tiles, a.cap_tiles);
  // `at`: the sequence of the tile
  auto follow = [&](int tile) {
    if (tile >= at.tiles && tile < at.tiles + seq_tiles(at.n, at.ctx)) return;
    int x, y;
    find_place(a, at, x, y, [&](int, int, int, int, int from, int to) { return tile >= from && tile < to; });
  };
  // the latent of token `key` of a sequence: its page, and where it is
  auto page_of = [&](int b, int key) { return a.block_table[(size_t)b * a.max_pages + min(key >> a.pshift, a.max_pages - 1)]; };
  auto row_at = [&](int page, int key) { return a.k_cache + (((size_t)min(max(page, 0), a.num_pages - 1) << a.pshift) + (key & (P - 1))) * ROW; };
  int tile = blockIdx.y;
  const int step = gridDim.y;
  if (tile >= tiles) return;
  if (blockIdx.x == gridDim.x - 1) {       // the rotated parts, as they are
    constexpr int CH = R / 8;
    for (; tile < tiles; tile += step) {
      follow(tile);
      for (int i = threadIdx.x; i < TK * CH; i += 256) {
        const int key = min((tile - at.tiles) * TK + i / CH, at.ctx - 1);
        *reinterpret_cast<u32x4*>(a.kr + ((size_t)tile * TK + i / CH) * R + i % CH * 8) =
            *reinterpret_cast<const u32x4*>(row_at(page_of(at.b, key), key) + RANK + i % CH * 8);
      }
    }
    return;
  }
  const int gb = min((int)blockIdx.x * 4 + wave, a.H * NB - 1);      // (waves behind the last block of outputs make it again)
  const int head = gb / NB, ob = gb % NB;
  const bool keys = ob < KB;
  const bf16_t* wrow = (keys ? a.uk + ((size_t)head * D + 32 * ob + l32) * RANK : a.uv + ((size_t)head * V + 32 * (ob - KB) + l32) * RANK) + 8 * h;
  u32x4 w[EB];
#pragma unroll
  for (int s = 0; s < EB; s++) w[s] = *reinterpret_cast<const u32x4*>(wrow + 16 * s);
  // chunk threadIdx.x + 256 i of a stage is part c of row r; the chunk behind a row's last is padding (any bytes)
  // A tile's pages are looked up two tiles before it is worked on, in front of the copies of the tile between, and are waited
  // for in front of the stores: loads, copies and stores return in one order.
  const bf16_t* from[ECOPIES];
  int key[ECOPIES], page[ECOPIES], beyond = 0, later = 0, last = 0;      // beyond: a tile's first token minus the tokens that there are
  auto lookup = [&](int t) {
    follow(t);
#pragma unroll
    for (int i = 0; i < ECOPIES; i++) {
      key[i] = min((t - at.tiles) * TK + min((int)(threadIdx.x + 256 * i) / EROW, TK - 1), at.ctx - 1);
      page[i] = page_of(at.b, key[i]);
    }
    last = (t - at.tiles) * TK - at.ctx;
  };
  auto arrived = [&] {
#pragma unroll
    for (int i = 0; i < ECOPIES; i++) {
      const int c = (int)(threadIdx.x + 256 * i) % EROW;
      from[i] = row_at(page[i], key[i]) + (c < EROW - 1 ? c * 8 : 0);
      asm volatile("" : "+v"(from[i]));
    }
    beyond = later;
    later = last;
  };
  auto ask = [&](int buf) {
#pragma unroll
    for (int i = 0; i < ECOPIES; i++)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)from[i],
                                       (__attribute__((address_space(3))) void*)(le_smem + buf * ESTAGE + wave * 1024 + i * 4096), 16, 0, 0);
  };
  int buf = 0;
  lookup(tile);
  arrived();
  ask(0);
  lookup(min(tile + step, tiles - 1));
  arrived();
  bool first = true;
  for (; tile < tiles; tile += step) {
    // this wave's copies have landed (all but its four stores of the tile before, which came after them) and its reads are done;
    // behind the barrier all have, and nobody reads the other buffer
    if (first) __builtin_amdgcn_s_waitcnt(0x0070);
    else __builtin_amdgcn_s_waitcnt(0x0074);
    first = false;
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    lookup(min(tile + 2 * step, tiles - 1));
    __builtin_amdgcn_sched_barrier(0);
    ask(buf ^ 1);                      // (behind the last tile that one again: a branch would make the wait below one for the copies too)
    const int edge = beyond;
    const char* src = le_smem + buf * ESTAGE + (l32 * EROW + h) * 16;
#pragma unroll
    for (int k = 0; k < 2; k++, src += 32 * EROW * 16) {
      f32x16 acc = {};
      auto latent = [&](int s) { return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(src + 32 * s)); };
      bf16_t* dst;
      if (keys) {
#pragma unroll
        for (int s = 0; s < EB; s++) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, w[s]), latent(s), acc, 0, 0, 0);
        dst = a.kx + (((size_t)tile * a.H + head) * TK + 32 * k + l32) * D + 32 * ob + 8 * h;
      } else {
#pragma unroll
        for (int s = 0; s < EB; s++) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(latent(s), __builtin_bit_cast(bf16x8, w[s]), acc, 0, 0, 0);
        if (edge + TK > 0) {             // tokens that there are not have values of zero
#pragma unroll
          for (int r = 0; r < 16; r++)
            if (edge + 32 * k + 8 * (r / 4) + 4 * h + r % 4 >= 0) acc[r] = 0.f;
        }
        dst = a.vx + (((size_t)tile * a.H + head) * V + 32 * (ob - KB) + l32) * TK + 32 * k + 8 * h;
      }
      if (k == 0) {
        __builtin_amdgcn_sched_barrier(0);
        arrived();
        __builtin_amdgcn_sched_barrier(0);
      }
      // half h has entries 8 g + 4 h + 0..3: exchanged so that it has 16 j + 8 h + 0..7, a store of 16 bytes
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const auto lo = __builtin_amdgcn_permlane32_swap(pack2_bf16(acc[8 * j], acc[8 * j + 1]), pack2_bf16(acc[8 * j + 4], acc[8 * j + 5]), false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap(pack2_bf16(acc[8 * j + 2], acc[8 * j + 3]), pack2_bf16(acc[8 * j + 6], acc[8 * j + 7]), false, false);
        *reinterpret_cast<u32x4*>(dst + 16 * j) = u32x4{lo[0], hi[0], lo[1], hi[1]};
      }
    }
    buf ^= 1;
  }
  __builtin_amdgcn_s_waitcnt(0x0070);                        // the last copies are in before LDS is given back
#endif
}

// ---- attention ----------------------------------------------------------------------------------------------------------
// A workgroup of four waves has 128 queries of a head, 32 a wave; keys and values of 64 tokens go from memory straight to one
// of two LDS buffers while the other's are multiplied, one barrier a tile.  The two buffers take half of a compute unit's LDS to
// the byte: the two workgroups there run apart, one's softmax under the other's products.
// Scores are S^T = K Q^T on v_mfma_f32_32x32x16_bf16: a query is a column, shared by lanes l and l ^ 32.  Which key is row a of a
// block of 32 is free; it is the key whose number is a with bits 2 and 3 exchanged, so that registers 8 s .. 8 s + 7 of half h
// hold keys 16 s + 8 h + 0..7, rounded to bfloat16 the B operand of O^T += V^T P^T whose A operand is 16 bytes of V^T.
// The sixteen-byte chunks of a row are xor-swizzled by the row so that 16 rows meet every bank once.
// The reference maximum of the softmax may lag by 8 in the exponent (p <= 256, harmless in 32-bit sums and in bfloat16 p);
// sums are rescaled only when a column outgrows that.
//
// Work is dealt by tiles of keys: the tiles of all query tiles of a head stand in a row, cut into `slots` pieces of one length, a
// workgroup each, whatever the portions' lengths and prefixes; a query tile that lies in several pieces leaves its sums
// in `part` (a piece has at most two such: its first and its last).  Heads' pieces run on a die side by side and
// share their keys in its L2.  (A piece has at least four tiles: 4, 8, 16 and 32 of them 55, 62, 69 and 98 us for 1,377 tokens of
// 12 heads, 49, 48, 57 and 78 for 64 behind 4,000, the three launches together.)
//
// Measured, the launch alone: 2,048 tokens of 12 heads behind 4,096, sizes 128 + 64, 128 and 256: 98 us, 0.82 PFLOP/s; bound by the
// chain of a tile (operands from LDS, products, softmax) where two waves a SIMD are not enough to cover it, and 23 us of ends: a
// piece's first copies and queries, and its sums on their way out.  With both other launches 145 us, where attention in the
// latent's space, its queries' and outputs' products and their copies took 454; 2,048 tokens without a prefix 73 and 211.
constexpr int K_BYTES = TK * D * 2, R_BYTES = TK * R * 2, V_BYTES = TK * V * 2, STAGE = K_BYTES + R_BYTES + V_BYTES;
constexpr int QS = (D + R) / 16, DS = D / 16, VT = V / 32, QG = QS % 4 == 0 ? 4 : 2;      // steps of a score, values' blocks; steps of a group
template <int N> __device__ __forceinline__ int swizzle(int row) { return N >= 16 ? row & 15 : (row / (16 / N)) & (N - 1); }   // N: chunks of a row

// Of eight bfloat16 values: all bits of those that are Inf or NaN (an exponent of ones carries into the sign's place).
__device__ __forceinline__ u32x4 odd_entries(u32x4 v) { return ((((v & 0x7f807f80u) + 0x00800080u) & 0x80008000u) >> 15) * 0xffffu; }

#ifdef __HIP_DEVICE_COMPILE__
template <int BYTES>
__device__ __forceinline__ void copy_block(const void* src, char* dst, uint32_t off) {
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(src), 0, BYTES, 0x00020000);
#pragma unroll
  for (int i = 0; i < BYTES / 4096; i++)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(dst + i * 4096), 16, off + i * 4096, 0, 0, 0);
}
#endif

__global__ __launch_bounds__(256, 2) void latent_prompt_kernel(const LatentArgs a) {
#ifdef __HIP_DEVICE_COMPILE__
  extern __shared__ __attribute__((aligned(16))) char lp_smem[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, col = lane & 31, h = lane >> 5;
  const int idx = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  if (idx >= a.H * a.slots) return;
  const int head = idx / a.slots, slot = idx - head * a.slots;
  Place at;
  int total, tiles;
  find_place(a, at, total, tiles, [](int, int, int, int, int, int) { return false; });
  const int per = piece(a, total), x0 = slot * per, x1 = min(total, x0 + per);
  if (x0 >= x1) return;
  if (!find_place(a, at, total, tiles, [&](int, int, int from, int to, int, int) { return x0 >= from && x0 < to; })) return;
  // the query tile of the first unit: the largest i with units_before(i) <= its place among the sequence's
  int first = seq_first(at.n, at.ctx), ntiles = (at.n + TQ - 1) / TQ, i = 0;
  {
    const int x = x0 - at.units;
    const float p = (float)(first + 1);
    i = min(max((int)((sqrtf(p * p + 4.f * (float)x) - p) * 0.5f), 0), ntiles - 1);
    while (i > 0 && units_before(i, first) > x) i--;
    while (i + 1 < ntiles && units_before(i + 1, first) <= x) i++;
  }
  int unit = x0 - at.units - units_before(i, first);         // the tile of keys that is next, of `count`
  auto count_of = [&](int tile) { return (min(at.ctx, at.ctx - at.n + (tile + 1) * TQ) + TK - 1) / TK; };

  // where this thread's chunks come from (a copy of 256 threads is 4 KB: whole periods of the swizzle)
  auto source = [&](auto chunks) {
    constexpr int N = decltype(chunks)::value;
    const int row = threadIdx.x / N;
    return (uint32_t)((row * N + ((threadIdx.x % N) ^ swizzle<N>(row))) * 16);
  };
  const uint32_t koff = source(Int<D / 8>()), roff = source(Int<R / 8>()), voff = source(Int<TK / 8>());
  auto ask = [&](int buf, int tile) {
    tile = min(tile, a.cap_tiles - 1);
    char* dst = lp_smem + buf * STAGE + wave * 1024;
    copy_block<K_BYTES>(a.kx + ((size_t)tile * a.H + head) * (TK * D), dst, koff);
    copy_block<R_BYTES>(a.kr + (size_t)tile * (TK * R), dst + K_BYTES, roff);
    copy_block<V_BYTES>(a.vx + ((size_t)tile * a.H + head) * (TK * V), dst + K_BYTES + R_BYTES, voff);
  };
  // where this lane's operands lie in a buffer
  const int krow = (col & ~12) | ((col & 4) << 1) | ((col & 8) >> 1);
  const int ksw = swizzle<D / 8>(krow), rsw = swizzle<R / 8>(krow), vsw = swizzle<TK / 8>(col);
  const int kat = krow * (D * 2), rat = K_BYTES + krow * (R * 2), vat = K_BYTES + R_BYTES + col * (TK * 2);
  const float c = a.scale * 1.4426950408889634f;

  int buf = 0;
  ask(0, at.tiles + unit);
  for (int x = x0; x < x1;) {
    const int count = count_of(i), from = unit, to = min(count, unit + x1 - x);
    const int prefix = at.ctx - at.n, wave_q0 = i * TQ + wave * 32, q_idx = wave_q0 + col, q_pos = prefix + q_idx;
    const bool q_ok = q_idx < at.n, active = wave_q0 < at.n;
    const int w_first = prefix + wave_q0, w_last = min(w_first + 31, at.ctx - 1);
    const size_t t = (size_t)(at.tok0 + (q_ok ? q_idx : 0));
    bf16x8 qf[QS];
    {
      const bf16_t* qrow = a.q + t * a.q_stride + (size_t)head * (D + R) + 8 * h;
#pragma unroll
      for (int s = 0; s < QS; s++) {
        const uint2 lo = *reinterpret_cast<const uint2*>(qrow + 16 * s), hi = *reinterpret_cast<const uint2*>(qrow + 16 * s + 4);
        qf[s] = __builtin_bit_cast(bf16x8, u32x4{lo.x, lo.y, hi.x, hi.y});
      }
      const float* cs = a.cos_sin + t * R + 8 * h;         // the rotated part: neighbours in pairs
#pragma unroll
      for (int s = DS; s < QS; s++) {
        u32x4 v = __builtin_bit_cast(u32x4, qf[s]);
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const float co = cs[16 * (s - DS) + 2 * j], si = cs[16 * (s - DS) + 2 * j + 1];
          const float u = __uint_as_float(v[j] << 16), w = __uint_as_float(v[j] & 0xffff0000u);
          v[j] = pack2_bf16(u * co - w * si, w * co + u * si);
        }
        qf[s] = __builtin_bit_cast(bf16x8, v);
      }
    }
    float m = -INFINITY, l = 0.f;
    bool again = false;                                      // a value that is not finite was left out
    f32x16 o[VT];
#pragma unroll
    for (int tt = 0; tt < VT; tt++) o[tt] = f32x16{};

    auto attend = [&](int key0, bool partly) {
      const char* b = lp_smem + buf * STAGE;
      f32x16 s[2];
      // operands in groups, each asked for under the products of the group before (left to itself the compiler asks for all it has
      // registers for, and for more)
      {
        u32x4 ka[2][QG];
        auto read = [&](int set, int g) {
#pragma unroll
          for (int j = 0; j < QG; j++) {
            const int k = g * QG / QS, st = g * QG % QS + j;
            ka[set][j] = *reinterpret_cast<const u32x4*>(st < DS ? b + kat + k * (32 * D * 2) + (((2 * st + h) ^ ksw) << 4)
                                                                 : b + rat + k * (32 * R * 2) + (((2 * (st - DS) + h) ^ rsw) << 4));
          }
        };
        read(0, 0);
#pragma unroll
        for (int g = 0; g < 2 * QS / QG; g++) {
          if (g + 1 < 2 * QS / QG) read((g + 1) & 1, g + 1);
          __builtin_amdgcn_sched_barrier(0);
          const int k = g * QG / QS, st = g * QG % QS;
          if (st == 0) s[k] = f32x16{};
#pragma unroll
          for (int j = 0; j < QG; j++) s[k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, ka[g & 1][j]), qf[st + j], s[k], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if (partly) {
        const int last = q_pos - key0 - 8 * h;
#pragma unroll
        for (int k = 0; k < 2; k++)
#pragma unroll
          for (int r = 0; r < 16; r++)
            if (32 * k + 16 * (r / 8) + r % 8 > last) s[k][r] = -INFINITY;
      }
      float mx = -INFINITY;
#pragma unroll
      for (int k = 0; k < 2; k++)
#pragma unroll
        for (int r = 0; r < 16; r++) mx = fmaxf(mx, s[k][r]);
      mx = max_across_32(mx);
      const float m_new = fmaxf(m, mx);
      if (__builtin_amdgcn_ballot_w64((m_new - m) * c > 8.0f) != 0) {      // (also while the reference is -inf)
        const float alpha = __builtin_amdgcn_exp2f((m - (m_new == -INFINITY ? 0.f : m_new)) * c);
        l *= alpha;
        m = m_new;
#pragma unroll
        for (int tt = 0; tt < VT; tt++) o[tt] *= alpha;
      }
      const float mc = (m == -INFINITY ? 0.f : m) * c;
      bf16x8 p[4];
      float sum = 0.f;
#pragma unroll
      for (int k = 0; k < 2; k++) {
#pragma unroll
        for (int r = 0; r < 16; r++) {
          s[k][r] = __builtin_amdgcn_exp2f(fmaf(s[k][r], c, -mc));
          sum += s[k][r];
        }
#pragma unroll
        for (int g = 0; g < 2; g++)
          p[2 * k + g] = __builtin_bit_cast(bf16x8, u32x4{pack2_bf16(s[k][8 * g], s[k][8 * g + 1]), pack2_bf16(s[k][8 * g + 2], s[k][8 * g + 3]),
                                                          pack2_bf16(s[k][8 * g + 4], s[k][8 * g + 5]), pack2_bf16(s[k][8 * g + 6], s[k][8 * g + 7])});
      }
      l += sum;
      __builtin_amdgcn_sched_barrier(0);
      auto value = [&](int ks, int tt) { return *reinterpret_cast<const u32x4*>(b + vat + tt * (32 * TK * 2) + (((2 * ks + h) ^ vsw) << 4)); };
      u32x4 va[2][VT];
#pragma unroll
      for (int tt = 0; tt < VT; tt++) va[0][tt] = value(0, tt);
#pragma unroll
      for (int ks = 0; ks < 4; ks++) {
        if (ks < 3) {
#pragma unroll
          for (int tt = 0; tt < VT; tt++) va[(ks + 1) & 1][tt] = value(ks + 1, tt);
        }
        if (partly) {
          // a value that is not finite waits (below) for the columns that see its key: a weight of zero would not hide it
          u32x4 any{0, 0, 0, 0};
#pragma unroll
          for (int tt = 0; tt < VT; tt++) {
            const u32x4 odd = odd_entries(va[ks & 1][tt]);
            any |= odd;
            va[ks & 1][tt] &= ~odd;
          }
          again = again || __any((any[0] | any[1] | any[2] | any[3]) != 0);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int tt = 0; tt < VT; tt++)
          o[tt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, va[ks & 1][tt]), p[ks], o[tt], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    };

    // this query tile's parameters for the way out; `at`, i and unit go on with what is asked for next
    const int tok0 = at.tok0, here = i, tile0 = at.tiles;
    for (int u = from; u < to; u++, x++) {
      // the unit behind this one
      unit++;
      if (unit == count) {
        unit = 0;
        if (++i == ntiles && x + 1 < x1) {                   // the next sequence that brings tokens
          do {
            at.units += seq_units(at.n, at.ctx);
            at.tiles += seq_tiles(at.n, at.ctx);
            at.b++;
            at.tok0 = a.cu_seqlens[at.b];
            at.n = a.cu_seqlens[at.b + 1] - at.tok0;
            at.ctx = a.context_lens[at.b];
          } while (at.n == 0 && at.b + 1 < a.num_seqs);
          ntiles = (at.n + TQ - 1) / TQ;
          i = 0;
        }
      }
      __builtin_amdgcn_s_waitcnt(0x0070);                    // this wave's copies have landed and its reads are done; behind the barrier all have,
      __builtin_amdgcn_s_barrier();                          // and nobody reads the other buffer
      __builtin_amdgcn_sched_barrier(0);
      if (x + 1 < x1) ask(buf ^ 1, at.tiles + unit);
      const int key0 = u * TK;
      if (active && key0 <= w_last) attend(key0, key0 + TK - 1 > w_first);
      buf ^= 1;
    }
    if (again) {
      // any weight makes of a value that is not finite what it is (not a number, or infinite with its sign)
#pragma unroll 1
      for (int key = max(from * TK, w_first / TK * TK); key <= min(to * TK - 1, w_last); key++) {
        const bf16_t* v = a.vx + ((size_t)min(tile0 + key / TK, a.cap_tiles - 1) * a.H + head) * (TK * V) + key % TK + 4 * h * TK;
#pragma unroll
        for (int tt = 0; tt < VT; tt++)
#pragma unroll
          for (int r = 0; r < 16; r++) {
            const float x = bf16_to_f32(v[(32 * tt + 8 * (r / 4) + r % 4) * TK]);
            o[tt][r] += key <= q_pos && !(fabsf(x) < INFINITY) ? x : 0.f;
            __builtin_amdgcn_sched_barrier(0);               // (few registers, not many loads: this is rare)
          }
      }
    }
    l = sum_across_32(l);
    if (!q_ok) {                                             // (a column without a query)
    } else if (from > 0 || to < count) {
      float* row = a.part + ((((size_t)head * a.slots + slot) * 2 + (from > 0 ? 0 : 1)) * TQ + wave * 32 + col) * PART_ROW;
#pragma unroll
      for (int tt = 0; tt < VT; tt++)
#pragma unroll
        for (int g = 0; g < 4; g++)
          *reinterpret_cast<f32x4*>(row + 32 * tt + 8 * g + 4 * h) = f32x4{o[tt][4 * g], o[tt][4 * g + 1], o[tt][4 * g + 2], o[tt][4 * g + 3]};
      if (h == 0) {
        row[V] = m;
        row[V + 1] = l;
      }
    } else {
      const size_t row = (size_t)(tok0 + here * TQ + wave * 32 + col);
      float f = 1.0f / l;
      if (a.gate) f *= 1.0f / (1.0f + __expf(-bf16_to_f32(a.gate[row * a.gate_stride + head])));
      bf16_t* dst = a.out + row * a.out_stride + (size_t)head * V + 4 * h;
#pragma unroll
      for (int tt = 0; tt < VT; tt++)
#pragma unroll
        for (int g = 0; g < 4; g++)
          *reinterpret_cast<uint2*>(dst + 32 * tt + 8 * g) = make_uint2(pack2_bf16(o[tt][4 * g] * f, o[tt][4 * g + 1] * f), pack2_bf16(o[tt][4 * g + 2] * f, o[tt][4 * g + 3] * f));
    }
  }
#endif
}

// A wave a token and head: the parts of its query tile.  Tiles that lie in one piece have their result already.
__global__ __launch_bounds__(256) void latent_join_kernel(const LatentArgs a) {
  const int t = a.first_token + blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63, head = blockIdx.y;
  if (t >= a.num_tokens) return;
  Place at;
  int total, tiles;
  if (!find_place(a, at, total, tiles, [&](int t0, int n, int, int, int, int) { return t >= t0 && t < t0 + n; })) return;
  const int per = piece(a, total);
  const int i = (t - at.tok0) / TQ, u0 = at.units + units_before(i, seq_first(at.n, at.ctx));
  const int count = (min(at.ctx, at.ctx - at.n + (i + 1) * TQ) + TK - 1) / TK, s0 = u0 / per, n = (u0 + count - 1) / per + 1 - s0;
  if (n == 1) return;
  const float c = a.scale * 1.4426950408889634f;
  const float* base = a.part + (((size_t)head * a.slots + s0) * 2 * TQ + (t - at.tok0) % TQ) * PART_ROW;
  auto row_of = [&](int s) { return base + (s * 2 + ((s0 + s) * per > u0 ? 0 : 1)) * (TQ * PART_ROW); };
  // lane s: part s, s + 64, ..: its maximum and the sum of its weights
  float M = -INFINITY, L = 0.f;
  for (int s = lane; s < n; s += 64) M = fmaxf(M, row_of(s)[V]);
  M = wave_max(M);
  constexpr int PER_LANE = V <= 64 ? 1 : V / 64;
  float o[PER_LANE] = {};
  const int d = lane * PER_LANE < V ? lane * PER_LANE : 0;
  for (int first = 0; first < n; first += 64) {
    float w = 0.f;
    if (first + lane < n) {
      const float* row = row_of(first + lane);
      w = row[V] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((row[V] - M) * c);
      L += w * row[V + 1];
    }
    const int many = min(64, n - first);
#pragma unroll 8
    for (int s = 0; s < many; s++) {
      const float* row = row_of(first + s) + d;
      const float ws = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w), s));
#pragma unroll
      for (int j = 0; j < PER_LANE; j++) o[j] = fmaf(ws, row[j], o[j]);
    }
  }
  float f = 1.0f / wave_sum(L);
  if (a.gate) f *= 1.0f / (1.0f + __expf(-bf16_to_f32(a.gate[(size_t)t * a.gate_stride + head])));
  bf16_t* dst = a.out + (size_t)t * a.out_stride + (size_t)head * V + d;
  if (lane * PER_LANE < V) {
    if constexpr (PER_LANE == 2) *reinterpret_cast<uint32_t*>(dst) = pack2_bf16(o[0] * f, o[1] * f);
    else dst[0] = f32_to_bf16(o[0] * f);
  }
}

// kx, vx, kr: workspaces for cap_tiles tiles of 64 tokens (every sequence's last may be partly empty; the layouts stand at the top);
// part: slots pieces a head, of at least `least` tiles of keys.  block_table, cu_seqlens and context_lens begin with the first
// portion's sequence; cu_seqlens counts the step's tokens, of which the rows from first_token on are written.
extern "C" int pico_latent_prompt(const void* q, int q_stride, const float* cos_sin, const void* k_cache, const void* uk, const void* uv,
                                  const int* block_table, int max_pages, const int* cu_seqlens, const int* context_lens, int num_seqs,
                                  int first_token, int num_tokens, void* kx, void* vx, void* kr, int cap_tiles, float* part, int slots, int least,
                                  void* out, int out_stride, const void* gate, int gate_stride, int H, int d, int r, int v, int rank,
                                  int P, int num_pages, float scale, hipStream_t stream) {
  PICO_REQUIRE(d == D && r == R && v == V && rank == RANK, "pico_latent_prompt: built for %d + %d, %d and a latent of %d, asked for %d + %d, %d and %d",
               D, R, V, RANK, d, r, v, rank);
  PICO_REQUIRE(H > 0 && H <= 4096 && num_seqs > 0 && first_token >= 0 && num_tokens > first_token && num_tokens < (1 << 22) && max_pages > 0 &&
                   num_pages > 0 && slots > 0 && (long long)H * slots < (1 << 20), "pico_latent_prompt: bad sizes");
  PICO_REQUIRE(P >= 1 && (P & (P - 1)) == 0, "pico_latent_prompt: the page size must be a power of two, got %d", P);
  PICO_REQUIRE(cap_tiles > 0 && cap_tiles < (1 << 20), "pico_latent_prompt: room for %d tiles of keys", cap_tiles);
  PICO_REQUIRE(((long long)(num_tokens / TQ) + num_seqs) * cap_tiles < (1 << 30), "pico_latent_prompt: sizes beyond one launch");
  PICO_REQUIRE(q_stride >= H * (D + R) && q_stride % 4 == 0 && (uintptr_t)q % 8 == 0, "pico_latent_prompt: query rows must start on 8 bytes and hold all heads");
  PICO_REQUIRE(out_stride >= H * V && out_stride % 4 == 0 && (uintptr_t)out % 8 == 0, "pico_latent_prompt: output rows must start on 8 bytes and hold all heads");
  PICO_REQUIRE(gate == nullptr || gate_stride >= H, "pico_latent_prompt: gate rows must hold all heads");
  PICO_REQUIRE(((uintptr_t)k_cache | (uintptr_t)uk | (uintptr_t)uv | (uintptr_t)kx | (uintptr_t)vx | (uintptr_t)kr | (uintptr_t)part) % 16 == 0 &&
                   (uintptr_t)cos_sin % 4 == 0, "pico_latent_prompt: misaligned tensors");
  const LatentArgs a{(const bf16_t*)q, cos_sin, (const bf16_t*)k_cache, (const bf16_t*)uk, (const bf16_t*)uv, block_table, cu_seqlens, context_lens,
                     (bf16_t*)kx, (bf16_t*)vx, (bf16_t*)kr, (bf16_t*)out, part, (const bf16_t*)gate, q_stride, gate_stride, out_stride, H,
                     num_seqs, max_pages, num_pages, 31 - __builtin_clz(P), cap_tiles, slots, least, num_tokens, first_token, scale};
  static const hipError_t room = hipFuncSetAttribute((const void*)&latent_prompt_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * STAGE);
  PICO_REQUIRE(room == hipSuccess, "pico_latent_prompt: %s", hipGetErrorString(room));
  const int gx = (H * ((D + V) / 32) + 3) / 4 + 1;
  const int gy = 512 / gx < 1 ? 1 : 512 / gx < cap_tiles ? 512 / gx : cap_tiles;             // two workgroups a compute unit
  static const hipError_t more = hipFuncSetAttribute((const void*)&latent_expand_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * ESTAGE);
  PICO_REQUIRE(more == hipSuccess, "pico_latent_prompt: %s", hipGetErrorString(more));
  latent_expand_kernel<<<dim3(gx, gy), 256, 2 * ESTAGE, stream>>>(a);
  PICO_LAUNCH_CHECK();
  latent_prompt_kernel<<<(H * slots + 7) / 8 * 8, 256, 2 * STAGE, stream>>>(a);
  PICO_LAUNCH_CHECK();
  latent_join_kernel<<<dim3((num_tokens - first_token + 3) / 4, H), 256, 0, stream>>>(a);
  PICO_LAUNCH_CHECK();
  return 0;
}
