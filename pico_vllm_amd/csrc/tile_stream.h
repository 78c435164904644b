// The inner part of a tiled bfloat16 product on the matrix cores: tiles of 64 MB rows of X by 64 NB rows of W, both
// contiguous along k, four waves (2 x 2), each with MB x NB blocks of v_mfma_f32_32x32x16_bf16; one workgroup a compute
// unit, or two that hide each other's waits (ts_share).  Every sum runs over k in the same order whatever the tile: one chain,
// or SETS of them, the stage s in chain s % SETS, which `done` adds up.
//
// A stage is 64 k of all rows of the tile.  Its 128-byte rows go from memory straight to LDS (buffer_load .. lds, sixteen
// bytes a lane, whole lines), the sixteen-byte chunks of a row xor-swizzled by the row so that the operand reads (32 rows,
// one chunk each) meet every bank once.  What lies outside a matrix (rows behind the last, k behind K) is an offset behind
// the buffer's end and arrives as zeros: no clamps, no selects.
//
// With one or two waves a SIMD little else hides a wait, so the products of a quarter stage (16 k) run while the operands of the
// next are read, and the only barrier of a stage stands where its last operands are in registers: behind it the next
// stage has landed and this one's buffer is asked to fill for the stage after.  The stages of all of a workgroup's tiles
// are one sequence, so the next tile's first stages travel under the last products and the epilogue of this one.
//
// What bounds it, measured: operands that the L2 holds, a 256 x 128 stage takes 1,290 cycles (1,024 of products, 1,175 for
// its 48 KB at the 41 bytes a cycle at which a compute unit takes in lines), a 256 x 256 one 2,230 (2,048); from memory the
// latency of a copy shows, because LDS holds two or three stages (four of a 128 x 128 tile, BUFS): 0.8 to 0.9 us a 256 x 128 stage.  Lines asked for
// further ahead (four bytes each into the L2, 2 to 6 stages before their copies) made it slower (113 to 117 us and 122 to
// 145): the copies' counter retires in order, behind the far lines.
#pragma once
#include "common.h"

typedef __bf16 ts_bf16x8 __attribute__((ext_vector_type(8)));
typedef float ts_f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t ts_u32x4 __attribute__((ext_vector_type(4)));

#define TS_BK 64
#define TS_OUT 0x80000000u          // added to an offset: behind the end of any buffer (at most 2^31 - 1 bytes)

constexpr int ts_stage_bytes(int MB, int NB) { return (MB + NB) * 64 * TS_BK * 2; }
// workgroups that share a compute unit, and buffers of a workgroup
constexpr int ts_share(int MB, int NB) { return MB * NB <= 6 ? 2 : 1; }
constexpr int ts_buffers(int MB, int NB) { return ts_stage_bytes(MB, NB) * 3 * ts_share(MB, NB) <= 160 * 1024 ? 3 : 2; }
constexpr int ts_lds_bytes(int MB, int NB) { return ts_stage_bytes(MB, NB) * ts_buffers(MB, NB); }
// s_waitcnt: at most n vector memory operations outstanding; with `lds` also no LDS read
constexpr int ts_wait(int n, bool lds) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | ((lds ? 0 : 15) << 8); }

// workgroups for so many tiles where `most` run at once
constexpr int ts_grid(long long tiles, int most) { return tiles < most ? (int)((tiles + 7) / 8 * 8) : most; }

// Of `rows` rows dealt out in blocks of whole eights to `workers` workgroups: how many a block has (the last workgroups may have none).
__host__ __device__ inline int ts_bring_rows(int rows, int workers) { return ((rows + workers - 1) / workers + 7) / 8 * 8; }

#ifdef __HIP_DEVICE_COMPILE__      // (buffer resources exist on the device only)
// The rows of one operand of a tile, as what a lane asks for: `rsrc` over the matrix from the tile's first row on, and the
// byte offset of this lane's chunk in its row of each of the wave's copies (eight rows each), at k = 0.
template <int B>
struct TileRowsSource {
  __amdgpu_buffer_rsrc_t rsrc;
  uint32_t off[2 * B];
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t ts_buffer(const void* base, long long bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)min(bytes, (long long)0x7fffffff), 0x00020000);
}

// The tile a workgroup takes in round r of `tiles`, or -1.  Workgroups go to the dies in turn (the grid is a multiple of eight,
// ts_grid), and a die's share of a round is a run of neighbouring tiles; so is its share of a last round that is not full: an
// eighth of what is left, for the workgroups that came to the die first, one a compute unit while there are units.  (Dealt from the
// first die on, and grids that are no multiple of eight left as they came: gelu of 13,440 columns, K 1,536, 832 rows 55 us, 45
// so; 11,008 pairs, K 2,048, 832 rows 101, 86; 18,944 pairs, K 3,584, 300 rows 135, 117; the two products of 2,754 rows over 16
// experts of 2,240 x 1,536 149, 134; calls of whole rounds the same.)
__device__ __forceinline__ int ts_tile(int r, int tiles) {
  const int die = blockIdx.x & 7, place = blockIdx.x >> 3, from = r * (int)gridDim.x, left = tiles - from;
  const int share = left >= (int)gridDim.x ? (int)gridDim.x >> 3 : (left + 7) >> 3, at = die * share + place;
  return place < share && at < left ? from + at : -1;
}

template <int FROM, int TO> struct Range { static constexpr int from = FROM, to = TO; };

// ENDS: tiles end at a k of their own (k_end).  BUFS: buffers of a stage each, all but one of them on their way.
template <int MB, int NB, int SETS = 1, bool ENDS = false, int BUFS = ts_buffers(MB, NB)>
struct TileStream {
  static constexpr int NBUF = BUFS, STAGE = ts_stage_bytes(MB, NB), LOADS = 2 * (MB + NB);
  char* lds;
  int wave, lane;
  int k_end;                            // ENDS: k from here on is asked for as zeros, set by `aim` (at most `run`'s K)
  uint32_t kbyte;                       // the byte of this lane's chunk within a row's 128 bytes
  const char *xrd, *wrd;                // this wave's operand rows in buffer 0
  int sw[4];                            // where lane (row l, half h) finds the chunk of quarter ks
  ts_f32x16 acc[SETS][NB][MB];
  ts_u32x4 w[2][NB], x[2][MB];

  __device__ __forceinline__ TileStream(char* smem) : lds(smem) {
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    lane = threadIdx.x & 63;
    const int rho = lane >> 3, pos = lane & 7, l = lane & 31, h = lane >> 5;
    kbyte = (uint32_t)((pos ^ rho) << 4);
#pragma unroll
    for (int s = 0; s < 4; s++) sw[s] = l * 128 + (((4 * h + s) ^ (l & 7)) << 4);
    xrd = smem + (wave >> 1) * (MB * 32 * 128);
    wrd = smem + MB * 64 * 128 + (wave & 1) * (NB * 32 * 128);
  }
  // the tile row behind this lane in the wave's copy j
  __device__ __forceinline__ int row(int j) const { return (4 * j + wave) * 8 + (lane >> 3); }

  // Copies FROM .. TO - 1 of the 2 (MB + NB) that bring 64 k from k0 on of the rows of `xs` and `ws` into buffer b
  // (k0 >= K: zeros).
  template <int FROM, int TO>
  __device__ __forceinline__ void ask(int b, const TileRowsSource<MB>& xs, const TileRowsSource<NB>& ws, int k0, int K) {
    const uint32_t k = (uint32_t)k0 * 2 + kbyte;
    const uint32_t at = k < (uint32_t)K * 2 ? k : TS_OUT;
    char* dst = lds + b * STAGE + wave * 1024;
#pragma unroll
    for (int j = FROM; j < TO; j++) {
      if (j < 2 * MB)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(xs.rsrc, (__attribute__((address_space(3))) void*)(dst + j * 4096), 16, xs.off[j < 2 * MB ? j : 0] + at, 0, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ws.rsrc, (__attribute__((address_space(3))) void*)(dst + j * 4096), 16, ws.off[j < 2 * MB ? 0 : j - 2 * MB] + at, 0, 0, 0);
    }
  }
  // in the order in which the products want them
  __device__ __forceinline__ void read(int set, int b, int ks) {
    w[set][0] = *reinterpret_cast<const ts_u32x4*>(wrd + b * STAGE + sw[ks]);
#pragma unroll
    for (int i = 0; i < MB; i++) x[set][i] = *reinterpret_cast<const ts_u32x4*>(xrd + b * STAGE + sw[ks] + i * 4096);
#pragma unroll
    for (int j = 1; j < NB; j++) w[set][j] = *reinterpret_cast<const ts_u32x4*>(wrd + b * STAGE + sw[ks] + j * 4096);
  }
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int v = 0; v < SETS; v++)
#pragma unroll
      for (int j = 0; j < NB; j++)
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
          for (int r = 0; r < 16; r++) acc[v][j][i][r] = 0.f;
  }
  template <int V>
  __device__ __forceinline__ void multiply(int set) {
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
      for (int i = 0; i < MB; i++)
        acc[V][j][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(ts_bf16x8, w[set][j]),
                                                               __builtin_bit_cast(ts_bf16x8, x[set][i]), acc[V][j][i], 0, 0, 0);
  }
  // The MB NB products of a quarter with its operand reads between the first and its copies between the last of them: the
  // reads are back long before their products (and before the barrier), and a copy is never asked for faster than a compute
  // unit takes them in (about 41 bytes a cycle of whole lines; a wave that asks faster stands still, its products with it).
  // Copies write LDS, so the compiler keeps them behind the reads in any case.
  template <int READS, int COPIES, int I = 0>
  __device__ __forceinline__ void weave() {
    constexpr int P = MB * NB, H = READS < P ? (READS > 0 ? READS : 0) : P - 1, L = P - H;
    if constexpr (I < P) {
      constexpr int R = I < H ? (I + 1) * READS / (H > 0 ? H : 1) - I * READS / (H > 0 ? H : 1) : 0;
      constexpr int C = I < H ? 0 : (I - H + 1) * COPIES / L - (I - H) * COPIES / L;
      if constexpr (R > 0) __builtin_amdgcn_sched_group_barrier(0x100, R, 0);
      if constexpr (C > 0) __builtin_amdgcn_sched_group_barrier(0x020, C, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      weave<READS, COPIES, I + 1>();
    }
  }
  // The copies that take the place of a finished stage go out in PARTS quarters from its last one on: all four where there
  // are three buffers, else three, so that the last has a quarter to land.
  static constexpr int PARTS = NBUF >= 3 ? 4 : 3;
  static constexpr int part(int i) { return LOADS * i / PARTS; }
  // The products of the stage in buffer b, whose first operands are in set 0; leaves the first operands of the stage in
  // buffer `next` there.  `copies` is called with the numbers of the copies to ask for: first what is left of those that
  // have begun, then `on` (they are all on their way), then the first of those that fill b again.
  template <int V, typename Copies, typename On>
  __device__ __forceinline__ void stage(int b, int next, Copies copies, On on) {
    __builtin_amdgcn_sched_barrier(0);
    read(1, b, 1);
    copies(Range<part(1), part(2)>());
    multiply<V>(0);
    weave<MB + NB, part(2) - part(1)>();
    __builtin_amdgcn_sched_barrier(0);
    read(0, b, 2);
    copies(Range<part(2), part(3)>());
    multiply<V>(1);
    weave<MB + NB, part(3) - part(2)>();
    __builtin_amdgcn_sched_barrier(0);
    if (PARTS == 3) on();
    read(1, b, 3);
    if (PARTS == 4) copies(Range<part(3), LOADS>());
    multiply<V>(0);
    weave<MB + NB, PARTS == 4 ? LOADS - part(3) : 0>();
    __builtin_amdgcn_sched_barrier(0);
    if (PARTS == 4) on();
    // this wave's copies of the next stage have landed and its reads of this one are done; then so are all waves'
    __builtin_amdgcn_s_waitcnt(ts_wait((NBUF - 2) * LOADS, true));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    read(0, next, 0);
    copies(Range<0, part(1)>());
    multiply<V>(1);
    weave<MB + NB, part(1)>();
    __builtin_amdgcn_sched_barrier(0);
  }
  // Stages s, s + 1, .. of a tile (those there are), one a chain.
  template <int V> struct Sets {};
  template <int V, typename Copies, typename On>
  __device__ __forceinline__ void round(Sets<V>, int s, int stages, int& buf, Copies copies, On on) {
    if constexpr (V < SETS) {
      if (V > 0 && s + V >= stages) return;
      const int next = buf + 1 == NBUF ? 0 : buf + 1;
      stage<V>(buf, next, copies, on);
      buf = next;
      round(Sets<V + 1>(), s, stages, buf, copies, on);
    }
  }
  // This workgroup's tiles of so many (ts_tile), each over K: `aim(t)` points xs and ws at tile t, `done(t)` takes its sums.
  template <typename Aim, typename Done>
  __device__ __forceinline__ void run(int tiles, int K, const TileRowsSource<MB>& xs, const TileRowsSource<NB>& ws, Aim aim, Done done) {
    const int stages = (K + TS_BK - 1) / TS_BK;
    int at_round = 0, at_tile = ts_tile(0, tiles), at_stage = 0, fill = 0;      // the stage that is asked for next, into buffer `fill`
    auto copies = [&](auto r) { ask<decltype(r)::from, decltype(r)::to>(fill, xs, ws, at_tile >= 0 ? at_stage * TS_BK : K, ENDS ? k_end : K); };
    auto on = [&] {
      fill = fill + 1 == NBUF ? 0 : fill + 1;
      if (++at_stage == stages && at_tile >= 0) {
        at_stage = 0;
        at_tile = ts_tile(++at_round, tiles);
        if (at_tile >= 0) aim(at_tile);
      }
    };
    aim(at_tile);
#pragma unroll
    for (int b = 0; b < NBUF - 1; b++) {
      copies(Range<0, LOADS>());
      on();
    }
    __builtin_amdgcn_s_waitcnt(ts_wait((NBUF - 2) * LOADS, true));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    copies(Range<0, part(1)>());
    read(0, 0, 0);
    int buf = 0;
    for (int turn = 0, t; (t = ts_tile(turn, tiles)) >= 0; turn++) {
      clear();
      for (int s = 0; s < stages; s += SETS) round(Sets<0>(), s, stages, buf, copies, on);
      done(t);
    }
    __builtin_amdgcn_s_waitcnt(ts_wait(0, true));          // the last copies (zeros) are in before LDS is given back
  }
};

// Copies of this worker's block of rows of stride ld, their first `most` k, to nobody's place in LDS: the memory-side cache then
// has them.  Tiles that wait for memory stage after stage get theirs from there in half the time, so workgroups without a tile do this for the
// others' matrix, in the order in which those want it.
__device__ __forceinline__ void ts_bring(const bf16_t* base, int rows, int ld, int most, int worker, int workers, char* lds) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const __amdgpu_buffer_rsrc_t r = ts_buffer(base, ((long long)(rows - 1) * ld + most) * 2);
  const int each = ts_bring_rows(rows, workers), r0 = worker * each, r1 = min(rows, r0 + each);
  for (int k = 0; k < most; k += TS_BK)
    for (int i = r0 + 8 * wave; i < r1; i += 32) {                 // eight rows of 128 bytes a copy
      const int row = i + (lane >> 3), col = k + (lane & 7) * 8;
      const uint32_t off = row < r1 && col < most ? (uint32_t)(row * ld + col) * 2 : TS_OUT;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)(lds + wave * 1024), 16, off, 0, 0, 0);
    }
  __builtin_amdgcn_s_waitcnt(ts_wait(0, true));
}

// Tile t of the order in which tiles are dealt out: strips of up to TS_STRIP tiles of rows, inside a strip column by column, so
// that the 32 tiles (64 where two share a unit) a die works on at a time are about as wide as high and share their operands in its
// L2.  (Strips of 3, 4, 5, 6, 7, 8, 10, 12, 16: 2,048 rows of 8,960 pairs, K 1,536, 107.5, 108.8, 107.7, 108.2, 108.8, 110.6, 108.5, 110, 114 us;
// of 13,440 columns 102.5, 103.1, 103.8, 103.3, 103.2, 105.3, 106.2, 105.3, 105.6; 1,400 rows of 18,944 pairs, K 3,584, 359, 357, 360, 350, 350, 347, 347,
// 350, 349; prompts of five designs 0.4 to 0.6 % faster with 6 than with 8.)
#define TS_STRIP 6
__device__ __forceinline__ void ts_place(int m_tiles, int n_tiles, int t, int& m, int& n) {
  const int per = TS_STRIP * n_tiles, strip = t / per, rest = t - strip * per, rows = min(TS_STRIP, m_tiles - strip * TS_STRIP);
  n = rest / rows;
  m = strip * TS_STRIP + rest - n * rows;
}
#endif
