// A routed feed-forward in bfloat16: the kernels that serve it.
//
// Few rows (a row is one (token, chosen expert) pair; single tokens and small steps): the matrices of the experts that they chose are
// streamed, once an expert where enough rows meet in one, 16 bytes a lane, sixteen lanes to an output element.
//
// More rows: they are sorted by expert on the device (nothing comes back to the host), every expert's rows padded to whole
// tiles, and two grouped products run on the matrix cores, tiles as tile_stream.h has them:
//   first:  y[p, f] = act(gate_e[f] . h[token of p], up_e[f] . h[token of p], w_p)      (rows gathered by the copies to LDS)
//   second: out[slot of p][token of p][n] = down_e[n] . y[p]                             (float32, scattered)
// While experts have few rows the matrices' stream bounds it: 128 rows over 32 experts of 4,736 x 3,584, 368 and 188 us the two
// products (5.8 TB/s) against 478 and 250 with operands that pass through registers; from about 100 rows an expert the
// latency of the copies: 4,096 rows over 16 experts of 2,240 x 1,536 92 and 47 us against 145 and 75, 2,754 rows 93 and 48
// against 101 and 54 (tiles of 128 rows are 69 and 65 percent full then).
//
// A row's result does not depend on which other rows share its tile: a matrix instruction keeps rows apart and the sums
// over k run in the same order for every row.
#include "tile_stream.h"

// mode 0: the clipped activation, the row's weight w on its input; mode 1: w silu(g) u (the weight on the expert's
// output, taken in front of the linear second product); mode 2: w times the clipped activation.  The same operations as
// expert_act of the plain kernels, so that an expert's activation has the same bits by every kernel.  (With times_sigmoid 2,048 rows of two
// experts each over 16 experts of 2,240 x 1,536 take 148 us, so 151; but then a prompt's rows move by their last bit, and of 260
// batches of 32 requests decoding behind such prompts 13 had one row whose fourth and fifth router scores lay closer than that, which
// took another expert and moved by a sixth of its size.)
__device__ __forceinline__ float moe_act(float g, float u, float limit, float alpha, int mode, float w) {
  if (mode == 1) return w * (g / (1.0f + expf(-g))) * u;
  if (mode == 0) { g *= w; u *= w; }
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return (mode == 2 ? w : 1.0f) * (g / (1.0f + expf(-alpha * g)) * (u + 1.0f));
}

__device__ __forceinline__ void unpack8(const uint4& v, float* f) {
  f[0] = __uint_as_float(v.x << 16); f[1] = __uint_as_float(v.x & 0xffff0000u);
  f[2] = __uint_as_float(v.y << 16); f[3] = __uint_as_float(v.y & 0xffff0000u);
  f[4] = __uint_as_float(v.z << 16); f[5] = __uint_as_float(v.z & 0xffff0000u);
  f[6] = __uint_as_float(v.w << 16); f[7] = __uint_as_float(v.w & 0xffff0000u);
}

__device__ __forceinline__ float dot8(const uint4& a, const float* x, float acc) {
  float f[8];
  unpack8(a, f);
#pragma unroll
  for (int i = 0; i < 8; i++) acc = fmaf(f[i], x[i], acc);
  return acc;
}

// the sum over a row of 16 lanes, in every lane of the row
__device__ __forceinline__ float row16_sum(float v) {
  v += lane_pattern<LANE_XOR_1>(v);
  v += lane_pattern<LANE_XOR_2>(v);
  v += lane_pattern<HALF_ROW_MIRROR>(v);
  v += lane_pattern<ROW_MIRROR>(v);
  return v;
}

// ---------------------------------------------------------------------------
// Few rows, SHARED: an expert's matrices are streamed once for all of its rows.  Workgroup (tile, j) looks the rows' experts over and takes the j-th
// that occurs for the first time; the last workgroups of a grid for as many experts as rows find none.  Tiles run along the grid's first
// index, so that an expert's workgroups go to all dies at one time.  The sums of a row are made as if it were alone.  Bound by the matrices' stream.
// Otherwise a row streams its expert's matrices itself, rows along the grid's first index (pico_moe_rows_shared says which).
// live (or null): the context of every token; a token without one pads a recorded step: its rows choose no expert and come out as zeros.
// ---------------------------------------------------------------------------
#define MOE_LANES 64
struct MoeRows {
  unsigned long long mask;                            // row numbers: base + the bits' numbers
  unsigned long long dead;                            // rows of padding, of whoever is to write their zeros
  int base, expert, tile;                             // expert < 0: nothing to do
};
template <bool SHARED>
__device__ __forceinline__ MoeRows moe_rows_of(const int* __restrict__ experts, const int* __restrict__ live, int R, int top, int E) {
  MoeRows m;
  m.dead = 0;
  if (!SHARED) {
    m.base = blockIdx.x; m.tile = blockIdx.y; m.mask = 1;
    const int e = experts[m.base];
    const bool there = !live || live[m.base / top] > 0;
    m.dead = there ? 0 : 1;
    m.expert = there && e < E ? e : -1;
    return m;
  }
  const int lane = threadIdx.x & 63;
  int e = lane < R ? experts[lane] : -1;
  const bool there = lane >= R || !live || live[lane / top] > 0;
  if (e >= E || !there) e = -1;
  m.base = 0; m.tile = blockIdx.x; m.expert = -1; m.mask = 0;
  if (blockIdx.y == 0) m.dead = __ballot(!there);
  // (the walk is the same for all lanes: a lane is read while all of them are on, as what one holds that is off is nobody's promise)
  unsigned long long left = __ballot(e >= 0);
  for (int j = blockIdx.y; left; j--) {
    const int next = __builtin_amdgcn_readlane(e, __builtin_ctzll(left));
    const unsigned long long same = __ballot(e == next);
    if (j == 0) { m.expert = next; m.mask = same; break; }
    left &= ~same;
  }
  return m;
}
// the next M rows of the mask; the last one again where there are fewer
template <int M>
__device__ __forceinline__ void moe_next_rows(unsigned long long& mask, int base, int (&r)[M]) {
#pragma unroll
  for (int i = 0; i < M; i++) {
    r[i] = base + __builtin_ctzll(mask);
    if (mask & (mask - 1)) mask &= mask - 1;
  }
}

constexpr int moe_up_out(bool shared) { return shared ? 8 : 16; }
// First half: 16 lanes make one f (its gate and its up) of M rows.
template <int M>
__device__ __forceinline__ void moe_up_some(const bf16_t* __restrict__ h, int ldh, const bf16_t* __restrict__ wg, const bf16_t* __restrict__ wu,
                                            const float* __restrict__ weights, bf16_t* __restrict__ y, unsigned long long& mask, int base,
                                            int top, int F, int D, int f, float limit, float alpha, int mode) {
  const int sub = threadIdx.x & 15, n = min(M, (int)__popcll(mask));
  int r[M];
  moe_next_rows(mask, base, r);
  const bf16_t* x[M];
  float g[M], u[M], w[M];
#pragma unroll
  for (int i = 0; i < M; i++) {
    x[i] = h + (size_t)(r[i] / top) * ldh;
    w[i] = weights[r[i]];
    g[i] = u[i] = 0.f;
  }
#pragma unroll 2
  for (int k = sub * 8; k < D; k += 128) {
    const uint4 gv = *reinterpret_cast<const uint4*>(wg + k);
    const uint4 uv = *reinterpret_cast<const uint4*>(wu + k);
    uint4 xv[M];
#pragma unroll
    for (int i = 0; i < M; i++) xv[i] = *reinterpret_cast<const uint4*>(x[i] + k);
#pragma unroll
    for (int i = 0; i < M; i++) {
      float xf[8];
      unpack8(xv[i], xf);
      g[i] = dot8(gv, xf, g[i]);
      u[i] = dot8(uv, xf, u[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < M; i++) {
    g[i] = row16_sum(g[i]);
    u[i] = row16_sum(u[i]);
    if (sub == 0 && i < n) y[(size_t)r[i] * F + f] = f32_to_bf16(moe_act(g[i], u[i], limit, alpha, mode, w[i]));
  }
}
template <bool SHARED>
__global__ __launch_bounds__(16 * moe_up_out(SHARED)) void moe_up_rows_kernel(const bf16_t* __restrict__ h, int ldh, const bf16_t* __restrict__ gate_up,
                                                          const int* __restrict__ experts, const float* __restrict__ weights,
                                                          const int* __restrict__ live, bf16_t* __restrict__ y, int R, int top, int E,
                                                          int F, int D, float limit, float alpha, int mode) {
  MoeRows m = moe_rows_of<SHARED>(experts, live, R, top, E);
  const int f = m.tile * moe_up_out(SHARED) + (threadIdx.x >> 4);
  if (m.expert < 0 || f >= F) return;
  const bf16_t* wg = gate_up + ((size_t)m.expert * 2 * F + f) * D;
  const bf16_t* wu = wg + (size_t)F * D;
  if (!SHARED) return moe_up_some<1>(h, ldh, wg, wu, weights, y, m.mask, m.base, top, F, D, f, limit, alpha, mode);
  for (int left = __popcll(m.mask); left > 0; left -= 4) {
    if (left == 1) moe_up_some<1>(h, ldh, wg, wu, weights, y, m.mask, m.base, top, F, D, f, limit, alpha, mode);
    else if (left == 2) moe_up_some<2>(h, ldh, wg, wu, weights, y, m.mask, m.base, top, F, D, f, limit, alpha, mode);
    else moe_up_some<4>(h, ldh, wg, wu, weights, y, m.mask, m.base, top, F, D, f, limit, alpha, mode);
  }
}

// Second half: out[slot][t][n] = down_e[n] . y[(t, slot)] (a slab a slot; whoever reads it adds the slabs up).  A
// wave makes MOE_DOWN_OUT neighbouring outputs of M rows with all its lanes along k, so that a launch of one token still has a
// few hundred workgroups and a lane several loads on their way.
#define MOE_DOWN_OUT 2
template <int M>
__device__ __forceinline__ void moe_down_some(const bf16_t* __restrict__ y, const bf16_t* const (&wd)[MOE_DOWN_OUT], float* __restrict__ out,
                                              unsigned long long& mask, int base, int T, int top, int F, int D, int n) {
  const int lane = threadIdx.x & 63, rows = min(M, (int)__popcll(mask));
  int r[M];
  moe_next_rows(mask, base, r);
  float s[M][MOE_DOWN_OUT];
#pragma unroll
  for (int m = 0; m < M; m++)
#pragma unroll
    for (int i = 0; i < MOE_DOWN_OUT; i++) s[m][i] = 0.f;
#pragma unroll 3
  for (int j = lane * 8; j < F; j += 512) {
    uint4 wv[MOE_DOWN_OUT], yv[M];
#pragma unroll
    for (int i = 0; i < MOE_DOWN_OUT; i++) wv[i] = *reinterpret_cast<const uint4*>(wd[i] + j);
#pragma unroll
    for (int m = 0; m < M; m++) yv[m] = *reinterpret_cast<const uint4*>(y + (size_t)r[m] * F + j);
#pragma unroll
    for (int m = 0; m < M; m++) {
      float yf[8];
      unpack8(yv[m], yf);
#pragma unroll
      for (int i = 0; i < MOE_DOWN_OUT; i++) s[m][i] = dot8(wv[i], yf, s[m][i]);
    }
  }
#pragma unroll
  for (int m = 0; m < M; m++) {
    float* o = out + ((size_t)(r[m] % top) * T + r[m] / top) * D + n;
#pragma unroll
    for (int i = 0; i < MOE_DOWN_OUT; i++) {
      const float total = wave_sum(s[m][i]);
      if (lane == 0 && n + i < D && m < rows) o[i] = total;
    }
  }
}
template <bool SHARED>
__global__ __launch_bounds__(256) void moe_down_rows_kernel(const bf16_t* __restrict__ y, const bf16_t* __restrict__ down,
                                                            const int* __restrict__ experts, const int* __restrict__ live,
                                                            float* __restrict__ out, int T, int top, int E, int F, int D) {
  MoeRows m = moe_rows_of<SHARED>(experts, live, T * top, top, E);
  const int n = (m.tile * 4 + (threadIdx.x >> 6)) * MOE_DOWN_OUT;
  if (n >= D) return;
  for (; m.dead; m.dead &= m.dead - 1) {
    const int r = m.base + __builtin_ctzll(m.dead), i = threadIdx.x & 63;
    if (i < MOE_DOWN_OUT && n + i < D) out[((size_t)(r % top) * T + r / top) * D + n + i] = 0.f;
  }
  if (m.expert < 0) return;
  const bf16_t* wd[MOE_DOWN_OUT];
#pragma unroll
  for (int i = 0; i < MOE_DOWN_OUT; i++) wd[i] = down + ((size_t)m.expert * D + min(n + i, D - 1)) * F;
  if (!SHARED) return moe_down_some<1>(y, wd, out, m.mask, m.base, T, top, F, D, n);
  for (int left = __popcll(m.mask); left > 0; left -= 4) {
    if (left == 1) moe_down_some<1>(y, wd, out, m.mask, m.base, T, top, F, D, n);
    else if (left == 2) moe_down_some<2>(y, wd, out, m.mask, m.base, T, top, F, D, n);
    else moe_down_some<4>(y, wd, out, m.mask, m.base, T, top, F, D, n);
  }
}

// Whether rows share their experts' streams: from four tokens on, as far as a wave has lanes, where T tokens that choose at random name an
// expert again so often that 80 MB less are asked for, of matrices (what is met at all) that the dies' L2s do not hold anyway.  To look
// the experts over takes 0.5 us a launch, and the rows of one workgroup more registers.  Microseconds for both halves, every row for itself / shared, by
// tokens x chosen experts: 16 experts of 2,240 x 1,536 4x2 31.9 / 30.3 (29 MB again), 8x2 54.9 / 53.1 (114 MB); of 4,480 x 1,536 4x2 56.9 / 55.4 (57 MB),
// 8x2 100.1 / 85.4 (227); 32 of 2,368 x 3,584 4x2 66.0 / 69.2 (37), 8x1 72.8 / 76.2 (42), 4x4 122.1 / 115.4 (140); 64 of 704 x 2,048 16x1 29.2 / 34.3 (15); eight
// of 704 x 2,048 16x1 26.0 / 27.4 (77); four of 1,536 x 1,536 8x2 35.3 / 25.2 (170); two of 512 x 1,024 8x2 11.4 / 16.2 (44, of 6 MB).  Over 321
// such sizes 10 % less in the mean than every row for itself, and at most 1.5 % more.
extern "C" int pico_moe_rows_shared(int T, int top, int E, int F, int D) {
  const double rows = (double)T * top, bytes = 6.0 * F * D;
  const double met = E * (1.0 - pow(1.0 - fmin(1.0, (double)top / E), T));
  return T > 3 && rows <= MOE_LANES && (rows - met) * bytes >= 80e6 && met * bytes >= 32e6;
}

// share: 1 or 0, or as pico_moe_rows_shared says (-1)
extern "C" int pico_moe_experts_rows(const void* h, int ldh, const void* gate_up, const void* down, const int* experts,
                                     const float* weights, const int* live, void* y, float* out, int T, int top, int E, int F, int D,
                                     float limit, float alpha, int mode, int share, hipStream_t stream) {
  PICO_REQUIRE(T >= 0 && top > 0 && E > 0 && F > 0 && D > 0 && ldh >= D, "pico_moe_experts_rows: bad sizes");
  PICO_REQUIRE(mode >= 0 && mode <= 2, "pico_moe_experts_rows: unknown mode %d", mode);
  PICO_REQUIRE(F % 8 == 0 && D % 8 == 0 && ldh % 8 == 0, "pico_moe_experts_rows: sizes must be multiples of 8");
  PICO_REQUIRE(((uintptr_t)h | (uintptr_t)gate_up | (uintptr_t)down | (uintptr_t)y) % 16 == 0,
               "pico_moe_experts_rows: operands must start on 16 bytes");
  if (T == 0) return 0;
  const long long R = (long long)T * top;
  PICO_REQUIRE(share <= 0 || R <= MOE_LANES, "pico_moe_experts_rows: up to %d rows share", MOE_LANES);
  const bool shared = share < 0 ? pico_moe_rows_shared(T, top, E, F, D) : share;
  const unsigned out_up = moe_up_out(shared), up = (F + out_up - 1) / out_up, dn = (D + 4 * MOE_DOWN_OUT - 1) / (4 * MOE_DOWN_OUT);
  // (tiles lie along the grid's first index where rows share: 2^32 threads there, 65,535 workgroups along the second)
  const unsigned most = shared ? 1u << 24 : 65536u;
  PICO_REQUIRE(R < (1ll << 30) && up < most && dn < most, "pico_moe_experts_rows: sizes beyond the grid");
  const unsigned met = (unsigned)min(R, (long long)E);
  const dim3 g1 = shared ? dim3(up, met) : dim3((unsigned)R, up), g2 = shared ? dim3(dn, met) : dim3((unsigned)R, dn);
#define LAUNCH(SHARED)                                                                                                                             \
  moe_up_rows_kernel<SHARED><<<g1, 16 * moe_up_out(SHARED), 0, stream>>>((const bf16_t*)h, ldh, (const bf16_t*)gate_up, experts, weights, live,      \
                                                                         (bf16_t*)y, (int)R, top, E, F, D, limit, alpha, mode);                    \
  moe_down_rows_kernel<SHARED><<<g2, 256, 0, stream>>>((const bf16_t*)y, (const bf16_t*)down, experts, live, out, T, top, E, F, D)
  if (shared) { LAUNCH(true); } else { LAUNCH(false); }
#undef LAUNCH
  PICO_LAUNCH_CHECK();
  return 0;
}

// ---------------------------------------------------------------------------
// Sorting the rows by expert.  One workgroup an expert: it counts every expert's rows (to know where its own begin),
// then writes its own rows' numbers in ascending order; its last tile is filled up with -1.
//   sorted[tiles_cap * bm]: row numbers (token * top + slot) or -1;  sorted_w: their weights;
//   tiles[2 t]: MOE_TILE(expert, rows) of tile t;  tiles[2 t + 1]: MOE_STRIP(first tile, tiles) of the strip it is in, up to
//   MOE_STRIP_TILES neighbouring tiles of one expert;  tiles[2 tiles_cap]: how many tiles there are
// ---------------------------------------------------------------------------
#define MOE_SORT_THREADS 1024
#define MOE_SORT_MAX_E 1024
#define MOE_TILE(e, rows) ((e) << 10 | (rows))
#define MOE_STRIP(first, n) ((first) << 4 | (n))
#define MOE_STRIP_TILES 8

__global__ __launch_bounds__(MOE_SORT_THREADS) void moe_sort_kernel(const int* __restrict__ experts,
                                                                    const float* __restrict__ weights, int R, int E, int bm,
                                                                    int tiles_cap, int* __restrict__ sorted,
                                                                    float* __restrict__ sorted_w, int* __restrict__ tiles_out,
                                                                    const int* __restrict__ live, int top, float* __restrict__ out, int T, int D) {
  __shared__ int hist[MOE_SORT_MAX_E];
  __shared__ int wave_count[MOE_SORT_THREADS / 64];
  __shared__ int base_tiles;
  const int e = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = MOE_SORT_THREADS / 64;
  // (a token without a context pads a recorded step: its rows, of MOE_LANES, have no expert and come out as zeros)
  auto expert = [&](int r) {
    const int x = experts[r];
    return (live ? live[r / top] : 1) > 0 ? x : -1;
  };
  if (live) {
    int turn = 0;
    for (unsigned long long dead = __ballot(lane < R && live[min(lane, R - 1) / top] <= 0); dead; dead &= dead - 1) {
      if (turn == e) {
        const int r = __builtin_ctzll(dead);
        float* o = out + ((size_t)(r % top) * T + r / top) * D;
        for (int n = tid; n < D; n += MOE_SORT_THREADS) o[n] = 0.f;
      }
      turn = turn + 1 == E ? 0 : turn + 1;
    }
  }
  for (int i = tid; i < E; i += MOE_SORT_THREADS) hist[i] = 0;
  if (tid == 0) base_tiles = 0;
  __syncthreads();
  for (int r = tid; r < R; r += MOE_SORT_THREADS) {
    const int x = expert(r);
    if (x >= 0 && x < E) atomicAdd(&hist[x], 1);
  }
  __syncthreads();
  int before = 0;
  for (int i = tid; i < e; i += MOE_SORT_THREADS) before += (hist[i] + bm - 1) / bm;
  if (before) atomicAdd(&base_tiles, before);
  __syncthreads();
  const int count = hist[e], tiles = (count + bm - 1) / bm, base = base_tiles;
  for (int i = tid; i < tiles; i += MOE_SORT_THREADS) {
    const int first = i / MOE_STRIP_TILES * MOE_STRIP_TILES;
    tiles_out[2 * (base + i)] = MOE_TILE(e, min(bm, count - i * bm));
    tiles_out[2 * (base + i) + 1] = MOE_STRIP(base + first, min(MOE_STRIP_TILES, tiles - first));
  }
  if (e == E - 1 && tid == 0) tiles_out[2 * tiles_cap] = base + tiles;
  // every wave takes a stretch of the rows: counts its own, then writes them behind those of the waves before it
  const int seg = ((R + nw - 1) / nw + 63) / 64 * 64, lo = wave * seg, hi = min(R, lo + seg);
  int mine = 0;
  for (int r0 = lo; r0 < hi; r0 += 64) {
    const int r = r0 + lane;
    const bool is = r < hi && expert(r) == e;
    mine += __popcll(__ballot(is));
  }
  if (lane == 0) wave_count[wave] = mine;
  __syncthreads();
  int at = 0;
  for (int i = 0; i < wave; i++) at += wave_count[i];
  int* dst = sorted + (size_t)base * bm;
  float* dst_w = sorted_w + (size_t)base * bm;
  for (int r0 = lo; r0 < hi; r0 += 64) {
    const int r = r0 + lane;
    const bool is = r < hi && expert(r) == e;
    const unsigned long long m = __ballot(is);
    if (is) {
      const int to = at + __popcll(m & ((1ull << lane) - 1ull));
      dst[to] = r;
      dst_w[to] = weights[r];
    }
    at += __popcll(m);
  }
  for (int i = count + tid; i < tiles * bm; i += MOE_SORT_THREADS) { dst[i] = -1; dst_w[i] = 0.f; }
}

// ---------------------------------------------------------------------------
// The grouped product: tiles as tile_stream.h has them, of 64 MB sorted rows of one expert by 64 NB rows of its matrix.
// UP:   X = gathered rows of h (K = D); the matrix's rows in blocks of 16 gate rows and the 16 up rows of the same columns;
//       act(gate, up) to y[p, f] (bfloat16).
// DOWN: X = y rows of the tile (K = F); float32 to out[slot][token][n].
// ---------------------------------------------------------------------------
struct MoeArgs {
  const bf16_t* X;
  const bf16_t* W;
  const int* sorted;
  const float* sorted_w;
  const int* tiles;
  bf16_t* y;
  float* out;
  int tiles_cap, ldx, T, top, F, D, n_tiles, mode;
  float limit, alpha;
};

#ifdef __HIP_DEVICE_COMPILE__
// a read of what an earlier kernel wrote, at an address that is the same in all lanes: it goes through the scalar cache and
// so does not wait behind the copies, which the vector loads' counter retires in order
__device__ __forceinline__ int moe_scalar(const int* p) {
  return *(const __attribute__((address_space(4))) int*)(uintptr_t)p;
}

// Tile t of the order in which tiles are dealt out: strip by strip, inside a strip column by column.  The tiles that share rows
// of a matrix are neighbours, so they run on one die at one time, and a matrix is read from memory once; a die at work on
// one strip also holds all of its rows in its L2.  (Strips of 8 tiles across experts read the rows on all dies and a matrix
// twice where a strip ends in it.)
__device__ __forceinline__ void moe_place(const MoeArgs& a, int t, int& m, int& n) {
  const int strip = moe_scalar(a.tiles + 2 * (t / a.n_tiles) + 1), first = strip >> 4, rows = strip & 15, rest = t - first * a.n_tiles;
  n = rest / rows;
  m = first + rest - n * rows;
}
#endif

template <int MB, int NB, bool UP, int SHARE = ts_share(MB, NB), int BUFS = ts_buffers(MB, NB)>
__global__ __launch_bounds__(256, SHARE) void moe_grouped_kernel(const MoeArgs a) {
#ifdef __HIP_DEVICE_COMPILE__
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  typedef TileStream<MB, NB, 1, false, BUFS> TS;
  TS ts(smem);
  constexpr int TM = 64 * MB, TN = 64 * NB, COLS = UP ? TN / 2 : TN;
  const int K = UP ? a.D : a.F, tiles = moe_scalar(a.tiles + 2 * a.tiles_cap) * a.n_tiles;
  if (ts_tile(0, tiles) < 0) return;
  TileRowsSource<MB> xs;
  TileRowsSource<NB> ws;
  auto aim = [&](int t) {
    int m, n;
    moe_place(a, t, m, n);
    const int tile = moe_scalar(a.tiles + 2 * m), e = tile >> 10, rows = tile & 1023;
    const int c0 = n * COLS;
    if (UP) {
      xs.rsrc = ts_buffer(a.X, ((long long)(a.T - 1) * a.ldx + K) * 2);
      ws.rsrc = ts_buffer(a.W + (size_t)e * 2 * a.F * K, (long long)a.F * K * 4);
#pragma unroll
      for (int j = 0; j < 2 * MB; j++) {
        const int* list = a.sorted + (size_t)m * TM + (4 * j + ts.wave) * 8;
        int r = moe_scalar(list);
#pragma unroll
        for (int i = 1; i < 8; i++) {
          const int v = moe_scalar(list + i);
          r = (ts.lane >> 3) == i ? v : r;
        }
        xs.off[j] = r < 0 ? TS_OUT : (uint32_t)(r / a.top * a.ldx) * 2;
      }
#pragma unroll
      for (int j = 0; j < 2 * NB; j++) {
        const int r = ts.row(j), c = c0 + (r >> 5) * 16 + (r & 15);
        ws.off[j] = c < a.F ? (uint32_t)((c + ((r & 16) ? a.F : 0)) * K) * 2 : TS_OUT;
      }
    } else {
      xs.rsrc = ts_buffer(a.X + (size_t)m * TM * K, (long long)rows * K * 2);
      ws.rsrc = ts_buffer(a.W + ((size_t)e * a.D + c0) * K, (long long)(a.D - c0) * K * 2);
#pragma unroll
      for (int j = 0; j < 2 * MB; j++) xs.off[j] = (uint32_t)(ts.row(j) * K) * 2;
#pragma unroll
      for (int j = 0; j < 2 * NB; j++) ws.off[j] = (uint32_t)(ts.row(j) * K) * 2;
    }
  };
  ts.run(tiles, K, xs, ws, aim, [&](int t) {
    // lane (l, h): row l of a block of X, tile rows 8 (r / 4) + 4 h + r % 4 of a block of W in register r
    int mt, nt;
    moe_place(a, t, mt, nt);
    const int l = ts.lane & 31, h = ts.lane >> 5, rows = moe_scalar(a.tiles + 2 * mt) & 1023;
#pragma unroll
    for (int i = 0; i < MB; i++) {
      const int in = (ts.wave >> 1) * (32 * MB) + 32 * i;      // the block's first row in its tile
      if (in >= rows) continue;
      const size_t p0 = (size_t)mt * TM + in;
      int mine = 0;                                            // the row's weight (UP) or number
#pragma unroll
      for (int j = 0; j < 32; j++) {
        const int v = moe_scalar((UP ? (const int*)a.sorted_w : a.sorted) + p0 + j);
        mine = l == j ? v : mine;
      }
      const bool there = in + l < rows;
      const float w = __int_as_float(mine);
      float* o = UP ? nullptr : a.out + ((size_t)(there ? mine % a.top : 0) * a.T + (there ? mine / a.top : 0)) * a.D;
#pragma unroll
      for (int j = 0; j < NB; j++) {
        const ts_f32x16& v = ts.acc[0][j][i];
        const int blk = (ts.wave & 1) * NB + j;
        if (UP) {
          uint32_t p[4];
#pragma unroll
          for (int q = 0; q < 4; q++)
            p[q] = pack2_bf16(moe_act(v[2 * q], v[8 + 2 * q], a.limit, a.alpha, a.mode, w),
                              moe_act(v[2 * q + 1], v[8 + 2 * q + 1], a.limit, a.alpha, a.mode, w));
          // the halves of the wave hold columns 0..3 and 8..11, 4..7 and 12..15: swapped, eight neighbours each
          const auto s0 = __builtin_amdgcn_permlane32_swap(p[0], p[2], false, false);
          const auto s1 = __builtin_amdgcn_permlane32_swap(p[1], p[3], false, false);
          const int c = nt * COLS + blk * 16 + 8 * h;
          if (there && c < a.F)
            *reinterpret_cast<uint4*>(a.y + (p0 + l) * a.F + c) = make_uint4(s0[0], s1[0], s0[1], s1[1]);
        } else {
#pragma unroll
          for (int q = 0; q < 4; q++) {
            const int n = nt * TN + blk * 32 + 8 * q + 4 * h;
            if (there && n < a.D) *reinterpret_cast<float4*>(o + n) = make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
          }
        }
      }
    }
  });
#endif
}

template <int MB, int NB, bool UP, int SHARE = ts_share(MB, NB), int BUFS = ts_buffers(MB, NB)>
static int moe_launch(MoeArgs a, hipStream_t stream) {
  constexpr int bytes = ts_stage_bytes(MB, NB) * BUFS;
  static const hipError_t room = hipFuncSetAttribute((const void*)&moe_grouped_kernel<MB, NB, UP, SHARE, BUFS>,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  PICO_REQUIRE(room == hipSuccess, "pico_moe_experts_grouped: %s", hipGetErrorString(room));
  const int cols = UP ? 32 * NB : 64 * NB, n = UP ? a.F : a.D;
  a.n_tiles = (n + cols - 1) / cols;
  const long long tiles = (long long)a.tiles_cap * a.n_tiles;
  PICO_REQUIRE(tiles < (1LL << 30), "pico_moe_experts_grouped: sizes beyond one launch");
  moe_grouped_kernel<MB, NB, UP, SHARE, BUFS><<<ts_grid(tiles, 256 * SHARE), 256, bytes, stream>>>(a);
  return 0;
}

// Rows of a tile: 64 up to 48 rows an expert (most experts then have one tile), else 128.  37 rows an expert of 2,240 x 1,536:
// 56 and 26 us the two products with tiles of 64, 54 and 35 with 128; 87 of 4,736 x 3,584: 495 and 263 with 64, 426 and 217
// with 128; 256 of 2,240 x 1,536: 119 and 67, 92 and 47.  Taller tiles pad more than they save.
extern "C" int pico_moe_tile_rows(long long rows, int E) { return rows <= 48LL * E ? 64 : 128; }

// Columns of a tile: as many rounds of workgroups as a call is expected to take (its rows spread over the experts at
// random), at the cost of a stage in a full round and in a last one that leaves a compute unit at most one workgroup, in
// microseconds; the operands come from memory, so a stage costs its latency more than its products.
struct MoeTile { int nb, share; float each, lone; };
static const MoeTile moe_tiles[2][2] = {{{1, 2, 0.72f, 0.6f}, {2, 2, 1.3f, 1.1f}}, {{3, 2, 1.9f, 1.65f}, {4, 1, 1.4f, 1.4f}}};

static double moe_live(double rows, int E, int bm) {           // tiles that are expected to have rows
  const double mean = rows / E;
  double tiles = E * -expm1(-mean);
  for (int j = 1; j * (double)bm < rows; j++) {
    const double p = 0.5 * erfc((j * bm - mean) / sqrt(2 * mean));
    if (p < 1e-3) break;
    tiles += E * p;
  }
  return tiles;
}

// ... and if experts are chosen unevenly: their shares of the rows grow in even steps, the last's e^4 (55) times the first's.
static double moe_live_uneven(double rows, int E, int bm) {
  const double step = exp(4.0 / E);
  double share = rows * (step - 1.0) / (exp(4.0) - 1.0), tiles = 0;
  for (int e = 0; e < E; e++, share *= step) tiles += ceil(share / bm);
  return tiles;
}

// The second product where its tiles of 128 or 192 columns are a single round: its rows are read as they lie and its ends are stores alone, so a unit is
// better left to one workgroup with three or four stages on their way (the first product's activations hide behind the other workgroup of a
// unit: 2,754 rows 84 us, with one 86).  0: no; else the blocks of 64 columns, by the number of stages: microseconds as two workgroups of 192 columns / one
// of 256, two stages on their way / of 192, three / of 128, four: 16 experts of 2,240 x 1,536, 1,400 rows 46 / 41 / 36 / 34, 2,754 47 / 44 / 39 / 50 (two
// rounds), 4,096 61 / 47 / 60 / 52 (two rounds of both); of 4,480 x 1,536 89 / 78 / 68 / 58, 92 / 77 / 69 / 97, 112 / 80 / 114 / 98.  A tile too many is a
// second round, so the round is to hold the tiles of rows at random and those of uneven choices.  Both products of 468 sizes and choices, even and
// not, 8 % less in the mean and none slower; with half a tile an expert for uneven choices 2,000 rows over 32 experts of 8,960 x 1,536 with some chosen
// more than others 560 us became 625, of 2,240 x 1,536 171 186.
extern "C" int pico_moe_down_round(long long rows, int E, int D) {
  const double live = fmax(ceil(moe_live((double)rows, E, 128)), moe_live_uneven((double)rows, E, 128));
  for (int nb = 2; nb <= 3; nb++)
    if (live * ((D + 64 * nb - 1) / (64 * nb)) <= 256) return nb;
  return 0;
}

template <bool UP>
static int moe_product(int bm, int E, const MoeArgs& a, hipStream_t stream) {
  const long long rows = (long long)a.T * a.top;
  if (!UP && bm == 128) {
    const int round = pico_moe_down_round(rows, E, a.D);
    if (round == 2) return moe_launch<2, 2, false, 1, 5>(a, stream);
    if (round == 3) return moe_launch<2, 3, false, 1, 4>(a, stream);
  }
  const double live = moe_live((double)rows, E, bm);
  double cost[2];
  for (int i = 0; i < 2; i++) {
    const MoeTile& t = moe_tiles[bm == 128][i];
    const int cols = (UP ? 32 : 64) * t.nb, n = UP ? a.F : a.D;
    const double rounds = ceil(live) * ((n + cols - 1) / cols) / (256.0 * t.share), full = floor(rounds), rest = rounds - full;
    cost[i] = full * t.each + (rest == 0 ? 0 : rest * t.share <= 1 ? t.lone : t.each);
  }
  const bool second = cost[1] < cost[0];
  if (bm == 64) return second ? moe_launch<1, 2, UP>(a, stream) : moe_launch<1, 1, UP>(a, stream);
  return second ? moe_launch<2, 4, UP>(a, stream) : moe_launch<2, 3, UP>(a, stream);
}

// sorted: int32 [2 tiles_cap bm] (row numbers, then weights), tiles: int32 [2 tiles_cap + 1]
extern "C" int pico_moe_experts_grouped(const void* h, int ldh, const void* gate_up, const void* down, const int* experts,
                                        const float* weights, const int* live, int* sorted, int* tiles, int tiles_cap, int bm, void* y,
                                        float* out, int T, int top, int E, int F, int D, float limit, float alpha,
                                        int mode, hipStream_t stream) {
  PICO_REQUIRE(mode >= 0 && mode <= 2, "pico_moe_experts_grouped: unknown mode %d", mode);
  PICO_REQUIRE(T >= 0 && top > 0 && E > 0 && F > 0 && D > 0 && ldh >= D, "pico_moe_experts_grouped: bad sizes");
  PICO_REQUIRE(E <= MOE_SORT_MAX_E, "pico_moe_experts_grouped: at most %d experts", MOE_SORT_MAX_E);
  PICO_REQUIRE(F % 8 == 0 && D % 8 == 0 && ldh % 8 == 0, "pico_moe_experts_grouped: sizes must be multiples of 8");
  PICO_REQUIRE(((uintptr_t)h | (uintptr_t)gate_up | (uintptr_t)down | (uintptr_t)y | (uintptr_t)out) % 16 == 0,
               "pico_moe_experts_grouped: operands must start on 16 bytes");
  if (T == 0) return 0;
  const long long R = (long long)T * top;
  PICO_REQUIRE(R < (1ll << 30), "pico_moe_experts_grouped: too many rows");
  PICO_REQUIRE((long long)T * ldh < (1ll << 30) && (long long)F * D < (1ll << 29),
               "pico_moe_experts_grouped: the activations or an expert's matrix span 2^31 bytes or more");
  PICO_REQUIRE(bm == pico_moe_tile_rows(R, E), "pico_moe_experts_grouped: tiles of %d rows", bm);
  const long long need = (R + (long long)E * (bm - 1)) / bm;
  PICO_REQUIRE(tiles_cap >= need, "pico_moe_experts_grouped: room for %d tiles, %lld may be needed", tiles_cap, need);
  float* sorted_w = (float*)sorted + (size_t)tiles_cap * bm;
  // (with more rows every expert has some either way, and to look for padding takes longer than it gives)
  if (R > MOE_LANES || R > 2 * E) live = nullptr;
  moe_sort_kernel<<<E, MOE_SORT_THREADS, 0, stream>>>(experts, weights, (int)R, E, bm, tiles_cap, sorted, sorted_w, tiles, live, top, out, T, D);
  const MoeArgs up{(const bf16_t*)h, (const bf16_t*)gate_up, sorted, sorted_w, tiles, (bf16_t*)y, nullptr, tiles_cap, ldh, T, top, F, D, 0, mode, limit, alpha};
  MoeArgs dn = up;
  dn.X = (const bf16_t*)y; dn.W = (const bf16_t*)down; dn.out = out;
  int rc = moe_product<true>(bm, E, up, stream);
  if (!rc) rc = moe_product<false>(bm, E, dn, stream);
  if (rc) return rc;
  PICO_LAUNCH_CHECK();
  return 0;
}
