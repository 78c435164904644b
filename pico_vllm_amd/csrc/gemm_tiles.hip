// Tiled bfloat16 product (prompt portions): C = X W^T (+ bias) and an epilogue, tiles as tile_stream.h has them, the tiles of
// a call dealt out to workgroups that stay.  What an activation behind the library's product costs is a pass over [T, 2 I]
// and back; here it is made of the sums in registers.  2,048 rows, 8,960 pairs, K 1,536: 115 us (0.98 PFLOP/s) against 117 and
// 20 for product and pass; 832 rows, 18,944 pairs, K 3,584: 223 against 266 and 20; 65 rows of a 152,064 x 3,584 output matrix in
// float32: 225 against 965 with the kernel for few rows (which reads the matrix once a 64 rows and unstaged).
#include "tile_stream.h"

// what becomes of the sums (the numbers are those of the weight-streaming product)
#define GT_BF16 0     // + bias
#define GT_F32 1      // + bias, float32
#define GT_SWIGLU 2   // W = [gate rows; up rows]: silu(gate) up, N / 2 columns
#define GT_RELU2 3    // max(x W^T + bias, 0)^2
#define GT_CLIPPED 5  // W = [gate rows; up rows]: g sigmoid(alpha g) (u + 1), g = min(gate, limit), u = up within -limit .. limit
#define GT_GELU 7     // gelu(x W^T + bias) with the error function
#define GT_PARTS 8    // float32 sums of a part of K (of the launches here alone)

struct GemmArgs {
  const bf16_t* X;
  const bf16_t* W;
  const float* bias;
  void* out;
  int M, cols, K, ldx, ldw, ldo;     // cols: output columns of this launch
  int up;                            // paired epilogues: from a gate row of W to the up row of the same column
  int m_tiles, n_tiles;
  int bring;                         // so much of k is read ahead by workgroups without a tile (unpaired, whole K; the grid has some)
  int splits, part;                  // of K: so many parts of `part` each, a part's sums in out + s M ldo (GT_PARTS; else one)
  float limit, alpha;
};

#define GT_COLS(NB, EPI) (gt_paired(EPI) ? 32 * (NB) : 64 * (NB))     // output columns of a tile
constexpr bool gt_paired(int epi) { return epi == GT_SWIGLU || epi == GT_CLIPPED; }
constexpr bool gt_float(int epi) { return epi == GT_F32 || epi == GT_PARTS; }

// FEW: with the exponential of the weight-streaming product
template <int EPI, bool FEW>
__device__ __forceinline__ float gt_pair(float g, float u, const GemmArgs& a) {
  if (EPI == GT_SWIGLU) return FEW ? g / (1.0f + __expf(-g)) * u : silu_f(g) * u;
  g = fminf(g, a.limit);
  u = fminf(fmaxf(u, -a.limit), a.limit);
  return (FEW ? g / (1.0f + __expf(-a.alpha * g)) : times_sigmoid(g, a.alpha * g)) * (u + 1.0f);
}
// z times the normal distribution's share below z, without a branch: a thread has up to 144 of them in a row, and erff has two
// branches, both taken by every wave.  13,440 outputs with a bias, K 1,536, microseconds with erff and the bias read between the
// outputs / so / library and pass: 300 rows 49 / 29 / 33, 1,024 100 / 60 / 63, 2,048 182 / 112 / 115.  With x = |z| / sqrt 2 the share beyond |z| is
// exp(-x^2) t Q(t), t = 1 / (1 + 0.3 x), Q of degree 8 fitted to erfc(x) exp(x^2) / (2 t) for equal relative error on 0 .. 10
// (2e-8).  Error against 64 bits over normal z 4.1e-8, 3.8e-8 with erff; of the smallest results (z below -4) 1e-6 of
// their size, where 1 + erf has lost all of it.
__device__ __forceinline__ float gt_gelu(float z) {
  const float t = __builtin_amdgcn_rcpf(fmaf(fabsf(z), 0.212132034f, 1.0f));
  float q = -0.06476139f;
  q = fmaf(q, t, 0.24278131f);
  q = fmaf(q, t, -0.25613844f);
  q = fmaf(q, t, 0.27385935f);
  q = fmaf(q, t, -0.047324907f);
  q = fmaf(q, t, 0.10746284f);
  q = fmaf(q, t, 0.07416963f);
  q = fmaf(q, t, 0.085357606f);
  q = fmaf(q, t, 0.084594004f);
  const float beyond = q * t * __builtin_amdgcn_exp2f(z * z * -0.72134752f);
  return z * (z > 0.f ? 1.0f - beyond : beyond);
}
template <int EPI>
__device__ __forceinline__ float gt_one(float v) {
  if (EPI == GT_RELU2) { v = fmaxf(v, 0.f); return v * v; }
  return EPI == GT_GELU ? gt_gelu(v) : v;
}
typedef float gt_f32x4 __attribute__((ext_vector_type(4), aligned(4)));

template <int MB, int NB, int EPI, int SETS, int SHARE, int BUFS>
__global__ __launch_bounds__(256, SHARE) void gemm_tiles_kernel(const GemmArgs a) {
#ifdef __HIP_DEVICE_COMPILE__      // (buffer resources exist on the device only)
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  typedef TileStream<MB, NB, SETS, EPI == GT_PARTS, BUFS> TS;
  TS ts(smem);
  constexpr int TM = 64 * MB, TN = 64 * NB, COLS = gt_paired(EPI) ? TN / 2 : TN;      // output columns of a tile
  const int tiles = a.m_tiles * a.n_tiles * (EPI == GT_PARTS ? a.splits : 1);
  if (ts_tile(0, tiles) < 0) {
    // (a single round: the first `busy` places of a die have its tiles)
    const int busy = (tiles + 7) >> 3;
    if (a.bring > 0 && (int)(blockIdx.x >> 3) >= busy)
      ts_bring(a.W, a.cols, a.ldw, a.bring, (int)blockIdx.x - 8 * busy, (int)gridDim.x - 8 * busy, smem);
    return;
  }
  TileRowsSource<MB> xs;
  TileRowsSource<NB> ws;
  auto aim = [&](int t) {
    int m, n;
    ts_place(a.m_tiles, a.n_tiles * (EPI == GT_PARTS ? a.splits : 1), t, m, n);
    const int m0 = m * TM, s = EPI == GT_PARTS ? n / a.n_tiles : 0, k0 = s * a.part, k = EPI == GT_PARTS ? min(a.part, a.K - k0) : a.K;
    n -= s * a.n_tiles;
    if (EPI == GT_PARTS) ts.k_end = k;
    xs.rsrc = ts_buffer(a.X + (size_t)m0 * a.ldx + k0, ((long long)(a.M - m0 - 1) * a.ldx + k) * 2);
#pragma unroll
    for (int j = 0; j < 2 * MB; j++) xs.off[j] = (uint32_t)(ts.row(j) * a.ldx) * 2;
    if (gt_paired(EPI)) {
      // blocks of 32 tile rows are 16 gate rows and the 16 up rows of the same columns
      const int c0 = n * COLS;
      ws.rsrc = ts_buffer(a.W, ((long long)(a.up + a.cols - 1) * a.ldw + a.K) * 2);
#pragma unroll
      for (int j = 0; j < 2 * NB; j++) {
        const int r = ts.row(j), c = c0 + (r >> 5) * 16 + (r & 15);
        ws.off[j] = c < a.cols ? (uint32_t)((c + ((r & 16) ? a.up : 0)) * a.ldw) * 2 : TS_OUT;
      }
    } else {
      const int n0 = n * TN;
      ws.rsrc = ts_buffer(a.W + (size_t)n0 * a.ldw + k0, ((long long)(a.cols - n0 - 1) * a.ldw + k) * 2);
#pragma unroll
      for (int j = 0; j < 2 * NB; j++) ws.off[j] = (uint32_t)(ts.row(j) * a.ldw) * 2;
    }
  };
  ts.run(tiles, EPI == GT_PARTS ? a.part : a.K, xs, ws, aim, [&](int t) {
    // lane (l, h): row l of a block of X, tile rows 8 (r / 4) + 4 h + r % 4 of a block of W in register r
    int mt, nt;
    ts_place(a.m_tiles, a.n_tiles * (EPI == GT_PARTS ? a.splits : 1), t, mt, nt);
    const int split = EPI == GT_PARTS ? nt / a.n_tiles : 0;
    nt -= split * a.n_tiles;
    const int l = ts.lane & 31, h = ts.lane >> 5;
    // of the bias what this lane adds, all of it asked for at once (a pair at a time between the outputs it was waited for each
    // time: 32 us of a call of 2,048 rows, 13,440 columns).  Not with float32 results, which do
    // little but store: of a 152,064 x 3,584 output matrix without a bias 740 rows took 943 us so, 762 to 805 without, 32 rows 221 and 211.
    constexpr bool AHEAD = !gt_paired(EPI) && !gt_float(EPI);
    gt_f32x4 bias[AHEAD ? NB : 1][4];
    if (AHEAD) {
#pragma unroll
      for (int j = 0; j < NB; j++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const int n = nt * TN + ((ts.wave & 1) * NB + j) * 32 + 8 * q + 4 * h;
          bias[AHEAD ? j : 0][q] = a.bias && n < a.cols ? *reinterpret_cast<const gt_f32x4*>(a.bias + n) : gt_f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
#pragma unroll
    for (int i = 0; i < MB; i++) {
      const int m = mt * TM + (ts.wave >> 1) * (32 * MB) + 32 * i + l;
#pragma unroll
      for (int j = 0; j < NB; j++) {
        ts_f32x16 v = ts.acc[0][j][i];
        if (SETS > 1) {
#pragma unroll
          for (int r = 0; r < 16; r++) {
            float sum = 0.f;
#pragma unroll
            for (int c = 0; c < SETS; c++) sum += ts.acc[c][j][i][r];
            v[r] = sum;
          }
        }
        const int blk = (ts.wave & 1) * NB + j;
        if (gt_float(EPI)) {
          float* o = (float*)a.out + ((size_t)split * a.M + m) * a.ldo;
#pragma unroll
          for (int q = 0; q < 4; q++) {
            const int n = nt * TN + blk * 32 + 8 * q + 4 * h;
            if (m < a.M && n < a.cols) {
              float4 f = make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
              if (a.bias) { f.x += a.bias[n]; f.y += a.bias[n + 1]; f.z += a.bias[n + 2]; f.w += a.bias[n + 3]; }
              *reinterpret_cast<float4*>(o + n) = f;
            }
          }
        } else {
          constexpr int G = gt_paired(EPI) ? 1 : 2;            // groups of 16 output columns in a block
#pragma unroll
          for (int g = 0; g < G; g++) {
            const int n = nt * COLS + blk * (16 * G) + 16 * g;
            uint32_t p[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
              float u0, u1;
              if (gt_paired(EPI)) {
                u0 = gt_pair<EPI, (SETS > 1)>(v[2 * q], v[8 + 2 * q], a);
                u1 = gt_pair<EPI, (SETS > 1)>(v[2 * q + 1], v[8 + 2 * q + 1], a);
              } else {
                const gt_f32x4 b = bias[AHEAD ? j : 0][2 * g + (q >> 1)];      // columns n + 8 (q / 2) + 4 h ..
                u0 = gt_one<EPI>(v[8 * g + 2 * q] + b[2 * (q & 1)]);
                u1 = gt_one<EPI>(v[8 * g + 2 * q + 1] + b[2 * (q & 1) + 1]);
              }
              p[q] = pack2_bf16(u0, u1);
            }
            // the halves of the wave hold columns 0..3 and 8..11, 4..7 and 12..15: swapped, eight neighbours each
            const auto s0 = __builtin_amdgcn_permlane32_swap(p[0], p[2], false, false);
            const auto s1 = __builtin_amdgcn_permlane32_swap(p[1], p[3], false, false);
            const int c = n + 8 * h;
            if (m < a.M && c < a.cols)
              *reinterpret_cast<uint4*>((bf16_t*)a.out + (size_t)m * a.ldo + c) = make_uint4(s0[0], s1[0], s0[1], s1[1]);
          }
        }
      }
    }
  });
#endif
}

// Of a single round that leaves an eighth of its places idle: how much of k the workgroups there read ahead, all of it or what each of
// them can while a tile reads GT_BRING times as much (their one wave of copies a SIMD waits for itself); 0: nothing.  That pays where the
// tiles wait for memory and several of them want the same rows of W; where the flow into the compute units is the bound it only adds to
// it.  So, microseconds without and with (recorded launches, matrices from memory):
// * not for parts of K (65 rows of 1,536 x 13,440 21.2 / 27.1, 256 28.2 / 31.0, 832 of 3,584 x 18,944 135 / 134) nor tiles of 192 or 256 rows
//   (832 rows of 6,144 x 1,536 with gelu 26.8 / 28.3, 352 of 18,944 x 3,584 60 / 66),
// * a single tile of rows up to GT_BRING_LONE tiles (96 rows, gelu: 6,144 x 1,536 15.2 / 13.4, 8,960 15.9 / 15.4, 13,440 17.0 / 17.9),
// * not what two share some units for, if K is long (1,700 rows of 1,536 x 13,440 to float32 118 / 133),
// * where a helper gets through most of its rows of W (384 rows of 7,168 x 3,584 36.6 / 32.3, 300 of 8,960 x 1,536, with a helper's rows in two
//   fifths of the time, 17.3 / 18.6),
// * from few elements on, and not where the last tiles have next to no rows, which wait for W alone and so read ahead themselves (2,052 rows of
//   1,536 x 8,960 62 either way).
// Of 420 points drawn over the single rounds below 196 are left: 11 % faster in the geometric mean, the slowest 2 % behind; the others
// the same.
#define GT_BRING 0.4f
#define GT_BRING_MOST 0.5f
#define GT_BRING_LONE 160
#define GT_BRING_K 4096
#define GT_BRING_LEAST (4 << 20)
extern "C" int pico_gemm_tiles_ahead(int M, int cols, int K, int splits, int mb, int nb, int share) {
  const int m_tiles = (M + 64 * mb - 1) / (64 * mb), slots = 256 * share, last = (M - 1) % (64 * mb);
  const long long tiles = (long long)m_tiles * ((cols + 64 * nb - 1) / (64 * nb)), idle = slots - (tiles + 7) / 8 * 8;
  if (splits > 1 || mb != 2 || idle < slots / 8 || (long long)cols * K < GT_BRING_LEAST) return 0;
  if (last < 32) return 0;
  if ((m_tiles == 1 && tiles > GT_BRING_LONE) || (tiles > 256 && K > GT_BRING_K)) return 0;
  const float each = (float)ts_bring_rows(cols, (int)idle) / (64 * (mb + nb));
  if (each > GT_BRING_MOST) return 0;
  return each <= GT_BRING ? K : (int)(K * GT_BRING / each) / TS_BK * TS_BK;
}

template <int MB, int NB, int EPI, int SETS = 1, int SHARE = ts_share(MB, NB), int BUFS = ts_buffers(MB, NB)>
static int gt_launch(GemmArgs a, hipStream_t stream) {
  constexpr int bytes = ts_stage_bytes(MB, NB) * BUFS;
  const auto kernel = gemm_tiles_kernel<MB, NB, EPI, SETS, SHARE, BUFS>;
  static const hipError_t room = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  PICO_REQUIRE(room == hipSuccess, "pico_gemm_tiles: %s", hipGetErrorString(room));
  a.m_tiles = (a.M + 64 * MB - 1) / (64 * MB);
  a.n_tiles = (a.cols + GT_COLS(NB, EPI) - 1) / GT_COLS(NB, EPI);
  const long long tiles = (long long)a.m_tiles * a.n_tiles * a.splits;
  PICO_REQUIRE(tiles < (1LL << 30), "pico_gemm_tiles: %d x %d outputs are too many for one launch", a.M, a.cols);
  a.bring = gt_paired(EPI) ? 0 : pico_gemm_tiles_ahead(a.M, a.cols, a.K, a.splits, MB, NB, SHARE);
  kernel<<<a.bring ? 256 * SHARE : ts_grid(tiles, 256 * SHARE), 256, bytes, stream>>>(a);
  PICO_LAUNCH_CHECK();
  return 0;
}

// Which tile.  All make the same sums, so it is a question of how many rounds of workgroups a call takes and what one costs:
// microseconds `each` a stage + `more`, fitted to calls of 24 and 56 stages with operands from memory.  A tile of which
// two share a compute unit costs `lone` a stage where a unit has one.  Outputs a microsecond of a full round are alike
// (0.34 to 0.36 million a microsecond and 24 stages), so what is left idle in the last round decides.
struct GtTile { int mb, nb, share; float each, lone, more; };
static const GtTile gt_tiles[] = {{2, 3, 2, 1.45f, 1.20f, 3.f}, {4, 2, 1, 0.84f, 0.84f, 3.8f}, {3, 3, 1, 1.00f, 1.00f, 2.f}, {2, 1, 2, 0.80f, 0.35f, 3.f}};

// The tile for M rows and `cols` columns and its cost.  `first`: how many columns to make in whole rounds with it, the
// others being better left to a launch of their own with the tile that suits them (2,052 rows of 8,960 pairs: three rounds
// and 62 tiles; the 62 as a fourth round cost 32 us, as 170 tiles of a third their size 12); else all.
static int gt_choose(int M, int cols, int stages, bool paired, bool split, int& first, float& cost, int parts = 1) {
  int best = 0;
  cost = 3e38f;
  for (int i = 0; i < 4; i++) {
    const GtTile& t = gt_tiles[i];
    const int tile_cols = GT_COLS(t.nb, paired ? GT_SWIGLU : GT_BF16), m_tiles = (M + 64 * t.mb - 1) / (64 * t.mb);
    const long long tiles = (long long)m_tiles * ((cols + tile_cols - 1) / tile_cols) * parts, round = 256 * t.share, full = tiles / round, rest = tiles % round;
    const float whole = (float)full * (t.each * stages + t.more);
    const float c = whole + (rest ? (rest <= 256 ? t.lone : t.each) * stages + t.more : 0.f);
    if (c < cost) { cost = c; best = i; first = cols; }
    const int n1 = (int)(full * round / m_tiles) * tile_cols;
    if (split && rest && n1 > 0 && n1 < cols) {
      int all;
      float other;
      gt_choose(M, cols - n1, stages, paired, false, all, other);
      if (whole + other + 3.f < cost) { cost = whole + other + 3.f; best = i; first = n1; }      // 3 us: a launch
    }
  }
  return best;
}

template <int EPI>
static int gt_run(GemmArgs a, hipStream_t stream) {
  const int stages = (a.part + TS_BK - 1) / TS_BK, cols = a.cols;
  int first, all, rc = 0;
  float cost;
  const int tile = gt_choose(a.M, cols, stages, gt_paired(EPI), a.splits == 1, first, cost, a.splits);
  auto run = [&](int i) {
    switch (i) {
      case 0: return gt_launch<2, 3, EPI>(a, stream);
      case 1: return gt_launch<4, 2, EPI>(a, stream);
      case 2: return gt_launch<3, 3, EPI>(a, stream);
      default: return gt_launch<2, 1, EPI>(a, stream);
    }
  };
  a.cols = first;
  rc = run(tile);
  if (rc || first == cols) return rc;
  a.W += (size_t)first * a.ldw;
  if (a.bias) a.bias += first;
  a.out = (char*)a.out + (size_t)first * (gt_float(EPI) ? 4 : 2);
  a.cols = cols - first;
  return run(gt_choose(a.M, a.cols, stages, gt_paired(EPI), false, all, cost));
}

// Plain products that are a single round of small tiles.  What such a call takes is the stages' latency from memory, so its
// workgroups have a compute unit each and as many stages on their way as LDS holds (128 x 128, K 1,536, 192 tiles: two buffers
// and two workgroups a unit 21.3 us, three, four, five buffers 15.5, 15.5, 16.3), and where an eighth of the units has no tile
// those read the matrix ahead (pico_gemm_tiles_ahead).  Microseconds, library / so without / with W read ahead, matrices from memory: 2,048 rows of
// 1,536 x 1,536 15.8 / 13.4, x 4,480 37.5 / 39.4 / 31.8, x 8,960 71.2 / 74.8 / 65.4; 640 rows of 3,584 x 4,736 40.5 / 44.3 / 34.1, 832 38.4 / 39.8,
// of 3,584 x 3,584 31.0 / 30.7; 352 of 7,168 x 3,584 34.9 / 35.0 / 30.3.  Of up to
// 128 such tiles 128 x 64 are a single round too; each is as long a chain as the larger, so they pay for short K alone and from
// where the library's fewer, longer workgroups run out: 700 rows of 1,536 x 1,536 12.8 / 11.1 (640 10.2 / 11.4), 400 of 3,072 x 1,536 13.0 /
// 11.5, 300 of 4,608 x 1,536 14.0 / 11.6, 832 of 2,048 x 2,048 15.2 / 14.2, of 1,536 x 2,240 16.5 / 14.7, of 1,536 x 3,072 17.8 / 18.9.  Of 420
// points drawn over these ranges the geometric mean is 12 % ahead of the library; 44 are behind it, most of them with up to 32 rows in
// the last tiles, where it depends on how the library's come out (129 rows of 5,120 x 2,560 16.1 / 20.2, the worst, of 6,144 x 2,048 21.5 / 16.8).
#define GT_ROUND 256
#define GT_NARROW 144                                // the library is as fast up to so many tiles of 128 x 64
#define GT_NARROW_K 2560
static int gt_small(int M, int N, int mb, int nb) { return ((M + 64 * mb - 1) / (64 * mb)) * ((N + 64 * nb - 1) / (64 * nb)); }
// 0: more or fewer tiles than that; 1: tiles of 128 x 64; 2: of 128 x 128
extern "C" int pico_gemm_tiles_round(int M, int N, int K) {
  if (M <= 64 || N <= 0 || K <= 0 || (long long)M * N > (long long)GT_ROUND * 128 * 128) return 0;
  const int narrow = gt_small(M, N, 2, 1), square = gt_small(M, N, 2, 2);
  if (narrow <= GT_ROUND) return K <= GT_NARROW_K && narrow > GT_NARROW ? 1 : 0;
  return square <= GT_ROUND && square > GT_ROUND / 2 ? 2 : 0;
}

// Up to 64 rows of a large matrix: the stream of W bounds a call, and tiles of 64 rows carry it.  32 rows of a 152,064 x 3,584
// output matrix in float32 203 us (5.4 TB/s; the weight-streaming product 244), of 28,416 pairs, K 3,584, 74 (89).  A row must not
// depend on how many others the call has, and fewer rows or a smaller matrix go through the weight-streaming product: so its
// sums are made here, four chains that take 64 k after 64 k in turn, added up in its order (as fast as one chain).
// 128 columns of W while that leaves no second round, then 64, which round up less (those two calls with the other width: 224 and
// 76).
template <int EPI>
static int gt_few(const GemmArgs& a, hipStream_t stream) {
  return a.cols <= 512 * GT_COLS(2, EPI) ? gt_launch<1, 2, EPI, 4>(a, stream) : gt_launch<1, 1, EPI, 4>(a, stream);
}

// X [M, K] row stride ldx, W [N, K] row stride ldw, bfloat16; out [M, N] (N / 2 columns for the paired epilogues) row stride
// ldo, bfloat16 or (GT_F32) float32.  All strides, K and the columns multiples of 8, the pointers on 16 bytes, each
// operand's span below 2^31 bytes.  few: up to 64 rows with the weight-streaming product's sums (float32 and paired epilogues).
extern "C" int pico_gemm_tiles(const void* X, const void* W, const float* bias, void* out, int epi, int M, int N,
                               int K, int ldx, int ldw, int ldo, float limit, float alpha, int few, hipStream_t stream) {
  PICO_REQUIRE(M >= 0 && N > 0 && K > 0, "pico_gemm_tiles: bad sizes M=%d N=%d K=%d", M, N, K);
  const int cols = gt_paired(epi) ? N / 2 : N;
  PICO_REQUIRE(ldx >= K && ldw >= K && ldo >= cols, "pico_gemm_tiles: a row stride is smaller than its row");
  PICO_REQUIRE(K % 8 == 0 && ldx % 8 == 0 && ldw % 8 == 0 && ldo % 8 == 0 && cols % 8 == 0 && (!gt_paired(epi) || N % 2 == 0),
               "pico_gemm_tiles: sizes and strides must be multiples of 8");
  PICO_REQUIRE(((uintptr_t)X | (uintptr_t)W | (uintptr_t)out) % 16 == 0, "pico_gemm_tiles: operands must start on 16 bytes");
  PICO_REQUIRE((long long)M * ldx < (1LL << 30) && (long long)N * ldw < (1LL << 30), "pico_gemm_tiles: an operand spans 2^31 bytes or more");
  PICO_REQUIRE(!bias || !gt_paired(epi), "pico_gemm_tiles: the paired epilogues take no bias");
  if (M == 0) return 0;
  GemmArgs a{(const bf16_t*)X, (const bf16_t*)W, bias, out, M, cols, K, ldx, ldw, ldo, N - cols, 0, 0, 0, 1, K, limit, alpha};
  if (few) {
    PICO_REQUIRE(M <= 64, "pico_gemm_tiles: %d rows are not few", M);
    switch (epi) {
      case GT_F32: return gt_few<GT_F32>(a, stream);
      case GT_SWIGLU: return gt_few<GT_SWIGLU>(a, stream);
      case GT_CLIPPED: return gt_few<GT_CLIPPED>(a, stream);
    }
    PICO_REQUIRE(false, "pico_gemm_tiles: no epilogue %d for few rows", epi);
  }
  switch (epi) {
    case GT_BF16:
      switch (pico_gemm_tiles_round(M, N, K)) {
        case 1: return gt_launch<2, 1, GT_BF16>(a, stream);
        case 2: return gt_launch<2, 2, GT_BF16, 1, 1, 4>(a, stream);
      }
      return gt_run<GT_BF16>(a, stream);
    case GT_F32: return gt_run<GT_F32>(a, stream);
    case GT_SWIGLU: return gt_run<GT_SWIGLU>(a, stream);
    case GT_RELU2: return gt_run<GT_RELU2>(a, stream);
    case GT_CLIPPED: return gt_run<GT_CLIPPED>(a, stream);
    case GT_GELU: return gt_run<GT_GELU>(a, stream);
  }
  PICO_REQUIRE(false, "pico_gemm_tiles: unknown epilogue %d", epi);
}

// A long K with few tiles: K in parts that run side by side, each into float32 rows of its own, and one pass that adds a row's
// parts up in their order and rounds once.  832 rows of 3,584 outputs, K 18,944: two parts 125 us (0.90 PFLOP/s), whole
// 215 with 112 to 392 tiles on 256 compute units, the library's product 175.
// The pass, eight neighbours a thread, is bound by memory.
__global__ __launch_bounds__(256) void gemm_join_kernel(const float* __restrict__ parts, int splits, const float* __restrict__ bias,
                                                        bf16_t* __restrict__ out, long long eights, int N) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= eights) return;
  const gt_f32x4* p = reinterpret_cast<const gt_f32x4*>(parts) + 2 * i;
  gt_f32x4 lo = p[0], hi = p[1];
  for (int s = 1; s < splits; s++) {
    lo += p[2 * s * eights];
    hi += p[2 * s * eights + 1];
  }
  if (bias) {
    const gt_f32x4* b = reinterpret_cast<const gt_f32x4*>(bias + 8 * i % N);
    lo += b[0];
    hi += b[1];
  }
  reinterpret_cast<uint4*>(out)[i] = make_uint4(pack2_bf16(lo[0], lo[1]), pack2_bf16(lo[2], lo[3]), pack2_bf16(hi[0], hi[1]), pack2_bf16(hi[2], hi[3]));
}

#define GT_SPLITS 8
static int gt_part(int K, int splits) { return ((K + splits - 1) / splits + TS_BK - 1) / TS_BK * TS_BK; }

// Into how many parts: by the tiles' cost (gt_choose) and the pass's, which moves 4 bytes a part and output and 2 at 4.5 TB/s.
// 1: whole, without a pass.
extern "C" int pico_gemm_tiles_parts(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0) return 1;
  int best = 1, first;
  float least = 3e38f;
  for (int s = 1; s <= GT_SPLITS; s++) {
    const int part = gt_part(K, s);
    if (s > 1 && (long long)(s - 1) * part >= K) break;
    float cost;
    gt_choose(M, N, part / TS_BK, false, s == 1, first, cost, s);
    if (s > 1) cost += 3.f + (float)M * N * (4 * s + 2) / 4.5e6f;
    if (cost < least) { least = cost; best = s; }
  }
  return best;
}

// out [M, N] bfloat16 = X W^T + bias with K in `splits` parts; parts float32 [splits, M, N].  Operands as pico_gemm_tiles.
extern "C" int pico_gemm_tiles_split(const void* X, const void* W, const float* bias, float* parts, void* out, int splits, int M, int N,
                                     int K, int ldx, int ldw, hipStream_t stream) {
  PICO_REQUIRE(M >= 0 && N > 0 && K > 0, "pico_gemm_tiles_split: bad sizes M=%d N=%d K=%d", M, N, K);
  PICO_REQUIRE(splits > 1 && splits <= GT_SPLITS && (long long)(splits - 1) * gt_part(K, splits) < K, "pico_gemm_tiles_split: %d parts of %d", splits, K);
  PICO_REQUIRE(ldx >= K && ldw >= K && K % 8 == 0 && ldx % 8 == 0 && ldw % 8 == 0 && N % 8 == 0,
               "pico_gemm_tiles_split: sizes and strides must be multiples of 8");
  PICO_REQUIRE(((uintptr_t)X | (uintptr_t)W | (uintptr_t)out | (uintptr_t)parts | (uintptr_t)bias) % 16 == 0, "pico_gemm_tiles_split: operands must start on 16 bytes");
  PICO_REQUIRE((long long)M * ldx < (1LL << 30) && (long long)N * ldw < (1LL << 30), "pico_gemm_tiles_split: an operand spans 2^31 bytes or more");
  if (M == 0) return 0;
  GemmArgs a{(const bf16_t*)X, (const bf16_t*)W, nullptr, parts, M, N, K, ldx, ldw, N, 0, 0, 0, 0, splits, gt_part(K, splits), 0.f, 0.f};
  const int rc = gt_run<GT_PARTS>(a, stream);
  if (rc) return rc;
  const long long eights = (long long)M * N / 8;
  gemm_join_kernel<<<(unsigned)((eights + 255) / 256), 256, 0, stream>>>(parts, splits, bias, (bf16_t*)out, eights, N);
  PICO_LAUNCH_CHECK();
  return 0;
}
