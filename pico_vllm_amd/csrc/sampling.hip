// Sampling from float32 logits with per-row parameters:
//   temperature == 0        argmax, lowest index on a tie            (pico_vllm/sampler.py:8)
//   top_p >= 1              draw from softmax(logits / T)             (sampler.py:16-17)
//   top_p <  1              keep the tokens whose preceding cumulative mass, in descending
//                           order of probability, is < top_p (the token that crosses stays),
//                           renormalise, draw                          (sampler.py:25-36)
// The draw is the inverse CDF in vocabulary order at the uniform number u[row] that the
// host supplies (the reference calls torch.multinomial; only the distribution is shared).
// The kept set of top-p is found without sorting: with e_i = exp((x_i - max) / T) and
// f(t) = sum of e_i > t, the kept tokens are those with e_i > t*, t* being the smallest
// float with f(t*) < top_p * sum(e), and of the tokens with e_i == t* exactly (the token that
// crosses, and any tied with it) the first ceil((top_p * sum - f(t*)) / t*) in vocabulary order:
// a sort keeps a prefix of tied tokens, not all of them (sampler.py:25-32; which of them is the
// sort's choice there, the lowest indices here, as a stable sort would).
//
// A row is read by SAMPLE_CHUNKS workgroups, one per chunk of the vocabulary (one workgroup reads a row no
// faster than one compute unit takes data in: 19 us for 151,936 logits), in a chain of launches whose
// workgroups never wait for one another: what a launch needs of the launch before it lies in memory.
//   1. the first maximum of every chunk (argmax_part_kernel);
//   2. for rows with top_p < 1, the mass of e by its bit pattern (e lies in (0, 1], where the patterns' order is the order of
//      the values): 2,033 classes of 2^19 patterns, a sixteenth of a factor of two each (sample_classes_kernel);
//   3. every workgroup finds from them the class in which f drops below the target, sums what its chunk has above that class, in
//      double, and lists what it has in it (sample_collect_kernel);
//   4. one workgroup a row finds t* among what is listed (classes of 2^9 patterns, then of one), then the chunk, the
//      thread, and the token at which the running sum of the kept e passes u times their total, ties counted in
//      vocabulary order (sample_pick_kernel).
// The search sums e as whole numbers of 2^-40 (fewer bits beyond 2^23 tokens): such sums are the same in any order, so they are
// made with atomics.  Each term is rounded down by less than 2^-40 of the largest, which is 1: V tokens lose less than V 2^-40 of a mass
// of 1 or more, 1.4e-7 at 151,936 tokens (7e-8 on average), 7.6e-6 at 2^23.  All other sums run in a fixed order: a row's result
// depends on its inputs only.  e is the hardware's exponential (__expf: 2^(x log2 e)) in every launch alike: what a token weighs
// must be the same bits wherever it is asked.
// (Five rounds of 63 thresholds and float sums, each a launch that read the row, in place of 2 and the search of 4: the chain 62 us for 8 rows
// of 151,936 logits with top_p < 1, 32 so; 64 rows 159, 65; one row 63, 30; 5,000 logits 34, 24.  Where a class holds most of a row
// the last launch's one workgroup has it all: logits within a twentieth of each other 61, 58.  Where a chunk's elements are most of it
// and all alike they are listed once: all logits equal 28, one by one 93.)
#include <chrono>

#include "common.h"

#define SAMPLE_CHUNKS 32            // as ARGMAX_CHUNKS below: the two share the first launch
#define ARGMAX_CHUNKS 32
#define SAMPLE_THREADS 256
#define SAMPLE_PICK_THREADS 1024    // of the last launch where it searches (else SAMPLE_THREADS)
#define SAMPLE_PIECE 8192           // the elements of the chosen chunk that the last launch holds in registers
#define SAMPLE_HELD 32              // the elements of a chunk that a thread of the third launch holds in registers
#define SAMPLE_CLASSES 2048         // of patterns: b >> SAMPLE_LOW; no e is above 1.0f, the first of class 2032
#define SAMPLE_LOW 19
#define SAMPLE_MID 9                // the last launch's classes: 2^(19 - 9) of 2^9 patterns, 2^9 of one
#define SAMPLE_ONE 0x3f800000u      // the bit pattern of 1.0f
#define SAMPLE_LISTED 4864          // elements of a class that a chunk lists at most (all of a chunk up to 155,648 tokens); more are read again
#define SAMPLE_ROWS 256             // rows with a list at a time
#define SAMPLE_ALIKE 256            // from so many on, and half of it, a chunk looks whether they are one value, and then lists it once

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct SampleChunk {
  int begin, end;
};
__device__ __forceinline__ SampleChunk sample_chunk(int V, int c) {
  const int len = (V + SAMPLE_CHUNKS - 1) / SAMPLE_CHUNKS;
  const int begin = min(V, c * len);
  return {begin, min(V, begin + len)};
}

// a lane's of the row's chunks' maxima (each stands in two lanes): the row's is their wave_max, in every lane of every wave
__device__ __forceinline__ float sample_chunk_max(const float* __restrict__ part_val, int row) {
  static_assert(SAMPLE_CHUNKS == 32, "a chunk in two lanes");
  return part_val[row * SAMPLE_CHUNKS + (threadIdx.x & 31)];
}

// e as a whole number of 2^-bits, rounded down
__device__ __forceinline__ unsigned long long sample_fixed(uint32_t b, int bits) {
  const uint32_t off = 127u - min(b >> 23, 127u);          // e in [2^-off, 2^(1 - off))
  const unsigned long long m = (unsigned long long)((b & 0x7fffffu) | 0x800000u) << (bits - 23);
  return off < 64u ? m >> off : 0ull;
}
__device__ __forceinline__ uint32_t sample_class(uint32_t b) { return min(b >> SAMPLE_LOW, (uint32_t)SAMPLE_CLASSES - 1); }

// What the launches before the last leave of a row's search: the class, the mass above it, and the target.
struct SampleRow {
  unsigned long long above;
  float target;
  uint32_t cls;
};

// Sum over the threads behind this one, and of all, of a workgroup of `waves` waves; whole numbers.
__device__ __forceinline__ unsigned long long block_behind(unsigned long long v, unsigned long long* scratch, int waves, unsigned long long& total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  unsigned long long incl = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const unsigned long long o = __shfl_down(incl, off, 64);
    if (lane + off < 64) incl += o;
  }
  __syncthreads();
  if (lane == 0) scratch[wave] = incl;
  __syncthreads();
  unsigned long long behind = 0;
  total = 0;
  for (int k = 0; k < waves; k++) {
    if (k > wave) behind += scratch[k];
    total += scratch[k];
  }
  return behind + incl - v;
}
// Of N classes a thread, in ascending order, with `above` behind them: the one at which the sum from above reaches the target.
template <int N>
__device__ __forceinline__ void sample_cross(const unsigned long long (&h)[N], unsigned long long above, double target, int first, int* cls,
                                             unsigned long long* mass) {
#pragma unroll
  for (int j = N - 1; j >= 0; j--) {
    if ((double)above < target && (double)(above + h[j]) >= target) {
      *cls = first + j;
      *mass = above;
    }
    above += h[j];
  }
}

// Additions to classes in LDS, a run of one class at a time: rows of equal or nearly equal logits send all lanes to one place.
struct SampleRun {
  unsigned long long* hist;
  uint32_t at = 0;
  unsigned long long sum = 0;
  __device__ __forceinline__ void add(uint32_t cls, unsigned long long f) {
    if (cls != at) {
      if (sum) atomicAdd(&hist[at], sum);
      at = cls;
      sum = 0;
    }
    sum += f;
  }
  __device__ __forceinline__ void end() {
    if (sum) atomicAdd(&hist[at], sum);
  }
};

// Sums of a chunk's e by class, added to the row's (which the first launch has cleared).
__global__ __launch_bounds__(SAMPLE_THREADS) void sample_classes_kernel(
    const float* __restrict__ logits, int ld, int V, const float* __restrict__ temperature, const float* __restrict__ top_p,
    const float* __restrict__ part_val, unsigned long long* __restrict__ classes, int bits) {
  __shared__ unsigned long long hist[SAMPLE_CLASSES];
  const int row = blockIdx.x, c = blockIdx.y, tid = threadIdx.x;
  // everything the workgroup needs from memory is asked for at once, whatever it turns out to need, without branches of lanes and
  // before anything is waited for: what the launch before wrote comes from memory, a microsecond or two away, and asking one after
  // the other would add them up
  const float mine = sample_chunk_max(part_val, row), temp = temperature[row], tp = top_p[row];
  const float* x = logits + (size_t)row * ld;
  const SampleChunk ch = sample_chunk(V, c);
  constexpr int AT_ONCE = 24;                              // elements of a thread: all of a chunk up to vocabularies of 196,608
  float v[AT_ONCE];
  // (In eights, as many as the chunk has.  With all of them always the chain for 8 rows of 157 and 5,000 logits 22.7 and 24.3 us, so 22.1 and 23.7,
  // 300 rows of 157 and 1,000 90 and 91, so 82 and 85, 64 rows of 50,257 47.2, so 45.7; 8 rows of 151,936 30.7 and 30.8.)
  auto fetch = [&](int from) {
#pragma unroll
    for (int g = 0; g < AT_ONCE; g += 8)
      if (from + g * SAMPLE_THREADS < ch.end) {
#pragma unroll
        for (int k = g; k < g + 8; k++) v[k] = x[min(from + tid + k * SAMPLE_THREADS, V - 1)];
      }
  };
  fetch(ch.begin);
  const float mx = wave_max(mine);
  if (!(temp > 0.f) || !(tp < 1.0f)) return;
  const float inv_t = 1.0f / temp;
#pragma unroll
  for (int j = 0; j < SAMPLE_CLASSES / SAMPLE_THREADS; j++) hist[j * SAMPLE_THREADS + tid] = 0ull;
  __syncthreads();
  SampleRun run{hist};
  for (int from = ch.begin;;) {
#pragma unroll
    for (int g = 0; g < AT_ONCE; g += 8)
      if (from + g * SAMPLE_THREADS < ch.end) {
#pragma unroll
        for (int k = g; k < g + 8; k++) {
          const float e = from + tid + k * SAMPLE_THREADS < ch.end ? __expf((v[k] - mx) * inv_t) : 0.f;
          if (e > 0.f) run.add(sample_class(__float_as_uint(e)), sample_fixed(__float_as_uint(e), bits));
        }
      }
    from += AT_ONCE * SAMPLE_THREADS;
    if (from >= ch.end) break;
    fetch(from);
  }
  run.end();
  __syncthreads();
#pragma unroll
  for (int j = 0; j < SAMPLE_CLASSES / SAMPLE_THREADS; j++) {
    const unsigned long long f = hist[j * SAMPLE_THREADS + tid];
    if (f) atomicAdd(&classes[(size_t)row * SAMPLE_CLASSES + j * SAMPLE_THREADS + tid], f);
  }
}

__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}
__device__ __forceinline__ int wave_sum_i32(int v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// exclusive prefix sums over the workgroup's threads, in a fixed order; `total` gets the sum of all
template <int THREADS>
__device__ __forceinline__ double block_prefix_f64(double v, double* wave_tot, double& total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double incl = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const double o = __shfl_up(incl, off, 64);
    if (lane >= off) incl += o;
  }
  __syncthreads();
  if (lane == 63) wave_tot[wave] = incl;
  __syncthreads();
  double before = 0.0;
  total = 0.0;
  for (int k = 0; k < THREADS / 64; k++) {
    if (k < wave) before += wave_tot[k];
    total += wave_tot[k];
  }
  return before + incl - v;
}
template <int THREADS>
__device__ __forceinline__ int block_prefix_i32(int v, int* wave_tot, int& total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int incl = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int o = __shfl_up(incl, off, 64);
    if (lane >= off) incl += o;
  }
  __syncthreads();
  if (lane == 63) wave_tot[wave] = incl;
  __syncthreads();
  int before = 0;
  total = 0;
#pragma unroll
  for (int k = 0; k < THREADS / 64; k++) {
    if (k < wave) before += wave_tot[k];
    total += wave_tot[k];
  }
  return before + incl - v;
}

// Per chunk: the sum (double) of the e above the row's class, and a list of those in it, a thread's behind the last thread's; the
// number that there are.  Where they are many and all alike (equal logits) one stands for them, and the number is its complement.
// Rows with top_p >= 1: the sum of all.
template <bool SEARCH>
__global__ __launch_bounds__(SAMPLE_THREADS) void sample_collect_kernel(
    const float* __restrict__ logits, int ld, int V, const float* __restrict__ temperature, const float* __restrict__ top_p,
    const float* __restrict__ part_val, const unsigned long long* __restrict__ classes, int bits, double* __restrict__ fin_s,
    int* __restrict__ fin_n, uint32_t* __restrict__ list, int room, SampleRow* __restrict__ rows) {
  __shared__ unsigned long long scratch[SAMPLE_THREADS / 64], mass;
  __shared__ int cls;
  __shared__ double ws[SAMPLE_THREADS / 64];
  __shared__ int wn[SAMPLE_THREADS / 64];
  __shared__ uint32_t ends[2][SAMPLE_THREADS / 64];
  const int row = blockIdx.x, c = blockIdx.y, tid = threadIdx.x;
  // (asked for at once and without branches, as in the launch before)
  const float own_max = sample_chunk_max(part_val, row), temp = temperature[row], tp = SEARCH ? top_p[row] : 1.0f;
  const float* x = logits + (size_t)row * ld;
  const SampleChunk ch = sample_chunk(V, c);
  // the terms of the elements begin + thread, begin + thread + SAMPLE_THREADS, .., all asked for at once: one load at a
  // time, each used at once, is a chain of memory latencies (6 us for the 19 elements a thread has of a chunk of 151,936 logits)
  const bool held = ch.end - ch.begin <= SAMPLE_HELD * SAMPLE_THREADS;     // the same for all threads
  const int rounds = held ? (ch.end - ch.begin + 8 * SAMPLE_THREADS - 1) / (8 * SAMPLE_THREADS) : 0;      // of eight elements a thread
  float mine[SAMPLE_HELD];
#pragma unroll
  for (int g = 0; g < SAMPLE_HELD / 8; g++) {
    if (g < rounds) {
#pragma unroll
      for (int k = 8 * g; k < 8 * g + 8; k++) mine[k] = x[min(ch.begin + tid + k * SAMPLE_THREADS, V - 1)];
    }
  }
  constexpr int OWN = SEARCH ? SAMPLE_CLASSES / SAMPLE_THREADS : 1;
  unsigned long long h[OWN];                               // the row's classes that this thread looks at
#pragma unroll
  for (int j = 0; SEARCH && j < OWN; j++) h[j] = classes[(size_t)row * SAMPLE_CLASSES + tid * OWN + j];
  const float mx = wave_max(own_max);
  if (!(temp > 0.f)) return;
  const float inv_t = 1.0f / temp;
  int above = -1;                                          // keep what is above this class, list what is in it
  if (SEARCH && tp < 1.0f) {
    unsigned long long own = 0, total;
#pragma unroll
    for (int j = 0; j < OWN; j++) own += h[j];
    if (tid == 0) cls = SAMPLE_ONE >> SAMPLE_LOW, mass = 0;                // (a target that is not above zero: the largest alone)
    const unsigned long long behind = block_behind(own, scratch, SAMPLE_THREADS / 64, total);
    const double one = (double)(1ull << bits);
    const float target = tp * (float)((double)total / one);
    sample_cross(h, behind, (double)target * one, tid * OWN, &cls, &mass);
    __syncthreads();
    above = cls;
    if (c == 0 && tid == 0) rows[row] = {mass, target, (uint32_t)above};
  }
  double s = 0.0;
  int n = 0;
  auto each = [&](auto use) {
    if (held) {
#pragma unroll
      for (int g = 0; g < SAMPLE_HELD / 8; g++) {
        if (g < rounds) {
#pragma unroll
          for (int k = 8 * g; k < 8 * g + 8; k++)
            if (ch.begin + tid + k * SAMPLE_THREADS < ch.end) use(mine[k]);
        }
      }
    } else {
      for (int i0 = ch.begin + tid; i0 < ch.end; i0 += 8 * SAMPLE_THREADS) {
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
          const int i = i0 + k * SAMPLE_THREADS;
          v[k] = i < ch.end ? x[i] : 0.f;
        }
#pragma unroll
        for (int k = 0; k < 8; k++)
          if (i0 + k * SAMPLE_THREADS < ch.end) use(__expf((v[k] - mx) * inv_t));
      }
    }
  };
#pragma unroll
  for (int g = 0; g < SAMPLE_HELD / 8; g++) {
    if (g < rounds) {
#pragma unroll
      for (int k = 8 * g; k < 8 * g + 8; k++) mine[k] = __expf((mine[k] - mx) * inv_t);
    }
  }
  if (!SEARCH || above < 0) {
    each([&](float e) {
      if (e > 0.f) s += (double)e;
    });
  } else {
    each([&](float e) {
      const int k = (int)sample_class(__float_as_uint(e));
      if (k > above && e > 0.f) s += (double)e;
      n += k == above;
    });
    int all;
    const int before = block_prefix_i32<SAMPLE_THREADS>(n, wn, all);
    uint32_t* mylist = list + ((size_t)row * SAMPLE_CHUNKS + c) * room;
    int at = before;
    bool alike = false;
    if (all >= SAMPLE_ALIKE && 2 * all >= ch.end - ch.begin) {      // the same for all threads; fewer are listed as fast as they are looked at
      uint32_t lo = 0xffffffffu, hi = 0u;
      each([&](float e) {
        const uint32_t b = __float_as_uint(e);
        if ((int)sample_class(b) == above) lo = min(lo, b), hi = max(hi, b);
      });
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) {
        lo = min(lo, (uint32_t)__shfl_xor((int)lo, off, 64));
        hi = max(hi, (uint32_t)__shfl_xor((int)hi, off, 64));
      }
      if ((tid & 63) == 0) ends[0][tid >> 6] = lo, ends[1][tid >> 6] = hi;
      __syncthreads();
#pragma unroll
      for (int k = 0; k < SAMPLE_THREADS / 64; k++) lo = min(lo, ends[0][k]), hi = max(hi, ends[1][k]);
      alike = lo == hi;
      if (alike && tid == 0) mylist[0] = lo;
    }
    if (!alike)
      each([&](float e) {
        if ((int)sample_class(__float_as_uint(e)) == above) {
          if (at < room) mylist[at] = __float_as_uint(e);
          at++;
        }
      });
    if (tid == 0) fin_n[(size_t)row * SAMPLE_CHUNKS + c] = alike ? ~all : all;
  }
  s = wave_sum_f64(s);
  if ((tid & 63) == 0) ws[tid >> 6] = s;
  __syncthreads();
  if (tid == 0) {
    for (int k = 1; k < SAMPLE_THREADS / 64; k++) s += ws[k];
    fin_s[(size_t)row * SAMPLE_CHUNKS + c] = s;
  }
}

// Where tokens go beside `out`: host memory that the GPU reaches, a word a row, the launch's stamp above the token (null: nowhere).
// Written past the caches, so that the host sees a token a microsecond after it is chosen, without a copy, and knows by the
// stamp whose it is, without an event.
struct SampleLanding {
  unsigned long long* words;
  uint32_t stamp;
};
__device__ __forceinline__ void sample_leave(int token, int row, int* out, const SampleLanding& to) {
  out[row] = token;
  if (to.words != nullptr)
    __hip_atomic_store(to.words + row, (unsigned long long)to.stamp << 32 | (uint32_t)token, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <int THREADS, bool SEARCH>
__global__ __launch_bounds__(THREADS) void sample_pick_kernel(
    const float* __restrict__ logits, int ld, int V, const float* __restrict__ temperature, const float* __restrict__ top_p,
    const float* __restrict__ u, const float* __restrict__ part_val, const int* __restrict__ part_idx,
    const double* __restrict__ fin_s, const int* __restrict__ fin_n, const uint32_t* __restrict__ list, int room,
    const SampleRow* __restrict__ rows, int bits, int* __restrict__ out, const SampleLanding landing) {
  constexpr int WAVES = THREADS / 64, PER = THREADS / SAMPLE_CHUNKS, PIECE = SAMPLE_PIECE / THREADS;     // PER: threads a chunk
  __shared__ unsigned long long hist[SEARCH ? 1 << (SAMPLE_LOW - SAMPLE_MID) : 1], scratch[WAVES], mass;
  __shared__ int cls;
  __shared__ double wave_tot[WAVES];
  __shared__ int wave_cnt[WAVES];
  __shared__ int chosen_chunk, chosen_ties_before;
  __shared__ int wave_first[WAVES], wave_last[WAVES];
  __shared__ int chunk_n[SAMPLE_CHUNKS];
  __shared__ double chunk_s[SAMPLE_CHUNKS];
  __shared__ double chosen_before, chosen_target;
  const int row = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  // (asked for at once and without branches, as in the launches before; rows without a search find in `r`, `number` and `head` what they do
  // not look at)
  const size_t base = (size_t)row * SAMPLE_CHUNKS;
  const int my_chunk = tid / PER, part = tid % PER;
  float mx = part_val[base + (lane & 31)];
  int mi = part_idx[base + (lane & 31)];
  const float temp = temperature[row], u_row = u[row];
  const float tp = SEARCH ? top_p[row] : 1.0f;
  double kept_s = fin_s[base + my_chunk];
  SampleRow r{};
  int number = 0;
  u32x4 head{0, 0, 0, 0};
  if (SEARCH) {
    r = rows[row];
    number = fin_n[base + my_chunk];
    head = reinterpret_cast<const u32x4*>(list + (base + my_chunk) * room)[min(part, room / 4 - 1)];
  }
  // the row's first maximum: what a greedy row gives, and what a draw falls back on
  wave_first_max(mx, mi);
  if (!(temp > 0.f)) {
    if (tid == 0) sample_leave(mi, row, out, landing);
    return;
  }
  const float inv_t = 1.0f / temp;
  const float* x = logits + (size_t)row * ld;
  float thr = 0.f;                            // keep e > thr, and the first `ties_kept` tokens with e == thr
  int ties_kept = 0x7fffffff;
  int kept_n = 0;
  if constexpr (SEARCH) if (tp < 1.0f) {
    // the patterns of this chunk's elements of the class, PER threads side by side, four neighbours each: from the list, of which
    // each thread holds the first ones, or, where it did not have room for all, from the logits
    const u32x4* mylist = reinterpret_cast<const u32x4*>(list + (base + my_chunk) * room);
    const u32x4 held = 4 * part < number ? head : u32x4{0, 0, 0, 0};
    auto entries = [&](auto use) {                        // use(pattern, how many of it)
      if ((uint32_t)number <= (uint32_t)room) {
#pragma unroll
        for (int j = 0; j < 4; j++)
          if (4 * part + j < number) use(held[j], 1);
        for (int k0 = part + PER; 4 * k0 < number; k0 += 4 * PER) {
          u32x4 v[4];
#pragma unroll
          for (int k = 0; k < 4; k++) v[k] = 4 * (k0 + k * PER) < number ? mylist[k0 + k * PER] : u32x4{0, 0, 0, 0};
#pragma unroll
          for (int k = 0; k < 4; k++)
#pragma unroll
            for (int j = 0; j < 4; j++)
              if (4 * (k0 + k * PER) + j < number) use(v[k][j], 1);
        }
      } else if (number < 0) {
        if (part == 0) use(mylist[0][0], ~number);
      } else {
        const SampleChunk ch = sample_chunk(V, my_chunk);
        for (int i0 = ch.begin + part; i0 < ch.end; i0 += 16 * PER) {
          float v[16];
#pragma unroll
          for (int k = 0; k < 16; k++) v[k] = i0 + k * PER < ch.end ? x[i0 + k * PER] : 0.f;
#pragma unroll
          for (int k = 0; k < 16; k++) {
            const uint32_t b = __float_as_uint(__expf((v[k] - mx) * inv_t));
            if (i0 + k * PER < ch.end && sample_class(b) == r.cls) use(b, 1);
          }
        }
      }
    };
    // among 2^(LOW - MID) classes of 2^MID patterns, then among the patterns of one
    static_assert(PER == 32 && (1 << (SAMPLE_LOW - SAMPLE_MID)) == THREADS && (1 << SAMPLE_MID) <= THREADS, "half a wave a chunk, a class a thread");
    const double one = (double)(1ull << bits), target = (double)r.target * one;
    uint32_t found = r.cls;                   // the leading bits of t*
    unsigned long long above = r.above, all;
    bool any = true;
#pragma unroll
    for (int level = 0; level < 2; level++) {
      const int shift = level ? 0 : SAMPLE_MID, width = level ? SAMPLE_MID : SAMPLE_LOW - SAMPLE_MID;
      hist[tid] = 0ull;
      if (tid == 0) cls = -1;
      __syncthreads();
      SampleRun run{hist};
      entries([&](uint32_t b, int copies) {
        if (b >> (shift + width) == found) run.add((b >> shift) & ((1u << width) - 1), sample_fixed(b, bits) * copies);
      });
      run.end();
      __syncthreads();
      const unsigned long long h[1] = {hist[tid]};
      sample_cross(h, above + block_behind(h[0], scratch, WAVES, all), target, tid, &cls, &mass);
      __syncthreads();
      any = any && cls >= 0;
      found = found << width | (uint32_t)max(cls, 0);
      if (cls >= 0) above = mass;
      __syncthreads();                        // (cls and hist are written again)
    }
    if (!any) found = SAMPLE_ONE, above = 0;  // a target that is not above zero: the first of the largest
    thr = __uint_as_float(found);
    // the mass above the threshold is below the target; tied tokens are taken, in vocabulary order, while
    // the mass before them still is
    ties_kept = max(1, (int)ceilf((r.target - (float)((double)above / one)) / thr));
    double s = 0.0;
    entries([&](uint32_t b, int copies) {
      const float e = __uint_as_float(b);
      if (e > thr) s += (double)e * copies;
      if (e == thr) kept_n += copies;
    });
#pragma unroll
    for (int off = PER / 2; off > 0; off >>= 1) {
      s += __shfl_xor(s, off, 64);
      kept_n += __shfl_xor(kept_n, off, 64);
    }
    kept_s += s;
  }
  if (part == 0) {
    chunk_n[my_chunk] = kept_n;
    chunk_s[my_chunk] = kept_s;
  }
  __syncthreads();
  if (tid < 64) {
    // what every chunk keeps, a chunk a lane: its e > thr, and of its ties those that still are among the first `ties_kept`
    const bool real = lane < SAMPLE_CHUNKS;
    const int n = real ? chunk_n[lane] : 0;
    int ties = n;
#pragma unroll
    for (int off = 1; off < SAMPLE_CHUNKS; off <<= 1) {
      const int o = __shfl_up(ties, off, 64);
      if (lane >= off) ties += o;
    }
    const int before = ties - n, taken = min(n, max(0, ties_kept - min(before, ties_kept)));
    const double kept = real ? chunk_s[lane] + (double)thr * (double)taken : 0.0;
    double run = kept;
#pragma unroll
    for (int off = 1; off < SAMPLE_CHUNKS; off <<= 1) {
      const double o = __shfl_up(run, off, 64);
      if (lane >= off) run += o;
    }
    const double target = (double)u_row * __shfl(run, SAMPLE_CHUNKS - 1, 64);
    double in_front = __shfl_up(run, 1, 64);
    if (lane == 0) in_front = 0.0;
    const unsigned long long some = __ballot(kept > 0.0), reaches = __ballot(kept > 0.0 && run > target);
    const int c = reaches ? __ffsll((long long)reaches) - 1 : some ? 63 - __clzll((long long)some) : 0;
    if (lane == c) {
      chosen_chunk = c;
      chosen_before = in_front;
      chosen_target = target;
      chosen_ties_before = before;
    }
  }
  __syncthreads();
  const SampleChunk ch = sample_chunk(V, chosen_chunk);
  // A thread owns a contiguous piece of the chunk and goes through it three times.  One element after the other from
  // memory, each pass is a chain of latencies (2 to 2.6 us each for the 19 elements a thread has of a chunk of
  // 151,936 logits): a piece of a chunk of up to SAMPLE_PIECE elements (vocabularies up to 262,144) is asked for at once and
  // its terms wait in registers.
  auto term = [&](int i) { return __expf((x[i] - mx) * inv_t); };
  const int piece = (ch.end - ch.begin + THREADS - 1) / THREADS;
  const int b = min(ch.end, ch.begin + tid * piece), e_ = min(ch.end, b + piece);
  const bool held = piece <= PIECE;                                 // the same for all threads
  float mine[PIECE];
  if (held) {
#pragma unroll
    for (int k = 0; k < PIECE; k++) mine[k] = b + k < e_ ? x[b + k] : 0.f;
#pragma unroll
    for (int k = 0; k < PIECE; k++) mine[k] = __expf((mine[k] - mx) * inv_t);
  }
  // use(i, e) for the elements of the piece in their order, until it returns false
  auto each = [&](auto use) {
    if (held) {
#pragma unroll
      for (int k = 0; k < PIECE; k++) {
        if (b + k >= e_ || !use(b + k, mine[k])) break;
      }
    } else {
      for (int i = b; i < e_; i++)
        if (!use(i, term(i))) break;
    }
  };
  int my_ties = 0;
  each([&](int, float e) { my_ties += e == thr; return true; });
  int all_ties;
  const int ties_before = chosen_ties_before + block_prefix_i32<THREADS>(my_ties, wave_cnt, all_ties);
  double s = 0.0;
  {
    int tie = ties_before;
    each([&](int, float e) {
      if (e > thr || (e == thr && tie++ < ties_kept)) s += (double)e;
      return true;
    });
  }
  double chunk_total;
  const double before = chosen_before + block_prefix_f64<THREADS>(s, wave_tot, chunk_total);
  const double target = chosen_target;
  // the first thread whose piece reaches the target, and the last that keeps anything (a vote in each wave, then
  // the waves side by side: every thread asking for one word of LDS at once takes 4 us)
  {
    const unsigned long long keeps = __ballot(s > 0.0), reaches = __ballot(s > 0.0 && before + s > target);
    if (lane == 0) {
      wave_last[tid >> 6] = keeps ? (tid | 63) - __clzll(keeps) : -1;
      wave_first[tid >> 6] = reaches ? tid + __ffsll(reaches) - 1 : 0x7fffffff;
    }
  }
  __syncthreads();
  int first = 0x7fffffff, last = -1;
#pragma unroll
  for (int w = 0; w < WAVES; w++) {
    first = min(first, wave_first[w]);
    last = max(last, wave_last[w]);
  }
  const int who = first != 0x7fffffff ? first : last;
  if (who < 0) {                              // nothing kept in the chunk (cannot be, but a token must come out)
    if (tid == 0) sample_leave(mi, row, out, landing);
    return;
  }
  if (tid == who) {
    double run = before;
    int pick = -1, last_kept = mi, tie = ties_before;
    each([&](int i, float e) {
      if (e > thr || (e == thr && tie++ < ties_kept)) {
        if (e > 0.f) last_kept = i;           // a token whose probability underflowed to zero is never the fallback
        run += (double)e;
        if (run > target) { pick = i; return false; }
      }
      return true;
    });
    sample_leave(pick >= 0 ? pick : last_kept, row, out, landing);
  }
}

// ---------------------------------------------------------------------------
// Greedy rows only: the argmax in two launches.  One workgroup per row reads the row no faster than
// one compute unit takes data in (19 us for 151,936 logits); ARGMAX_CHUNKS workgroups per row find the
// first maximum of a chunk each, a second launch picks among them (the lowest index on a tie, as above).
// ---------------------------------------------------------------------------
// What a step's rows are sampled with, as it travels with a launch: temperature, top_p, uniform number of up to N rows.
template <int N>
struct SampleGiven {
  float v[3][N];
};
template <>
struct SampleGiven<0> {};

// N > 0: leaves the rows' options in params [3][stride] for the launches behind it.  clear: the classes of the second launch of sampling.
template <int N>
__global__ __launch_bounds__(256) void argmax_part_kernel(const float* __restrict__ logits, int ld, int V, float* __restrict__ part_val,
                                                          int* __restrict__ part_idx, unsigned long long* __restrict__ clear,
                                                          const SampleGiven<N> given, float* __restrict__ params, int stride) {
  __shared__ float vals[4];
  __shared__ int idxs[4];
  const int row = blockIdx.x, c = blockIdx.y, tid = threadIdx.x;
  constexpr int SHARE = SAMPLE_CLASSES / ARGMAX_CHUNKS;
  if constexpr (N > 0) {
    if (c == 0 && tid < 3) params[(size_t)tid * stride + row] = given.v[tid][row];
  }
  if (clear != nullptr && tid < SHARE) clear[(size_t)row * SAMPLE_CLASSES + c * SHARE + tid] = 0ull;
  const float* x = logits + (size_t)row * ld;
  const int len = (V + ARGMAX_CHUNKS - 1) / ARGMAX_CHUNKS;
  const int begin = min(V, c * len), end = min(V, begin + len);
  float mx = -INFINITY;
  int mi = 0x7fffffff;
  // four loads in flight per thread; indices rise within a thread, so ">" keeps the first maximum
  for (int i0 = begin + tid; i0 < end; i0 += 4 * 256) {
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int i = i0 + j * 256;
      v[j] = i < end ? x[i] : -INFINITY;
    }
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (v[j] > mx) { mx = v[j]; mi = i0 + j * 256; }
  }
  wave_first_max(mx, mi);
  if ((tid & 63) == 0) { vals[tid >> 6] = mx; idxs[tid >> 6] = mi; }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < 4; w++) keep_first_max(mx, mi, vals[w], idxs[w]);
    part_val[row * ARGMAX_CHUNKS + c] = mx;
    part_idx[row * ARGMAX_CHUNKS + c] = mi;
  }
}

__global__ __launch_bounds__(64) void argmax_final_kernel(const float* __restrict__ part_val, const int* __restrict__ part_idx,
                                                          int* __restrict__ out, const SampleLanding landing) {
  const int row = blockIdx.x, lane = threadIdx.x;
  float mx = lane < ARGMAX_CHUNKS ? part_val[row * ARGMAX_CHUNKS + lane] : -INFINITY;
  int mi = lane < ARGMAX_CHUNKS ? part_idx[row * ARGMAX_CHUNKS + lane] : 0x7fffffff;
  wave_first_max(mx, mi);
  if (lane == 0) sample_leave(mi, row, out, landing);
}

// part_val, part_idx: workspace of R * pico_argmax_chunks() entries each
extern "C" int pico_argmax_chunks() { return ARGMAX_CHUNKS; }

// landing, stamp: SampleLanding
extern "C" int pico_argmax_rows(const float* logits, int ld, int R, int V, float* part_val, int* part_idx, int* out,
                                unsigned long long* landing, uint32_t stamp, hipStream_t stream) {
  PICO_REQUIRE(R >= 0 && V > 0 && ld >= V, "pico_argmax: bad sizes R=%d V=%d ld=%d", R, V, ld);
  PICO_REQUIRE(R <= 65535, "pico_argmax: too many rows");
  if (R == 0) return 0;
  argmax_part_kernel<0><<<dim3(R, ARGMAX_CHUNKS), 256, 0, stream>>>(logits, ld, V, part_val, part_idx, nullptr, SampleGiven<0>{}, nullptr, 0);
  argmax_final_kernel<<<R, 64, 0, stream>>>(part_val, part_idx, out, SampleLanding{landing, stamp});
  PICO_LAUNCH_CHECK();
  return 0;
}
extern "C" int pico_argmax(const float* logits, int ld, int R, int V, float* part_val, int* part_idx, int* out, hipStream_t stream) {
  return pico_argmax_rows(logits, ld, R, V, part_val, part_idx, out, nullptr, 0, stream);
}

// The address at which kernels reach pinned host memory; null: they do not.
extern "C" void* pico_host_on_device(void* host) {
  void* p = nullptr;
  if (hipHostGetDevicePointer(&p, host, 0) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  return p;
}

// Waits on the host, for `limit_us` at most, until the n words of landing bear the stamp; their tokens.  0: they do not yet.
extern "C" int pico_landed(const unsigned long long* landing, int n, uint32_t stamp, int* tokens, int limit_us) {
  const auto end = std::chrono::steady_clock::now() + std::chrono::microseconds(limit_us);
  for (int i = 0; i < n; i++) {
    unsigned long long w;
    for (int spins = 0; (uint32_t)((w = __atomic_load_n(landing + i, __ATOMIC_RELAXED)) >> 32) != stamp; spins++) {
      if (spins % 64 == 63 && std::chrono::steady_clock::now() > end) return 0;
      __builtin_ia32_pause();
    }
    tokens[i] = (int)(uint32_t)w;
  }
  return 1;
}

// The counter-based generator: u in [0, 1) of 24 random bits from (seed, index of the token in its request).
static uint64_t splitmix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}
static float sample_uniform(uint64_t seed, uint64_t index) {
  return (float)(splitmix64(splitmix64(seed) ^ index * 0xD6E8FEB86659FD93ull) >> 40) / (float)(1 << 24);
}
extern "C" void pico_sample_uniforms(const uint64_t* seeds, const uint64_t* indices, int n, float* u) {
  for (int i = 0; i < n; i++) u[i] = sample_uniform(seeds[i], indices[i]);
}

// Words of a chunk's list: none are missing up to SAMPLE_LISTED elements a chunk.  (A class that is not listed whole is read again, three
// times: nearly flat rows of 151,936 102 us in place of 58 with a list of half a chunk.)
static int sample_room(int V) {
  const long long len = ((long long)V + SAMPLE_CHUNKS - 1) / SAMPLE_CHUNKS;
  return len < SAMPLE_LISTED ? (int)((len + 3) / 4 * 4) : SAMPLE_LISTED;
}

// work: pico_sample_workspace_words(R, V, top_p_rows) 4-byte words, 16-byte aligned: 640 bytes a row, and with top_p_rows for up to
// SAMPLE_ROWS rows 16 KB of classes and a row's length of floats (at most 623 KB).  top_p_rows == 0: no row has top_p < 1
// (every row is treated so), and the launch that looks for the threshold is left out.
extern "C" long long pico_sample_workspace_words(int R, int V, int top_p_rows) {
  static_assert(sizeof(SampleRow) == 16, "four words a row");
  const long long at_once = R < SAMPLE_ROWS ? R : SAMPLE_ROWS;
  return (long long)R * SAMPLE_CHUNKS * (2 + 1 + 1 + 1) + (top_p_rows ? at_once * (2 * SAMPLE_CLASSES + 4 + SAMPLE_CHUNKS * (long long)sample_room(V)) : 0);
}

// What the launches of a call share
struct SampleCall {
  const float* logits;
  int ld, R, V;
  const float *temperature, *top_p, *u;
  int* out;
  SampleLanding landing;
  void* work;
  int top_p_rows;
  hipStream_t stream;
};

// first(row, rows, part_val, part_idx, classes or null): the first launch, for `most` rows at most
template <typename First>
static int sample_launches(const SampleCall& a, int most, First first) {
  static_assert(SAMPLE_CHUNKS == ARGMAX_CHUNKS, "the first launch is the argmax's");
  PICO_REQUIRE(a.R >= 0 && a.V > 0 && a.ld >= a.V, "pico_sample: bad sizes R=%d V=%d ld=%d", a.R, a.V, a.ld);
  PICO_REQUIRE(a.R <= 65535, "pico_sample: too many rows");
  if (a.R == 0) return 0;
  // (every part of the workspace is a multiple of 16 bytes long)
  PICO_REQUIRE(a.work != nullptr && (uintptr_t)a.work % 16 == 0, "pico_sample: the workspace is missing or not 16-byte aligned");
  const size_t n = (size_t)a.R * SAMPLE_CHUNKS;
  double* fin_s = (double*)a.work;
  float* part_val = (float*)(fin_s + n);
  int* part_idx = (int*)(part_val + n);
  int* fin_n = part_idx + n;
  unsigned long long* classes = (unsigned long long*)(fin_n + n);
  const int room = sample_room(a.V), at_once = a.R < SAMPLE_ROWS ? a.R : SAMPLE_ROWS;
  SampleRow* rows = (SampleRow*)(classes + (size_t)at_once * SAMPLE_CLASSES);
  uint32_t* list = (uint32_t*)(rows + at_once);
  int bits = 40;                              // a row's sum of whole numbers of 2^-bits stays below 2^63
  while (bits > 31 && a.V > (1LL << (63 - bits))) bits--;
  for (int r = 0; r < a.R; r += most) {                        // rows with a list side by side; the next ones write it again behind them
    const int m = a.R - r < most ? a.R - r : most;
    const size_t c = (size_t)r * SAMPLE_CHUNKS;
    const float* x = a.logits + (size_t)r * a.ld;
    const SampleLanding landing{a.landing.words ? a.landing.words + r : nullptr, a.landing.stamp};
    const dim3 grid(m, SAMPLE_CHUNKS);
    first(r, m, part_val + c, part_idx + c, a.top_p_rows ? classes : nullptr);
    if (!a.top_p_rows) {
      sample_collect_kernel<false><<<grid, SAMPLE_THREADS, 0, a.stream>>>(x, a.ld, a.V, a.temperature + r, nullptr, part_val + c, nullptr, bits, fin_s + c,
                                                                         fin_n + c, nullptr, 0, nullptr);
      sample_pick_kernel<SAMPLE_THREADS, false><<<m, SAMPLE_THREADS, 0, a.stream>>>(x, a.ld, a.V, a.temperature + r, nullptr, a.u + r, part_val + c,
                                                                                   part_idx + c, fin_s + c, fin_n + c, nullptr, 0, nullptr, bits, a.out + r,
                                                                                   landing);
      continue;
    }
    sample_classes_kernel<<<grid, SAMPLE_THREADS, 0, a.stream>>>(x, a.ld, a.V, a.temperature + r, a.top_p + r, part_val + c, classes, bits);
    sample_collect_kernel<true><<<grid, SAMPLE_THREADS, 0, a.stream>>>(x, a.ld, a.V, a.temperature + r, a.top_p + r, part_val + c, classes, bits, fin_s + c,
                                                                      fin_n + c, list, room, rows);
    sample_pick_kernel<SAMPLE_PICK_THREADS, true><<<m, SAMPLE_PICK_THREADS, 0, a.stream>>>(x, a.ld, a.V, a.temperature + r, a.top_p + r, a.u + r,
                                                                                          part_val + c, part_idx + c, fin_s + c, fin_n + c, list, room, rows,
                                                                                          bits, a.out + r, landing);
  }
  PICO_LAUNCH_CHECK();
  return 0;
}

extern "C" int pico_sample(const float* logits, int ld, int R, int V, const float* temperature, const float* top_p,
                           const float* u, int* out, void* work, int top_p_rows, hipStream_t stream) {
  return sample_launches({logits, ld, R, V, temperature, top_p, u, out, {nullptr, 0}, work, top_p_rows, stream}, top_p_rows ? SAMPLE_ROWS : 65535,
                         [&](int r, int m, float* val, int* idx, unsigned long long* classes) {
                           argmax_part_kernel<0><<<dim3(m, SAMPLE_CHUNKS), 256, 0, stream>>>(logits + (size_t)r * ld, ld, V, val, idx, classes,
                                                                                             SampleGiven<0>{}, nullptr, 0);
                         });
}

template <int N>
static void launch_given(const float* x, int ld, int V, float* val, int* idx, unsigned long long* classes, const float* temperature, const float* top_p,
                         const uint64_t* seeds, const uint64_t* indices, int m, float* params, int stride, hipStream_t stream) {
  SampleGiven<N> given;
  for (int i = 0; i < m; i++) {
    given.v[0][i] = temperature[i];
    given.v[1][i] = top_p[i];
    given.v[2][i] = temperature[i] > 0.f ? sample_uniform(seeds[i], indices[i]) : 0.f;
  }
  for (auto& row : given.v)
    for (int i = m; i < N; i++) row[i] = 0.f;
  argmax_part_kernel<N><<<dim3(m, SAMPLE_CHUNKS), 256, 0, stream>>>(x, ld, V, val, idx, classes, given, params, stride);
}

// The same with temperature, top_p, seeds and token indices [R] in ordinary host memory: they travel with the first launch, which leaves them in
// params (float [3][stride], stride >= R, device memory), so there is no copy in front of it.  (8 rows, half of them with top_p: a step with its
// copies and an event 63 us from call to tokens, so, and with landing, 48.)  A launch carries 768 bytes of options up to 64 rows, else 3 KB.
extern "C" int pico_sample_rows(const float* logits, int ld, int R, int V, const float* temperature, const float* top_p, const uint64_t* seeds,
                                const uint64_t* indices, float* params, int stride, int* out, unsigned long long* landing,
                                uint32_t stamp, void* work, int top_p_rows, hipStream_t stream) {
  PICO_REQUIRE(stride >= R && params && temperature && top_p && seeds && indices, "pico_sample_rows: room for %d rows' options, got %d", R, stride);
  return sample_launches({logits, ld, R, V, params, params + stride, params + 2 * (size_t)stride, out, {landing, stamp}, work, top_p_rows, stream}, SAMPLE_ROWS,
                         [&](int r, int m, float* val, int* idx, unsigned long long* classes) {
                           const auto launch = m <= 64 ? launch_given<64> : launch_given<SAMPLE_ROWS>;
                           launch(logits + (size_t)r * ld, ld, V, val, idx, classes, temperature + r, top_p + r, seeds + r, indices + r, m, params + r, stride,
                                  stream);
                         });
}

// ---------------------------------------------------------------------------
// The same two launches with the chunk maxima in memory of the library's own (no_alloc.h).
// ---------------------------------------------------------------------------
#include "no_alloc.h"

#include <mutex>

#define NOALLOC_ENTRIES (PICO_NOALLOC_MAX_ROWS * ARGMAX_CHUNKS)
#define NOALLOC_MAX_DEVICES 64

// [values: NOALLOC_ENTRIES floats][indices: NOALLOC_ENTRIES ints].  In host code this name is only a handle
// for hipGetSymbolAddress; the address that kernels and copies take is g_scratch_ptr[device].
static __device__ __align__(256) unsigned char scratch[NOALLOC_ENTRIES * (sizeof(float) + sizeof(int))];

static void* g_scratch_ptr[NOALLOC_MAX_DEVICES];     // per device: where that GPU's copy of the array lies
static std::mutex g_scratch_mutex;

// The address of the current device's copy, looked up once per device with that device current.
static int noalloc_scratch(void** ptr) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  PICO_REQUIRE(e == hipSuccess, "pico_noalloc: hipGetDevice failed: %s", hipGetErrorString(e));
  PICO_REQUIRE(dev >= 0 && dev < NOALLOC_MAX_DEVICES, "pico_noalloc: device %d is beyond the %d this library keeps", dev,
               NOALLOC_MAX_DEVICES);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (g_scratch_ptr[dev] == nullptr) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    PICO_REQUIRE(e == hipSuccess && p != nullptr, "pico_noalloc: hipGetSymbolAddress failed on device %d: %s", dev,
                 hipGetErrorString(e));
    g_scratch_ptr[dev] = p;
  }
  *ptr = g_scratch_ptr[dev];
  return 0;
}

extern "C" int pico_noalloc_max_rows() { return PICO_NOALLOC_MAX_ROWS; }

extern "C" int pico_noalloc_init() {
  void* p = nullptr;
  return noalloc_scratch(&p);
}

extern "C" int pico_argmax_noalloc(const float* logits, int ld, int R, int V, int* out, hipStream_t stream) {
  PICO_REQUIRE(R >= 0 && V > 0 && ld >= V, "pico_argmax_noalloc: bad sizes R=%d V=%d ld=%d", R, V, ld);
  PICO_REQUIRE(R <= PICO_NOALLOC_MAX_ROWS, "pico_argmax_noalloc: %d rows, the library's own memory holds %d; "
               "use pico_argmax with a workspace", R, PICO_NOALLOC_MAX_ROWS);
  PICO_REQUIRE(logits != nullptr && out != nullptr, "pico_argmax_noalloc: null pointer");
  if (R == 0) return 0;
  void* base = nullptr;
  if (noalloc_scratch(&base) != 0) return -1;
  float* part_val = reinterpret_cast<float*>(base);
  int* part_idx = reinterpret_cast<int*>(reinterpret_cast<unsigned char*>(base) + NOALLOC_ENTRIES * sizeof(float));
  // the first launch writes entries [0, R * ARGMAX_CHUNKS), the second reads exactly those: nothing to clear
  argmax_part_kernel<0><<<dim3(R, ARGMAX_CHUNKS), 256, 0, stream>>>(logits, ld, V, part_val, part_idx, nullptr, SampleGiven<0>{}, nullptr, 0);
  argmax_final_kernel<<<R, 64, 0, stream>>>(part_val, part_idx, out, SampleLanding{nullptr, 0});
  PICO_LAUNCH_CHECK();
  return 0;
}
