// Sampling of one token per row of logits, one block per row, all in float.
//
// Order as in the reference (src/sampler/mod.rs:194-238): temperature <= 0 is
// the argmax (of equal maxima the last index, as `max_by` keeps it, :60-68);
// else z = logit / T, top-k on z (:93-119, ties at the threshold kept in index
// order), softmax, top-p on the probabilities (:144-170), then the first index
// whose running sum reaches r, else the last index (:225-238).  The reference
// draws r from an unseeded generator; here r comes from Philox4x32-10 keyed by
// the seed with the counter (step, sequence), so a sequence's draws do not
// depend on its batch-mates.
#include "common.hpp"

namespace tl {

constexpr int SNT = 1024;

__device__ __forceinline__ uint32_t order_key(float v) {
  const uint32_t b = __float_as_uint(v);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);   // ascending with the value
}

__device__ inline float philox_uniform(uint32_t seed_lo, uint32_t seed_hi, uint32_t step,
                                       uint32_t seq) {
  uint32_t c0 = step, c1 = seq, c2 = 0u, c3 = 0u, k0 = seed_lo, k1 = seed_hi;
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    if (r > 0) {
      k0 += 0x9E3779B9u;
      k1 += 0xBB67AE85u;
    }
    const uint32_t hi0 = __umulhi(0xD2511F53u, c0), lo0 = 0xD2511F53u * c0;
    const uint32_t hi1 = __umulhi(0xCD9E8D57u, c2), lo1 = 0xCD9E8D57u * c2;
    const uint32_t n0 = hi1 ^ c1 ^ k0, n1 = lo1, n2 = hi0 ^ c3 ^ k1, n3 = lo0;
    c0 = n0; c1 = n1; c2 = n2; c3 = n3;
  }
  return (float)(c0 >> 8) * (1.0f / 16777216.0f);      // [0, 1)
}

// Four floats of a row from index i on (i a multiple of 4); `n` of them lie in the row.  VEC: rows are
// aligned to 16 bytes and a multiple of 4 long; else whole fours by one load all the same (global memory takes
// 16 bytes at any multiple of 4), and the row's end one by one: 64 rows of 50,257, greedy 9 us, a plain draw 50, where
// loads one by one took 17 and 103.
typedef f32x4 __attribute__((aligned(4))) f32x4_at4;
template <bool VEC> __device__ __forceinline__ int load4(const float* __restrict__ p, int i, int V, float v[4]) {
  if (VEC ? i >= V : i + 4 > V) {
    const int n = VEC ? 0 : max(0, V - i);
    if (!VEC) {
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = j < n ? p[i + j] : 0.f;
    }
    return n;
  }
  const f32x4 t = VEC ? *(const f32x4*)(p + i) : (f32x4) * (const f32x4_at4*)(p + i);
  v[0] = t[0]; v[1] = t[1]; v[2] = t[2]; v[3] = t[3];
  return 4;
}
template <bool VEC> __device__ __forceinline__ void store4(float* __restrict__ p, int i, int n, const float v[4]) {
  if (VEC) {
    if (n) *(f32x4*)(p + i) = f32x4{v[0], v[1], v[2], v[3]};
  } else if (n == 4) {
    *(f32x4_at4*)(p + i) = f32x4{v[0], v[1], v[2], v[3]};
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j < n) p[i + j] = v[j];
  }
}

// f(index, value) over a row, every thread on its own elements, in any order; `update` stores what f returns.
// Eight loads of 16 bytes a thread are under way at a time: a row is read by one compute unit, whose way to
// L2 (64 bytes a cycle) is what a pass over a long row takes.
constexpr int ROW_LOADS = 8;
template <bool VEC, typename F> __device__ __forceinline__ void visit(const float* __restrict__ p, int V, F f) {
  for (int base = threadIdx.x * 4; base < V; base += SNT * 4 * ROW_LOADS) {
    float v[ROW_LOADS][4];
    int n[ROW_LOADS];
#pragma unroll
    for (int u = 0; u < ROW_LOADS; ++u) n[u] = load4<VEC>(p, base + u * SNT * 4, V, v[u]);
#pragma unroll
    for (int u = 0; u < ROW_LOADS; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (j < n[u]) f(base + u * SNT * 4 + j, v[u][j]);
  }
}
template <bool VEC, typename F>
__device__ __forceinline__ void update(const float* __restrict__ src, float* __restrict__ dst, int V, F f) {
  for (int base = threadIdx.x * 4; base < V; base += SNT * 4 * ROW_LOADS) {
    float v[ROW_LOADS][4];
    int n[ROW_LOADS];
#pragma unroll
    for (int u = 0; u < ROW_LOADS; ++u) n[u] = load4<VEC>(src, base + u * SNT * 4, V, v[u]);
#pragma unroll
    for (int u = 0; u < ROW_LOADS; ++u) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (j < n[u]) v[u][j] = f(base + u * SNT * 4 + j, v[u][j]);
      store4<VEC>(dst, base + u * SNT * 4, n[u], v[u]);
    }
  }
}

template <typename T> __device__ __forceinline__ T wave_incl_scan(T v) {
  const int lane = threadIdx.x % WAVE;
#pragma unroll
  for (int o = 1; o < WAVE; o <<= 1) {
    const T t = __shfl_up(v, o, WAVE);
    if (lane >= o) v += t;
  }
  return v;
}
// exclusive prefix over the threads of the block, in thread order; `sh` holds SNT / WAVE values
template <typename T> __device__ __forceinline__ T block_excl_scan(T v, T* sh, T* total) {
  const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const T incl = wave_incl_scan(v);
  __syncthreads();
  if (lane == WAVE - 1) sh[w] = incl;
  __syncthreads();
  T before = 0, all = 0;
#pragma unroll
  for (int i = 0; i < SNT / WAVE; ++i) {
    if (i == w) before = all;
    all += sh[i];
  }
  *total = all;
  return before + incl - v;
}

// a probability as a whole number of 2^-60: sums of these are exact whatever their order
constexpr double FIX = 1152921504606846976.0;
__device__ __forceinline__ unsigned long long fixed60(float p) { return (unsigned long long)((double)p * FIX); }

struct SampleShared {
  unsigned long long hist[2048];
  unsigned long long scan[SNT / WAVE];
  unsigned long long above;
  int reached[2][SNT / WAVE][16];
  int digit;
  int count;
  int pick;
  int wave_count[SNT / WAVE];
  double wave_sum[SNT / WAVE];
  float red[SNT / WAVE];
};
__device__ __forceinline__ float from_order_key(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? k & 0x7fffffffu : ~k);
}
// The largest multiple of 2^12 that at least k of the block's NT values reach (0 if there is none above it), four bits and one
// barrier a round: 3.3 us over 1,024 threads.
template <int NT> __device__ __forceinline__ uint32_t bound_of_kth(uint32_t mine, int k, int (*reached)[SNT / WAVE][16]) {
  const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  uint32_t bound = 0u;
#pragma unroll
  for (int round = 0; round < 5; ++round) {
    const int shift = 28 - 4 * round;
    int c = 0;
#pragma unroll
    for (int j = 1; j < 16; ++j) {
      const int n = __popcll(__ballot(mine >= (bound | (uint32_t)j << shift)));
      if (lane == j) c = n;
    }
    if (lane < 16) reached[round % 2][w][lane] = c;
    __syncthreads();                                    // (the other half is written before the next one, so one a round is enough)
    int all = 0;
#pragma unroll
    for (int i = 0; i < NT / WAVE; ++i) all += reached[round % 2][i][lane % 16];
    const unsigned long long enough = __ballot(lane > 0 && lane < 16 && all >= k);
    if (enough) bound |= (uint32_t)(63 - __clzll((long long)enough)) << shift;
  }
  return bound;
}
// The passes over logits go by the logits themselves (a division is 14 instructions, 12 us a pass over 131,072): two logits whose
// quotients round to one number lie within 2 units in the last place of each other, so 4 are a margin.
__device__ __forceinline__ uint32_t with_margin(uint32_t bound) { return bound > 4u ? bound - 4u : 0u; }
// a candidate: by its quotient, of equal ones the smaller index first
__device__ __forceinline__ unsigned long long candidate(float quotient, int i) { return (unsigned long long)order_key(quotient) << 32 | ~(uint32_t)i; }

// Rows in parts: workgroups of their own look through PART_RUN logits each for what may be among the row's k largest. A part's
// list: how many there are, then the first PART_KEEP of them in any order.
constexpr int PART_NT = 512, PART_LOADS = 4, PART_RUN = PART_NT * PART_LOADS * 4, PART_KEEP = 511, PART_TOP_K = 256;
static_assert(2 * PART_TOP_K <= PART_NT, "the k-th largest of the threads' maxima, which little more than k logits reach");
typedef unsigned long long PartList[1 + PART_KEEP];

// the short lists of the way by candidates
constexpr int CANDIDATES = 2048;
constexpr int MOST_TOP_K = 1024;
static_assert(MOST_TOP_K == SNT, "one kept candidate a thread");
struct Lists {
  unsigned long long c[CANDIDATES];      // order_key of the quotient, and below it what is larger the smaller the index
  float top_z[MOST_TOP_K];
  int top_i[MOST_TOP_K];
};

// The n <= CANDIDATES numbers of c (none is 0) sorted down, by a bitonic network over the next power of two; a thread a pair.  Pairs
// less than a wave apart are the wave's own 128 places, so that only the wider steps need a barrier.  Up to RANKED a rank by
// comparison with all others is as fast.  A row of equal logits, microseconds, by comparison / this: 256 41 / 42, 512 46 / 45,
// 2,048 (two a thread, their keys made for every comparison, before) 531 / 60; 131,072 logits with top-k 400 108 / 76.
constexpr int RANKED = 256;
__device__ __forceinline__ void sort_down(unsigned long long* c, int n) {
  static_assert(CANDIDATES == 2 * SNT, "one pair a thread");
  int places = 2 * WAVE;
  while (places < n) places *= 2;
  for (int i = n + threadIdx.x; i < places; i += SNT) c[i] = 0;
  bool wide = true;
  for (int size = 2; size <= places; size *= 2)
    for (int apart = size / 2; apart > 0; apart /= 2) {
      if (wide || apart > WAVE) __syncthreads();
      else __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      wide = apart > WAVE;
      const int a = (threadIdx.x & ~(apart - 1)) * 2 + (threadIdx.x & (apart - 1)), b = a + apart;
      if (b < places) {
        const unsigned long long x = c[a], y = c[b];
        if ((x < y) == ((a & size) == 0)) { c[a] = y; c[b] = x; }
      }
    }
  __syncthreads();
}

// The largest t with (weights of the keys >= t) >= target, digit by digit from the top (11, 11 and 10 bits) through
// a histogram in LDS; 0 if no t reaches the target.  `above` returns the weights of the keys > t, `at` those of t.
template <bool VEC, typename Key, typename Weight>
__device__ __forceinline__ uint32_t select_key(const float* __restrict__ p, int V, unsigned long long target, Key key, Weight weight,
                                               SampleShared& sh, unsigned long long* above, unsigned long long* at) {
  uint32_t prefix = 0u;
  unsigned long long over = 0;
#pragma unroll 1
  for (int round = 0; round < 3; ++round) {
    const int shift = round == 0 ? 21 : (round == 1 ? 10 : 0);
    const uint32_t bins = round == 2 ? 1024u : 2048u;
    const uint32_t known = round == 0 ? 0u : (round == 1 ? 0xffe00000u : 0xfffffc00u);
    __syncthreads();
    sh.hist[threadIdx.x] = 0;
    sh.hist[threadIdx.x + SNT] = 0;
    if (threadIdx.x == 0) sh.digit = -1;
    __syncthreads();
    visit<VEC>(p, V, [&](int, float v) {
      const uint32_t k = key(v);
      if ((k & known) == prefix) atomicAdd(&sh.hist[(k >> shift) & (bins - 1u)], weight(v));
    });
    __syncthreads();
    // thread t has the bins 2047 - 2 t and 2046 - 2 t, so that prefixes run from the largest key down
    const int hi = 2047 - 2 * (int)threadIdx.x;
    const unsigned long long wh = sh.hist[hi], wl = sh.hist[hi - 1];
    unsigned long long total;
    const unsigned long long before = over + block_excl_scan<unsigned long long>(wh + wl, sh.scan, &total);
    if (before < target && before + wh + wl >= target) {
      const bool first = before + wh >= target;
      sh.digit = first ? hi : hi - 1;
      sh.above = first ? before : before + wh;
    }
    __syncthreads();
    if (sh.digit < 0) {                                  // all of them together do not reach the target
      *above = total;                                    // (only the first digit can miss)
      *at = 0;
      return 0u;
    }
    over = sh.above;
    *at = sh.hist[sh.digit];
    prefix |= (uint32_t)sh.digit << shift;
  }
  *above = over;
  return prefix;
}

// Keep the first `room` (in the order of the row) of the elements with key == thr, and those with a larger key:
// the others become `gone`.  Waves take the row in equal runs, one after the other.
template <bool VEC, typename Key, typename Kept>
__device__ __forceinline__ void keep_ties(float* __restrict__ p, int V, uint32_t thr, int room, float gone, Key key, Kept kept, SampleShared& sh) {
  const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const int run = ((V + SNT / WAVE - 1) / (SNT / WAVE) + 255) / 256 * 256;
  const int lo = min(V, w * run), hi = min(V, lo + run);
  int c = 0;
  for (int base = lo; base < hi; base += 256) {
    float v[4];
    const int n = load4<VEC>(p, base + lane * 4, V, v);
    for (int j = 0; j < n; ++j) c += key(v[j]) == thr;
  }
#pragma unroll
  for (int o = WAVE / 2; o > 0; o >>= 1) c += __shfl_xor(c, o, WAVE);
  __syncthreads();
  if (lane == 0) sh.wave_count[w] = c;
  __syncthreads();
  int rank = 0;
  for (int i = 0; i < w; ++i) rank += sh.wave_count[i];
  for (int base = lo; base < hi; base += 256) {
    float v[4];
    const int n = load4<VEC>(p, base + lane * 4, V, v);
    int mine = 0;
    for (int j = 0; j < n; ++j) mine += key(v[j]) == thr;
    const int incl = wave_incl_scan(mine);
    int at = rank + incl - mine;
    for (int j = 0; j < n; ++j) {
      const uint32_t k = key(v[j]);
      if (k < thr || (k == thr && at++ >= room)) v[j] = gone;
      else v[j] = kept(v[j]);
    }
    store4<VEC>(p, base + lane * 4, n, v);
    rank += __shfl(incl, WAVE - 1, WAVE);
  }
  __syncthreads();
}

// Where a row's token goes: device memory, and host memory that the device can write (or null).
struct Tokens {
  int* device;
  int* host;
  __device__ __forceinline__ void put(int b, int token) const {
    device[b] = token;
    if (host) __hip_atomic_store(host + b, token, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
};

// The draw over a whole row of probabilities: the first index whose running sum reaches r, else the last.
template <bool VEC> __device__ __forceinline__ void draw_row(const float* __restrict__ p, int V, float r, SampleShared& sh, int b, Tokens out) {
  const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const int run = ((V + SNT / WAVE - 1) / (SNT / WAVE) + 255) / 256 * 256;
  const int lo = min(V, w * run), hi = min(V, lo + run);
  double s = 0.0;
#pragma unroll 8
  for (int base = lo; base < hi; base += 256) {
    float v[4];
    const int n = load4<VEC>(p, base + lane * 4, V, v);
    for (int j = 0; j < n; ++j) s += (double)v[j];
  }
#pragma unroll
  for (int o = WAVE / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, WAVE);
  __syncthreads();
  if (lane == 0) sh.wave_sum[w] = s;
  if (threadIdx.x == 0) sh.pick = V - 1;
  __syncthreads();
  double before = 0.0;
  for (int i = 0; i < w; ++i) before += sh.wave_sum[i];
  if (lo < hi && before < (double)r && before + s >= (double)r) {      // (one wave at most: sums only grow)
    int pick = hi - 1;
    double so_far = before;
    for (int base = lo; base < hi; base += 256) {
      float v[4];
      const int n = load4<VEC>(p, base + lane * 4, V, v);
      double mine = 0.0;
      for (int j = 0; j < n; ++j) mine += (double)v[j];
      const double incl = wave_incl_scan(mine);
      const unsigned long long reached = __ballot(n > 0 && so_far + incl >= (double)r);
      if (reached) {
        const int first = __ffsll((long long)reached) - 1;
        double t = so_far + incl - mine;
        int at = base + lane * 4;
        for (int j = 0; j < n; ++j) {
          t += (double)v[j];
          if (t >= (double)r) break;
          if (j + 1 < n) ++at;
        }
        pick = __shfl(at, first, WAVE);
        break;
      }
      so_far += __shfl(incl, WAVE - 1, WAVE);
    }
    if (lane == 0) sh.pick = pick;
  }
  __syncthreads();
  if (threadIdx.x == 0) out.put(b, r > 0.f ? sh.pick : 0);   // (index 0's running sum reaches a draw of 0)
}

// One part of a row, its logits in registers: the k-th largest of the threads' maxima bounds the part's k-th largest from below, and
// the row's k largest are among their parts'.  What lies at or above the bound goes to the part's list, zeros to its probabilities.
template <bool VEC>
__global__ void __launch_bounds__(PART_NT)
sample_part_kernel(const float* __restrict__ logits, int V, int run, float temperature, int top_k, float* __restrict__ probs, PartList* __restrict__ lists) {
  __shared__ int reached[2][SNT / WAVE][16];
  __shared__ int count;
  const int b = blockIdx.x, tid = threadIdx.x, lo = blockIdx.y * run, hi = min(V, lo + run);
  const float* z = logits + (size_t)b * V;
  float* p = probs + (size_t)b * V;
  unsigned long long* list = lists[(size_t)b * gridDim.y + blockIdx.y];
  float v[PART_LOADS][4];
  int n[PART_LOADS];
#pragma unroll
  for (int u = 0; u < PART_LOADS; ++u) n[u] = load4<VEC>(z, lo + (u * PART_NT + tid) * 4, hi, v[u]);
  if (tid == 0) count = 0;
  uint32_t mine = 0u;
#pragma unroll
  for (int u = 0; u < PART_LOADS; ++u)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j < n[u]) mine = max(mine, order_key(v[u][j]));
  const uint32_t bound = with_margin(bound_of_kth<PART_NT>(mine, top_k, reached));
  const float zeros[4] = {0.f, 0.f, 0.f, 0.f};
  int c = 0;
#pragma unroll
  for (int u = 0; u < PART_LOADS; ++u) {
    store4<VEC>(p, lo + (u * PART_NT + tid) * 4, n[u], zeros);
#pragma unroll
    for (int j = 0; j < 4; ++j) c += j < n[u] && order_key(v[u][j]) >= bound;
  }
  const int upto = wave_incl_scan(c);                   // one request a wave for places: one a logit took 3.4 us of a part's 6.4
  int at = 0;
  if (tid % WAVE == WAVE - 1) at = atomicAdd(&count, upto);
  at = __shfl(at, WAVE - 1, WAVE) + upto - c;
#pragma unroll
  for (int u = 0; u < PART_LOADS; ++u)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j < n[u] && order_key(v[u][j]) >= bound) {
        if (at < PART_KEEP) list[1 + at] = candidate(v[u][j] / temperature, lo + (u * PART_NT + tid) * 4 + j);
        ++at;
      }
  __syncthreads();
  if (tid == 0) list[0] = count;
}

// One workgroup of 1,024 threads a row.  What bounds it is one compute unit's work on a row (131,072 logits are
// 512 KB, 3.5 us a pass at 64 bytes a cycle from L2, and more where an element costs a division or an exponential)
// times the number of passes, so passes are what was taken out:
//   * top-k of at most 1,024 (two passes): the k-th largest of the threads' own maxima bounds the k-th largest of the
//     row from below; what lies at or above it, little more than k elements, goes to a list in LDS and is sorted
//     there; softmax, top-p and the draw run over the list.
//   * everything else: thresholds by a histogram of the key's bits, three passes whatever the row holds, where
//     bisection took one a bit.  top-p adds probabilities as whole numbers of 2^-60.
// With `lists` the first way begins with the parts' candidates (sample_part_kernel) in place of its two passes.
// Microseconds of the kernels (by bisection, a bit a pass, before): 16 rows of 131,072 logits at T = 0.7 with top-k 50
// and top-p 0.95 22 in parts (1,612; 32 by one workgroup a row), top-p 0.9 alone 136 (840), neither 82 (166), top-k 2,000 134 (939),
// greedy 12 (24); 64 rows of 32,000 18 (443), 46 (238), 27 (54), 44 (257), 7 (9.1).
template <bool VEC>
__global__ void __launch_bounds__(SNT)
sample_kernel(const float* __restrict__ logits, int V, float temperature, int top_k, float top_p,
              uint32_t seed_lo, uint32_t seed_hi, const int* __restrict__ counters,
              float* __restrict__ probs, Tokens out, const PartList* __restrict__ lists, int n_parts) {
  __shared__ SampleShared sh;
  __shared__ Lists li;
  const int b = blockIdx.x, tid = threadIdx.x, w = tid / WAVE, lane = tid % WAVE;
  const float* z_in = logits + (size_t)b * V;
  float* p = probs + (size_t)b * V;

  if (!(temperature > 0.f)) {                           // greedy: of equal maxima the last index
    float best = -INFINITY;
    int bi = -1;
    visit<VEC>(z_in, V, [&](int i, float v) {
      if (bi < 0 || v >= best) { best = v; bi = i; }
    });
#pragma unroll
    for (int o = WAVE / 2; o > 0; o >>= 1) {
      const float v2 = __shfl_xor(best, o, WAVE);
      const int i2 = __shfl_xor(bi, o, WAVE);
      if (i2 >= 0 && (bi < 0 || v2 > best || (v2 == best && i2 > bi))) { best = v2; bi = i2; }
    }
    if (lane == 0) { sh.red[w] = best; sh.wave_count[w] = bi; }
    __syncthreads();
    if (tid == 0) {
      for (int i = 1; i < SNT / WAVE; ++i) {
        const float v2 = sh.red[i];
        const int i2 = sh.wave_count[i];
        if (i2 >= 0 && (bi < 0 || v2 > best || (v2 == best && i2 > bi))) { best = v2; bi = i2; }
      }
      out.put(b, bi);
    }
    return;
  }
  const float r = philox_uniform(seed_lo, seed_hi, (uint32_t)counters[2 * b + 1], (uint32_t)counters[2 * b]);
  const auto order = [](float v) { return order_key(v); };
  const auto bits = [](float v) { return __float_as_uint(v); };

  if (top_k > 0 && top_k < V && top_k <= MOST_TOP_K) {
    const PartList* parts = lists ? lists + (size_t)b * n_parts : nullptr;
    if (tid == 0) sh.count = 0;
    // A wave takes parts w and w + 16: their counts and each lane's first candidate come in one trip, the others, which lists of more
    // than a wave's lanes have, behind it
    // (counts, candidates and again for the second pass: 16.4 us the kernel, 15.9 now).
    constexpr int MINE = 2;
    static_assert(MINE * (SNT / WAVE) >= 32, "tl_sample_parts gives at most 32");
    int counts[MINE] = {};
    unsigned long long first[MINE] = {};
    if (parts) {
#pragma unroll
      for (int q = 0; q < MINE; ++q) {
        const unsigned long long* l = parts[min(w + q * (SNT / WAVE), n_parts - 1)];
        counts[q] = (int)l[0];
        first[q] = l[1 + lane];
      }
#pragma unroll
      for (int q = 0; q < MINE; ++q)
        if (w + q * (SNT / WAVE) >= n_parts) counts[q] = 0;
    }
    // (a part with more than its list holds, equal logits for instance: as without parts)
    if (parts && !__syncthreads_or(max(counts[0], counts[1]) > PART_KEEP)) {
      const auto each = [&](auto f) {
#pragma unroll
        for (int q = 0; q < MINE; ++q) {
          if (lane < counts[q]) f(first[q]);
          for (int j = lane + WAVE; j < counts[q]; j += WAVE) f(parts[w + q * (SNT / WAVE)][1 + j]);
        }
      };
      uint32_t mine = 0u;
      each([&](unsigned long long c) { mine = max(mine, (uint32_t)(c >> 32)); });
      const uint32_t bound = bound_of_kth<SNT>(mine, top_k, sh.reached);
      each([&](unsigned long long c) {
        if ((uint32_t)(c >> 32) >= bound) {
          const int at = atomicAdd(&sh.count, 1);
          if (at < CANDIDATES) li.c[at] = c;
        }
      });
    } else {
      uint32_t mine = 0u;
      visit<VEC>(z_in, V, [&](int, float v) { mine = max(mine, order_key(v)); });
      const uint32_t bound = with_margin(bound_of_kth<SNT>(mine, top_k, sh.reached));
      update<VEC>(z_in, p, V, [&](int i, float v) {
        if (order_key(v) >= bound) {
          const int at = atomicAdd(&sh.count, 1);
          if (at < CANDIDATES) li.c[at] = candidate(v / temperature, i);
        }
        return 0.f;
      });
    }
    __syncthreads();
    const int n = sh.count;
    if (n <= CANDIDATES) {
      // by value, of equal ones the smaller index first: the first k are kept
      if (n <= RANKED) {
        if (tid < n) {
          const unsigned long long mine_c = li.c[tid];
          int rank = 0;
#pragma unroll 8
          for (int o = 0; o < n; ++o) rank += li.c[o] > mine_c;
          if (rank < top_k) { li.top_z[rank] = from_order_key(mine_c >> 32); li.top_i[rank] = (int)~(uint32_t)mine_c; }
        }
      } else {
        sort_down(li.c, n);
        if (tid < top_k) { li.top_z[tid] = from_order_key(li.c[tid] >> 32); li.top_i[tid] = (int)~(uint32_t)li.c[tid]; }
      }
      __syncthreads();
      const float mx = li.top_z[0], least = li.top_z[top_k - 1];
      // (NaN fails the first; a last kept quotient among the denormals may be that of many logits)
      if (mx < INFINITY && least > -INFINITY && fabsf(least) > 1e-30f) {
        const bool have = tid < top_k;
        const int my_i = have ? li.top_i[tid] : 0;
        float e = have ? expf(li.top_z[tid] - mx) : 0.f;
        const float sum = block_sum<SNT>(e, sh.red);
        e = e / sum;
        bool kept = have;
        if (top_p > 0.f && top_p < 1.f) {
          // by probability, of equal ones the smaller index first: the list's order unless quotients that differ have
          // exponentials that do not
          __syncthreads();
          if (have) li.top_z[tid] = e;
          __syncthreads();
          const float e_next = have && tid + 1 < top_k ? li.top_z[tid + 1] : -1.f;
          const bool turned = e_next > e || (e_next == e && li.top_i[tid + 1] < my_i);
          double before = 0.0, total;
          if (__syncthreads_or(turned)) {
            for (int o = 0; o < top_k; ++o)
              before += li.top_z[o] > e || (li.top_z[o] == e && li.top_i[o] < my_i) ? (double)li.top_z[o] : 0.0;
          } else {
            before = block_excl_scan<double>((double)e, sh.wave_sum, &total);
          }
          kept = have && before < (double)top_p;
          const float new_sum = block_sum<SNT>(kept ? e : 0.f, sh.red);
          e = kept ? e / new_sum : 0.f;
        }
        __syncthreads();
        if (have) li.top_z[tid] = e;
        if (tid == 0) sh.pick = V - 1;
        __syncthreads();
        if (kept) {
          double run = 0.0;
          for (int o = 0; o < top_k; o += 8) {          // (loads first: an addition that waits for its own takes 80 ns)
            float z[8];
            int i[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) { z[q] = li.top_z[o + q]; i[q] = li.top_i[o + q]; }
#pragma unroll
            for (int q = 0; q < 8; ++q) run += o + q < top_k && i[q] <= my_i ? (double)z[q] : 0.0;
          }
          if (run >= (double)r) atomicMin(&sh.pick, my_i);
          p[my_i] = e;                                  // (behind the zeros of the pass above: barriers lie between)
        }
        __syncthreads();
        if (tid == 0) out.put(b, r > 0.f ? sh.pick : 0);
        return;
      }
    }
    __syncthreads();
  }

  update<VEC>(z_in, p, V, [&](int, float v) { return v / temperature; });
  __syncthreads();
  if (top_k > 0 && top_k < V) {
    unsigned long long n_gt, n_at;
    const uint32_t thr = select_key<VEC>(p, V, (unsigned long long)top_k, order, [](float) { return 1ull; }, sh, &n_gt, &n_at);
    __syncthreads();
    if (n_gt + n_at <= (unsigned long long)top_k) {
      update<VEC>(p, p, V, [&](int, float v) { return order_key(v) < thr ? -INFINITY : v; });
      __syncthreads();
    } else {
      keep_ties<VEC>(p, V, thr, top_k - (int)n_gt, -INFINITY, order, [](float v) { return v; }, sh);
    }
  }

  // softmax
  float mx = -INFINITY;
  visit<VEC>(p, V, [&](int, float v) { mx = fmaxf(mx, v); });
  mx = block_max<SNT>(mx, sh.red);
  float sum = 0.f;
  update<VEC>(p, p, V, [&](int, float v) {
    const float e = expf(v - mx);
    sum += e;
    return e;
  });
  sum = block_sum<SNT>(sum, sh.red);
  update<VEC>(p, p, V, [&](int, float v) { return v / sum; });
  __syncthreads();
  if (!(sum > 0.f && sum < INFINITY)) {                 // infinities or NaN among the logits: no draw
    if (tid == 0) out.put(b, V - 1);
    return;
  }

  if (top_p > 0.f && top_p < 1.f) {
    // the largest t with sum(p_i >= t) >= top_p is the smallest kept probability
    unsigned long long w_gt, w_at;
    const uint32_t thr = select_key<VEC>(p, V, fixed60(top_p), bits, [](float v) { return fixed60(v); }, sh, &w_gt, &w_at);
    const double thr_d = (double)__uint_as_float(thr), sum_gt = (double)w_gt / FIX;
    int ties = 0;
    visit<VEC>(p, V, [&](int, float v) { ties += __float_as_uint(v) == thr; });
    int n_ties;
    block_excl_scan<int>(ties, sh.wave_count, &n_ties);
    int room = thr_d > 0.0 ? (int)fmin(ceil(((double)top_p - sum_gt) / thr_d), (double)n_ties) : n_ties;
    room = max(1, min(room, n_ties));
    const float new_sum = (float)(sum_gt + (double)room * thr_d);
    const auto scaled = [&](float v) { return new_sum > 0.f ? v / new_sum : v; };
    if (room >= n_ties) {
      __syncthreads();
      update<VEC>(p, p, V, [&](int, float v) { return __float_as_uint(v) < thr ? 0.f : scaled(v); });
      __syncthreads();
    } else {
      keep_ties<VEC>(p, V, thr, room, 0.f, bits, scaled, sh);
    }
  }
  draw_row<VEC>(p, V, r, sh, b, out);
}

}  // namespace tl

using namespace tl;

// The parts a row is looked through in, or 0: none, a row is one workgroup's.  Long rows, and not so many that one workgroup each fills
// the chip.  Microseconds of the kernels, one workgroup a row / in parts, at T = 0.7 and top-k 50: 16 rows of 131,072
// 28 / 20, 64 of them 30 / 31, 16 rows of 32,000 16 / 18.  lists: room for [B][parts] lists of tl_sample_list_bytes() each.
extern "C" int tl_sample_parts(int B, int V, float temperature, int top_k) {
  if (B <= 0 || !(temperature > 0.f) || top_k <= 0 || top_k > PART_TOP_K || V <= 8 * PART_RUN || V > 32 * PART_RUN) return 0;
  const int parts = (V + PART_RUN - 1) / PART_RUN;
  return (long long)B * parts <= 512 ? parts : 0;
}
extern "C" int tl_sample_list_bytes() { return (int)sizeof(PartList); }

// counters [B][2] and host_out [B] (or null) may lie in pinned host memory: a row's workgroup reads 8 bytes of the one and writes 4 of the
// other while it has half a megabyte of logits to go through, where a copy each costs the stream 8 us and the host 5.
extern "C" int tl_sample(const float* logits, int B, int V, float temperature, int top_k, float top_p,
                         unsigned long long seed, const int* counters, float* probs, int* out, int* host_out, void* lists, int n_parts,
                         hipStream_t st) {
  TL_REQUIRE(B >= 0 && V > 0, "sample: bad sizes B=%d V=%d", B, V);
  TL_REQUIRE(n_parts == 0 || (lists != nullptr && n_parts == tl_sample_parts(B, V, temperature, top_k)), "sample: %d parts of a row of %d", n_parts, V);
  if (B == 0) return 0;
  const bool vec = V % 4 == 0 && ((uintptr_t)logits | (uintptr_t)probs) % 16 == 0;
  if (n_parts) {
    const int run = ((V + n_parts - 1) / n_parts + 3) / 4 * 4;
    const auto part = vec ? sample_part_kernel<true> : sample_part_kernel<false>;
    part<<<dim3(B, n_parts), PART_NT, 0, st>>>(logits, V, run, temperature, top_k, probs, (PartList*)lists);
    TL_LAUNCH_CHECK("sample_part");
  }
  const auto kernel = vec ? sample_kernel<true> : sample_kernel<false>;
  kernel<<<B, SNT, 0, st>>>(logits, V, temperature, top_k, top_p, (uint32_t)(seed & 0xffffffffu),
                            (uint32_t)(seed >> 32), counters, probs, Tokens{out, host_out}, (const PartList*)(n_parts ? lists : nullptr), n_parts);
  TL_LAUNCH_CHECK("sample");
  return 0;
}
