// Products of many rows with one of several matrices each, C[p] = A[row(p)] * W[group(p)]^T on the matrix cores:
// the experts of a routed feed-forward over the rows that chose them, without a copy of the rows and without
// the host knowing how many there are.
//
//  * group_pairs: the (row, chosen expert) pairs in the order of their experts, a row's place kept within one.
//  * gemm_grouped: tiles of up to 160 positions of one group by 256 of its channels.  What a tile does with its sums is the
//    kernel's template: an expert's activation times the row's weight into bfloat16, gated or not, or the sums as
//    they are.
//  * combine_pairs: a row's results from its experts added up in the order in which it chose them.
//
// A shared expert, which every row uses, can run along as slices of at most an expert's size: groups E, E + 1, ... of all
// rows each, at the positions behind the pairs', whose results are added behind the chosen experts'.
#include "experts.hpp"

namespace tl {

#define TL_AS1 __attribute__((address_space(1)))      // global memory and LDS, as global_load_lds takes them
#define TL_AS3 __attribute__((address_space(3)))

// ---- the order of the pairs --------------------------------------------------------------------------------
// chosen [n_pairs] expert numbers -> offsets [E + 1], order [n_pairs]: position -> pair, place [n_pairs]: pair ->
// position.  A workgroup an expert: it counts the pairs of smaller experts and its own (every workgroup reads all
// of `chosen`, a few tens of KB from L2), then deals its pairs their positions, wave after wave.  6 us for 9,248 pairs
// of 16 experts, where a sort, a count and their index kernels took 80.  A number that is no expert's counts as the
// nearest expert's, so that `order` and `place` are a permutation, and what goes by them stays in its buffers, whatever
// `chosen` holds.
constexpr int GP_WAVES = 16;
__global__ void __launch_bounds__(GP_WAVES * WAVE)
group_pairs_kernel(const int* __restrict__ chosen, int n_pairs, int E, int* __restrict__ offsets, int* __restrict__ order,
                   int* __restrict__ place) {
  __shared__ int s_less[GP_WAVES], s_mine[GP_WAVES];
  const int e = blockIdx.x, wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  // waves take the pairs in equal runs, one after the other
  const int run = ((n_pairs + GP_WAVES - 1) / GP_WAVES + WAVE - 1) / WAVE * WAVE;
  const int lo = min(n_pairs, wave * run), hi = min(n_pairs, lo + run);
  int less = 0, mine = 0;
#pragma unroll 4
  for (int i = lo + lane; i < hi; i += WAVE) {
    const int c = min(max(chosen[i], 0), E - 1);
    less += c < e;
    mine += c == e;
  }
#pragma unroll
  for (int o = WAVE / 2; o > 0; o >>= 1) {
    less += __shfl_xor(less, o, WAVE);
    mine += __shfl_xor(mine, o, WAVE);
  }
  if (lane == 0) { s_less[wave] = less; s_mine[wave] = mine; }
  __syncthreads();
  int first = 0, before = 0, all = 0;
#pragma unroll
  for (int w = 0; w < GP_WAVES; ++w) {
    first += s_less[w];
    if (w < wave) before += s_mine[w];
    all += s_mine[w];
  }
  if (threadIdx.x == 0) {
    offsets[e] = first;
    if (e == E - 1) offsets[E] = first + all;
  }
  int at = first + before;
  for (int base = lo; base < hi; base += WAVE) {
    const int i = base + lane;
    const bool hit = i < hi && min(max(chosen[i], 0), E - 1) == e;
    const unsigned long long hits = __ballot(hit);
    if (hit) {
      const int pos = at + __popcll(hits & ((1ull << lane) - 1ull));
      order[pos] = i;
      place[i] = pos;
    }
    at += __popcll(hits);
  }
}

// out[n, :] (+)= sum over slots k of z[place[n * top + k], :], in the order of k, then of the slices of the shared expert,
// z[rows * top + j * rows + n, :]
__global__ void __launch_bounds__(256)
combine_pairs_kernel(const float* __restrict__ z, const int* __restrict__ place, int rows, int top, int slices, int H, int accumulate,
                     float* __restrict__ out) {
  const int n = blockIdx.x, c = (blockIdx.y * 256 + threadIdx.x) * 4;
  if (c >= H) return;
  f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k = 0; k < top; ++k) sum += *(const f32x4*)(z + (size_t)place[(size_t)n * top + k] * H + c);
#pragma unroll 4
  for (int j = 0; j < slices; ++j) sum += *(const f32x4*)(z + ((size_t)rows * (top + j) + n) * H + c);
  f32x4* o = (f32x4*)(out + (size_t)n * H + c);
  *o = accumulate ? *o + sum : sum;
}

// ---- the product --------------------------------------------------------------------------------------------
constexpr int GG_STORE = 0;    // C float [position, N] = sums
constexpr int GG_UNARY = 1;    // C bfloat16 [position, N] = act(sums) * weight
constexpr int GG_GATED = 2;    // W's rows of a group are [gate (N) | up (N)]: C bfloat16 [position, N] = act(gate, up, weight)

struct Grouped {
  const bf16* A;
  const bf16* W;
  void* C;
  long long w_step;            // elements from one group's weights to the next's
  int lda, ldw, K, N;
  const int* offsets;          // [E + 1] first positions of the experts
  const int* order;            // position -> pair, or null: A has a row a position
  int E, rows, top;            // experts, rows of the step, chosen experts a row
  int slices, last;            // groups of all rows behind the experts', and the size of the last (its N, or with `slice_k` its K)
  int slice_k;
  long long up_step;           // gated: elements from a slice's gate rows to its up rows
  const bf16* gated_slices;    // gated: the slices' gate rows (they lie otherwise than an expert's)
  int stagger;                 // tiles of other channels begin with other stages of K
  const float* weights;        // [row, E] the router's
  const float* row_weight;     // [row] a weight on the slices' output, or null
  int squared;                 // the activation of one argument: max(., 0), or its square
  GateTerms gate;
};

__device__ __forceinline__ int group_first(const Grouped& g, int x) {
  return x < g.E ? g.offsets[x] : g.rows * (g.top + x - g.E);
}
__device__ __forceinline__ int group_size(const Grouped& g, int x) { return x < g.E ? g.offsets[x + 1] - g.offsets[x] : g.rows; }

constexpr int GG_BM = 160, GG_BN = 256, GG_BK = 64, GG_NS = 3, GG_WAVES = 4;
constexpr int GG_ROWB = GG_BK * 2, GG_STAGE = (GG_BM + GG_BN) * GG_ROWB, GG_LDS = GG_NS * GG_STAGE;
static_assert(GG_LDS <= 160 * 1024, "a compute unit's LDS");

// Where the operands of a tile come from, and its place.
struct Tile {
  const bf16* asrc[GG_BM / 32];      // this lane's sources: of the 8 rows wave + 4 x of A's, and of the wave's 64 rows of W
  const bf16* wsrc[8];
  int e, m0, m_rows, n0;
  int K, N;                          // of its group
  int row0;                          // what a position of a slice lies past its row
  int first;                         // the stage of K it begins with
};

// All of K for 16 MU rows of A (MU: an even number of 16-row blocks, those that hold positions) by the wave's 64 rows of W.
template <int EPI, int MU>
__device__ __forceinline__ void gg_tile(const Grouped& g, const Tile& t, unsigned char* smem) {
  constexpr int AI = MU / 2, LPS = AI + 8;                     // loads of a wave a stage: A's, and all
  constexpr int EARLY = MU < 4 ? MU : 4;                       // blocks of A that are in registers before their turn
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE, li = lane % 16, kg = lane / 16;
  const int stages = (t.K + GG_BK - 1) / GG_BK;
  const int chunk = (lane % 8) ^ ((lane / 16) & 3);            // of an 8-row load's even half of 16 rows; the odd half's differs in bit 2
  const auto issue = [&](int i) {
    unsigned char* slot = smem + (i % GG_NS) * GG_STAGE;
    int k = i + t.first;
    if (k >= stages) k -= stages;
    k *= GG_BK;
    // (past the end of a row its last chunk again, see `cut`)
    const int even = min(k + chunk * 8, t.K - 8), odd = min(k + (chunk ^ 4) * 8, t.K - 8), mine = wave % 2 ? odd : even;
#pragma unroll
    for (int x = 0; x < 8; ++x)
      __builtin_amdgcn_global_load_lds((const TL_AS1 void*)(t.wsrc[x] + (x % 2 ? odd : even)),
                                       (TL_AS3 void*)(slot + GG_BM * GG_ROWB + (wave * 8 + x) * 1024), 16, 0, 0);
#pragma unroll
    for (int x = 0; x < AI; ++x)
      __builtin_amdgcn_global_load_lds((const TL_AS1 void*)(t.asrc[x] + mine), (TL_AS3 void*)(slot + (wave + 4 * x) * 1024), 16, 0, 0);
  };
  f32x4 acc[MU][4];
#pragma unroll
  for (int u = 0; u < MU; ++u)
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[u][v] = f32x4{0.f, 0.f, 0.f, 0.f};
  // chunk c of row r of a stage lies at place c ^ (r / 2 % 8) of its 128 bytes
  const int row_at = li * GG_ROWB, place[2] = {(kg ^ (li / 2)) * 16, ((4 + kg) ^ (li / 2)) * 16};
  const auto fetch_w = [&](int i, int half, bf16x8 (&w)[4]) {
    const unsigned char* slot = smem + (i % GG_NS) * GG_STAGE + GG_BM * GG_ROWB + wave * 8192 + row_at + place[half];
#pragma unroll
    for (int v = 0; v < 4; ++v) w[v] = *reinterpret_cast<const bf16x8*>(slot + v * 2048);
  };
  const auto fetch_a = [&](int i, int half, int u) {
    return *reinterpret_cast<const bf16x8*>(smem + (i % GG_NS) * GG_STAGE + row_at + place[half] + u * 2048);
  };
  // half a stage (32 k): the operands of its first products are in registers; the others come from LDS between the products (a
  // wave is alone on its SIMD, and a row of reads would let the matrix core idle), and behind them the next half's first
  const auto multiply = [&](int i, int half, bool more, bool cut, const bf16x8 (&a)[EARLY], const bf16x8 (&w)[4], bf16x8 (&an)[EARLY], bf16x8 (&wn)[4]) {
    bf16x8 b[MU];
#pragma unroll
    for (int u = 0; u < EARLY; ++u) b[u] = a[u];
#pragma unroll
    for (int u = EARLY; u < MU; ++u) b[u] = fetch_a(i, half, u);
    if (more) {
      fetch_w(i + half, 1 - half, wn);
#pragma unroll
      for (int u = 0; u < EARLY; ++u) an[u] = fetch_a(i + half, 1 - half, u);
    }
    if (cut && (stages - 1) * GG_BK + (half * 4 + kg) * 8 >= t.K) {      // what lies past the end of K (a multiple of 8)
#pragma unroll
      for (int u = 0; u < MU; ++u)
#pragma unroll
        for (int j = 0; j < 8; ++j) b[u][j] = (bf16)0.f;
    }
#pragma unroll
    for (int u = 0; u < MU; ++u)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[u][v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[v], b[u], acc[u][v], 0, 0, 0);
    constexpr int READS = MU + 4, EACH = MU * 4 / READS;
#pragma unroll
    for (int r = 0; r < READS; ++r) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, EACH, 0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");         // this wave's reads have returned, before the next barrier
  };
  issue(0);
  if (stages > 1) {
    issue(1);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LPS) : "memory");
  } else {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  __builtin_amdgcn_s_barrier();
  bf16x8 a0[EARLY], a1[EARLY], w0[4], w1[4];
  fetch_w(0, 0, w0);
#pragma unroll
  for (int u = 0; u < EARLY; ++u) a0[u] = fetch_a(0, 0, u);
  for (int i = 0; i + 1 < stages; ++i) {
    __builtin_amdgcn_s_barrier();                              // everyone has left stage i - 1
    if (i + 2 < stages) issue(i + 2);                          // into its place
    multiply(i, 0, true, false, a0, w0, a1, w1);
    // stage i + 1 is here when only the loads behind it are under way
    if (i + 2 < stages) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LPS) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    multiply(i, 1, true, false, a1, w1, a0, w0);
  }
  const bool cut = t.K % GG_BK != 0;
  multiply(stages - 1, 0, true, cut, a0, w0, a1, w1);
  multiply(stages - 1, 1, false, cut, a1, w1, a0, w0);

  // acc[u][v][r]: position 16 u + li of the tile, row 64 wave + 16 v + 4 kg + r of W's tile
#pragma unroll
  for (int u = 0; u < MU; ++u) {
    const int m = u * 16 + li;
    if (m >= t.m_rows) continue;
    const int pos = t.m0 + m;
    if constexpr (EPI == GG_STORE) {
      float* out = (float*)g.C + (size_t)pos * g.N;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int n = t.n0 + wave * 64 + v * 16 + kg * 4;
        if (n < t.N) *reinterpret_cast<f32x4*>(out + n) = acc[u][v];
      }
    } else {
      const bool slice = t.e >= g.E;
      const int row = slice ? pos - t.row0 : g.order[pos] / g.top;
      const float s = slice ? 1.f : g.weights[(size_t)row * g.E + t.e];
      const float after = slice && g.row_weight ? g.row_weight[row] : 1.f;
      bf16* out = (bf16*)g.C + (size_t)pos * g.N;
      if constexpr (EPI == GG_UNARY) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int n = t.n0 + wave * 64 + v * 16 + kg * 4;
          if (n >= t.N) continue;
          bf16x4 h;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float z = fmaxf(acc[u][v][r], 0.f);
            h[r] = (bf16)((g.squared ? z * z : z) * s * after);
          }
          *reinterpret_cast<bf16x4*>(out + n) = h;
        }
      } else {
#pragma unroll
        for (int v = 0; v < 4; v += 2) {
          const int n = t.n0 + wave * 32 + v * 8 + kg * 4;
          if (n >= t.N) continue;
          bf16x4 h;
#pragma unroll
          for (int r = 0; r < 4; ++r) h[r] = (bf16)(gated_value(acc[u][v][r], acc[u][v + 1][r], s, slice ? g.gate.limit_shared : g.gate.limit, g.gate) * after);
          *reinterpret_cast<bf16x4*>(out + n) = h;
        }
      }
    }
  }
}

// A workgroup of 4 waves, one to a SIMD, has a tile of up to 160 positions of a group x 256 rows of W; a wave has all of the
// positions and 64 of the rows (160 sums a lane), so that a tile with fewer positions costs the matrix cores that much
// less, in steps of 32.  A group's positions are dealt to its tiles evenly.  Stages of 64 k (52 KB, whole lines of 128 bytes:
// halves of 64 were fetched twice) go from memory straight into a ring of three in LDS.  Chunk c of row r of a stage lies at
// place c ^ (r / 2 % 8): 16 lanes that read one chunk of 16 rows fall on all banks once.  Rows of A come from where the
// pair's row lies (a lane gives its own address).
// What bounds it: the products of a stage are 1,280 cycles of the matrix cores, the reads and writes of LDS 1,310, and they
// overlap in part only: a stage takes 1.5 us with the chip full, 1.26 with the loads taken out, 0.9 with the products.
// Other tiles measured (2,312 rows, 16 experts of 3,584 channels, 4 a row, up / down, microseconds; this one 444 / 361):
// 128 x 256 with stages of 32 k and two workgroups a unit 461 / 407, 256 x 256 with 4 waves 462 / 450, with 8 waves 438 / 383
// (1,024 rows: 256 / 224 against 189 / 164 here, since 257 rows take two of its tiles), W from memory into registers 472 / 442.
template <int EPI>
__global__ void __launch_bounds__(GG_WAVES * WAVE, 1)
gemm_grouped_kernel(Grouped g) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char gg_smem[];
  constexpr int CT = EPI == GG_GATED ? GG_BN / 2 : GG_BN;      // channels of C a tile
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const int nt = (g.N + CT - 1) / CT;

  // which tile: an expert's tiles follow each other, of its tiles those of the same channels; each of the 8 XCDs
  // (workgroups go round them) has a run of tiles of its own, whose operands its L2 then serves
  Tile t;
  t.e = t.m0 = t.m_rows = t.n0 = t.first = 0;
  t.row0 = 0;
  {
    const int groups = g.E + g.slices, per = (groups + WAVE - 1) / WAVE;      // groups of a lane
    int tiles = 0;
    for (int i = 0; i < per; ++i) {
      const int x = lane * per + i;
      if (x < groups) tiles += (group_size(g, x) + GG_BM - 1) / GG_BM;
    }
    int incl = tiles;
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
      const int up = __shfl_up(incl, o, WAVE);
      if (lane >= o) incl += up;
    }
    const int total = __shfl(incl, WAVE - 1, WAVE) * nt;
    const int chunk = (total + 7) / 8, id = blockIdx.x;
    const int at_tile = (id % 8) * chunk + id / 8;
    if (id / 8 >= chunk || at_tile >= total) return;           // (the same for all of the workgroup)
    const unsigned long long behind = __ballot(incl * nt > at_tile);
    const int owner = __ffsll((long long)behind) - 1;
    int left = at_tile - (__shfl(incl, owner, WAVE) - __shfl(tiles, owner, WAVE)) * nt;
    for (int i = 0; i < per; ++i) {
      const int x = owner * per + i;
      if (x >= groups) break;
      const int at = group_first(g, x), count = group_size(g, x);
      const int mt = (count + GG_BM - 1) / GG_BM;
      if (left < mt * nt) {
        const int share = ((count + mt - 1) / mt + 15) / 16 * 16;      // positions of a tile (the last may have fewer)
        t.e = x;
        t.row0 = at;
        t.m0 = at + left % mt * share;
        t.m_rows = min(share, at + count - t.m0);
        t.n0 = left / mt * CT;
        t.first = left / mt;
        break;
      }
      left -= mt * nt;
    }
  }
  const bool slice = t.e >= g.E, last = t.e + 1 == g.E + g.slices && slice;
  t.K = last && g.slice_k ? g.last : g.K;
  t.N = last && !g.slice_k ? g.last : g.N;
  if (t.n0 >= t.N) return;                                     // (the last slice may have fewer channels)
  t.first = g.stagger ? (int)((long)t.first * ((t.K + GG_BK - 1) / GG_BK) / nt) : 0;

  const int sub = lane / 8;                                    // a load takes 8 rows of 128 bytes
#pragma unroll
  for (int x = 0; x < GG_BM / 32; ++x) {
    const int pos = t.m0 + min((wave + 4 * x) * 8 + sub, t.m_rows - 1);
    const int row = !g.order ? pos : slice ? pos - t.row0 : g.order[pos] / g.top;
    t.asrc[x] = g.A + (size_t)row * g.lda;
  }
  const bool apart = EPI == GG_GATED && slice;
  const bf16* We = apart ? g.gated_slices + (size_t)(t.e - g.E) * g.N * g.ldw : g.W + (size_t)t.e * g.w_step;
  const size_t up_at = EPI == GG_GATED ? (apart ? (size_t)g.up_step : (size_t)g.N * g.ldw) : 0;
#pragma unroll
  for (int x = 0; x < 8; ++x) {
    const int r16 = wave * 4 + x / 2, r = x % 2 * 8 + sub;     // row r of 16 rows of the tile
    if (EPI == GG_GATED)                                       // gate and up in turn
      t.wsrc[x] = We + (size_t)min(t.n0 + r16 / 2 * 16 + r, t.N - 1) * g.ldw + (r16 % 2 ? up_at : 0);
    else
      t.wsrc[x] = We + (size_t)min(t.n0 + r16 * 16 + r, t.N - 1) * g.ldw;
  }
  switch ((t.m_rows + 31) / 32) {
    case 1: gg_tile<EPI, 2>(g, t, gg_smem); break;
    case 2: gg_tile<EPI, 4>(g, t, gg_smem); break;
    case 3: gg_tile<EPI, 6>(g, t, gg_smem); break;
    case 4: gg_tile<EPI, 8>(g, t, gg_smem); break;
    default: gg_tile<EPI, 10>(g, t, gg_smem); break;
  }
}

template <int EPI> static int launch_grouped(const Grouped& g, hipStream_t st) {
  // every call: the attribute belongs to the function on the current device, and setting it costs well under a microsecond
  const hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_grouped_kernel<EPI>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, GG_LDS);
  if (err != hipSuccess) {
    set_error("gemm_grouped: cannot have %d bytes of LDS: %s", GG_LDS, hipGetErrorString(err));
    return 2;
  }
  constexpr int CT = EPI == GG_GATED ? GG_BN / 2 : GG_BN;
  const long nt = (g.N + CT - 1) / CT;
  // at most this many tiles, whatever the experts' sizes
  const long pairs = (long)g.rows * g.top;
  const long most = nt * (pairs / GG_BM + (g.E < pairs ? g.E : pairs) + (long)g.slices * ((g.rows + GG_BM - 1) / GG_BM));
  const long grid = (most + 7) / 8 * 8;
  TL_REQUIRE(grid < (1l << 31), "gemm_grouped: rows=%d N=%d have more tiles than a grid holds", g.rows, g.N);
  gemm_grouped_kernel<EPI><<<(unsigned)grid, GG_WAVES * WAVE, GG_LDS, st>>>(g);
  TL_LAUNCH_CHECK("gemm_grouped");
  return 0;
}

}  // namespace tl

using namespace tl;

extern "C" {

// chosen int [n, top] -> offsets int [E + 1], order and place int [n * top] (see group_pairs_kernel)
int tl_group_pairs(const int* chosen, int n_pairs, int E, int* offsets, int* order, int* place, hipStream_t st) {
  TL_REQUIRE(n_pairs > 0 && E > 0 && E <= 65535, "group_pairs: bad sizes pairs=%d E=%d", n_pairs, E);
  TL_REQUIRE(chosen && offsets && order && place, "group_pairs: a buffer is missing");
  group_pairs_kernel<<<E, GP_WAVES * WAVE, 0, st>>>(chosen, n_pairs, E, offsets, order, place);
  TL_LAUNCH_CHECK("group_pairs");
  return 0;
}

// z float [n * (top + slices), H] -> out float [n, H], stored or added to
int tl_combine_pairs(const float* z, const int* place, int n, int top, int slices, int H, int accumulate, float* out, hipStream_t st) {
  TL_REQUIRE(n >= 0 && top > 0 && slices >= 0 && H > 0 && H % 4 == 0, "combine_pairs: bad sizes n=%d top=%d H=%d (H a multiple of 4)", n, top, H);
  TL_REQUIRE(z && place && out && ((uintptr_t)z | (uintptr_t)out) % 16 == 0, "combine_pairs: a buffer is missing or off 16 bytes");
  if (n == 0) return 0;
  combine_pairs_kernel<<<dim3(n, (H + 1023) / 1024), 256, 0, st>>>(z, place, n, top, slices, H, accumulate, out);
  TL_LAUNCH_CHECK("combine_pairs");
  return 0;
}

// The positions of a step of n rows: its n * top pairs in the order of their experts (offsets, order as tl_group_pairs leaves
// them), then n for each of `slices` slices of a shared expert of `shared` channels, ff channels each (the last the rest).
// first half: A bfloat16 [n, K = H], W the stacked matrix [E * ff + shared, H] (gated: twice the rows, an expert's [gate | up] and
// the shared one's behind them); C bfloat16 [positions, ff].  epilogue 1: the square of max(., 0) (act_code 0) or max(., 0)
// (1), times the row's weight of the expert; 2: the gated activation.
// second half (epilogue 0): A bfloat16 [positions, ff], W [H, E * ff + shared]; C float [positions, H].
int tl_gemm_grouped(const void* A, const void* W, void* C, int n, int H, int E, int ff, int shared, int slices, int top, const int* offsets,
                    const int* order, const float* weights, const float* row_weight, int epilogue, int act_code, float limit,
                    float limit_shared, float alpha, float shift, int on_input, hipStream_t st) {
  TL_REQUIRE(n >= 0 && H > 0 && E > 0 && ff > 0 && shared >= 0 && top > 0 && slices >= 0, "gemm_grouped: bad sizes n=%d H=%d E=%d ff=%d shared=%d top=%d slices=%d",
             n, H, E, ff, shared, top, slices);
  TL_REQUIRE(H % 8 == 0 && ff % 8 == 0 && shared % 8 == 0, "gemm_grouped: H=%d ff=%d shared=%d must be multiples of 8", H, ff, shared);
  TL_REQUIRE(slices == 0 || slices == (shared + ff - 1) / ff, "gemm_grouped: %d slices of %d are not a shared expert of %d", slices, ff, shared);
  TL_REQUIRE((long)n * (top + slices) < (1l << 31), "gemm_grouped: %d rows have too many positions", n);
  TL_REQUIRE(A && W && C && offsets && ((uintptr_t)A | (uintptr_t)W | (uintptr_t)C) % 16 == 0, "gemm_grouped: an operand is missing or off 16 bytes");
  TL_REQUIRE(epilogue >= 0 && epilogue <= 2 && act_code >= 0 && act_code <= 1, "gemm_grouped: unknown epilogue %d or activation %d", epilogue, act_code);
  TL_REQUIRE(epilogue == GG_STORE || (order && weights), "gemm_grouped: the pairs' order or weights are missing");
  if (n == 0) return 0;
  const bool down = epilogue == GG_STORE;
  const int total = E * ff + shared;
  Grouped g{};
  g.A = (const bf16*)A; g.W = (const bf16*)W; g.C = C;
  g.w_step = down ? ff : (long long)(epilogue == GG_GATED ? 2 : 1) * ff * H;
  g.lda = down ? ff : H; g.ldw = down ? total : H; g.K = down ? ff : H; g.N = down ? H : ff;
  g.offsets = offsets; g.order = down ? nullptr : order; g.E = E; g.rows = n; g.top = top;
  g.slices = slices; g.last = shared - (slices - 1) * ff; g.slice_k = down;
  g.up_step = (long long)shared * H;
  g.gated_slices = g.W + (long long)2 * E * ff * H;
  // where an expert has few positions the weights come from memory, row after row at one distance: workgroups that go along K
  // in step would ask the same channels of the memory at a time (130 rows of 16 experts: 113 to 86 us; K's tail has to be the last stage)
  g.stagger = g.K % GG_BK == 0 && (!down || slices == 0 || g.last % GG_BK == 0) && (long)n * top <= (long)E * GG_BM;
  g.weights = weights; g.row_weight = row_weight;
  g.squared = act_code == 0;
  g.gate = GateTerms{limit, limit_shared, alpha, shift, on_input};
  if (epilogue == GG_STORE) return launch_grouped<GG_STORE>(g, st);
  if (epilogue == GG_UNARY) return launch_grouped<GG_UNARY>(g, st);
  return launch_grouped<GG_GATED>(g, st);
}

}  // extern "C"
