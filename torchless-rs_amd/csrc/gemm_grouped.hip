// Products of many rows with one of several matrices each, C[p] = A[row(p)] * W[group(p)]^T on the matrix cores:
// the experts of a routed feed-forward over the rows that chose them, without a copy of the rows and without
// the host knowing how many there are.
//
//  * group_pairs: the (row, chosen expert) pairs in the order of their experts, a row's place kept within one.
//  * gemm_grouped: tiles of up to 224 positions of one group by 256 of its channels.  What a tile does with its sums is the
//    kernel's template: an expert's activation times the row's weight into bfloat16, gated or not, or the sums as
//    they are.
//  * combine_pairs: a row's results from its experts added up in the order in which it chose them.
//
// A shared expert, which every row uses, can run along as slices of at most an expert's size: groups E, E + 1, ... of all
// rows each, at the positions behind the pairs', whose results are added behind the chosen experts'.
#include "experts.hpp"
#include "tile_loop.hpp"

namespace tl {

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

constexpr int GG_BM = 224, GG_BN = 256, GG_WN = 4, GG_NA = 2, GG_NW = 3;
constexpr int GG_LDS = tile_lds<GG_WN, GG_BM / 32, GG_NA, GG_NW>();
static_assert(GG_LDS <= 160 * 1024, "a compute unit's LDS");
// Tiles of few positions wait for the weights: what A's ring does not need of the LDS goes to another stage of W under way.
// A decode step of 19 rows of the 1,792-channel design (5 positions an expert): with the rings of the large tiles 3 % behind the
// four-wave tiles (1,404 against 1,364 us in one run), so 3 % ahead (1,304 against 1,343 in another); of 40 rows 1,386 against 1,429.
template <int MU> struct GGRings {
  static constexpr int A = MU == 1 ? 4 : MU == 2 ? 3 : GG_NA, W = MU <= 2 ? 4 : GG_NW;
  static_assert(tile_lds<GG_WN, MU, A, W>() <= GG_LDS, "the workgroup's LDS");
};

// A tile and its place.
struct Tile {
  int e, m0, m_rows, n0;
  int K, N;                          // of its group
  int row0;                          // what a position of a slice lies past its row
  int first;                         // the stage of K it begins with
};

// All of K for 32 MU rows of A (those that hold positions, and up to 31 more) by 256 rows of W.
template <int EPI, int MU>
__device__ __forceinline__ void gg_tile(const Grouped& g, const Tile& t, unsigned char* smem) {
  using S = TileShape<GG_WN, MU>;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE, li = lane % 16, kg = lane / 16;
  const int wm = wave / GG_WN, wn = wave % GG_WN, sub = lane / 8;
  const bool slice = t.e >= g.E;
  const char* asrc[S::A_PER];
#pragma unroll
  for (int x = 0; x < S::A_PER; ++x) {
    const int pos = t.m0 + min(tile_load<S::A_LOADS>(wave, x) * 8 + sub, t.m_rows - 1);
    const int row = !g.order ? pos : slice ? pos - t.row0 : g.order[pos] / g.top;
    asrc[x] = reinterpret_cast<const char*>(g.A + (size_t)row * g.lda);
  }
  const bool apart = EPI == GG_GATED && slice;
  const bf16* We = apart ? g.gated_slices + (size_t)(t.e - g.E) * g.N * g.ldw : g.W + (size_t)t.e * g.w_step;
  const size_t up_at = EPI == GG_GATED ? (apart ? (size_t)g.up_step : (size_t)g.N * g.ldw) : 0;
  const char* wsrc[S::W_PER];
#pragma unroll
  for (int x = 0; x < S::W_PER; ++x) {
    const int r = (wave + TILE_WAVES * x) * 8 + sub;           // row of the tile
    if (EPI == GG_GATED)                                       // 16 gate rows and their 16 up rows in turn
      wsrc[x] = reinterpret_cast<const char*>(We + (size_t)min(t.n0 + r / 32 * 16 + r % 16, t.N - 1) * g.ldw + (r / 16 % 2 ? up_at : 0));
    else
      wsrc[x] = reinterpret_cast<const char*>(We + (size_t)min(t.n0 + r, t.N - 1) * g.ldw);
  }
  f32x4 acc[MU][4];
#pragma unroll
  for (int u = 0; u < MU; ++u)
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[u][v] = f32x4{0.f, 0.f, 0.f, 0.f};
  tile_loop<GG_WN, MU, GGRings<MU>::A, GGRings<MU>::W, 0>(smem, [&](int x, unsigned at) { return asrc[x] + at; }, [&](int x, unsigned at) { return wsrc[x] + at; }, t.K, 0,
                                        (t.K + TILE_K - 1) / TILE_K, t.first, acc);

  // acc[u][v][r]: position 16 (wm MU + u) + li of the tile, row 64 wn + 16 v + 4 kg + r of W's tile
  float s[MU], after[MU];
  if constexpr (EPI != GG_STORE) {
#pragma unroll
    for (int u = 0; u < MU; ++u) {
      const int pos = t.m0 + min((wm * MU + u) * 16 + li, t.m_rows - 1);
      const int row = slice ? pos - t.row0 : g.order[pos] / g.top;
      s[u] = slice ? 1.f : g.weights[(size_t)row * g.E + t.e];
      after[u] = slice && g.row_weight ? g.row_weight[row] : 1.f;
    }
  }
#pragma unroll
  for (int u = 0; u < MU; ++u) {
    const int m = (wm * MU + u) * 16 + li;
    if (m >= t.m_rows) continue;
    const int pos = t.m0 + m;
    if constexpr (EPI == GG_STORE) {
      float* out = (float*)g.C + (size_t)pos * g.N;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int n = t.n0 + wn * 64 + v * 16 + kg * 4;
        if (n < t.N) *reinterpret_cast<f32x4*>(out + n) = acc[u][v];
      }
    } else {
      bf16* out = (bf16*)g.C + (size_t)pos * g.N;
      if constexpr (EPI == GG_UNARY) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int n = t.n0 + wn * 64 + v * 16 + kg * 4;
          if (n >= t.N) continue;
          bf16x4 h;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float z = fmaxf(acc[u][v][r], 0.f);
            h[r] = (bf16)((g.squared ? z * z : z) * s[u] * after[u]);
          }
          *reinterpret_cast<bf16x4*>(out + n) = h;
        }
      } else {
#pragma unroll
        for (int v = 0; v < 4; v += 2) {
          const int n = t.n0 + wn * 32 + v * 8 + kg * 4;
          if (n >= t.N) continue;
          bf16x4 h;
#pragma unroll
          for (int r = 0; r < 4; ++r) h[r] = (bf16)(gated_value(acc[u][v][r], acc[u][v + 1][r], s[u], slice ? g.gate.limit_shared : g.gate.limit, g.gate) * after[u]);
          *reinterpret_cast<bf16x4*>(out + n) = h;
        }
      }
    }
  }
}

// A workgroup of 8 waves has a tile of up to 224 positions of a group x 256 rows of W (see tile_loop.hpp; 256 positions would
// spill); a tile with fewer positions costs the matrix cores that much less, in steps of 32.  A group's positions are dealt to its
// tiles evenly.  Rows of A come from where the pair's row lies (a lane gives its own address).
// Bound by the products' rate with the chip full, and with few positions an expert by the weights (5.7 TB/s at 130 rows).  16
// experts, 4 a row, microseconds, up / down, before with four waves of 160 x 64, a wave alone on its SIMD: 3,584 channels at 600 rows
// 125 / 188 and 110 / 113 now, 2,312 rows 381 / 325 and 287 / 272 (0.95 and 1.0 PFLOP/s), 8,192 rows 1,144 / 1,081 and 862 / 891
// (1.1); 1,792 gated ones at 2,312 rows 386 / 183 and 292 / 153; 130 and 300 rows as they were.
template <int EPI>
__global__ void __launch_bounds__(TILE_WAVES * WAVE)
gemm_grouped_kernel(Grouped g) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char gg_smem[];
  constexpr int CT = EPI == GG_GATED ? GG_BN / 2 : GG_BN;      // channels of C a tile
  const int lane = threadIdx.x % WAVE;
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
  t.first = g.stagger ? (int)((long)t.first * ((t.K + TILE_K - 1) / TILE_K) / nt) : 0;

  switch ((t.m_rows + 31) / 32) {
    case 1: gg_tile<EPI, 1>(g, t, gg_smem); break;
    case 2: gg_tile<EPI, 2>(g, t, gg_smem); break;
    case 3: gg_tile<EPI, 3>(g, t, gg_smem); break;
    case 4: gg_tile<EPI, 4>(g, t, gg_smem); break;
    case 5: gg_tile<EPI, 5>(g, t, gg_smem); break;
    case 6: gg_tile<EPI, 6>(g, t, gg_smem); break;
    default: gg_tile<EPI, 7>(g, t, gg_smem); break;
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
  gemm_grouped_kernel<EPI><<<(unsigned)grid, TILE_WAVES * WAVE, GG_LDS, st>>>(g);
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
  g.stagger = g.K % TILE_K == 0 && (!down || slices == 0 || g.last % TILE_K == 0) && (long)n * top <= (long)E * GG_BM;
  g.weights = weights; g.row_weight = row_weight;
  g.squared = act_code == 0;
  g.gate = GateTerms{limit, limit_shared, alpha, shift, on_input};
  if (epilogue == GG_STORE) return launch_grouped<GG_STORE>(g, st);
  if (epilogue == GG_UNARY) return launch_grouped<GG_UNARY>(g, st);
  return launch_grouped<GG_GATED>(g, st);
}

}  // extern "C"
