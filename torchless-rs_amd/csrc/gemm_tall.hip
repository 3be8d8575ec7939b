// bfloat16 products of more than 128 rows on the matrix cores, C[M,N] (+)= A[M,K] * W[N,K]^T, where they are faster than the BLAS
// library's (ops.tall_plan): tiles of 128 to 256 rows by 128 or 256 channels (tile_loop.hpp), K cut over workgroups into
// partial sums where the tiles are too few for the chip, the activation of a paired product in the epilogue.
#include "epilogues.hpp"
#include "experts.hpp"
#include "tile_loop.hpp"

namespace tl {

struct Tall {
  const bf16* A;
  const bf16* W;
  float* C;                    // float [splits, M, N], or with a paired epilogue bfloat16 [M, N / 2]
  int M, N, K, lda, ldw;
  int mt, nt;                  // tiles along the rows and the channels
  int share;                   // rows of a tile (the last may have fewer)
  int splits, stages;          // slices of K, and a slice's stages of 64 k
  int stagger;                 // tiles of other channels begin with other stages
  int whole, parts;            // the tiles behind the first `whole` ones are cut in `parts` (2 or 4); 0: none is
  Epi epi;
  // TALL_UNARY, TALL_GATED: the activation of an expert on the sums, times a factor of the row (null: 1); C is bfloat16
  UnaryAct unary;              // [M, N]
  GateTerms gate;              // [M, N / 2]; W is [gate | up] by rows, paired as the tile is loaded: channels in groups of 64,
                               // 32 of gate and the 32 rows N / 2 further
  const float* row_weight;
};
constexpr int TALL_UNARY = 6, TALL_GATED = 7;   // epilogues beside those of `Epi`

constexpr int TALL_GROUP = 8;  // tiles of rows that go side by side through the channels

// m_rows rows from m0 by the channels from n0 on, slice `split` of K
template <int WN, int MU, int NA, int NW, int W_AUX>
__device__ __forceinline__ void tall_tile(const Tall& g, int m0, int m_rows, int n0, int split, int first, unsigned char* smem) {
  using S = TileShape<WN, MU>;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE, li = lane % 16, kg = lane / 16;
  const int wm = wave / WN, wn = wave % WN, sub = lane / 8;
  const int t0 = split * g.stages, n_t = min((g.K + TILE_K - 1) / TILE_K - t0, g.stages);
  // a lane's rows as distances from the first of the tile's that its wave loads: at most 256 rows of K.  Gate and up rows that lie
  // apart go by 32 in turn, four waves' loads each: of all its loads a wave has gate rows or up rows.
  const char* A0 = reinterpret_cast<const char*>(g.A + (size_t)m0 * g.lda);
  const bool apart = g.epi == TALL_GATED;
  const char* W0 = reinterpret_cast<const char*>(g.W + (size_t)(apart ? n0 / 2 + (wave & 4 ? g.N / 2 : 0) : n0) * g.ldw);
  unsigned aoff[S::A_PER], woff[S::W_PER];
#pragma unroll
  for (int x = 0; x < S::A_PER; ++x) aoff[x] = (unsigned)min(tile_load<S::A_LOADS>(wave, x) * 8 + sub, m_rows - 1) * (unsigned)g.lda * 2u;
#pragma unroll
  for (int x = 0; x < S::W_PER; ++x) {
    const int c = min((wave + TILE_WAVES * x) * 8 + sub, g.N - 1 - n0);
    woff[x] = (unsigned)(apart ? c / 64 * 32 + c % 32 : c) * (unsigned)g.ldw * 2u;
  }

  f32x4 acc[MU][4];
#pragma unroll
  for (int u = 0; u < MU; ++u)
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[u][v] = f32x4{0.f, 0.f, 0.f, 0.f};
  tile_loop<WN, MU, NA, NW, W_AUX>(smem, [&](int x, unsigned at) { return A0 + (aoff[x] + at); }, [&](int x, unsigned at) { return W0 + (woff[x] + at); },
                                   g.K, t0, n_t, first % n_t, acc);

  // acc[u][v][r]: row 16 (wm MU + u) + li of the tile, channel 64 wn + 16 v + 4 kg + r
  const int c0 = n0 + wn * 64 + kg * 4;
  // a wave's 64 channels are 32 gate rows and their 32 up rows; value(gate, up, row)
  const auto paired = [&](auto value) {
#pragma unroll
    for (int u = 0; u < MU; ++u) {
      const int m = (wm * MU + u) * 16 + li;
      if (m >= m_rows) continue;
      bf16* out = reinterpret_cast<bf16*>(g.C) + (size_t)(m0 + m) * (g.N / 2);
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        const int n = (n0 + wn * 64) / 2 + v * 16 + kg * 4;
        if (n >= g.N / 2) continue;
        bf16x4 h;
#pragma unroll
        for (int r = 0; r < 4; ++r) h[r] = (bf16)value(acc[u][v][r], acc[u][v + 2][r], m0 + m);
        *reinterpret_cast<bf16x4*>(out + n) = h;
      }
    }
  };
  // (a loop for each: with one that chose for every value the short one came with the long ones around it, 393 us for gate|up of 2,048
  // rows by 28,672, K = 4,096, and 355 so)
  if (g.epi == EPI_SILU_PAIR) return paired([&](float x, float y, int) { return pair_value_near(x, y, Epi(EPI_SILU_PAIR)); });
  if (is_pair(g.epi)) return paired([&](float x, float y, int) { return pair_value(x, y, g.epi); });
  if (apart)
    return paired([&](float x, float y, int m) {
      return gated_value(x, y, 1.f, g.gate.limit_shared, g.gate) * (g.row_weight ? g.row_weight[m] : 1.f);
    });
  if (g.epi == TALL_UNARY) {
#pragma unroll
    for (int u = 0; u < MU; ++u) {
      const int m = (wm * MU + u) * 16 + li;
      if (m >= m_rows) continue;
      bf16* out = reinterpret_cast<bf16*>(g.C) + (size_t)(m0 + m) * g.N;
      const float after = g.row_weight ? g.row_weight[m0 + m] : 1.f;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        if (c0 + v * 16 >= g.N) continue;
        bf16x4 h;
#pragma unroll
        for (int r = 0; r < 4; ++r) h[r] = (bf16)(unary_act(acc[u][v][r], g.unary) * after);
        *reinterpret_cast<bf16x4*>(out + c0 + v * 16) = h;
      }
    }
    return;
  }
  float* C = g.C + (size_t)split * g.M * g.N + (size_t)m0 * g.N;
  if (g.epi == EPI_ACCUMULATE) {               // what is added to comes from memory for several blocks of rows at a time
    constexpr int UB = MU < 7 ? 4 : 2;                   // (in the registers that the operands had)
#pragma unroll
    for (int b = 0; b < MU; b += UB) {
      f32x4 old[UB][4];
#pragma unroll
      for (int u = 0; u < UB && b + u < MU; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          old[u][v] = *reinterpret_cast<const f32x4*>(C + (size_t)min((wm * MU + b + u) * 16 + li, m_rows - 1) * g.N + min(c0 + v * 16, g.N - 4));
#pragma unroll
      for (int u = 0; u < UB && b + u < MU; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[b + u][v] = old[u][v] + acc[b + u][v];
    }
  }
#pragma unroll
  for (int u = 0; u < MU; ++u) {
    const int m = (wm * MU + u) * 16 + li;
    if (m >= m_rows) continue;
#pragma unroll
    for (int v = 0; v < 4; ++v)
      if (c0 + v * 16 < g.N) *reinterpret_cast<f32x4*>(C + (size_t)m * g.N + c0 + v * 16) = acc[u][v];
  }
}

// PARTS: the launch may have tiles in parts, see `Tall::whole`.
template <int WN, int MU, int NA, int NW, int W_AUX, bool PARTS>
__global__ void __launch_bounds__(TILE_WAVES * WAVE)
gemm_tall_kernel(Tall g) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char tall_smem[];
  constexpr int CHANNELS = TileShape<WN, MU>::CHANNELS;
  // each of the 8 XCDs (workgroups go round them) has a run of tiles of its own; the tiles go by groups of TALL_GROUP of rows, in
  // a group from channels to channels, so that an XCD's workgroups share rows and channels in its L2.  Where K is cut, a slice's tiles
  // follow each other: an XCD then reads a slice or two of A instead of all of it.
  const int total = g.mt * g.nt, whole = PARTS ? g.whole : total * g.splits;
  const bool cut = PARTS && (int)blockIdx.x >= whole;          // (whole is a multiple of 8 where tiles are cut)
  const int id = cut ? blockIdx.x - whole : blockIdx.x, count = cut ? (total - whole) * g.parts : whole;
  const int chunk = (count + 7) / 8, at = id % 8 * chunk + id / 8;
  if (id / 8 >= chunk || at >= count) return;
  const int split = PARTS ? 0 : at / total, t = cut ? whole + at / g.parts : at - split * total;
  const int group = t / (TALL_GROUP * g.nt), gm = group * TALL_GROUP, gs = min(TALL_GROUP, g.mt - gm), in = t - gm * g.nt;
  const int nb = in / gs, m0 = (gm + in % gs) * g.share, m_rows = min(g.share, g.M - m0), n0 = nb * CHANNELS;
  if constexpr (PARTS) {
    if (cut) {
      const int part = at % g.parts, n1 = n0 + part % 2 * (CHANNELS / 2);
      if (n1 >= g.N) return;
      if (g.parts == 2) {
        tall_tile<WN / 2, 4, 3, 4, W_AUX>(g, m0, m_rows, n1, 0, 0, tall_smem);
      } else {
        const int upper = (m_rows + 31) / 32 * 16, m1 = part / 2 * upper;
        if (m1 < m_rows) tall_tile<WN / 2, 2, 5, 5, W_AUX>(g, m0 + m1, part / 2 ? m_rows - upper : upper, n1, 0, 0, tall_smem);
      }
      return;
    }
  }
  tall_tile<WN, MU, NA, NW, W_AUX>(g, m0, m_rows, n0, split, g.stagger ? nb : 0, tall_smem);
}

template <int WN, int MU, int NA, int NW, int W_AUX, bool PARTS = false> static int launch_tall(Tall g, int n_split, hipStream_t st) {
  using S = TileShape<WN, MU>;
  constexpr int LDS = PARTS ? 160 * 1024 : tile_lds<WN, MU, NA, NW>();
  static_assert(LDS <= 160 * 1024 && tile_lds<2, 4, 3, 4>() <= 160 * 1024 && tile_lds<2, 2, 5, 5>() <= 160 * 1024, "a compute unit's LDS");
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_tall_kernel<WN, MU, NA, NW, W_AUX, PARTS>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  if (e != hipSuccess) {
    set_error("gemm_tall: cannot have %d bytes of LDS: %s", LDS, hipGetErrorString(e));
    return 2;
  }
  g.mt = (int)(((long)g.M + S::ROWS - 1) / S::ROWS);
  g.nt = (int)(((long)g.N + S::CHANNELS - 1) / S::CHANNELS);
  g.share = ((g.M + g.mt - 1) / g.mt + 15) / 16 * 16;
  g.splits = n_split;
  const long tiles = (long)g.mt * g.nt;
  TL_REQUIRE(!PARTS || (g.whole % 8 == 0 && g.whole >= 0 && g.whole <= tiles), "gemm_tall: %d of %ld tiles whole (a multiple of 8)", g.whole, tiles);
  const long grid = PARTS ? g.whole + ((tiles - g.whole) * g.parts + 7) / 8 * 8 : (tiles * n_split + 7) / 8 * 8;
  TL_REQUIRE(grid * TILE_WAVES * WAVE < (1l << 32), "gemm_tall: M=%d N=%d have more tiles than a grid holds", g.M, g.N);
  gemm_tall_kernel<WN, MU, NA, NW, W_AUX, PARTS><<<(unsigned)grid, TILE_WAVES * WAVE, LDS, st>>>(g);
  TL_LAUNCH_CHECK("gemm_tall");
  return 0;
}

}  // namespace tl

using namespace tl;

// A [M, K] with rows lda apart, W [N, K] with rows ldw apart; K, lda, ldw multiples of 8, N of 4 (with a paired epilogue of 64).
// n_split == 1: C as in tl_gemm_bf16; more: C float [n_split][M][N] receives partial sums (epilogue 0), every split with one
// stage of 64 k at least.  rows, channels: the tile, one of 256, 224, 192, 160 x 256 and 256, 192, 128 x 128.  once: W is read by
// one tile of rows only (tiles of 128 channels mark its loads non-temporal; the rule has no such product in wider ones); stagger: tiles of other channels begin with other stages of K
// (K a multiple of 64, not cut).  parts: 0, or 2 or 4 (tiles of 256 channels, K not cut): the tiles behind the first `whole`, a
// multiple of 8, are cut into so many.
static int run_tall(Tall g, int rows, int channels, int n_split, int once, hipStream_t st) {
  const int M = g.M, N = g.N, K = g.K, lda = g.lda, ldw = g.ldw, stagger = g.stagger, whole = g.whole, parts = g.parts, epilogue = g.epi;
  const void *A = g.A, *W = g.W, *C = g.C;
  TL_REQUIRE(M > 0 && N > 0 && K > 0 && K % 8 == 0 && N % 4 == 0, "gemm_tall: bad sizes M=%d N=%d K=%d (K a multiple of 8, N of 4)", M, N, K);
  TL_REQUIRE(lda >= K && ldw >= K && lda % 8 == 0 && ldw % 8 == 0 && lda < (1 << 22) && ldw < (1 << 22),
             "gemm_tall: rows %d and %d apart for K=%d (multiples of 8 below 2^22)", lda, ldw, K);
  TL_REQUIRE(A && W && C && ((uintptr_t)A | (uintptr_t)W | (uintptr_t)C) % 16 == 0, "gemm_tall: operands must be 16-byte aligned");
  TL_REQUIRE(epilogue >= 0 && epilogue <= TALL_GATED && (n_split == 1 || epilogue == EPI_STORE), "gemm_tall: epilogue %d cannot go with %d splits", epilogue, n_split);
  TL_REQUIRE(!(is_pair(epilogue) || epilogue == TALL_GATED) || N % 64 == 0, "gemm_tall: the paired epilogue needs N=%d to be a multiple of 64", N);
  const int stages = (K + TILE_K - 1) / TILE_K, per = (stages + n_split - 1) / (n_split > 0 ? n_split : 1);
  TL_REQUIRE(n_split >= 1 && n_split <= 65535 && (long)(n_split - 1) * per < stages, "gemm_tall: %d splits of K=%d would leave one without a stage", n_split, K);
  TL_REQUIRE(!stagger || (n_split == 1 && K % TILE_K == 0), "gemm_tall: stages in turn need K=%d uncut and a multiple of %d", K, TILE_K);
  TL_REQUIRE(parts == 0 || ((parts == 2 || parts == 4) && n_split == 1 && channels == 256 && !once && !stagger && whole >= 0),
             "gemm_tall: tiles in %d parts (2 or 4, of 256 channels, K not cut)", parts);
  g.stages = per;
#define TL_TALL(R, CH, WN, MU, NA, NW)                                                         \
  if (rows == R && channels == CH) {                                                           \
    if (parts) return launch_tall<4, MU, 2, 3, 0, true>(g, n_split, st);                       \
    return launch_tall<WN, MU, NA, NW, 0>(g, n_split, st);                                     \
  }
  TL_TALL(256, 256, 4, 8, 2, 3)
  TL_TALL(224, 256, 4, 7, 2, 3)
  TL_TALL(192, 256, 4, 6, 2, 3)
  TL_TALL(160, 256, 4, 5, 3, 3)
#undef TL_TALL
#define TL_TALL(R, MU, NA, NW)                                                                 \
  if (rows == R && channels == 128)                                                            \
    return once ? launch_tall<2, MU, NA, NW, 2>(g, n_split, st) : launch_tall<2, MU, NA, NW, 0>(g, n_split, st);
  // (W, from memory, three stages ahead and A, from L2, two: 226 rows by 28,672, K = 4,096, 60 us; A three and W one ahead 71, A one and W five 70)
  TL_TALL(256, 4, 3, 4)
  TL_TALL(192, 3, 4, 4)
  TL_TALL(128, 2, 5, 5)
#undef TL_TALL
  TL_REQUIRE(false, "gemm_tall: no tiles of %d x %d", rows, channels);
}

extern "C" int tl_gemm_tall(const void* A, int lda, const void* W, int ldw, void* C, int M, int N, int K, int rows, int channels, int n_split,
                            int once, int stagger, int whole, int parts, int epilogue, hipStream_t st) {
  TL_REQUIRE(epilogue >= 0 && epilogue <= 5, "gemm_tall: unknown epilogue %d", epilogue);
  Tall g{};
  g.A = (const bf16*)A; g.W = (const bf16*)W; g.C = (float*)C;
  g.M = M; g.N = N; g.K = K; g.lda = lda; g.ldw = ldw;
  g.stagger = stagger; g.whole = whole; g.parts = parts;
  g.epi = epi_of(epilogue);
  return run_tall(g, rows, channels, n_split, once, st);
}

// The same with an expert's activation on the sums, times row_weight[m] (or null): gated == 0: C bfloat16 [M, N] = act(product) (codes
// of `UnaryAct`); gated == 1: W [gate | up], N / 2 rows each, C bfloat16 [M, N / 2] = act(gate, up) (`gated_value`; N a multiple of 64).
extern "C" int tl_gemm_tall_act(const void* A, int lda, const void* W, int ldw, void* C, int M, int N, int K, int rows, int channels, int once,
                                int stagger, int whole, int parts, int gated, int act_code, float act_a, float act_b, float limit, float alpha,
                                float shift, const float* row_weight, hipStream_t st) {
  TL_REQUIRE(act_code >= 0 && act_code <= 2, "gemm_tall_act: unknown activation %d", act_code);
  Tall g{};
  g.A = (const bf16*)A; g.W = (const bf16*)W; g.C = (float*)C;
  g.M = M; g.N = N; g.K = K; g.lda = lda; g.ldw = ldw;
  g.stagger = stagger; g.whole = whole; g.parts = parts;
  g.epi = Epi(gated ? TALL_GATED : TALL_UNARY);
  g.unary = UnaryAct{act_code, act_a, act_b};
  g.gate = GateTerms{limit, limit, alpha, shift, 0};
  g.row_weight = row_weight;
  return run_tall(g, rows, channels, 1, once, st);
}
