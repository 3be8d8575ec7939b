// C[M,N] (+)= A[M,K] * W[N,K]^T of 32-bit operands by tiles on the matrix cores, for more rows than gemm_plain.hip's kernels for few.
//
// v_mfma_f32_16x16x4_f32 adds its four products one after the other, each a fused multiply-add rounded to 32 bits (checked
// bit for bit against a chain of fmaf: ordinary numbers, 40 powers of two apart, denormals, infinities), at twice the rate of the
// vector pipes (138 TFLOP/s measured over the chip).  So the sums have the order, and the bits, of the plain path's other kernels: runs
// of K in ascending order, a group over its runs, the result over its groups.
// Microseconds, tiles on the vector pipes (gemm_plain.hip, which keep the operands that do not fit here) / these: N x K = 16,384 x 2,048 at
// 32 / 80 / 512 / 2,048 rows 48 / 47, 123 / 73, 569 / 332, 2,221 / 1,285 (107 TFLOP/s); 2,048 x 8,192 70 / 27, 75 / 40, 268 / 194, 1,031 / 631;
// 3,072 x 2,048 20 / 16, 34 / 23, 107 / 99, 397 / 258.  Up to 96 rows or so a unit has one workgroup, whose waves wait at a barrier
// a stage together: half of the matrix cores' rate.
#include "gemm_f32.hpp"

namespace tl {

constexpr int FK = 32;                            // k of a stage: 128 bytes of a row
constexpr int FROW = FK * 4;
constexpr int FN = 64;                            // channels of a tile, 16 a wave
constexpr int FWAVES = 8;                         // two on a SIMD, each with half of the rows
constexpr int F_ROWS = 8;                         // most blocks of 16 rows of a tile
constexpr int F_LDS = 79 * 1024;                  // two workgroups a compute unit

template <int MT> struct F32Shape {
  static constexpr int ROWS = 16 * MT + FN, STAGE = ROWS * FROW, LOADS = ROWS / 8, PER = (LOADS + FWAVES - 1) / FWAVES;
  static constexpr int FIT = (F_LDS - 1024) / STAGE, NS = FIT > 6 ? 6 : FIT, LDS = NS * STAGE + 1024;
  static_assert(NS >= 3 && (NS - 1) * PER <= 63, "stages under way");
};

struct F32Product {
  const float *A, *W;
  float* C;
  int M, N, K, lda, ldw, ldc;
  int m_tiles;                                    // tiles of rows
  long total;                                     // tiles
  int groups;                                     // a workgroup's groups of K
  int accumulate;
};

// MW blocks of 16 rows from block `first` of the tile on by 16 channels: a wave's share.
// A stage is two halves of 16 k.  While the products of a half are issued, the operands of the next come from LDS into other registers;
// one barrier a stage, between the halves: behind it every wave has all of the stage in registers, so that its place takes the loads of
// another, and the next stage is there.
template <int MT, int MW, bool DIRECT>
__device__ __forceinline__ void f32_tile(const F32Product& p, int m0, int n0, int first, int wave, unsigned char* smem) {
  using S = F32Shape<MT>;
  constexpr int SPARE = S::NS * S::STAGE;         // 1 KB that takes the loads of shares that do not exist
  constexpr int BLOCKS = MW > 0 ? MW : 1, HALF = BK / 4;
  const int lane = threadIdx.x % WAVE, li = lane % 16, kg = lane / 16, wn = wave % 4;
  const int L = run_length(p.K), group_len = PR * L;
  const int k_begin = (int)blockIdx.y * p.groups * group_len, k_end = min(p.K, k_begin + p.groups * group_len), n_t = (k_end - k_begin) / FK;

  const char* src[S::PER];
  int dst[S::PER];
#pragma unroll
  for (int x = 0; x < S::PER; ++x) {
    const int q = wave + FWAVES * x, r = 8 * q + lane / 8, c = (lane % 8) ^ (r / 2 % 8);
    const float* row = r < 16 * MT ? p.A + (size_t)min(m0 + r, p.M - 1) * p.lda : p.W + (size_t)min(n0 + r - 16 * MT, p.N - 1) * p.ldw;
    src[x] = reinterpret_cast<const char*>(row + k_begin) + c * 16;
    dst[x] = q < S::LOADS ? q * 1024 : -1;
  }
  const auto issue = [&](int i) {
    unsigned char* slot = smem + i % S::NS * S::STAGE;
#pragma unroll
    for (int x = 0; x < S::PER; ++x)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src[x] + (size_t)i * FROW),
                                       (__attribute__((address_space(3))) void*)(dst[x] >= 0 ? slot + dst[x] : smem + SPARE), 16, 0, 0);
  };
  f32x4 acc[BLOCKS], group[BLOCKS], sum[BLOCKS];
#pragma unroll
  for (int u = 0; u < MW; ++u) acc[u] = group[u] = sum[u] = f32x4{0.f, 0.f, 0.f, 0.f};
  // this lane's channels of C: n0 + 16 wn + 4 kg + r; its row of block u: m0 + 16 (first + u) + li
  const int n = n0 + wn * 16 + kg * 4;
  const auto store = [&](float* out, size_t ld, f32x4 (&v)[BLOCKS], bool add) {
    const bool whole = n + 4 <= p.N && ld % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0;
#pragma unroll
    for (int u = 0; u < MW; ++u) {
      const int m = m0 + (first + u) * 16 + li;
      if (m >= p.M) continue;
      float* c = out + (size_t)m * ld + n;
      if (whole) {
        *reinterpret_cast<f32x4*>(c) = add ? *reinterpret_cast<const f32x4*>(c) + v[u] : v[u];
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < p.N) c[r] = add ? c[r] + v[u][r] : v[u][r];
      }
    }
  };
  const auto read = [&](int i, int half, float (&w)[HALF], float (&a)[BLOCKS][HALF]) {
    const unsigned char* slot = smem + i % S::NS * S::STAGE + kg * 4;
#pragma unroll
    for (int s = 0; s < HALF; ++s) {
      const int c = ((half * HALF + s) ^ (li / 2)) * 16;
      w[s] = *reinterpret_cast<const float*>(slot + (16 * MT + wn * 16 + li) * FROW + c);
#pragma unroll
      for (int u = 0; u < MW; ++u) a[u][s] = *reinterpret_cast<const float*>(slot + ((first + u) * 16 + li) * FROW + c);
    }
  };
  int in_run = 0, in_group = 0, g = (int)blockIdx.y * p.groups;
  // the products of a half; `last`: of all of the workgroup's k (K's end is a stage's)
  const auto multiply = [&](const float (&w)[HALF], const float (&a)[BLOCKS][HALF], bool last) {
#pragma unroll
    for (int s = 0; s < HALF; ++s)
#pragma unroll
      for (int u = 0; u < MW; ++u) acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[s], a[u][s], acc[u], 0, 0, 0);
    in_run += BK;
    in_group += BK;
    if (in_run != L && !last) return;
    in_run = 0;
#pragma unroll
    for (int u = 0; u < MW; ++u) {
      group[u] += acc[u];
      acc[u] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    if (in_group != group_len && !last) return;
    in_group = 0;
    if constexpr (DIRECT) {
#pragma unroll
      for (int u = 0; u < MW; ++u) sum[u] += group[u];
    } else {
      store(p.C + (size_t)g * p.M * p.N, p.N, group, false);
      ++g;
    }
#pragma unroll
    for (int u = 0; u < MW; ++u) group[u] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  const auto meet = [&]() {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

#pragma unroll
  for (int i = 0; i < S::NS; ++i)
    if (i < n_t) issue(i);
  if (n_t >= S::NS) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S::NS - 1) * S::PER) : "memory");
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  meet();
  float w0[HALF], w1[HALF], a0[BLOCKS][HALF], a1[BLOCKS][HALF];
  read(0, 0, w0, a0);
  for (int i = 0; i < n_t; ++i) {
    read(i, 1, w1, a1);
    multiply(w0, a0, false);
    if (i + 1 < n_t) {
      // stage i + 1 has arrived for this wave when only those behind it are under way, and it has read stage i
      if (i + S::NS <= n_t) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((S::NS - 2) * S::PER) : "memory");
      else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      meet();
      if (i + S::NS < n_t) issue(i + S::NS);
      read(i + 1, 0, w0, a0);
    }
    multiply(w1, a1, i + 1 == n_t);
  }
  if constexpr (DIRECT) store(p.C, p.ldc, sum, p.accumulate != 0);
}

// A tile of 16 MT rows by 64 channels: both operands through a ring of stages in LDS (global_load_lds).  Waves w and w + 4 have the
// same 16 channels, the first the larger half of the blocks of rows, the second the rest: they lie on one SIMD, where one reads LDS while
// the other multiplies (four waves with all of the rows each and no half ahead: 96 rows of 16,384 x 2,048 105 us, so 83).  Within a
// row of a stage the 16-byte chunk c lies at place c ^ (row / 2 % 8): the 64 lanes of a read, 16 rows by four neighbouring k, fall on all
// of the banks.
// DIRECT: a workgroup goes through all groups of K and stores (or adds to) C; else through `groups` of them from
// blockIdx.y * groups on, and leaves each one's sums in C = parts [PG][M][N].
template <int MT, bool DIRECT>
__global__ void __launch_bounds__(FWAVES * WAVE)
gemm_f32_tiles_kernel(F32Product p) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char f32_smem[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  // each of the 8 XCDs (workgroups go round them) has a run of tiles of its own, a channel block's tiles of rows next to each other
  const long id = (long)blockIdx.z * gridDim.x + blockIdx.x, chunk = (p.total + 7) / 8, at = id % 8 * chunk + id / 8;
  if (id / 8 >= chunk || at >= p.total) return;
  const int n0 = (int)(at / p.m_tiles) * FN, m0 = (int)(at % p.m_tiles) * (16 * MT);
  if (MT % 2 == 0 || wave < 4) f32_tile<MT, (MT + 1) / 2, DIRECT>(p, m0, n0, wave / 4 * ((MT + 1) / 2), wave, f32_smem);
  else f32_tile<MT, MT / 2, DIRECT>(p, m0, n0, (MT + 1) / 2, wave, f32_smem);
}

// the groups' sums in their order
template <int V>
__global__ void __launch_bounds__(256)
gemm_f32_groups_kernel(const float* __restrict__ parts, float* __restrict__ C, int M, int N, int ldc, int accumulate) {
  typedef __attribute__((ext_vector_type(V))) float part;
  const size_t all = (size_t)M * N, e = ((size_t)blockIdx.x * 256 + threadIdx.x) * V;
  if (e >= all) return;
  part p[PG], t = {};
#pragma unroll
  for (int g = 0; g < PG; ++g) p[g] = *reinterpret_cast<const part*>(parts + g * all + e);
#pragma unroll
  for (int g = 0; g < PG; ++g) t += p[g];
  part* c = reinterpret_cast<part*>(C + e / N * ldc + e % N);
  *c = accumulate ? *c + t : t;
}

static int f32_rows(int M) {                      // blocks of 16 rows a tile, in equal shares
  const int blocks = (M + 15) / 16, tiles = (blocks + F_ROWS - 1) / F_ROWS;
  return (blocks + tiles - 1) / tiles;
}

bool f32_tiles_fit(const float* A, const float* W, int K, int lda, int ldw) {
  return K % FK == 0 && lda % 4 == 0 && ldw % 4 == 0 && ((uintptr_t)A | (uintptr_t)W) % 16 == 0;
}

// As few as give every compute unit a workgroup, if there are so many groups with something in them.
int f32_tiles_split(int M, int N, int K) {
  const long tiles = ((long)N + FN - 1) / FN * ((M + 16L * f32_rows(M) - 1) / (16 * f32_rows(M)));
  if (K % FK != 0 || (long)(PG - 1) * PR * run_length(K) >= K) return 1;
  int split = 1;
  while (split < PG && tiles * split < compute_units()) split *= 2;
  return split;
}

template <int MT>
static int launch_f32(const float* A, const float* W, float* C, float* parts, int M, int N, int K, int lda, int ldw, int ldc, int accumulate,
                      int split, hipStream_t st) {
  using S = F32Shape<MT>;
  const auto kernel = split > 1 ? gemm_f32_tiles_kernel<MT, false> : gemm_f32_tiles_kernel<MT, true>;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, S::LDS);
  if (e != hipSuccess) {
    set_error("gemm_f32: cannot have %d bytes of LDS: %s", S::LDS, hipGetErrorString(e));
    return 2;
  }
  const int m_tiles = (M + 16 * MT - 1) / (16 * MT);
  const long total = ((long)N + FN - 1) / FN * m_tiles, grid = (total + 7) / 8 * 8;
  TL_REQUIRE(total < (1l << 31), "gemm: M=%d N=%d have more tiles than a grid holds", M, N);
  const dim3 dims((unsigned)(grid < GRID_X ? grid : GRID_X), split, (unsigned)((grid + GRID_X - 1) / GRID_X));
  kernel<<<dims, FWAVES * WAVE, S::LDS, st>>>(F32Product{A, W, split > 1 ? parts : C, M, N, K, lda, ldw, ldc, m_tiles, total, PG / split, accumulate});
  TL_LAUNCH_CHECK("gemm_f32_tiles");
  if (split > 1) {
    const bool four = N % 4 == 0 && ldc % 4 == 0 && (uintptr_t)C % 16 == 0;
    const size_t all = (size_t)M * N / (four ? 4 : 1);
    const auto add = four ? gemm_f32_groups_kernel<4> : gemm_f32_groups_kernel<1>;
    add<<<(unsigned)((all + 255) / 256), 256, 0, st>>>(parts, C, M, N, ldc, accumulate);
    TL_LAUNCH_CHECK("gemm_f32_groups");
  }
  return 0;
}

int f32_tiles(const float* A, const float* W, float* C, float* parts, int M, int N, int K, int lda, int ldw, int ldc, int accumulate,
              hipStream_t st) {
  const int split = parts != nullptr ? f32_tiles_split(M, N, K) : 1;
  switch (f32_rows(M)) {
    case 1: return launch_f32<1>(A, W, C, parts, M, N, K, lda, ldw, ldc, accumulate, split, st);
    case 2: return launch_f32<2>(A, W, C, parts, M, N, K, lda, ldw, ldc, accumulate, split, st);
    case 3: return launch_f32<3>(A, W, C, parts, M, N, K, lda, ldw, ldc, accumulate, split, st);
    case 4: return launch_f32<4>(A, W, C, parts, M, N, K, lda, ldw, ldc, accumulate, split, st);
    case 5: return launch_f32<5>(A, W, C, parts, M, N, K, lda, ldw, ldc, accumulate, split, st);
    case 6: return launch_f32<6>(A, W, C, parts, M, N, K, lda, ldw, ldc, accumulate, split, st);
    case 7: return launch_f32<7>(A, W, C, parts, M, N, K, lda, ldw, ldc, accumulate, split, st);
    default: return launch_f32<8>(A, W, C, parts, M, N, K, lda, ldw, ldc, accumulate, split, st);
  }
}

}  // namespace tl
