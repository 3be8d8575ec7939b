// The inner loop of the products of many rows: a tile of a workgroup's rows of A by its rows of W over a run of K, both operands
// bfloat16 with K along memory, the sums in the matrix cores' layout.
//
// Eight waves, two on a SIMD: one wave alone issues 16x16x32 products at two thirds of the matrix cores' rate (1.57 against 2.3
// PFLOP/s over the chip), two side by side fill them, and what one spends on reading LDS the other multiplies.  The waves lie WM x WN
// over the tile, a wave has 16 MU rows of A and 64 rows of W.  Stages of 64 k (whole lines of 128 bytes) go from memory straight
// into two rings in LDS (global_load_lds), one for each operand, NA and NW stages long, so that the operand that comes from
// memory can be a stage further ahead than the one that L2 holds.  Within a row of a stage the 16-byte chunk c lies at place
// c ^ (row / 2 % 8): the 16 lanes that LDS serves at a time fall on all of its banks.
//
// A stage is two halves of 32 k.  While the products of a half are issued, the operands of the next half come from LDS into
// another set of registers, so that no product waits for a read; one barrier a stage, before the second half: behind
// it every wave has what it needs of the stage in registers, the places of the stage take the loads of a later one, and the
// next stage's are there to be read.  The order of reads, loads and products is pinned (sched_barrier): left to itself the
// compiler gathers the loads at the front, where both waves of a SIMD would wait for them.
//
// Measured for 256 x 256 rows and stages in both rings (K = 14,336): 1.07 us a stage with half of the chip's units at work (the
// products alone 0.88), 1.55 with all of them on numbers as they occur, 1.2 on zeros: there the chip's power is the bound, as it is
// for the BLAS library.
#pragma once
#include "common.hpp"

namespace tl {

constexpr int TILE_K = 64;                     // k of a stage
constexpr int TILE_ROW = TILE_K * 2;           // bytes of a row in a stage
constexpr int TILE_WAVES = 8;

template <int WN, int MU> struct TileShape {
  static constexpr int WM = TILE_WAVES / WN, ROWS = WM * MU * 16, CHANNELS = WN * 64;
  // loads a wave issues for a stage, of 8 rows each
  static constexpr int A_LOADS = ROWS / 8, A_PER = (A_LOADS + TILE_WAVES - 1) / TILE_WAVES, W_PER = CHANNELS / 64;
  static constexpr int A_SLOT = ROWS * TILE_ROW, W_SLOT = CHANNELS * TILE_ROW;
};
template <int WN, int MU, int NA, int NW> constexpr int tile_lds() {
  return NA * TileShape<WN, MU>::A_SLOT + NW * TileShape<WN, MU>::W_SLOT;
}

// Which 8 of the tile's rows of A (or W) load x of a wave takes, LOADS in all: wave + 8 x.  Where there are none left the wave takes
// the same again as another, even or odd like its own, since on that the places of the chunks go.
template <int LOADS> __device__ __forceinline__ int tile_load(int wave, int x) {
  const int q = wave + TILE_WAVES * x;
  return q < LOADS ? q : q - (LOADS >= TILE_WAVES ? TILE_WAVES : LOADS);
}

// acc[u][v][r] += the sum over stages t0 .. t0 + n_t - 1 for row wm * 16 MU + 16 u + lane % 16 of A's tile and row
// wn * 64 + 16 v + 4 (lane / 16) + r of W's.  a_at(x, at), w_at(x, at): byte `at` of this lane's row of load x (row
// lane / 8 of the eight of `tile_load`).
// first: the stage (from t0 on) it begins with, going round.  K: whole rows' length, a multiple of 8; the stage that holds K's
// end, if that is no multiple of 64, has to come last (first = 0).  n_t >= 1.
template <int WN, int MU, int NA, int NW, int W_AUX, typename AAt, typename WAt>
__device__ __forceinline__ void tile_loop(unsigned char* smem, AAt a_at, WAt w_at, int K, int t0, int n_t, int first, f32x4 (&acc)[MU][4]) {
  using S = TileShape<WN, MU>;
  constexpr int LOADS = S::A_PER + S::W_PER, W_RING = NA * S::A_SLOT, DEEP = NA > NW ? NA : NW;
  // A's loads of a turn go before W's where W's ring is the longer one, else behind: those still under way when a stage has
  // to be there are the last ones
  constexpr bool A_FIRST = NA <= NW;
  constexpr int AHEAD = NA < NW ? (NA - 2) * LOADS + S::W_PER : NA > NW ? (NW - 2) * LOADS + S::A_PER : (NA - 2) * LOADS;
  static_assert(NA >= 2 && NW >= 2 && AHEAD + LOADS <= 63, "a place to read and one to fill, and a count of six bits");
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE, li = lane % 16, kg = lane / 16;
  const int wm = wave / WN, wn = wave % WN;
  const int chunk = ((lane % 8) ^ (4 * wave + lane / 16) % 8) * 16;      // this lane's chunk of its rows, in bytes: the same for every load
  const int most = K * 2 - 16 - chunk;                                   // (past the end of a row its last chunk again, see `cut`)
  const auto bytes_at = [&](int i) { return (unsigned)(min((t0 + (i + first < n_t ? i + first : i + first - n_t)) * TILE_ROW, most) + chunk); };
  // places in the rings, in bytes: where a stage's operands lie, and where the next stage's do
  struct Place { int a, w; };
  const auto behind_of = [](Place p) {
    return Place{p.a + S::A_SLOT < NA * S::A_SLOT ? p.a + S::A_SLOT : 0, p.w + S::W_SLOT < NW * S::W_SLOT ? p.w + S::W_SLOT : 0};
  };
  const auto load_a = [&](int place, int x, unsigned at) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)a_at(x, at),
                                     (__attribute__((address_space(3))) void*)(smem + place + tile_load<S::A_LOADS>(wave, x) * 1024), 16, 0, 0);
  };
  const auto load_w = [&](int place, int x, unsigned at) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)w_at(x, at),
                                     (__attribute__((address_space(3))) void*)(smem + W_RING + place + (wave + TILE_WAVES * x) * 1024), 16, 0, W_AUX);
  };
  const int a_row = (wm * MU * 16 + li) * TILE_ROW, w_row = W_RING + (wn * 64 + li) * TILE_ROW;
  // read r of a half's MU + 4, W's first
  const auto read = [&](Place p, int half, int r, bf16x8 (&a)[MU], bf16x8 (&w)[4]) {
    const int c = ((half * 4 + kg) ^ (li / 2)) * 16;
    if (r < 4) w[r] = *reinterpret_cast<const bf16x8*>(smem + p.w + w_row + c + r * 16 * TILE_ROW);
    else a[r - 4] = *reinterpret_cast<const bf16x8*>(smem + p.a + a_row + c + (r - 4) * 16 * TILE_ROW);
  };
  constexpr int READS = MU + 4, PART = MU > 3 ? MU - 2 : 1;              // the last products cover the reads' way
  constexpr int READS_EACH = (READS + PART - 1) / PART, LOADS_EACH = (LOADS + MU - 1) / MU;
  // The products of a half; between them, if `more`, the reads of half rh at `from`, and with `la`, `lw` the loads of turn i into
  // `into`.
  const auto half = [&](const bf16x8 (&a)[MU], const bf16x8 (&w)[4], bool more, Place from, int rh, bf16x8 (&an)[MU], bf16x8 (&wn_)[4], bool la, bool lw,
                        int i, Place into) {
    const unsigned at_a = la ? bytes_at(i + NA) : 0, at_w = lw ? bytes_at(i + NW) : 0;
#pragma unroll
    for (int u = 0; u < MU; ++u) {
      if (more) {
#pragma unroll
        for (int r = u * READS_EACH; r < (u + 1) * READS_EACH && r < READS; ++r) read(from, rh, r, an, wn_);
      }
#pragma unroll
      for (int q = u * LOADS_EACH; q < (u + 1) * LOADS_EACH && q < LOADS; ++q) {
        if (A_FIRST ? q < S::A_PER : q >= S::W_PER) {
          if (la) load_a(into.a, A_FIRST ? q : q - S::W_PER, at_a);
        } else if (lw) {
          load_w(into.w, A_FIRST ? q - S::A_PER : q, at_w);
        }
      }
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        const int v = u % 2 ? 3 - i4 : i4;
        acc[u][v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[v], a[u], acc[u][v], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // this wave's reads have returned; as a builtin, so that the compiler knows and places no wait of its own behind the next read
  const auto reads_back = [&]() {
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_sched_barrier(0);
  };
  const auto meet = [&]() {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
#pragma unroll
  for (int e = -DEEP; e < 0; ++e) {                            // the turns before the first: stages 0 .. of both rings
    const auto fill_a = [&]() {
      if (e + NA >= 0 && e + NA < n_t) {
        const unsigned at = bytes_at(e + NA);
#pragma unroll
        for (int x = 0; x < S::A_PER; ++x) load_a((e + NA) * S::A_SLOT, x, at);
      }
    };
    if (A_FIRST) fill_a();
    if (e + NW >= 0 && e + NW < n_t) {
      const unsigned at = bytes_at(e + NW);
#pragma unroll
      for (int x = 0; x < S::W_PER; ++x) load_w((e + NW) * S::W_SLOT, x, at);
    }
    if (!A_FIRST) fill_a();
  }
  bf16x8 a0[MU], a1[MU], w0[4], w1[4];
  if (n_t >= DEEP) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(AHEAD + LOADS) : "memory");
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  meet();
  Place here{0, 0};
#pragma unroll
  for (int r = 0; r < READS; ++r) read(here, 0, r, a0, w0);
  reads_back();
  int i = 0;
  for (; i + DEEP < n_t; ++i) {
    const Place next = behind_of(here);
    half(a0, w0, true, here, 1, a1, w1, false, false, i, here);
    reads_back();
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(AHEAD) : "memory");         // stage i + 1 is here
    meet();
    half(a1, w1, true, next, 0, a0, w0, true, true, i, here);
    reads_back();
    here = next;
  }
  for (; i + 1 < n_t; ++i) {
    const Place next = behind_of(here);
    half(a0, w0, true, here, 1, a1, w1, false, false, i, here);
    reads_back();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    meet();
    half(a1, w1, true, next, 0, a0, w0, i + NA < n_t, i + NW < n_t, i, here);
    reads_back();
    here = next;
  }
  const int behind = (t0 + n_t) * TILE_K - K;                  // > 0: what lies past the end of K (a multiple of 8) counts as 0
  const auto cut = [&](int h, bf16x8 (&a)[MU]) {
    if (behind > 0 && (h * 4 + kg) * 8 >= TILE_K - behind) {
#pragma unroll
      for (int u = 0; u < MU; ++u)
#pragma unroll
        for (int j = 0; j < 8; ++j) a[u][j] = (bf16)0.f;
    }
  };
  cut(0, a0);
  half(a0, w0, true, here, 1, a1, w1, false, false, i, here);
  reads_back();
  cut(1, a1);
  half(a1, w1, false, here, 0, a0, w0, false, false, i, here);
}

}  // namespace tl
