// C[M,N] (+)= A[M,K] * W[N,K]^T with float accumulation in plain FMA: the
// product of the true 32-bit path, and the fallback for operand types that
// the MFMA kernels do not take.  Weights are row-major [out, in] as the
// checkpoint stores them (out[r] = sum_c W[r,c] x[c],
// src/loader/parameters.rs:551-594 of the reference).
//
// Every kernel here adds an output element in one order, which depends on K alone, so that a row's
// result does not depend on what else is in the batch: K is cut into 8 groups of 8 runs of `run_length(K)`
// channels; a run is summed over k in ascending order, a group over its runs, the result over its groups.
// (The runs are what lets few rows spread over the chip: a chain of 8,192 additions in one thread is the
// whole time of a product of one row.)
#include "gated.hpp"
#include "gemm_f32.hpp"

namespace tl {

// Few rows of floats: a workgroup of 8 waves has 8 outputs' rows of W and up to MR rows of A.  A wave has a group
// of K, its lanes the 64 pairs of an output and a run of the group; a lane's chain is one run long.  W comes in
// coalesced pieces, 128 bytes of each of the 64 pairs at a time through the wave's own part of LDS, and A's 128 bytes of the wave's 8
// runs with them; the next pieces are on their way in registers meanwhile.  (Loads come back in the order they were asked for: when
// a lane loaded its A where it used it, it waited for the next pieces of W with it.)  Bound by the stream of W.  N / 8 workgroups fill the
// chip from N = 2,048 on; tiles of 64 x 64 with a chain of all of K in a thread, which this replaced, made 32 workgroups there.
// Microseconds at one row, those tiles and so: N x K = 2,048 x 8,192 525 and 14.6, 2,048 x 2,048 130 and 5.6, 16,384 x 2,048 216 and
// 24.  At one / two / four rows with A loaded by each lane, and through LDS: 2,048 x 8,192 17.6 / 18.8 / 24.4 and 14.6 / 15.3 / 17.1, 4,096 x 14,336
// 45.7 / 52.2 / 66.2 and 39.6 / 40.3 / 47.6 (5.9 TB/s at one), 28,672 x 4,096 86.8 / 96.5 / 128.8 and 73.5 / 73.6 / 103 (6.4 TB/s), 3,072 x 2,048 7.3 / 8.4 /
// 11.4 and 6.6 / 7.3 / 11.  Two pieces ahead: 2,048 x 8,192 16.2 at one row, 17.6 at two, whose registers then last for one workgroup a
// compute unit only; three and four rows 19.1 and 18.6.
// LINES: W's loads take whole lines, each once, and are marked non-temporal (2,048 x 8,192 at 2 rows 20.0 us without, 18.2 with, A loaded by each lane).
constexpr int CHUNK = 32;                         // channels of a pair that a wave brings in at a time
constexpr int UNITS = CHUNK / 4;                  // of 16 bytes
template <int MR, bool ACCUMULATE, bool LINES>
__global__ void __launch_bounds__(512, 4)
gemm_plain_rows_kernel(const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C, int M, int N,
                       int K, int lda, int ldw, int ldc) {
  // a wave's pieces, 64 rows of W and 8 MR of A; unit u of W's row p lies at u ^ (p / 2) % 8, of A's run r at u ^ r: reads of 16 rows spread
  // over the banks.  Two rows' 80 KB are the most of which two workgroups lie on a compute unit
  __shared__ f32x4 stage[PG][(64 + MR * PR) * UNITS];
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const long first_n = ((long)blockIdx.z * gridDim.x + blockIdx.x) * 8;
  if (first_n >= N) return;
  const int n0 = (int)first_n, m0 = blockIdx.y * MR;
  const int L = run_length(K);
  const int rows = min(MR, M - m0);
  float acc[MR];
#pragma unroll
  for (int m = 0; m < MR; ++m) acc[m] = 0.f;

  // a load brings 128 bytes of 8 pairs: pair 8 i + lane / 8 (output lane / 8 of run i), 4 channels from 4 (lane % 8); of A those of run lane / 8
  const int l8 = lane / 8, lu = lane % 8, lq = lu * 4, ln = n0 + l8;
  const float* wp = W + (size_t)min(ln, N - 1) * ldw;
  f32x4 w[8], a[MR];
  const auto fetch = [&](int at) {
    const int off = at + lq, ka = (wave * PR + l8) * L + off;
#pragma unroll
    for (int m = 0; m < MR; ++m) {
      a[m] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (off < L && ka < K) a[m] = *(const f32x4*)(A + (size_t)(m0 + min(m, rows - 1)) * lda + ka);     // (K is a multiple of 4)
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int k = (wave * PR + i) * L + off;
      w[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (off < L && k < K && ln < N) w[i] = LINES ? __builtin_nontemporal_load((const f32x4*)(wp + k)) : *(const f32x4*)(wp + k);
    }
  };
  f32x4* mine = stage[wave];
  f32x4* mine_a = mine + 64 * UNITS;
  fetch(0);
  for (int at = 0; at < L; at += CHUNK) {
#pragma unroll
    for (int m = 0; m < MR; ++m) mine_a[(m * PR + l8) * UNITS + (lu ^ l8)] = a[m];
#pragma unroll
    for (int i = 0; i < 8; ++i) mine[(i * 8 + l8) * UNITS + (lu ^ ((i * 8 + l8) / 2 % 8))] = w[i];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (at + CHUNK < L) fetch(at + CHUNK);
    const int todo = min(UNITS, (L - at) / 4);    // (a run is a multiple of 16 long; what lies past K is 0 times 0)
    const int p = l8 * 8 + lu;                    // this lane's pair: output lane % 8, run lane / 8
#pragma unroll 2
    for (int u = 0; u < todo; ++u) {
      const f32x4 wv = mine[p * UNITS + (u ^ (p / 2 % 8))];
#pragma unroll
      for (int m = 0; m < MR; ++m) {
        const f32x4 av = mine_a[(m * PR + l8) * UNITS + (u ^ l8)];
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[m] = fmaf(av[j], wv[j], acc[m]);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
  // the runs of a group in order, then the groups, whose sums take the place of their wave's pieces
#pragma unroll
  for (int m = 0; m < MR; ++m) {
    float g = 0.f;
#pragma unroll
    for (int i = 0; i < PR; ++i) g += __shfl(acc[m], i * 8 + lane % 8, WAVE);
    if (lane < 8) reinterpret_cast<float*>(mine)[m * 8 + lane] = g;
  }
  __syncthreads();
  const int m = threadIdx.x / 8, n = n0 + threadIdx.x % 8;
  if (m < rows && n < N) {
    float t = 0.f;
#pragma unroll
    for (int g = 0; g < PG; ++g) t += reinterpret_cast<const float*>(stage[g])[m * 8 + threadIdx.x % 8];
    float* c = C + (size_t)(m0 + m) * ldc + n;
    *c = ACCUMULATE ? *c + t : t;
  }
}

// The same bits for one to four rows, K up to 2,048 and many outputs: a workgroup goes through a run of eights of outputs, the next
// eights' pieces under way while it sums the last's, and a lane keeps its run of A, one piece long, in registers.  With an
// eight a workgroup every workgroup waits for memory once and does nothing meanwhile, and brings A for each.  One / two rows,
// an eight a workgroup and so: 16,384 x 2,048 24.0 / 25.3 and 24.4 / 25.2 us, 32,000 x 2,048 43.3 / 46.2 and 44.1 / 44.5 (5.9 TB/s), 16,384 x 1,024 16.6 / 17.3 and
// 15.7 / 17.6; three / four rows, of which one workgroup lies on a compute unit, 37.8 / 40.7 and 26.6 / 26.1, 69.4 / 74.6 and 46.6 / 45.9.  With fewer
// eights than workgroups there is nothing to go on to (3,072 x 2,048 7.3 us at two rows, 9.3 so).
// At one row two workgroups of 128 registers lie on a compute unit; with more rows' A it is one, of at most 256, which fetches two eights
// ahead where the registers last (16,384 x 2,048: two rows 29.6 us with 512 workgroups and one eight ahead, 27.9 with 256, 26.2 with two
// ahead; four rows 30.1 and 25.8 with 256, 45 with two ahead, which spills).
//
// Around the product it can do what stands next to it in a step of single tokens, with the bits of the kernels of their own:
//   * the RMS norm of A's rows (`rmsnorm_reg_kernel`'s sums), by every workgroup for itself while its first weights are under way;
//   * PAIR: act(gate) * up, an eight being four gates and the four ups that belong to them;
//   * ROPE: the rotation of q and k, q into its rows and k, v into their pages (`rope_commit_kernel`); an eight is four pairs of channels.
// Each of these was a launch that moved some KB.  Microseconds at one / two / four rows, launches of their own and so: norm, 16,384 x
// 2,048 and gate 31.6 / 31.4 / 31.1 and 26.9 / 28.8 / 30.1; norm, 3,072 x 2,048 and rotation 12.5 / 14.0 / 17.8 and 9.8 / 11.1 / 13.0; at
// K = 1,024, 8,192 outputs 14.3 / 17.0 / 17.1 and 11.5 / 14.2 / 15.0.
constexpr int ROWS_WORKGROUPS = 512;
constexpr int short_ahead(int mr) { return mr == 2 || mr == 3 ? 2 : 1; }
constexpr int short_workgroups(int mr) { return mr == 1 ? ROWS_WORKGROUPS : ROWS_WORKGROUPS / 2; }
enum { DO_STORE, DO_ADD, DO_PAIR, DO_ROPE };
struct Around {
  const float* norm_w;                            // [K], or null: A's rows as they are
  float eps;
  int act;                                        // PAIR: W is [gate | up] by rows, C [M, N / 2]
  ActConstants constants;
  const int* row_pos;                             // ROPE: W is [q | k | v] by rows
  Rotation rot;
  const int* table;
  int table_stride, ring_pages, nq, nkv, d;
  float *q, *pages;
};
template <int MR, int DO, bool LINES>
__global__ void __launch_bounds__(512, MR == 1 ? 4 : 2)
gemm_plain_short_kernel(const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C, int N, int K, int lda, int ldw,
                        int ldc, Around f) {
  __shared__ float stage[PG][64][CHUNK + 4];      // rows 144 bytes apart: 16-byte reads of 64 rows spread over the banks
  __shared__ float sums[2][PG][MR][8];            // of this eight, and of the one before, which others may still read
  __shared__ float squares[MR][4];
  constexpr int AHEAD = short_ahead(MR);
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const long eights = (N - 1) / 8 + 1;
  const int from = (int)(blockIdx.x * eights / gridDim.x), to = (int)((blockIdx.x + 1) * eights / gridDim.x);
  const int L = run_length(K);                    // at most CHUNK
  const int run = lane / 8;                       // of this lane's pair: output lane % 8, run lane / 8
  const int k0 = (wave * PR + run) * L;
  // the row of W of an eight's output o; ROPE: pair 4 (eight % (d / 8)) + o % 4 of a head, its first channel or its second
  const auto row_of = [&](int eight, int o) {
    if constexpr (DO == DO_PAIR) return o < 4 ? 4 * eight + o : N / 2 + 4 * eight + o - 4;
    if constexpr (DO == DO_ROPE) {
      const int per = f.d / 8, head = eight / per;
      int a, b;
      pair_channels((eight - head * per) * 4 + o % 4, f.rot.rotary_dim, f.rot.interleaved, a, b);
      return head * f.d + (o < 4 ? a : b);
    }
    return eight * 8 + o;
  };
  // a load brings 128 bytes of 8 pairs: pair 8 i + lane / 8 (output lane / 8 of run i), 4 channels from 4 (lane % 8)
  const int lq = (lane % 8) * 4;
  f32x4 next[AHEAD][8];
  const auto fetch = [&](f32x4 (&into)[8], int eight) {
    const int ln = row_of(eight, lane / 8);
    const float* wp = W + (size_t)min(ln, N - 1) * ldw;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int k = (wave * PR + i) * L + lq;
      into[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (lq < L && k < K && ln < N) into[i] = LINES ? __builtin_nontemporal_load((const f32x4*)(wp + k)) : *(const f32x4*)(wp + k);
    }
  };
#pragma unroll
  for (int b = 0; b < AHEAD; ++b)
    if (from + b < to) fetch(next[b], from + b);
  // ROPE: the sine and cosine that the thread of output threadIdx.x % 8 of row threadIdx.x / 8 needs at the end of an eight
  const int row = threadIdx.x / 8, out = threadIdx.x % 8;
  float sn = 0.f, cs = 1.f;
  int pos = 0, page = 0;
  if (DO == DO_ROPE && row < MR) {
    pos = f.row_pos[row];
    page = f.table[(size_t)row * f.table_stride + (pos / PAGE) % f.ring_pages];
  }
  const auto angle = [&](int eight) {
    if (row >= MR) return;
    const int per = f.d / 8, head = eight / per, pair = (eight - head * per) * 4 + out % 4;
    if (head < f.nq + f.nkv && 2 * pair < f.rot.rotary_dim) sincosf(f.rot.inv_freq[pair] * (float)pos, &sn, &cs);
  };
  const float* a_rows = A;
  int a_stride = lda;
  if (DO >= DO_PAIR && f.norm_w != nullptr) {      // four waves a row; the normed rows take the stage's place for a while
    constexpr int MINE = (MR + 1) / 2;
    const int t = threadIdx.x % 256, nv = K / 4;  // (K is at most 2,048)
    const float4* wr = reinterpret_cast<const float4*>(f.norm_w);
    float4 v[MINE][2], g[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
      if (t + 256 * i < nv) g[i] = wr[t + 256 * i];
#pragma unroll
    for (int h = 0; h < MINE; ++h) {
      const int m = 2 * h + wave / 4;
      if (m >= MR) continue;
      const float4* xr = reinterpret_cast<const float4*>(A + (size_t)m * lda);
      float ss = 0.f;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int c = t + 256 * i;
        if (c < nv) {
          v[h][i] = xr[c];
          ss += v[h][i].x * v[h][i].x + v[h][i].y * v[h][i].y + v[h][i].z * v[h][i].z + v[h][i].w * v[h][i].w;
        }
      }
      ss = wave_sum(ss);
      if (lane == 0) squares[m][wave % 4] = ss;
    }
    __syncthreads();
    float* y = &stage[0][0][0];
#pragma unroll
    for (int h = 0; h < MINE; ++h) {
      const int m = 2 * h + wave / 4;
      if (m >= MR) continue;
      float r = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) r += squares[m][i];
      const float rms = sqrtf(r / (float)K + f.eps);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int c = t + 256 * i;
        if (c < nv)
          *reinterpret_cast<float4*>(y + m * K + 4 * c) =
              make_float4((v[h][i].x / rms) * g[i].x, (v[h][i].y / rms) * g[i].y, (v[h][i].z / rms) * g[i].z, (v[h][i].w / rms) * g[i].w);
      }
    }
    __syncthreads();
    a_rows = y;
    a_stride = K;
  }
  f32x4 a[MR][CHUNK / 4];                         // (what lies past the run or past K is 0 times 0)
#pragma unroll
  for (int q = 0; q < CHUNK / 4; ++q)
#pragma unroll
    for (int m = 0; m < MR; ++m)
      a[m][q] = 4 * q < L && k0 + 4 * q < K ? *(const f32x4*)(a_rows + (size_t)m * a_stride + k0 + 4 * q) : f32x4{0.f, 0.f, 0.f, 0.f};
  if (DO >= DO_PAIR && f.norm_w != nullptr) __syncthreads();
  if (DO == DO_ROPE && from < to) angle(from);
  const auto go = [&](f32x4 (&pieces)[8], int eight) {
#pragma unroll
    for (int i = 0; i < 8; ++i) *(f32x4*)&stage[wave][i * 8 + lane / 8][lq] = pieces[i];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (eight + AHEAD < to) fetch(pieces, eight + AHEAD);
    float acc[MR];
#pragma unroll
    for (int m = 0; m < MR; ++m) acc[m] = 0.f;
#pragma unroll
    for (int q = 0; q < CHUNK / 4; ++q) {
      const f32x4 w = *(const f32x4*)&stage[wave][run * 8 + lane % 8][4 * q];
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int m = 0; m < MR; ++m) acc[m] = fmaf(a[m][q][j], w[j], acc[m]);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    // the runs of a group in order, then the groups
    float (*mine)[MR][8] = sums[(eight - from) % 2];
#pragma unroll
    for (int m = 0; m < MR; ++m) {
      float g = 0.f;
#pragma unroll
      for (int i = 0; i < PR; ++i) g += __shfl(acc[m], i * 8 + lane % 8, WAVE);
      if (lane < 8) mine[wave][m][lane] = g;
    }
    __syncthreads();
    const int n = row_of(eight, out);
    if (row < MR && n < N) {
      float t = 0.f;
#pragma unroll
      for (int g = 0; g < PG; ++g) t += mine[g][row][out];
      if constexpr (DO == DO_PAIR) {
        const float up = __shfl_xor(t, 4, WAVE);
        if (out < 4) C[(size_t)row * ldc + n] = gate_times_up(t, up, f.act, f.constants);
      } else if constexpr (DO == DO_ROPE) {
        const float other = __shfl_xor(t, 4, WAVE);
        const int head = n / f.d, c = n - head * f.d, pair = (eight - head * (f.d / 8)) * 4 + out % 4;
        if (head < f.nq + f.nkv && 2 * pair < f.rot.rotary_dim) {
          float ra, rb;
          rotate_pair(out < 4 ? t : other, out < 4 ? other : t, cs, sn, ra, rb);
          t = out < 4 ? ra : rb;
        }
        float* kd = f.pages + (size_t)page * 2 * f.nkv * PAGE * f.d;
        const int r = pos % PAGE;
        if (head < f.nq) f.q[((size_t)row * f.nq + head) * f.d + c] = t;
        else if (head < f.nq + f.nkv) kd[((size_t)(head - f.nq) * PAGE + r) * f.d + c] = t;
        else kd[(size_t)f.nkv * PAGE * f.d + ((size_t)(head - f.nq - f.nkv) * f.d + c) * PAGE + r] = t;
      } else {
        float* c = C + (size_t)row * ldc + n;
        *c = DO == DO_ADD ? *c + t : t;
      }
    }
    if (DO == DO_ROPE && eight + 1 < to) angle(eight + 1);
  };
  for (int eight = from; eight < to; eight += AHEAD)
#pragma unroll
    for (int b = 0; b < AHEAD; ++b)
      if (eight + b < to) go(next[b], eight + b);
}

// 32 x 32 outputs a workgroup of 8 waves, each with a group of K and 4 x 4 outputs a lane, operands through the wave's
// own part of LDS, the groups' sums through LDS at the end.  16 multiply-adds for two 16-byte reads of LDS a lane: the
// vector pipes and LDS are about as busy as each other.  Eight times the waves of tiles of 64 x 64 with a thread's
// chain over all of K for a product of the same size, and faster at every size measured, 1 to 8,192 rows:
// N x K = 2,048 x 8,192 at 64 rows 76 us (563 with those), at 1,024 rows 582 (1,259), at 2,048 1,040 (1,790); 16,384 x
// 2,048 at 64 rows 78 (320), at 2,048 2,210 (3,600); bfloat16 4,096 x 4,097 at 2,048 rows 1,175 (1,373).
// VEC: rows of both operands may be read four channels at a time; else a channel a lane, 16 lanes along a row.
constexpr int GT = 32, GK = 16;
template <typename TA, typename TW, bool VEC, bool ACCUMULATE>
__global__ void __launch_bounds__(512)
gemm_plain_kernel(const TA* __restrict__ A, const TW* __restrict__ W, float* __restrict__ C, int M, int N,
                  int K, int lda, int ldw, int ldc) {
  __shared__ float shared[PG * 2 * GK * (GT + 4)];
  static_assert(PG * 2 * GK * (GT + 4) >= PG * GT * GT, "the sums of the groups take the operands' place");
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const unsigned tiles_n = (N + GT - 1) / GT, tile = blockIdx.y * gridDim.x + blockIdx.x;
  if (tile >= tiles_n * ((M + GT - 1) / GT)) return;
  const int m0 = (int)(tile / tiles_n) * GT, n0 = (int)(tile % tiles_n) * GT;
  float (*As)[GT + 4] = (float (*)[GT + 4])(shared + wave * 2 * GK * (GT + 4));
  float (*Ws)[GT + 4] = As + GK;
  const int tx = lane % 8, ty = lane / 8;
  const int L = run_length(K), first = wave * PR * L;
  float group[4][4], acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) group[i][j] = acc[i][j] = 0.f;
  // loads: rows lr, lr + RS, ..., VW channels from lk
  constexpr int VW = VEC ? 4 : 1, RS = WAVE * VW / GK, LOADS = GT / RS;
  const int lr = lane / (GK / VW), lk = lane % (GK / VW) * VW;
  typedef __attribute__((ext_vector_type(VW))) TA part_a;
  typedef __attribute__((ext_vector_type(VW))) TW part_w;
  part_a na[LOADS];                                // as they come: a conversion here would wait for the load
  part_w nw[LOADS];
  const auto fetch = [&](int k) {
#pragma unroll
    for (int h = 0; h < LOADS; ++h) {
      const int m = m0 + lr + RS * h, n = n0 + lr + RS * h;
      na[h] = m < M && k < K ? *(const part_a*)(A + (size_t)min(m, M - 1) * lda + k) : part_a{};
      nw[h] = n < N && k < K ? *(const part_w*)(W + (size_t)min(n, N - 1) * ldw + k) : part_w{};
    }
  };
  const int end = min(K, first + PR * L);
  fetch(first + lk);
  int in_run = 0;
  for (int k0 = first; k0 < end; k0 += GK) {
#pragma unroll
    for (int h = 0; h < LOADS; ++h)
#pragma unroll
      for (int j = 0; j < VW; ++j) {
        As[lk + j][lr + RS * h] = to_f32((TA)na[h][j]);
        Ws[lk + j][lr + RS * h] = to_f32((TW)nw[h][j]);
      }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (k0 + GK < end) fetch(k0 + GK + lk);
#pragma unroll
    for (int kk = 0; kk < GK; ++kk) {
      const f32x4 a = *(const f32x4*)&As[kk][ty * 4], b = *(const f32x4*)&Ws[kk][tx * 4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    in_run += GK;
    if (in_run == L || k0 + GK >= end) {
      in_run = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          group[i][j] += acc[i][j];
          acc[i][j] = 0.f;
        }
    }
  }
  __syncthreads();
  float* sums = shared + wave * GT * GT;
#pragma unroll
  for (int i = 0; i < 4; ++i) *(f32x4*)&sums[(ty * 4 + i) * GT + tx * 4] = f32x4{group[i][0], group[i][1], group[i][2], group[i][3]};
  __syncthreads();
  for (int e = threadIdx.x; e < GT * GT; e += 512) {
    const int m = m0 + e / GT, n = n0 + e % GT;
    if (m >= M || n >= N) continue;
    float t = 0.f;
#pragma unroll
    for (int g = 0; g < PG; ++g) t += shared[g * GT * GT + e];
    float* c = C + (size_t)m * ldc + n;
    *c = ACCUMULATE ? *c + t : t;
  }
}

template <typename TA, typename TW, bool VEC>
static int launch_tiles(const TA* A, const TW* W, float* C, int M, int N, int K, int lda, int ldw, int ldc,
                        int accumulate, hipStream_t st) {
  const long tiles = (long)((N + GT - 1) / GT) * ((M + GT - 1) / GT);
  TL_REQUIRE(tiles < (1l << 31), "gemm: M=%d N=%d have more tiles than a grid holds", M, N);
  const dim3 grid((unsigned)(tiles < GRID_X ? tiles : GRID_X), (unsigned)((tiles + GRID_X - 1) / GRID_X));
  if (accumulate)
    gemm_plain_kernel<TA, TW, VEC, true><<<grid, 512, 0, st>>>(A, W, C, M, N, K, lda, ldw, ldc);
  else
    gemm_plain_kernel<TA, TW, VEC, false><<<grid, 512, 0, st>>>(A, W, C, M, N, K, lda, ldw, ldc);
  TL_LAUNCH_CHECK("gemm_plain");
  return 0;
}

// gemm_plain_short_kernel's sizes (of one to four rows)
static bool goes_on(int N, int K) { return run_length(K) <= CHUNK && ((long)N + 7) / 8 > ROWS_WORKGROUPS; }

// (a run that is no multiple of 32 channels, or rows off whole lines, would take lines in halves: those are to stay in the caches)
static bool whole_lines(const float* W, int K, int ldw) { return ldw % 32 == 0 && run_length(K) % 32 == 0 && (uintptr_t)W % 128 == 0; }

// one to four rows of K up to 2,048 with what `f` does around the product
template <int DO>
static int launch_around(const char* what, const float* A, const float* W, float* C, int M, int N, int K, int ldc, const Around& f, hipStream_t st) {
  TL_REQUIRE(M > 0 && M <= 4 && N > 0 && K > 0 && K % 4 == 0 && run_length(K) <= CHUNK, "%s: M=%d N=%d K=%d (one to four rows of at most %d channels)", what, M,
             N, K, CHUNK * PG * PR);
  TL_REQUIRE(A && W && ((uintptr_t)A | (uintptr_t)W | (uintptr_t)f.norm_w) % 16 == 0, "%s: operands must be 16-byte aligned", what);
  const int grid = (int)min(((long)N + 7) / 8, (long)short_workgroups(M));
  const bool lines = whole_lines(W, K, K);
#define TL_AROUND(MR)                                                                                            \
  do {                                                                                                           \
    if (lines) gemm_plain_short_kernel<MR, DO, true><<<grid, 512, 0, st>>>(A, W, C, N, K, K, K, ldc, f);          \
    else gemm_plain_short_kernel<MR, DO, false><<<grid, 512, 0, st>>>(A, W, C, N, K, K, K, ldc, f);               \
  } while (0)
  if (M == 1) TL_AROUND(1);
  else if (M == 2) TL_AROUND(2);
  else if (M == 3) TL_AROUND(3);
  else TL_AROUND(4);
#undef TL_AROUND
  TL_LAUNCH_CHECK(what);
  return 0;
}

template <int MR>
static int launch_rows(const float* A, const float* W, float* C, int M, int N, int K, int lda, int ldw, int ldc,
                       int accumulate, hipStream_t st) {
  const long groups = ((long)N + 7) / 8;
  if constexpr (MR <= 4) {
    const bool lines = whole_lines(W, K, ldw);
    if (goes_on(N, K) && M == MR) {
#define TL_SHORT(DO, LN) gemm_plain_short_kernel<MR, DO, LN><<<short_workgroups(MR), 512, 0, st>>>(A, W, C, N, K, lda, ldw, ldc, Around{})
      if (accumulate && lines) TL_SHORT(DO_ADD, true);
      else if (accumulate) TL_SHORT(DO_ADD, false);
      else if (lines) TL_SHORT(DO_STORE, true);
      else TL_SHORT(DO_STORE, false);
#undef TL_SHORT
      TL_LAUNCH_CHECK("gemm_plain_short");
      return 0;
    }
    if (lines && MR <= 2) {
      const dim3 grid((unsigned)(groups < GRID_X ? groups : GRID_X), 1, (unsigned)((groups + GRID_X - 1) / GRID_X));
      if (accumulate) gemm_plain_rows_kernel<MR, true, true><<<grid, 512, 0, st>>>(A, W, C, M, N, K, lda, ldw, ldc);
      else gemm_plain_rows_kernel<MR, false, true><<<grid, 512, 0, st>>>(A, W, C, M, N, K, lda, ldw, ldc);
      TL_LAUNCH_CHECK("gemm_plain_rows");
      return 0;
    }
  }
  const dim3 grid((unsigned)(groups < GRID_X ? groups : GRID_X), (M + MR - 1) / MR, (unsigned)((groups + GRID_X - 1) / GRID_X));
  if (accumulate)
    gemm_plain_rows_kernel<MR, true, false><<<grid, 512, 0, st>>>(A, W, C, M, N, K, lda, ldw, ldc);
  else
    gemm_plain_rows_kernel<MR, false, false><<<grid, 512, 0, st>>>(A, W, C, M, N, K, lda, ldw, ldc);
  TL_LAUNCH_CHECK("gemm_plain_rows");
  return 0;
}

// The kernel for few rows reads W once for every 8 rows and has a thread's chain 64 times shorter than K.  Against it, microseconds
// (rows / tiles): the tiles on the matrix cores (`fit`), N x K = 2,048 x 2,048 at 8 rows 8.9 / 11, 3,072 x 2,048 at 4 11 / 12, at 6 14.0 / 13.3,
// 2,048 x 8,192 at 4 17 / 26, at 6 19.5 / 22.5, at 8 20.2 / 22.3, 4,096 x 4,096 at 6 22.8 / 22.5, at 8 23.0 / 22.6, 4,096 x 14,336 at 4 47 / 62, at 6 54 /
// 62, at 8 56 / 62, 28,672 x 4,096 at 6 134 / 103; the tiles on the vector pipes, 2,048 x 8,192 at 16 rows 52 / 68, at 32 96 / 72 (with A loaded by
// each lane); 3,072 x 2,048 at 16 21 / 19; 4,096 x 14,336 at 16 197 / 123; 16,384 x 2,048 at 4 41 / 36 (of up to four rows wide outputs are
// `goes_on`'s).
static bool few_rows(int M, int N, int K, bool fit) {
  if (fit) return M <= 4 || (M <= 8 && (long)M * N <= (K <= 4096 ? 16384 : 32768));
  return M <= 2 || (M <= 16 && (long)M * N <= 32768);
}

template <typename TA, typename TW>
static int launch_plain(const void* Av, const void* Wv, float* C, float* parts, int M, int N, int K, int lda, int ldw,
                        int ldc, int accumulate, hipStream_t st) {
  const TA* A = (const TA*)Av;
  const TW* W = (const TW*)Wv;
  const bool vec = K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && (uintptr_t)A % (4 * sizeof(TA)) == 0 &&
                   (uintptr_t)W % (4 * sizeof(TW)) == 0;
  if (!vec) return launch_tiles<TA, TW, false>(A, W, C, M, N, K, lda, ldw, ldc, accumulate, st);
  if constexpr (sizeof(TA) == 4 && sizeof(TW) == 4) {
    const bool fit = f32_tiles_fit(A, W, K, lda, ldw);
    if (few_rows(M, N, K, fit) || (M <= 4 && goes_on(N, K))) {
      if (M == 1) return launch_rows<1>(A, W, C, M, N, K, lda, ldw, ldc, accumulate, st);
      if (M == 2) return launch_rows<2>(A, W, C, M, N, K, lda, ldw, ldc, accumulate, st);
      if (M == 3) return launch_rows<3>(A, W, C, M, N, K, lda, ldw, ldc, accumulate, st);
      if (M <= 4) return launch_rows<4>(A, W, C, M, N, K, lda, ldw, ldc, accumulate, st);
      return launch_rows<8>(A, W, C, M, N, K, lda, ldw, ldc, accumulate, st);
    }
    if (fit) return f32_tiles(A, W, C, parts, M, N, K, lda, ldw, ldc, accumulate, st);
  }
  return launch_tiles<TA, TW, true>(A, W, C, M, N, K, lda, ldw, ldc, accumulate, st);
}

}  // namespace tl

using namespace tl;

constexpr int MOST_ROWS = 65535 * 64;      // what callers have always been held to; the tiles' own limit is `launch_tiles`'

// The floats of scratch that a product of 32-bit operands of these sizes can use (it goes without, but slower).
extern "C" long long tl_gemm_plain_parts(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0 || few_rows(M, N, K, true) || f32_tiles_split(M, N, K) == 1) return 0;
  return (long long)PG * M * N;
}

// parts: scratch of n_parts floats (null or too few: none), see tl_gemm_plain_parts.
extern "C" int tl_gemm_plain(const void* A, int a_dt, const void* W, int w_dt, float* C, float* parts, long long n_parts, int M, int N,
                             int K, int lda, int ldw, int ldc, int accumulate, hipStream_t st) {
  TL_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm: bad sizes M=%d N=%d K=%d", M, N, K);
  TL_REQUIRE(lda >= K && ldw >= K && ldc >= N, "gemm: leading dimensions lda=%d ldw=%d ldc=%d too small "
             "for K=%d N=%d", lda, ldw, ldc, K, N);
  TL_REQUIRE(M <= MOST_ROWS, "gemm: M=%d, products have at most %d rows", M, MOST_ROWS);
  if (M == 0) return 0;
  if (n_parts < (long long)PG * M * N || (uintptr_t)parts % 16 != 0) parts = nullptr;
  if (a_dt == DT_F32 && w_dt == DT_F32)
    return launch_plain<float, float>(A, W, C, parts, M, N, K, lda, ldw, ldc, accumulate, st);
  if (a_dt == DT_BF16 && w_dt == DT_BF16)
    return launch_plain<bf16, bf16>(A, W, C, parts, M, N, K, lda, ldw, ldc, accumulate, st);
  if (a_dt == DT_BF16 && w_dt == DT_F32)
    return launch_plain<bf16, float>(A, W, C, parts, M, N, K, lda, ldw, ldc, accumulate, st);
  if (a_dt == DT_F32 && w_dt == DT_BF16)
    return launch_plain<float, bf16>(A, W, C, parts, M, N, K, lda, ldw, ldc, accumulate, st);
  TL_REQUIRE(false, "gemm: unknown dtype codes a=%d w=%d", a_dt, w_dt);
}

// out[m, i] = act(g_i) * u_i of g|u = norm(A[m]) W^T (norm_w null: of A itself), W [2 I, K]; the codes of `act` are tl_act_mul's
extern "C" int tl_gemm_plain_pair(const float* A, const float* norm_w, float eps, const float* W, int act, float alpha, float limit, float shift,
                                  float* out, int M, int I, int K, hipStream_t st) {
  TL_REQUIRE(out && I > 0 && I % 4 == 0 && I < (1 << 30), "gemm_plain_pair: I=%d (a multiple of 4)", I);
  TL_REQUIRE(act == ACT_SILU || act == ACT_GELU_TANH || act == ACT_SWISH_CLAMPED || act == ACT_RELU, "gemm_plain_pair: no function of code %d", act);
  TL_REQUIRE(act != ACT_SWISH_CLAMPED || limit > 0.f, "gemm_plain_pair: the clamp needs a positive limit");
  Around f{};
  f.norm_w = norm_w; f.eps = eps; f.act = act; f.constants = ActConstants{alpha, limit, shift};
  return launch_around<DO_PAIR>("gemm_plain_pair", A, W, out, M, 2 * I, K, I, f, st);
}

// tl_rope_commit of q|k|v = norm(A) W^T (norm_w null: of A itself), W [(nq + 2 nkv) d, K]; pages of float
extern "C" int tl_gemm_plain_rope(const float* A, const float* norm_w, float eps, const float* W, int M, int K, const int* row_pos,
                                  const float* inv_freq, int rotary_dim, int interleaved, const int* table, int table_stride, int ring_pages,
                                  int nq, int nkv, int d, float* q, float* pages, hipStream_t st) {
  TL_REQUIRE(nq > 0 && nkv > 0 && d > 0 && d % 8 == 0 && d <= 256 && ring_pages > 0 && table_stride > 0 && (long)(nq + 2 * nkv) * d < (1 << 30),
             "gemm_plain_rope: bad sizes nq=%d nkv=%d d=%d ring_pages=%d table_stride=%d", nq, nkv, d, ring_pages, table_stride);
  TL_REQUIRE(rotary_dim >= 0 && rotary_dim <= d && rotary_dim % 2 == 0 && (rotary_dim == 0 || inv_freq != nullptr),
             "gemm_plain_rope: %d rotated channels of a head of %d (even, at most the head, with their frequencies)", rotary_dim, d);
  TL_REQUIRE(row_pos && table && q && pages, "gemm_plain_rope: a buffer is missing");
  Around f{};
  f.norm_w = norm_w; f.eps = eps;
  f.row_pos = row_pos; f.rot = Rotation{inv_freq, rotary_dim, interleaved != 0};
  f.table = table; f.table_stride = table_stride; f.ring_pages = ring_pages; f.nq = nq; f.nkv = nkv; f.d = d; f.q = q; f.pages = pages;
  return launch_around<DO_ROPE>("gemm_plain_rope", A, W, nullptr, M, (nq + 2 * nkv) * d, K, 0, f, st);
}
