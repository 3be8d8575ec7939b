// The recurrence of a state-space mixer (see state_space.hip) by chunks of rows on the matrix cores: bfloat16 steps in which
// sequences bring several rows.  With i, j the places in a chunk of at most SC = 64 rows, c_i the sum of log2 of the decays
// of rows 0 .. i, and S the state before the chunk,
//
//   y_i = 2^c_i S^T C_i + sum_{j <= i} (C_i . B_j) 2^(c_i - c_j) dt_j x_j + D x_i
//   S  <- 2^c_last S + sum_j B_j (2^(c_last - c_j) dt_j x_j)^T
//
// x, B and C are bfloat16 and enter the products as they are.  What is float beside them, the weights of the middle
// sum, the state, the weighted x of the last, goes in as THREE bfloat16 terms (x = hi + mid + lo: 24 bits, as many as a
// float has), and all sums are float; the logarithms are added in double, so that the difference of two of them has a
// float's precision however far down the chunk it lies.
//
// A workgroup has 16 columns of one head of one sequence a wave and goes through the sequence's chunks, the state in its
// accumulators: lane (li, kg) of a wave holds S[n][d] for d = li and n = 16 t + 4 kg + r.  Two such tiles are, as they lie,
// an operand of the first product, whose 32 terms a lane may name in any order as long as C's operand follows it.
//
// The products give every row of a chunk a term of every other, with weight 0 where there is none, and take floats apart
// into terms: a NaN or an infinity spreads to rows before its own, and an infinite state becomes NaN.  Whatever x, B, C, dt
// or state holds one, some y of the chunk is not finite then (each has its term in one, be it with weight 0).  The workgroup
// leaves the chunks there and goes on row by row from the state before that one.
// What bounds it: a chunk's way of phases (rows to LDS, weights, products), each short and behind the one before: 8 us a
// chunk, where its 130 products of 16 cycles a wave take 0.9, its splits about as long and its traffic in LDS 0.8; a
// second workgroup on the compute unit fills gaps (5 us a chunk).
// 128 heads of 128 x 64, microseconds, row by row before: one sequence of 2,048 rows 258 (1,215), four of 128 to 1,024 rows 117
// (838), one of 8,192 1,020 (5,580).  Relative error against float64 (2,000 rows): y 1.2e-7 (5.7e-7), state 1.0e-7 (3.3e-7).
#include "common.hpp"

namespace tl {

constexpr int SC = 64;                 // rows of a chunk

__device__ __forceinline__ float sc_softplus(float a) { return fmaxf(a, 0.f) + log1pf(expf(-fabsf(a))); }

// x = a + b + c, three bfloat16 terms
__device__ __forceinline__ void sc_split(float x, bf16& a, bf16& b, bf16& c) {
  a = (bf16)x;
  const float r = x - (float)a;
  b = (bf16)r;
  c = (bf16)(r - (float)b);
}

// Rows of 64 places j (128 bytes, 8 chunks of 16) of a matrix stored with its rows along the other index: chunk jc of row n
// lies at slot jc ^ key(n).  16 lanes that read a chunk of 16 rows, and 8 that write one place of rows 8 apart, fall on
// different banks.
__device__ __forceinline__ int sc_key(int n) { return ((n >> 3) ^ n) & 7; }

// By the rows of a chunk: the sum of log2 of the decays up to the row, in two floats, dt', what is left of the state before the
// chunk, and the weight of the row in the state behind it.
struct Decays {
  float hi[SC], lo[SC], dt[SC], grow[SC], weight[SC];
};

// NT: tiles of 16 rows of the state (N = 16 NT); WV: waves, 16 columns each
template <int NT, int WV>
__global__ void __launch_bounds__(WV * WAVE, WV / 2)
ssm_chunks_kernel(const bf16* __restrict__ u, int C, int inner, int G, int heads, int dv, const float* __restrict__ proj, int width,
                  int dt_off, const float* __restrict__ dt_bias, const float* __restrict__ A_log, const float* __restrict__ Dw,
                  float* __restrict__ state, long long stride, const int* __restrict__ cu_seqlens, const int* __restrict__ slots,
                  int least, float* __restrict__ y) {
  constexpr int N = 16 * NT, NC = N / 8, THREADS = WV * WAVE;          // NC: chunks of 8 of a row of B or C
  constexpr int CL = SC * NC / THREADS, BP = CL / 2;                   // loads of C, pairs of rows of B a thread
  static_assert(NT >= 2 && NT % 2 == 0 && CL % 2 == 0 && CL > 0, "whole pairs of rows a thread");
  __shared__ __attribute__((aligned(16))) bf16 Cs[SC * N], Bs[SC * N], Bt[N * SC], xT[16 * WV * SC];
  __shared__ __attribute__((aligned(16))) bf16 Ms[3][6 * 512];         // blocks of 16 rows x 32 places of the lower triangle
  __shared__ __attribute__((aligned(16))) Decays decays[2];            // of this chunk and of the next
  __shared__ int spoilt;                                               // a chunk's y were not all finite
  const int h = blockIdx.x, b = blockIdx.y, t = threadIdx.x, wave = t / WAVE, lane = t % WAVE, li = lane % 16, kg = lane / 16;
  const int d0 = blockIdx.z * (16 * WV), g = h / (heads / G);
  const int row0 = cu_seqlens[b], n_new = cu_seqlens[b + 1] - row0;
  if (n_new < least) return;
  const float neg_rate = -expf(A_log[h]);
  const double rate = (double)neg_rate * 1.4426950408889634;
  const float bias = dt_bias[h], skip = Dw[h];

  // the state: this lane's column and rows
  float* S_g = state + (long long)slots[b] * stride + ((size_t)h * dv + d0 + wave * 16 + li) * N + 4 * kg;
  f32x4 S[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) S[n] = *reinterpret_cast<const f32x4*>(S_g + 16 * n);

  bf16x8 cr[CL], br[2 * BP], xr[2];
  const auto load = [&](int i0) {
    const int rows = n_new - i0;
    const bf16* base = u + (size_t)(row0 + i0) * C;
    bf16x8 zero;
#pragma unroll
    for (int e = 0; e < 8; ++e) zero[e] = (bf16)0.f;
#pragma unroll
    for (int k = 0; k < CL; ++k) {
      const int e = t + THREADS * k, r = e / NC, c = e % NC;
      cr[k] = r < rows ? *reinterpret_cast<const bf16x8*>(base + (size_t)r * C + inner + (G + g) * N + c * 8) : zero;
    }
#pragma unroll
    for (int k = 0; k < 2 * BP; ++k) {                   // rows 2 p and 2 p + 1 of pair p
      const int e = t + THREADS * (k / 2), r = e / NC * 2 + k % 2, c = e % NC;
      br[k] = r < rows ? *reinterpret_cast<const bf16x8*>(base + (size_t)r * C + inner + g * N + c * 8) : zero;
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int r = t / (2 * WV) * 2 + k, c = t % (2 * WV);
      xr[k] = r < rows ? *reinterpret_cast<const bf16x8*>(base + (size_t)r * C + h * dv + d0 + c * 8) : zero;
    }
  };
  // by one wave, a row a lane (rows behind the chunk's last: dt 0, decay 1)
  float raw = 0.f;                                       // dt of the chunk after the one whose decays were taken last
  const auto load_dt = [&](int i0) { raw = i0 + lane < n_new ? proj[(size_t)(row0 + i0 + lane) * width + dt_off + h] : 0.f; };
  const auto decay = [&](int i0, Decays& out) {
    const bool row = i0 + lane < n_new;
    const float dt = row ? sc_softplus(raw + bias) : 0.f;
    load_dt(i0 + SC);
    // (a decay this small is 0 in a float: the cut keeps differences of sums finite; NaN stays)
    double c = row ? rate * (double)dt : 0.0;
    c = c < -1e6 ? -1e6 : c;
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
      const double p = __shfl_up(c, o, WAVE);
      if (lane >= o) c += p;
    }
    const double all = __shfl(c, WAVE - 1, WAVE);
    const float hi = (float)c, lo = (float)(c - (double)hi);
    out.hi[lane] = hi;
    out.lo[lane] = lo;
    out.dt[lane] = dt;
    out.grow[lane] = exp2f(hi) * exp2f(lo);
    out.weight[lane] = exp2f((float)(all - c)) * dt;
  };
  typedef __attribute__((ext_vector_type(2))) __bf16 pair;
  int from = n_new;                                      // the first row that this wave takes by itself
  if (t == 0) spoilt = 0;
  load(0);
  if (wave == WV - 1) {
    load_dt(0);
    decay(0, decays[0]);
  }
  // the blocks of zeros to the right of the diagonal's, which the products read beside it
  for (int e = t; e < 3 * 2 * 16 * 16; e += THREADS) {
    const int q = e / 512, block = e / 256 % 2 ? 2 + 1 : 0, row = e / 16 % 16, j = 16 + e % 16;      // of rows 0 .. 15 and 32 .. 47
    Ms[q][block * 512 + row * 32 + (((j / 8) ^ (row / 4)) & 3) * 8 + j % 8] = (bf16)0.f;
  }
  for (int i0 = 0; i0 < n_new; i0 += SC) {
    const Decays& dec = decays[i0 / SC % 2];
    const int rows = min(SC, n_new - i0);
    __syncthreads();                                     // the last chunk has been read
    const int leave = spoilt;
    // where registers are too few to keep the places in LDS over all chunks (eight waves a unit, states of 128 rows: 44 spilled), the
    // thread's number is opaque and the places are worked out anew: 64 sequences of 13 rows 173 us, with spills 293; where they are
    // not, that costs a tenth (one of 2,048 rows 279 against 255)
    int tl = t;
    if constexpr (NT == 8 && WV == 4) asm volatile("" : "+v"(tl));
    const int li = tl % 16, kg = tl / 16 % 4;
#pragma unroll
    for (int k = 0; k < CL; ++k) {
      const int e = tl + THREADS * k, r = e / NC, c = e % NC;
      *reinterpret_cast<bf16x8*>(Cs + r * N + ((c ^ r) & (NC - 1)) * 8) = cr[k];
    }
#pragma unroll
    for (int k = 0; k < BP; ++k) {
      const int e = tl + THREADS * k, r = e / NC * 2, c = e % NC;
      *reinterpret_cast<bf16x8*>(Bs + r * N + ((c ^ r) & (NC - 1)) * 8) = br[2 * k];
      *reinterpret_cast<bf16x8*>(Bs + (r + 1) * N + ((c ^ (r + 1)) & (NC - 1)) * 8) = br[2 * k + 1];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int n = c * 8 + q;
        *reinterpret_cast<pair*>(Bt + n * SC + ((r / 8) ^ sc_key(n)) * 8 + r % 8) = pair{br[2 * k][q], br[2 * k + 1][q]};
      }
    }
    {
      const int r = tl / (2 * WV) * 2, c = tl % (2 * WV);
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int d = c * 8 + q;
        *reinterpret_cast<pair*>(xT + d * SC + ((r / 8) ^ sc_key(d)) * 8 + r % 8) = pair{xr[0][q], xr[1][q]};
      }
    }
    if (leave) {
      from = min(from, i0);
      break;
    }
    __syncthreads();
    if (i0 + SC < n_new) load(i0 + SC);

    // the weights of the middle sum: the ten blocks (it, jt) of 16 x 16 on and below the diagonal, dealt to the waves; a lane has
    // row i = 16 it + li and places j = 16 jt + 4 kg + r
#pragma unroll
    for (int p0 = 0; p0 < 10; p0 += WV) {
      const int p = p0 + wave;
      if (p >= 10) break;
      const int it = p < 1 ? 0 : p < 3 ? 1 : p < 6 ? 2 : 3, jt = p - it * (it + 1) / 2;
      const int i = 16 * it + li, j = 16 * jt + li, j4 = 16 * jt + 4 * kg;
      f32x4 m = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < NT / 2; ++s)
        m = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(Bs + j * N + (((4 * s + kg) ^ j) & (NC - 1)) * 8),
                                                    *reinterpret_cast<const bf16x8*>(Cs + i * N + (((4 * s + kg) ^ i) & (NC - 1)) * 8), m, 0, 0, 0);
      const float ch = dec.hi[i], cl = dec.lo[i];
      const f32x4 jh = *reinterpret_cast<const f32x4*>(dec.hi + j4), jl = *reinterpret_cast<const f32x4*>(dec.lo + j4),
                  jd = *reinterpret_cast<const f32x4*>(dec.dt + j4);
      bf16x4 term[3];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float w = j4 + r <= i ? m[r] * exp2f((ch - jh[r]) + (cl - jl[r])) * jd[r] : 0.f;
        bf16 a, bb, c;
        sc_split(w, a, bb, c);
        term[0][r] = a; term[1][r] = bb; term[2][r] = c;
      }
      // block (it, jt / 2) of 16 rows of 32 places, chunk c of row li at slot c ^ (li / 4)
      const int block = (it < 2 ? it : 2 * it - 2) + jt / 2, chunk = jt % 2 * 2 + kg / 2;
      const int at = block * 512 + li * 32 + ((chunk ^ (li / 4)) & 3) * 8 + kg % 2 * 4;
#pragma unroll
      for (int q = 0; q < 3; ++q) *reinterpret_cast<bf16x4*>(&Ms[q][at]) = term[q];
    }
    if (wave == WV - 1 && i0 + SC < n_new) decay(i0 + SC, decays[(i0 / SC + 1) % 2]);
    // the state's terms: tiles 2 s and 2 s + 1 are a lane's 8 values of 32 rows n
    bf16x8 st[3][NT / 2];
#pragma unroll
    for (int s = 0; s < NT / 2; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        bf16 a, bb, c;
        sc_split(S[2 * s + e / 4][e % 4], a, bb, c);
        st[0][s][e] = a; st[1][s][e] = bb; st[2][s][e] = c;
      }
    __syncthreads();

    const int d = wave * 16 + li;
    float finite = 0.f;                                  // NaN once a y was not
    bf16x8 xf[2];                                        // x^T of column d, places 32 ks + 8 kg
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) xf[ks] = *reinterpret_cast<const bf16x8*>(xT + d * SC + ((4 * ks + kg) ^ sc_key(d)) * 8);
#pragma unroll
    for (int it = 0; it < SC / 16; ++it) {
      const int i = 16 * it + li, i4 = 16 * it + 4 * kg;
      f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < NT / 2; ++s) {
        // C of row i at n = 32 s + 4 kg .. and 32 s + 16 + 4 kg ..
        const int c0 = 4 * s + kg / 2, c1 = c0 + 2;
        const bf16x4 lo = *reinterpret_cast<const bf16x4*>(Cs + i * N + ((c0 ^ i) & (NC - 1)) * 8 + kg % 2 * 4);
        const bf16x4 hi = *reinterpret_cast<const bf16x4*>(Cs + i * N + ((c1 ^ i) & (NC - 1)) * 8 + kg % 2 * 4);
        const bf16x8 cf = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
        for (int q = 2; q >= 0; --q) o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cf, st[q][s], o, 0, 0, 0);
      }
      const f32x4 gr = *reinterpret_cast<const f32x4*>(dec.grow + i4);
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] *= gr[r];
#pragma unroll
      for (int ks = 0; ks <= it / 2; ++ks) {
        const int at = ((it < 2 ? it : 2 * it - 2) + ks) * 512 + li * 32 + ((kg ^ (li / 4)) & 3) * 8;
#pragma unroll
        for (int q = 2; q >= 0; --q) o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(&Ms[q][at]), xf[ks], o, 0, 0, 0);
      }
      // o[r]: row i4 + r, column d
      const bf16x4 xv = *reinterpret_cast<const bf16x4*>(xT + d * SC + ((i4 / 8) ^ sc_key(d)) * 8 + i4 % 8);
#pragma unroll
      for (int r = 0; r < 4; ++r) finite = fmaf(o[r], 0.f, finite);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (i4 + r < rows) y[(size_t)(row0 + i0 + i4 + r) * inner + h * dv + d0 + d] = fmaf(skip, (float)xv[r], o[r]);
    }

    if (__any(isnan(finite))) {
      from = i0;
      spoilt = 1;                                        // (read behind the next barrier)
      continue;
    }

    // the state behind the chunk
    const float all = dec.grow[SC - 1];
    bf16x8 xw[3][2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        bf16 a, bb, c;
        sc_split((float)xf[ks][e] * dec.weight[32 * ks + 8 * kg + e], a, bb, c);
        xw[0][ks][e] = a; xw[1][ks][e] = bb; xw[2][ks][e] = c;
      }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int n = 16 * nt + li;
#pragma unroll
      for (int r = 0; r < 4; ++r) S[nt][r] *= all;
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const bf16x8 bf = *reinterpret_cast<const bf16x8*>(Bt + n * SC + ((4 * ks + kg) ^ sc_key(n)) * 8);
#pragma unroll
        for (int q = 2; q >= 0; --q) S[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf, xw[q][ks], S[nt], 0, 0, 0);
      }
    }
  }
  if (from < n_new) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // the y that these rows' go over have arrived
    const int col = h * dv + d0 + wave * 16 + li;
    for (int i = from; i < n_new; ++i) {
      const bf16* row = u + (size_t)(row0 + i) * C;
      const bf16 *Br = row + inner + g * N + 4 * kg, *Cr = Br + G * N;
      const float dt = sc_softplus(proj[(size_t)(row0 + i) * width + dt_off + h] + bias), a = expf(neg_rate * dt);
      const float x = (float)row[col], dtx = dt * x;
      f32x4 sums = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const bf16x4 bv = *reinterpret_cast<const bf16x4*>(Br + 16 * n), cv = *reinterpret_cast<const bf16x4*>(Cr + 16 * n);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          S[n][r] = fmaf(a, S[n][r], (float)bv[r] * dtx);
          sums[r] = fmaf(S[n][r], (float)cv[r], sums[r]);
        }
      }
      float sum = (sums[0] + sums[1]) + (sums[2] + sums[3]);
      sum += __shfl_xor(sum, 16, WAVE);
      sum += __shfl_xor(sum, 32, WAVE);
      if (kg == 0) y[(size_t)(row0 + i) * inner + col] = fmaf(skip, x, sum);
    }
  }
#pragma unroll
  for (int n = 0; n < NT; ++n) *reinterpret_cast<f32x4*>(S_g + 16 * n) = S[n];
}

template <int NT, int WV>
static int launch_chunks(const bf16* u, int C, int inner, int G, int heads, int dv, const float* proj, int width, int dt_off,
                         const float* dt_bias, const float* A_log, const float* D, float* state, long long stride, const int* cu,
                         const int* slots, int B, int least, float* y, hipStream_t st) {
  ssm_chunks_kernel<NT, WV><<<dim3(heads, B, dv / (16 * WV)), WV * WAVE, 0, st>>>(u, C, inner, G, heads, dv, proj, width, dt_off, dt_bias, A_log, D,
                                                                                  state, stride, cu, slots, least, y);
  TL_LAUNCH_CHECK("ssm_chunks");
  return 0;
}

}  // namespace tl

using namespace tl;

extern "C" {

// Which sizes and buffers the chunks take: states of 32, 64 or 128 rows, columns in whole pairs of tiles, rows of whole 16-byte
// pieces.
int tl_ssm_chunks_serve(int dt, int C, int G, int N, int heads, int dv, const void* u, const void* state, long long stride) {
  return dt == DT_BF16 && (N == 32 || N == 64 || N == 128) && dv % 32 == 0 && heads % G == 0 && C == heads * dv + 2 * G * N &&
         stride % 4 == 0 && ((uintptr_t)u | (uintptr_t)state) % 16 == 0;
}

// as tl_ssm_scan, for buffers that tl_ssm_chunks_serve takes and the sequences of `least` rows or more (at least one); the
// others are left alone
int tl_ssm_chunks(const void* u, int C, int G, int N, int heads, int dv, const float* proj, int width, int dt_off, const float* dt_bias,
                  const float* A_log, const float* D, float* state, long long stride, const int* cu_seqlens, const int* slots, int n, int B,
                  int least, float* y, hipStream_t st) {
  TL_REQUIRE(n >= 0 && B >= 0 && heads > 0 && G > 0 && dv > 0 && least > 0, "ssm_chunks: bad sizes heads=%d G=%d N=%d dv=%d least=%d", heads, G, N, dv, least);
  TL_REQUIRE(tl_ssm_chunks_serve(DT_BF16, C, G, N, heads, dv, u, state, stride), "ssm_chunks: C=%d G=%d N=%d heads=%d dv=%d stride=%lld are not served", C,
             G, N, heads, dv, stride);
  TL_REQUIRE(dt_off >= 0 && dt_off + heads <= width && stride >= (long long)heads * N * dv, "ssm_chunks: bad sizes dt_off=%d width=%d stride=%lld", dt_off,
             width, stride);
  TL_REQUIRE(u && proj && dt_bias && A_log && D && state && cu_seqlens && slots && y, "ssm_chunks: a buffer is missing");
  if (n == 0 || B == 0) return 0;
  // 64 columns a workgroup share the weights' work; 32 where there would be fewer than one workgroup a compute unit
  const bool four = dv % 64 == 0 && (long)heads * B * (dv / 64) >= 256;
#define TL_CHUNKS(NN, WW) \
  return launch_chunks<NN, WW>((const bf16*)u, C, heads * dv, G, heads, dv, proj, width, dt_off, dt_bias, A_log, D, state, stride, cu_seqlens, slots, B, least, y, st)
  if (N == 32) {
    TL_CHUNKS(2, 2);
  } else if (N == 64) {
    if (four) TL_CHUNKS(4, 4);
    TL_CHUNKS(4, 2);
  }
  if (four) TL_CHUNKS(8, 4);
  TL_CHUNKS(8, 2);
#undef TL_CHUNKS
}

}  // extern "C"
