// Between the fused projection of an attention and the attention itself, head by head.
//
// A row of the projection is [q (nq*dk) | k (nkv*dk) | v (nkv*dv) | g (ng)] in float.  Per row:
//
//   * the biases are added (optional), and the values multiplied by `v_factor`;
//   * every head of q and of k is divided by ITS OWN root mean square over its dk channels,
//     eps inside the root, and multiplied by a weight of dk channels that all heads share
//     (optional; q and k have a weight each);
//   * the first `rotary_dim` channels of every head of q and k are rotated in pairs
//     (i, i + rotary_dim/2) by the angle pos * inv_freq[i];
//   * or (`unit_norm`) every head of q and of k is divided by its root mean square AFTER the
//     rotation, with no weight;
//   * the values are mixed with those that an earlier layer left for the same row:
//     v <- (1 - lambda) v + lambda v_first  (`mix` 2), or are left for later layers (`mix` 1);
//     v_first is float, unrounded;
//   * g -> 1 / (1 + exp(-g)), one gate per channel of the concatenated heads (ng = nq*dv) or
//     any other number.
//
// k and v go to rows of their own, or (pages != null: one token a sequence) straight into the
// page of the row's position; a mixer that reads another's keys and values has none of its own
// (nkv == 0: the row is [q | g]).  One wave takes one unit of work: a head of q, a head of k, a
// head of v, or 256 gate channels.
#include "common.hpp"

namespace tl {

constexpr int HP_MAX_D = 256;

struct HeadTerms {
  const float* bias;       // [Q + K + V + ng] or null
  const float* q_norm;     // [dk] or null
  const float* k_norm;     // [dk] or null
  float eps;
  int mix;                 // 0: none; 1: leave v in v_first; 2: mix with v_first
  float lambda;
  float* v_first;          // [n, nkv*dv] float
  int unit_norm;           // q and k heads divided by their root mean square after the rotation, no weight
  float v_factor;          // on the (biased) values
};

// A wave goes through units blockIdx.y * 4 + wave, 4 * gridDim.y further each, and keeps what a head's rotation takes of the row's
// position, J channels of a head a lane (dk <= 64 J): the sines and cosines are most of the instructions, and with a head a wave
// they were computed for every head.  Steps of few rows still go a head a wave: they wait for the longest chain, not for the
// units.  2,348 rows of 32 + 8 + 8 heads of 128 and 32 gates, 64 channels rotated and unit norms: 54.4 us before, 35.0 now; the same
// heads normed by weights with 4,096 gates, all rotated (164 MB) 68.9 and 61.5.
template <typename T, int J>
__global__ void __launch_bounds__(256)
head_prepare_kernel(const float* __restrict__ proj, int proj_stride, const int* __restrict__ row_pos, Rotation rot, HeadTerms t,
                    int nq, int nkv, int dk, int dv, int ng, T* __restrict__ q, T* __restrict__ k, T* __restrict__ v,
                    float* __restrict__ gate, const int* __restrict__ table, int table_stride, int ring_pages,
                    T* __restrict__ pages) {
  const int n = blockIdx.x;
  const int lane = threadIdx.x % WAVE;
  const int first = blockIdx.y * 4 + threadIdx.x / WAVE;
  const int Q = nq * dk, K = nkv * dk, V = nkv * dv;
  const int units = nq + 2 * nkv + (ng + 255) / 256;
  const float* row = proj + (size_t)n * proj_stride;
  const int pos = row_pos[n];
  auto at = [&](int i) { return row[i] + (t.bias ? t.bias[i] : 0.f); };

  int r = 0;
  T* kd = nullptr;
  T* vd = nullptr;
  if (pages) {
    const int page = table[(size_t)n * table_stride + (pos / PAGE) % ring_pages];
    kd = pages + (size_t)page * nkv * PAGE * (dk + dv);
    vd = kd + (size_t)nkv * PAGE * dk;
    r = pos % PAGE;
  }
  const int half = rot.rotary_dim / 2;
  float sn[J], cs[J];
  if (first < nq + nkv) {
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int c = lane + WAVE * j;
      if (c < 2 * half) sincosf((float)pos * rot.inv_freq[c < half ? c : c - half], &sn[j], &cs[j]);
    }
  }

  for (int unit = first; unit < units; unit += 4 * gridDim.y) {
    if (unit < nq + nkv) {                       // a head of q or of k
      const bool is_q = unit < nq;
      const int head = is_q ? unit : unit - nq;
      const int off = (is_q ? 0 : Q) + head * dk;
      const float* w = is_q ? t.q_norm : t.k_norm;
      float a[J], b[J];                          // this lane's channels, and those that they are rotated with
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const int c = lane + WAVE * j;
        a[j] = c < dk ? at(off + c) : 0.f;
        b[j] = c < 2 * half ? at(off + (c < half ? c + half : c - half)) : 0.f;
      }
      if (w) {
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < J; ++j)
          if (lane + WAVE * j < dk) ss += a[j] * a[j];
        const float f = 1.0f / sqrtf(wave_sum(ss) / (float)dk + t.eps);
#pragma unroll
        for (int j = 0; j < J; ++j) {
          const int c = lane + WAVE * j;
          if (c < dk) a[j] = a[j] * f * w[c];
          if (c < 2 * half) b[j] = b[j] * f * w[c < half ? c + half : c - half];
        }
      }
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const int c = lane + WAVE * j;
        if (c < 2 * half) {
          float ra, rb;
          rotate_pair(c < half ? a[j] : b[j], c < half ? b[j] : a[j], cs[j], sn[j], ra, rb);
          a[j] = c < half ? ra : rb;
        }
      }
      float after = 1.f;
      if (t.unit_norm) {
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < J; ++j)
          if (lane + WAVE * j < dk) ss += a[j] * a[j];
        after = 1.0f / sqrtf(wave_sum(ss) / (float)dk + t.eps);
      }
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const int c = lane + WAVE * j;
        if (c >= dk) continue;
        const T o = from_f32<T>(a[j] * after);
        if (is_q) q[(size_t)n * Q + head * dk + c] = o;
        else if (pages) kd[((size_t)head * PAGE + r) * dk + c] = o;
        else k[(size_t)n * K + head * dk + c] = o;
      }
    } else if (unit < nq + 2 * nkv) {            // a head of v
      const int head = unit - nq - nkv;
      for (int c = lane; c < dv; c += WAVE) {
        const int i = head * dv + c;
        float a = at(Q + K + i) * t.v_factor;
        if (t.mix == 1) t.v_first[(size_t)n * V + i] = a;
        else if (t.mix == 2) a = (1.0f - t.lambda) * a + t.lambda * t.v_first[(size_t)n * V + i];
        const T o = from_f32<T>(a);
        if (pages) vd[((size_t)head * dv + c) * PAGE + r] = o;
        else v[(size_t)n * V + i] = o;
      }
    } else {
      const int g0 = (unit - nq - 2 * nkv) * 256;  // gate channels
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i = g0 + lane + WAVE * j;
        if (i < ng) gate[(size_t)n * ng + i] = 1.0f / (1.0f + expf(-at(Q + K + V + i)));
      }
    }
  }
}

}  // namespace tl

using namespace tl;

extern "C" {

int tl_head_prepare(const float* proj, int proj_stride, const int* row_pos, const float* inv_freq, int rotary_dim, const float* bias,
                    const float* q_norm, const float* k_norm, float eps, int unit_norm, int mix, float lambda, float v_factor,
                    float* v_first, int n, int nq, int nkv, int dk, int dv, int ng, void* q, void* k, void* v, float* gate, int dt,
                    const int* table, int table_stride, int ring_pages, void* pages, hipStream_t st) {
  TL_REQUIRE(n >= 0 && nq > 0 && nkv >= 0 && dk > 0 && dv > 0 && ng >= 0 && dk <= HP_MAX_D && dv <= HP_MAX_D,
             "head_prepare: bad sizes n=%d nq=%d nkv=%d dk=%d dv=%d ng=%d (heads up to %d)", n, nq, nkv, dk, dv, ng, HP_MAX_D);
  TL_REQUIRE(proj_stride >= nq * dk + nkv * (dk + dv) + ng, "head_prepare: rows %d apart are too short", proj_stride);
  TL_REQUIRE(rotary_dim >= 0 && rotary_dim % 2 == 0 && rotary_dim <= dk,
             "head_prepare: %d rotated channels of a head of %d (even, at most the head)", rotary_dim, dk);
  TL_REQUIRE(rotary_dim == 0 || inv_freq, "head_prepare: a rotation without frequencies");
  TL_REQUIRE(proj && row_pos && q && (nkv == 0 || pages || (k && v)), "head_prepare: a buffer is missing");
  TL_REQUIRE(!unit_norm || (q_norm == nullptr && k_norm == nullptr), "head_prepare: a norm before the rotation or one after it");
  TL_REQUIRE(ng == 0 || gate, "head_prepare: %d gate channels and nowhere to put them", ng);
  TL_REQUIRE(mix >= 0 && mix <= 2 && (mix == 0 || v_first), "head_prepare: mixing values needs the buffer they are left in");
  TL_REQUIRE(pages == nullptr || (table && table_stride > 0 && ring_pages > 0), "head_prepare: pages without a page table");
  TL_REQUIRE(dt == DT_F32 || dt == DT_BF16, "head_prepare: unknown dtype code %d", dt);
  if (n == 0) return 0;
  const Rotation rot{inv_freq, rotary_dim, 0};
  const HeadTerms t{bias, q_norm, k_norm, eps, mix, lambda, v_first, unit_norm, v_factor};
  const int units = nq + 2 * nkv + (ng + 255) / 256;
  // units a wave: as many as leave 7 workgroups a compute unit, up to three; from 800 rows on a row in 200, at most 8.  32 + 8 + 8 heads of
  // 128 with 32 gates, one / two / three units: 100 rows 3.8 / 4.2 / 4.5 us, 150 4.5 / 4.4 / 4.7, 200 5.4 / 4.8 / 5.1, 300 6.8 / 6.6 / 6.2, 600
  // 11.4 / 10.3 / 9.9 (2,348 rows with three 34.8, with eight 33.1); 64 + 8 + 8 of 256 at 150 rows 10.6 / 8.8 / 9.2; 16 + 2 + 2 of 64
  // at 256 rows 3.8 / 4.0 / 4.7; with 4,096 gates, whose units are short, at 130 rows 5.8 / 6.2 and at 256 8.9 / 9.0 / 8.0
  const long workgroups = ((long)n * units + 3) / 4;
  const int each = max((int)min((workgroups + 1791) / 1792, 3l), min(n / 200, 8));
  const dim3 grid(n, (units + 4 * each - 1) / (4 * each));
#define TL_HP(T, J)                                                                                                          \
  head_prepare_kernel<T, J><<<grid, 256, 0, st>>>(proj, proj_stride, row_pos, rot, t, nq, nkv, dk, dv, ng, (T*)q, (T*)k, (T*)v, gate, \
                                                  table, table_stride, ring_pages, (T*)pages)
#define TL_HP_J(T)                  \
  do {                              \
    if (dk <= 64) TL_HP(T, 1);      \
    else if (dk <= 128) TL_HP(T, 2); \
    else TL_HP(T, 4);               \
  } while (0)
  if (dt == DT_F32) TL_HP_J(float);
  else TL_HP_J(bf16);
#undef TL_HP_J
#undef TL_HP
  TL_LAUNCH_CHECK("head_prepare");
  return 0;
}

}  // extern "C"
