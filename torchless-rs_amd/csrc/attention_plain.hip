// Attention over the cache and the keys of this step, one wave per (row, head):
// the kernel of the true 32-bit path and the reference that the faster
// kernels are checked against.  It serves any mix of rows: whole prompts, a
// prompt that goes on from cached context, single decoded tokens.
//
// For the query at position p of sequence b, key j is visible iff j <= p and
// (no window or j > p - W)  (src/model/modules/attention.rs:90 and
// src/model/models/gpt_oss.rs:168-175 of the reference).  Keys j < n_cached[b]
// are read from the sequence's pages, later ones from this step's k/v rows.
// score = (k.q) * scale, scale applied after the dot; softmax with running
// maximum over tiles of 64 keys, all in float
// (src/model/modules/attention.rs:82-121, src/kernels/mod.rs:494-543).
#include "common.hpp"

namespace tl {

constexpr int MAX_D = 256;

// VEC (steps that read everything from the pages, heads of a multiple of 4, aligned): four channels of a key a load, and where a tile of
// keys is one page's, four keys' values: the same sums in the same order, a quarter of the loads and many of them under way at once, where
// a lane waited for each.  (Tiles begin at the first key that a row sees: they are pages' while that is the sequence's first, and for a row
// past its window only where the window begins with a page; its values else come one by one.)  Without a window, 32 heads of 64 / 128, two
// rows: 50 keys 7.0 / 11.0 us before, 4.8 / 6.4 now, 300 28.0 / 49.5 and 13.8 / 21.6, 2,000 194 / 363 and 99 / 175.  Steps with rows of their
// own read those, in whole lines, as before: of many rows fewer waves of more registers were up to 6 percent slower (300 rows of 64 channels
// 63.0 and 66.7).
template <typename T, bool VEC>
__global__ void __launch_bounds__(64)
attn_plain_kernel(const T* __restrict__ q, const T* __restrict__ k_new, const T* __restrict__ v_new,
                  const T* __restrict__ pages, const int* __restrict__ table, int table_stride,
                  int ring_pages, const int* __restrict__ row_seq, const int* __restrict__ row_pos,
                  const int* __restrict__ cu_seqlens, const int* __restrict__ n_cached, int nq,
                  int nkv, int d, int window, float scale, T* __restrict__ out) {
  using vec4 = __attribute__((ext_vector_type(4))) T;
  __shared__ __attribute__((aligned(16))) float q_s[MAX_D];
  __shared__ __attribute__((aligned(16))) float p_s[WAVE];
  __shared__ const T* v_s[WAVE];
  __shared__ int vstride_s[WAVE];
  const int n = blockIdx.x / nq, h = blockIdx.x % nq;
  const int lane = threadIdx.x;
  const int b = row_seq[n], p = row_pos[n];
  const int kvh = h / (nq / nkv);
  const int cached = n_cached[b];
  const int row0 = cu_seqlens[b];
  const int lo = (window > 0 && p - window + 1 > 0) ? p - window + 1 : 0;
  const size_t head_elems = (size_t)PAGE * d;
  const size_t page_elems = 2 * (size_t)nkv * head_elems;
  const size_t v_off = (size_t)nkv * head_elems;

  const T* qr = q + ((size_t)n * nq + h) * d;
  for (int i = lane; i < d; i += WAVE) q_s[i] = to_f32(qr[i]);
  __syncthreads();

  float m = -INFINITY, l = 0.f;
  float acc[MAX_D / WAVE];
#pragma unroll
  for (int i = 0; i < MAX_D / WAVE; ++i) acc[i] = 0.f;

  for (int j0 = lo; j0 <= p; j0 += WAVE) {
    const int j = j0 + lane;
    float s = -INFINITY;
    const T* vp = nullptr;
    int vstride = 1;                 // values: [d][PAGE] in a page, [d] in the step's rows
    if (j <= p) {
      const T* kp;
      if (j < cached) {
        const int page = table[(size_t)b * table_stride + (j / PAGE) % ring_pages];
        kp = pages + (size_t)page * page_elems + (size_t)kvh * head_elems + (size_t)(j % PAGE) * d;
        vp = pages + (size_t)page * page_elems + v_off + (size_t)kvh * head_elems + (j % PAGE);
        vstride = PAGE;
      } else {
        const size_t r = ((size_t)(row0 + j - cached) * nkv + kvh) * d;
        kp = k_new + r;
        vp = v_new + r;
      }
      float dot = 0.f;
      if constexpr (VEC) {
#pragma unroll 8
        for (int t = 0; t < d; t += 4) {
          const vec4 kk = *reinterpret_cast<const vec4*>(kp + t);
          const f32x4 qq = *reinterpret_cast<const f32x4*>(&q_s[t]);
#pragma unroll
          for (int e = 0; e < 4; ++e) dot = fmaf(to_f32((T)kk[e]), qq[e], dot);
        }
      } else {
        for (int t = 0; t < d; ++t) dot = fmaf(to_f32(kp[t]), q_s[t], dot);
      }
      s = dot * scale;
    }
    const float m_new = fmaxf(m, wave_max(s));       // finite: key j0 is visible
    const float pj = (j <= p) ? expf(s - m_new) : 0.f;
    const float alpha = expf(m - m_new);              // 0 in the first tile (m = -inf)
    l = l * alpha + wave_sum(pj);
    m = m_new;
    __syncthreads();
    p_s[lane] = pj;
    v_s[lane] = vp;
    vstride_s[lane] = vstride;
    __syncthreads();
    const int cnt = (p - j0 + 1 < WAVE) ? p - j0 + 1 : WAVE;
    const bool one_page = VEC && j0 % PAGE == 0 && j0 + cnt <= cached;
#pragma unroll
    for (int i = 0; i < MAX_D / WAVE; ++i) {
      const int dim = lane + WAVE * i;
      if (dim < d) {
        float a = acc[i] * alpha;
        int jj = 0;
        if (one_page) {
          const T* vr = v_s[0] + (size_t)dim * PAGE;
#pragma unroll 4
          for (; jj + 3 < cnt; jj += 4) {
            const vec4 vv = *reinterpret_cast<const vec4*>(vr + jj);
            const f32x4 pp = *reinterpret_cast<const f32x4*>(&p_s[jj]);
#pragma unroll
            for (int e = 0; e < 4; ++e) a = fmaf(pp[e], to_f32((T)vv[e]), a);
          }
        }
        for (; jj < cnt; ++jj) a = fmaf(p_s[jj], to_f32(v_s[jj][(size_t)dim * vstride_s[jj]]), a);
        acc[i] = a;
      }
    }
  }
  T* o = out + ((size_t)n * nq + h) * d;
#pragma unroll
  for (int i = 0; i < MAX_D / WAVE; ++i) {
    const int dim = lane + WAVE * i;
    if (dim < d) o[dim] = from_f32<T>(acc[i] / l);
  }
}

}  // namespace tl

using namespace tl;

extern "C" int tl_attn_plain(const void* q, const void* k_new, const void* v_new, const void* pages,
                             int dt, const int* table, int table_stride, int ring_pages,
                             const int* row_seq, const int* row_pos, const int* cu_seqlens,
                             const int* n_cached, int n, int nq, int nkv, int d, int window,
                             float scale, void* out, hipStream_t st) {
  TL_REQUIRE(n >= 0 && nq > 0 && nkv > 0 && nq % nkv == 0, "attention: bad head counts nq=%d nkv=%d",
             nq, nkv);
  TL_REQUIRE(d > 0 && d <= MAX_D, "attention: head size %d is not served (1..%d)", d, MAX_D);
  TL_REQUIRE(ring_pages > 0 && table_stride > 0 && window >= 0,
             "attention: bad cache geometry ring_pages=%d table_stride=%d window=%d", ring_pages,
             table_stride, window);
  TL_REQUIRE((long long)n * nq < 2147483647LL, "attention: too many (row, head) pairs");
  if (n == 0) return 0;
  const size_t quad = dt == DT_F32 ? 16 : 8;
  const bool vec = k_new == nullptr && d % 4 == 0 && (uintptr_t)pages % quad == 0;
#define TL_PLAIN(T, VEC)                                                                                                     \
  attn_plain_kernel<T, VEC><<<n * nq, 64, 0, st>>>((const T*)q, (const T*)k_new, (const T*)v_new, (const T*)pages, table,     \
                                                   table_stride, ring_pages, row_seq, row_pos, cu_seqlens, n_cached, nq, nkv, \
                                                   d, window, scale, (T*)out)
  if (dt == DT_F32 && vec) TL_PLAIN(float, true);
  else if (dt == DT_F32) TL_PLAIN(float, false);
  else if (dt == DT_BF16 && vec) TL_PLAIN(bf16, true);
  else if (dt == DT_BF16) TL_PLAIN(bf16, false);
  else
    TL_REQUIRE(false, "attention: unknown dtype code %d", dt);
#undef TL_PLAIN
  TL_LAUNCH_CHECK("attn_plain");
  return 0;
}
