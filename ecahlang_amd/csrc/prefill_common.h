// What the matrix-core prefill kernels share: their parameters and work records, the global -> LDS
// copies, and the merge of split key ranges (16-bit caches: prefill_mfma.hip, fp32: prefill_f32.hip).
#pragma once
#include <type_traits>
#include "attn_common.h"

namespace pkv {
namespace pre {

constexpr int kMaxChunk = 8192;  // keys per item (its page ids are staged in LDS)
// Lazy running max (log2 units): a row's reference max moves only when its scores exceed it by
// more than this, so probabilities stay <= 2^kLazyMax (exact enough in fp16 / bf16 P, and far
// from fp32 overflow in the sums) and the output rows are rescaled only on such jumps.
constexpr float kLazyMax = 8.f;

// Source of the value rows that must read as zero (past the chunk, absent pages): P is 0 there,
// and 0 * NaN would poison P.V.
static __device__ uint4 g_zero_rows[64];

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// One wave-wide 16-byte-per-lane copy global -> LDS: lane l's 16 bytes at sbase + voff (a
// wave-uniform base in an SGPR pair plus a 32-bit per-lane byte offset) land at LDS byte
// m0 + 16 * l (m0 uniform).  Written as inline assembly so that the compiler does not track it:
// the caller orders it with explicit vmcnt waits and barriers (the compiler cannot tell which LDS
// array a later transposed read touches and would otherwise wait for every copy in flight,
// draining the prefetch pipeline).
__device__ __forceinline__ void lds_copy16(const void* sbase, unsigned voff, unsigned m0) {
  asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "s"(m0) : "memory", "m0");
}
// LDS byte address of a pointer into a __shared__ array.
__device__ __forceinline__ unsigned lds_addr(const char* p) {
  return (unsigned)(uintptr_t)(const __attribute__((address_space(3))) char*)(p);
}
constexpr int kItem = 12;    // int32 fields per work item
constexpr int kGroup = 8;    // int32 fields per split group

struct PrefillMfmaParams {
  const void* q;
  int64_t q_sn, q_sh;
  const void* k_cache;
  const void* v_cache;
  int64_t page_stride, num_pages;
  const int32_t* indices;
  int64_t num_indices;
  int32_t hq, hkv;
  int32_t causal;
  float scale_log2;
  void* out;
  int64_t o_sn, o_sh;
  const int32_t* items;
  float2* part_ml;  // [slot][rows of an item]
  float* part_o;    // [slot][rows of an item][D] (kHalfPartials: fp16 elements, else fp32)
  int32_t o_vec;
};

// Split groups' partial outputs are kept in fp16 when the cache is fp16 (averages of fp16 V
// rows, so they fit; half the bytes written by the items and read by the merge), else fp32.
// (the run-time groups, G = 0, keep fp32 partials: on the vector kernel, which ran them before, nothing
// between the scores and the output was rounded to 16 bits).
template <typename T, int G>
constexpr bool kHalfPartials = std::is_same<T, _Float16>::value && G != 0;

// Query rows per item: ROWS, or (run-time groups) the largest multiple of the group below it.
template <int G, int ROWS>
__device__ __forceinline__ int item_rows(int g) { return G ? ROWS : ROWS / g * g; }

// One query row over the keys [k0, lim) of its chunk by the whole wave, as the vector kernel computes
// it: fp32, no product for a key the row does not see.  The matrix-core kernels multiply a masked
// key's value row by a zero weight, which is NaN when that row holds an infinity or a NaN, so the
// kernels that took shapes over from the vector kernel redo a row that did not come out finite.
// store(dim of this lane, value, max, sum) gets D / 64 consecutive dims per lane.
template <typename T, int D, typename Store>
__device__ __forceinline__ void exact_row(const PrefillMfmaParams& P, const int* pages, int k0, int lim,
                                          int64_t hoff, const T* q, Store&& store) {
  constexpr int DPL = D / 64;
  const int lane = threadIdx.x & 63;
  const int64_t rowstride = (int64_t)P.hkv * D;
  const T* kc = reinterpret_cast<const T*>(P.k_cache) + hoff;
  const T* vc = reinterpret_cast<const T*>(P.v_cache) + hoff + lane * DPL;
  float m = -INFINITY, l = 0.f, acc[DPL];
#pragma unroll
  for (int j = 0; j < DPL; ++j) acc[j] = 0.f;
#pragma unroll 1
  for (int ts = k0; ts < lim; ts += 64) {
    const int t = ts + lane, page = t < lim ? pages[(t - k0) >> 4] : -1;
    float s = 0.f;
    if (page >= 0) {
      const T* kr = kc + page * P.page_stride + (t & 15) * rowstride;
#pragma unroll 1
      for (int d = 0; d < D; ++d) s += to_f32(q[d]) * P.scale_log2 * to_f32(kr[d]);
    }
    s = page >= 0 ? s : -INFINITY;
    const float mnew = fmaxf(m, wave_max(s));
    const float alpha = m == -INFINITY ? 0.f : exp2f(m - mnew);
    const float p = (page >= 0 && mnew != -INFINITY) ? exp2f(s - mnew) : 0.f;
    l = l * alpha + wave_sum(p);
    m = mnew;
#pragma unroll
    for (int j = 0; j < DPL; ++j) acc[j] *= alpha;
    const int n = min(64, lim - ts);
#pragma unroll 1
    for (int tt = 0; tt < n; ++tt) {
      const int pg = pages[(ts + tt - k0) >> 4];
      if (pg < 0) continue;
      const float w = __shfl(p, tt, 64);
      const T* vr = vc + pg * P.page_stride + ((ts + tt) & 15) * rowstride;
#pragma unroll
      for (int j = 0; j < DPL; ++j) acc[j] += w * to_f32(vr[j]);
    }
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
  for (int j = 0; j < DPL; ++j) store(lane * DPL + j, acc[j] * inv, m, l);
}

// Folds the partials of each split group: group = {first_slot, nslots, qo_start, t0, tq, h}.
// A workgroup takes merge_rows() rows of one group; D/8 lanes per row, 8 dims each (16-byte
// loads of fp16 partials).  Each round loads kMergeUnroll slots' (max, sum) and rows together,
// from clamped (always valid) addresses, and folds them under a running max: one memory round
// trip per round, and for a group of at most kMergeUnroll slots the plain fold under the
// group's max.
constexpr int kMergeUnroll = 4;
template <int D>
constexpr int merge_rows() { return 256 / (D / 8); }

template <typename T, int D, int G, int ROWS>
__global__ __launch_bounds__(256) void prefill_merge_kernel(PrefillMfmaParams P, const int32_t* groups) {
  constexpr int RB = merge_rows<D>(), TPR = D / 8;
  const int32_t* gr = groups + (int64_t)kGroup * (blockIdx.x / (ROWS / RB));
  const int s0 = gr[0], ns = gr[1], qo_start = gr[2], t0 = gr[3], tq = gr[4], h = gr[5];
  const int r = (blockIdx.x % (ROWS / RB)) * RB + threadIdx.x / TPR, d = (threadIdx.x % TPR) * 8;
  const int g = G ? G : P.hq / P.hkv, rows = item_rows<G, ROWS>(g);
  const int tt = r / g, hh = r % g;
  if (tt >= tq || ns <= 0) return;
  const float2* ml = P.part_ml + (int64_t)s0 * rows + r;
  const int64_t po = ((int64_t)s0 * rows + r) * D + d;  // element offset of slot s0's dims
  float M = -INFINITY;
  float den = 0.f;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < ns; s += kMergeUnroll) {
    float2 w[kMergeUnroll];
    float v[kMergeUnroll][8];
#pragma unroll
    for (int u = 0; u < kMergeUnroll; ++u) {
      const int64_t sl = min(s + u, ns - 1);
      w[u] = ml[sl * rows];
      if constexpr (kHalfPartials<T, G>) {
        const uint4 raw = *reinterpret_cast<const uint4*>(reinterpret_cast<const _Float16*>(P.part_o) + po + sl * rows * D);
        _Float16 hv[8];
        __builtin_memcpy(hv, &raw, 16);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[u][e] = (float)hv[e];
      } else {
        const float4* src = reinterpret_cast<const float4*>(P.part_o + po + sl * rows * D);
        const float4 a = src[0], b = src[1];
        v[u][0] = a.x; v[u][1] = a.y; v[u][2] = a.z; v[u][3] = a.w;
        v[u][4] = b.x; v[u][5] = b.y; v[u][6] = b.z; v[u][7] = b.w;
      }
    }
    // the running max over the slots loaded so far (repeats of the last slot included, as in a
    // separate max pass); what earlier rounds folded is rescaled to it
    float Mn = M;
#pragma unroll
    for (int u = 0; u < kMergeUnroll; ++u) Mn = fmaxf(Mn, w[u].x);
    if (Mn > M) {
      const float f = den > 0.f ? exp2f(M - Mn) : 0.f;
      den *= f;
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] *= f;
      M = Mn;
    }
#pragma unroll
    for (int u = 0; u < kMergeUnroll; ++u) {
      // a slot whose rows saw no key (l = 0) carries no weight; repeats past ns count zero
      // (such a slot's row may hold anything, hence the branch rather than a zero weight; a sum that
      // is NaN stays one)
      const float c = (s + u < ns && w[u].y != 0.f) ? exp2f(w[u].x - M) * w[u].y : 0.f;
      if (c != 0.f) {
        den += c;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += c * v[u][e];
      }
    }
  }
  const float inv = den > 0.f ? 1.f / den : 0.f;
  T* orow = reinterpret_cast<T*>(P.out) + (int64_t)(qo_start + t0 + tt) * P.o_sn + (int64_t)(h * g + hh) * P.o_sh + d;
  if (P.o_vec) {  // (rows aligned for four elements at a time)
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      T o4[4] = {from_f32<T>(acc[4 * half] * inv), from_f32<T>(acc[4 * half + 1] * inv),
                 from_f32<T>(acc[4 * half + 2] * inv), from_f32<T>(acc[4 * half + 3] * inv)};
      __builtin_memcpy(__builtin_assume_aligned(orow + 4 * half, 4 * sizeof(T)), o4, 4 * sizeof(T));
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) orow[e] = from_f32<T>(acc[e] * inv);
  }
}

}  // namespace pre
}  // namespace pkv
