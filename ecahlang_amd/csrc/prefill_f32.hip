// Paged chunked prefill over fp32 caches on the matrix cores (page_size 16, head_dim 64 or 128, GQA
// groups 1 to 16).  Same contract as the vector kernel (BatchPrefillWithPagedKVCacheWrapper.run,
// ecahlang/main.py:432-443, :68); everything stays in fp32: v_mfma_f32_16x16x4_f32 takes fp32 operands.
//
// Work items come from the host plan as for the 16-bit kernel (prefill_mfma.hip), of (128 / g) * g
// query rows of one KV head: 8 waves of 16 rows.  A step is SK keys, staged by all threads in LDS
// (two buffers, copied straight from global memory while the previous step is computed; one barrier
// a step).  With lane l = (lr = l % 16, lg = l / 16):
//   S^T[key][row] = K . Q^T     A: lane holds K[key lr][dim 16 s + 4 lg + e], B: Q[row lr][the same dims],
//                               one 16-byte read of each feeding the four products e = 0 .. 3 (the
//                               reduction may take the dims in any order that both operands share)
//   online softmax              lane: row lr, keys 4 lg + i of each 16-key tile
//   O^T[dim][row] += V^T . P    product i takes the keys 4 lg + i, which are the lane's own softmax
//                               weights: B is the score register itself.  A: V[key 4 lg + i][dim 64 c
//                               + 4 lr + e], one 16-byte read for the four output tiles e = 0 .. 3
// so the scores never leave their registers, and a lane ends with 16 consecutive dims of its row.
//
// What bounds it: the fp32 products, 64 flop a cycle and SIMD (157 TFLOP/s over the chip; a large fp32
// product of the installed library reaches 153).  A wave has 64 products of 2,048 flop in flight a
// step and phase, two waves a SIMD (head_dim 64: four) cover each other's reads and softmax.  Steps
// are 64 keys at head_dim 64 and 32 at 128: 64 KB of LDS, so two workgroups fit a CU.
// Measured at 32 / 8 heads of 64 dims, 6 prompts of 12 to 512 tokens on up to 300 cached ones (2.2
// GFLOP of valid pairs): 472 us on the vector kernel (a workgroup a query row), 47.7 us here, both
// 3.3e-7 off 64 bits.
#include "attn_common.h"
#include "mfma_common.h"
#include "prefill_common.h"
#include "../../include/pagedkv.h"

using namespace pkv;
using namespace pkv::mfma;
using namespace pkv::pre;

namespace {

constexpr int kRowsF = 128;  // query rows per item (8 waves x 16)

template <int D>
__global__ __launch_bounds__(512, 4) void prefill_f32_kernel(PrefillMfmaParams P) {
  constexpr int SK = 4096 / D, KT = SK / 16;  // keys and 16-key tiles per step
  constexpr int CPR = D / 4;                  // 16-byte chunks per row
  constexpr int ROWB = D * 4, TILEB = 16 * ROWB, STEPB = KT * TILEB;
  constexpr int RPI = 64 / CPR;               // rows per 1 KB copy
  constexpr int LPP = 16 / RPI;               // copies per page
  constexpr int KL = KT * LPP / 8;            // K (and V) copies per wave and step, all of one page
  static_assert(KT * LPP % 8 == 0 && LPP % KL == 0, "copies per wave");
  constexpr int QS = D / 16;                  // 16-dim pieces of a row
  constexpr int NC = D / 64;                  // 64-dim pieces of the output

  __shared__ __align__(16) char s_k[2 * STEPB];
  __shared__ __align__(16) char s_v[2 * STEPB];
  __shared__ int s_page[kMaxChunk / 16 + KT];  // the chunk's page ids, -1 = absent

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int g = P.hq / P.hkv;
  const int32_t* it = P.items + (int64_t)kItem * blockIdx.x;
  const int h = it[1], t0 = it[2], tq = it[3], k0 = it[4], k1 = it[5], slot = it[6];
  const int kv_len = it[7], qo_len = it[8], qo_start = it[9], kp0 = it[10];
  const int64_t npages_req = (kv_len + 15) / 16;
  const int64_t rowstride = (int64_t)P.hkv * D, hoff = (int64_t)h * D;

  // this wave's 16 rows
  const int r = 16 * wave + lr, rtok = r / g, rh = r % g;
  const bool row_ok = rtok < tq;
  const int64_t qrow = qo_start + t0 + (row_ok ? rtok : 0);
  const float* qsrc = reinterpret_cast<const float*>(P.q) + qrow * P.q_sn + (int64_t)(h * g + rh) * P.q_sh + 4 * lg;
  f4 qr[QS];
#pragma unroll
  for (int s = 0; s < QS; ++s) {
    const f4 v = *reinterpret_cast<const f4*>(qsrc + 16 * s);
    qr[s] = row_ok ? v : f4{0.f, 0.f, 0.f, 0.f};
  }
  int lim = P.causal ? t0 + rtok + kv_len - qo_len + 1 : kv_len;  // the row sees keys below lim
  lim = row_ok ? min(lim, k1) : -1;
  int lim_min = row_ok ? lim : INT_MAX;
#pragma unroll
  for (int x = 1; x < 64; x <<= 1) lim_min = min(lim_min, __shfl_xor(lim_min, x, 64));
  lim_min = __builtin_amdgcn_readfirstlane(lim_min);

  // (the plan keeps k1 - k0 <= kMaxChunk; the clamp keeps s_page in bounds regardless)
  const int nsteps = min((k1 - k0 + SK - 1) / SK, kMaxChunk / SK);
  for (int i = threadIdx.x; i < nsteps * KT; i += blockDim.x) {
    const int64_t pi = k0 / 16 + i;
    const int64_t e = kp0 + (pi < npages_req ? pi : npages_req - 1);  // (past the last page: masked)
    const int64_t pg = (uint64_t)e < (uint64_t)P.num_indices ? P.indices[e] : -1;
    s_page[i] = (pg >= 0 && pg < P.num_pages) ? (int)pg : -1;
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // the loads so far are in (compiler-visible vmcnt(0))
  lds_barrier();

  // This wave's copies of a step: KL KB of one page's K rows and of its V rows.  K chunks are
  // XOR-swizzled by their row (16 rows of one chunk position are read at once); V rows are read
  // whole, 16 lanes a row.  Absent pages read zero rows, and V rows past the chunk's end repeat its
  // last row inside it (a masked key's weight is 0, and 0 * NaN would poison the sum).
  const int my_page = wave * KL / LPP;
  const char* kbase = reinterpret_cast<const char*>(reinterpret_cast<const float*>(P.k_cache) + hoff);
  const char* vbase = reinterpret_cast<const char*>(reinterpret_cast<const float*>(P.v_cache) + hoff);
  const char* const zero_rows = reinterpret_cast<const char*>(g_zero_rows);
  const int64_t page_bytes = P.page_stride * 4;
  const unsigned sk = lds_addr(s_k), sv = lds_addr(s_v);
  auto issue = [&](int st, int pg) __attribute__((always_inline)) {
    const int vr = k1 - (k0 + SK * st) - 16 * my_page;  // rows of the page inside the chunk
    const bool have = pg >= 0, havev = have && vr > 0;
    const char* kb = have ? kbase + pg * page_bytes : zero_rows;
    const char* vb = havev ? vbase + pg * page_bytes : zero_rows;
#pragma unroll
    for (int x = 0; x < KL; ++x) {
      const int wi = wave * KL + x, row = RPI * (wi % LPP) + lane / CPR, pos = lane % CPR;
      const unsigned dst = (st & 1) * STEPB + my_page * TILEB + RPI * (wi % LPP) * ROWB;
      lds_copy16(kb, have ? (unsigned)((row * rowstride + 4 * (pos ^ row)) * 4) : 16u * lane, sk + dst);
      lds_copy16(vb, havev ? (unsigned)((min(row, vr - 1) * rowstride + 4 * pos) * 4) : 16u * lane, sv + dst);
    }
  };
  auto page_of = [&](int st) __attribute__((always_inline)) -> int { return s_page[min(st, nsteps - 1) * KT + my_page]; };

  f4 o[NC][4];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int e = 0; e < 4; ++e) o[c][e] = f4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, lsum = 0.f;
  const float scale = P.scale_log2;
  int pg_next = 0;
  if (nsteps > 0) {
    issue(0, __builtin_amdgcn_readfirstlane(page_of(0)));
    pg_next = page_of(1);
  }
#pragma unroll 1
  for (int j = 0; j < nsteps; ++j) {
    wait_vmcnt<0>();  // this wave's copies of step j have landed ...
    lds_barrier();    // ... and everybody's, and step j - 1's buffer has been read
    if (j + 1 < nsteps) issue(j + 1, __builtin_amdgcn_readfirstlane(pg_next));
    pg_next = page_of(j + 2);
    const int kb = k0 + SK * j;
    bool absent[KT];
    bool full = kb + SK <= lim_min;  // (uniform)
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      absent[kt] = __builtin_amdgcn_readfirstlane(s_page[j * KT + kt]) < 0;
      full = full && !absent[kt];
    }
    const char* kbuf = s_k + (j & 1) * STEPB;
    const char* vbuf = s_v + (j & 1) * STEPB;
    f4 sacc[KT];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) sacc[kt] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < QS; ++s) {
      f4 a[KT];
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
        a[kt] = *reinterpret_cast<const f4*>(kbuf + kt * TILEB + lr * ROWB + (((4 * s + lg) ^ lr) << 4));
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
          sacc[kt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[kt][e], qr[s][e], sacc[kt], 0, 0, 0);
    }
    if (!full) {
      const int rem = lim - kb - 4 * lg;
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (!(16 * kt + i < rem && !absent[kt])) sacc[kt][i] = -INFINITY;
    }
    float cmax = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
      cmax = max3f(cmax, max2f(sacc[kt][0], sacc[kt][1]), max2f(sacc[kt][2], sacc[kt][3]));
    const float cms = max_across_groups(cmax) * scale;
    const bool grow = cms > m + kLazyMax;  // (false while every score so far is masked)
    if (__ballot(grow)) {
      const float mnew = grow ? cms : m;
      // 0 from -inf; 1 if unchanged (also where no key has been seen: -inf less -inf is NaN)
      const float alpha = grow ? __builtin_amdgcn_exp2f(m - mnew) : 1.f;
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[c][e] *= alpha;
      lsum *= alpha;
      m = mnew;
    }
    const float nm = m == -INFINITY ? 0.f : -m;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
#pragma unroll
      for (int i = 0; i < 4; ++i) sacc[kt][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[kt][i], scale, nm));
      lsum += (sacc[kt][0] + sacc[kt][1]) + (sacc[kt][2] + sacc[kt][3]);
    }
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const f4 v = *reinterpret_cast<const f4*>(vbuf + kt * TILEB + (4 * lg + i) * ROWB + 256 * c + 16 * lr);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            o[c][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[e], sacc[kt][i], o[c][e], 0, 0, 0);
        }
      }
    }
  }

  // ---- rows out: lane holds dims 64 c + 16 lg + 4 i + e of row lr
  const float ltot = sum_across_groups(lsum);
  const float inv = ltot > 0.f ? 1.f / ltot : 0.f;
  float z = 0.f;  // (0, or NaN from an infinity or a NaN)
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < 4; ++i) z = __builtin_fmaf(o[c][e][i], 0.f, z);
  const uint64_t bad = __ballot(z != 0.f && row_ok);
  const int64_t pr = (int64_t)slot * item_rows<0, kRowsF>(g) + r;
  if (row_ok) {
    float* dst = slot < 0 ? reinterpret_cast<float*>(P.out) + qrow * P.o_sn + (int64_t)(h * g + rh) * P.o_sh
                          : P.part_o + pr * D;
    const bool vec = slot >= 0 || P.o_vec;
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float* d = dst + 64 * c + 16 * lg + 4 * i;
        if (vec) {
          *reinterpret_cast<float4*>(d) = make_float4(o[c][0][i] * inv, o[c][1][i] * inv, o[c][2][i] * inv, o[c][3][i] * inv);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) d[e] = o[c][e][i] * inv;
        }
      }
    if (slot >= 0 && lg == 0) P.part_ml[pr] = make_float2(m, ltot);
  }
  if (bad) {  // (wave-uniform) rows that did not come out finite: see exact_row
    wait_stores();
#pragma unroll 1
    for (uint32_t todo = (uint32_t)((bad | bad >> 16 | bad >> 32 | bad >> 48) & 0xFFFF); todo; todo &= todo - 1) {
      const int rr = 16 * wave + __builtin_ctz(todo), tt = rr / g, hh = rr % g;
      const int64_t row = qo_start + t0 + tt;
      const float* q = reinterpret_cast<const float*>(P.q) + row * P.q_sn + (int64_t)(h * g + hh) * P.q_sh;
      const int l = P.causal ? t0 + tt + kv_len - qo_len + 1 : kv_len;
      exact_row<float, D>(P, s_page, k0, min(l, k1), hoff, q, [&](int d, float x, float mx, float sum) {
        if (slot < 0) {
          reinterpret_cast<float*>(P.out)[row * P.o_sn + (int64_t)(h * g + hh) * P.o_sh + d] = x;
        } else {
          const int64_t p = (int64_t)slot * item_rows<0, kRowsF>(g) + rr;
          P.part_o[p * D + d] = x;
          if (d == 0) P.part_ml[p] = make_float2(mx, sum);
        }
      });
    }
  }
}

template <int D>
int launch(const PrefillMfmaParams& P, int n_items, const int32_t* groups, int n_groups, hipStream_t s) {
  if (n_items > 0) hipLaunchKernelGGL((prefill_f32_kernel<D>), dim3(n_items), dim3(512), 0, s, P);
  if (n_groups > 0)
    hipLaunchKernelGGL((prefill_merge_kernel<float, D, 0, kRowsF>), dim3(n_groups * (kRowsF / merge_rows<D>())),
                       dim3(256), 0, s, P, groups);
  return (int)hipGetLastError();
}

}  // namespace

namespace pkv {
int prefill_f32_launch(const pre::PrefillMfmaParams& P, int d, int n_items, const int32_t* groups, int n_groups,
                       hipStream_t s) {
  return d == 64 ? launch<64>(P, n_items, groups, n_groups, s) : launch<128>(P, n_items, groups, n_groups, s);
}
}  // namespace pkv
